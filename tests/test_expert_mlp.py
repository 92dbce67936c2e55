"""When the block-FP8 expert MLP's gate, up and SwiGLU may run as one launch:
only where nobody could tell it from calling the projections."""

from __future__ import annotations

import torch

from kairyu_amd.moe import BlockFp8ExpertMlp


def test_hooks_keep_the_projections_calls():
    mlp, x = BlockFp8ExpertMlp(256, 128), torch.zeros(4, 256, dtype=torch.bfloat16)
    assert mlp._fused_swiglu(x)
    every = torch.nn.modules.module
    for register in (mlp.gate_proj.register_forward_hook, mlp.up_proj.register_forward_pre_hook,
                     every.register_module_forward_hook, every.register_module_forward_pre_hook):
        handle = register(lambda *args: None)
        assert not mlp._fused_swiglu(x)
        handle.remove()
        assert mlp._fused_swiglu(x)


def test_a_symbolic_trace_records_the_projections():
    """The forward traces with the projections as leaves, and the traced module
    computes what it does."""

    class Leaves(torch.fx.Tracer):
        def is_leaf_module(self, module, name):
            return name.endswith("_proj")

    mlp = BlockFp8ExpertMlp(256, 128)
    for proj in (mlp.gate_proj, mlp.up_proj, mlp.down_proj):
        proj.weight.copy_(torch.randn(proj.weight.shape).to(torch.float8_e4m3fn))
    graph = Leaves().trace(mlp)
    assert [n.target for n in graph.nodes if n.op == "call_module"] == ["gate_proj", "up_proj", "down_proj"]
    x = torch.randn(3, 256).to(torch.bfloat16)
    assert torch.equal(torch.fx.GraphModule(mlp, graph)(x), mlp(x))
