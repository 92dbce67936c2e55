"""When the block-FP8 expert MLP's gate, up and SwiGLU may run as one launch:
only where nobody could tell it from calling the projections."""

from __future__ import annotations

import torch

from kairyu_amd.moe import BlockFp8ExpertMlp


def test_hooks_keep_the_projections_calls():
    mlp, x = BlockFp8ExpertMlp(256, 128), torch.zeros(4, 256, dtype=torch.bfloat16)
    assert mlp._fused_swiglu(x)
    for handle in (mlp.gate_proj.register_forward_hook(lambda *args: None),
                   mlp.up_proj.register_forward_pre_hook(lambda *args: None),
                   torch.nn.modules.module.register_module_forward_hook(lambda *args: None),
                   torch.nn.modules.module.register_module_forward_pre_hook(lambda *args: None)):
        assert not mlp._fused_swiglu(x)
        handle.remove()
        assert mlp._fused_swiglu(x)
