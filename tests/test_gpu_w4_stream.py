"""The W4A16 streaming GEMM (17 to 48 rows) against the CPU oracle.

Every column-tile form (4, 6, 8 and 10 tiles of 16 columns by N) at two and at
three row tiles, row-tile edges, K of fewer stages than waves, K splits, ragged
last tiles, both scale/zero tables, groups of two stages, act-order, rows at an
odd address and bf16 values past the fp16 range; each case says which form it
means and asks the dispatch.  Bounds are the W4A16 contract's
(``gpu_helpers.check_w4a16`` / ``check_swiglu``).
"""

from __future__ import annotations

import pytest
import torch

from gpu_helpers import banner, check_swiglu, check_w4a16
from kairyu_amd._native import w4a16_route
from kairyu_amd.quant import gptq as gptq_format
from kairyu_amd.quant.packed import QuantLinearPack
from test_gpu_w4a16 import _awq_module, _gptq_module

pytestmark = pytest.mark.gpu


def _module(kind, k, n, group, seed, bias):
    if kind == "awq":
        return _awq_module(k, n, group=group, seed=seed, bias=bias, random_packed=True)
    g_idx = None
    if "ao" in kind:
        order = torch.randperm(k, generator=torch.Generator().manual_seed(k))
        g_idx = (order // group).to(torch.int32)
    module = _gptq_module(k, n, group=group, seed=seed, bias=bias, g_idx=g_idx, random_packed=True)
    if g_idx is not None:
        module.g_idx.copy_(g_idx)
    if "sym" in kind:  # one zero for every group and column: the scale-only table
        module.qzeros.copy_(gptq_format.pack_gptq_cols(torch.full((module.qzeros.shape[0], n), 7)))
    return module


# tiles, splits of the streaming form; None: the tile kernel
@pytest.mark.parametrize("kind,m,n,k,group,dtype,form", [
    ("awq", 17, 8, 128, 128, torch.float16, (4, 1)),            # one stage, one partial tile
    ("gptq-sym", 32, 1048, 640, 128, torch.bfloat16, (4, 1)),   # ragged tile, five stages
    ("gptq", 33, 4096, 1536, 256, torch.float16, (4, 3)),       # two stages per group, K splits
    ("gptq-sym-ao", 48, 1024, 1280, 256, torch.float16, (4, 2)),
    ("awq", 48, 4096, 8320, 128, torch.bfloat16, None),         # past the bf16 limit
    ("awq", 34, 8456, 4096, 128, torch.bfloat16, None),         # K whole on few CUs, long for bf16
    ("awq", 20, 3584, 8320, 128, torch.bfloat16, (4, 4)),
    ("gptq-ao", 31, 24568, 256, 128, torch.bfloat16, (6, 1)),
    ("awq", 47, 28680, 256, 128, torch.float16, (8, 1)),
    ("gptq-sym", 34, 37896, 384, 128, torch.bfloat16, (10, 1)),
    ("awq", 17, 28680, 256, 128, torch.float16, (8, 1)),
    ("gptq-sym-ao", 32, 28680, 384, 128, torch.bfloat16, (8, 1)),
    ("gptq", 32, 37896, 256, 128, torch.bfloat16, (10, 1)),
    ("awq", 49, 1024, 512, 128, torch.float16, None),           # past the row limit
])
def test_linear_matches_oracle(cuda, kind, m, n, k, group, dtype, form):
    banner(f"w4 stream {kind} m={m} n={n} k={k} group={group} {dtype}")
    route = w4a16_route(dtype, "ao" in kind, m, n, k, group)
    assert (route.kernel, route.tiles, route.splits) == ("stream", *form) if form else route.kernel == "tile"
    module = _module(kind, k, n, group, seed=m + n, bias=m % 2 == 0).to(cuda)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(dtype)
    if dtype == torch.bfloat16:  # saturates to 65504, in one step of one row
        x[m // 2, 3] = 7.0e4
        x[m // 2, 70] = -3.0e38
    out = module(x.to(cuda))
    check_w4a16(out, module, x, label=f"{kind} m={m} n={n} k={k}")
    # a strided view (made contiguous before the launch), and contiguous rows at
    # an odd address, which no 16-byte load can read: the tile kernel's (or, with
    # an act-order, gathered before the streaming kernel)
    wide = torch.zeros(m, k + 8, dtype=dtype, device=cuda)
    wide[:, :k] = x.to(cuda)
    assert torch.equal(module(wide[:, :k]), out)
    odd = torch.zeros(m * k + 1, dtype=dtype, device=cuda)[1:].view(m, k)
    odd.copy_(x)
    assert odd.is_contiguous() and odd.data_ptr() % 16 == 2
    check_w4a16(module(odd), module, x, label=f"{kind} m={m} n={n} k={k} odd address")


# column tiles of the fused form; None: two passes, the plain product with its K
# split in five and in seven
@pytest.mark.parametrize("kind,m,width,k,dtype,tiles", [
    ("awq", 17, 16, 128, torch.float16, 4),
    ("gptq-ao", 32, 1040, 640, torch.bfloat16, 4),
    ("gptq-sym", 33, 12272, 256, torch.float16, 6),
    ("gptq", 48, 14352, 256, torch.bfloat16, 8),
    ("gptq-sym-ao", 40, 18944, 384, torch.float16, 10),
    ("awq", 20, 14352, 384, torch.bfloat16, 8),
    ("gptq-ao", 29, 18960, 256, torch.float16, 10),
    ("awq", 40, 1040, 2560, torch.bfloat16, None),
    ("gptq-ao", 24, 1040, 4352, torch.float16, None),
])
def test_swiglu_matches_oracle(cuda, kind, m, width, k, dtype, tiles):
    banner(f"w4 stream swiglu {kind} m={m} width={width} k={k} {dtype}")
    route = w4a16_route(dtype, "ao" in kind, m, 2 * width, k, 128, swiglu=True)
    assert (route.kernel, route.tiles) == ("stream", tiles) if tiles else route.kernel == "tile"
    gate, up = (_module(kind, k, width, 128, seed=7 * m + i, bias=m % 2 == 0).to(cuda) for i in range(2))
    pack = QuantLinearPack.create([gate, up])
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(dtype)
    check_swiglu(pack.swiglu(x.to(cuda)), gate, up, x, label=f"{kind} m={m} width={width} k={k}")
