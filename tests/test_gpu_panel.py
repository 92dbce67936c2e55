"""The panel GEMM (65 to 256 rows; from 33 with many weight rows) at the edges
of its forms: one and two row tiles per wave, panels of 2 to 16 weight tiles,
split K, K tails, ragged rows and columns, waves without rows.  Each case says
which form it means and asks the dispatch."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_helpers import banner, bits, check_block_fp8, check_fp8, np32
from kairyu_amd import _native
from kairyu_amd.kernels import quant_gemm_hip as hip
from kairyu_amd.moe import BlockFp8ExpertMlp
from kairyu_amd.quant.linear import BlockFp8Linear, Fp8Linear, Int8Linear
from kairyu_amd.quant.packed import QuantLinearPack
from oracle import linear as olinear
from test_gpu_stream import _fill, _gen

pytestmark = pytest.mark.gpu

# (m, n, k, panel tiles, K splits), each ragged in rows, columns or K: one and
# two row tiles per wave, every panel width that a product takes, split and
# whole; tiles None: past the panels (another kernel)
SHAPES = [(65, 6200, 144, 4, 1), (130, 1004, 2832, 4, 3), (200, 3500, 3088, 4, 2), (128, 8, 112, 4, 1),
          (256, 1024, 8208, 8, 8), (130, 4200, 5136, 8, 7), (96, 17000, 272, 8, 1), (250, 16500, 272, 8, 1),
          (100, 33000, 272, 12, 1), (128, 49300, 144, 16, 1), (40, 8600, 400, 4, 1), (64, 9000, 256, 4, 1),
          (129, 33000, 256, None, 1), (200, 50008, 128, None, 1)]


def _expect(route, tiles, splits):
    if tiles is None:
        assert route.kernel != "panel"
    else:
        assert (route.kernel, route.tiles, route.splits) == ("panel", tiles, splits)


@pytest.mark.parametrize("m,n,k,tiles,splits", SHAPES)
def test_int8_panels_are_exact(cuda, m, n, k, tiles, splits):
    banner(f"panel int8 m={m} n={n} k={k}")
    _expect(_native.w8a8_route(m, n, k), tiles, splits)
    module = _fill(Int8Linear(k, n, True), _gen(n + k)).to(cuda)
    x = torch.randn(m, k, generator=_gen(m)).to(torch.bfloat16)
    acc = torch.empty(m, n, dtype=torch.int32, device=cuda)
    out = hip.int8_linear_forward(x.to(cuda), module, accumulators=acc)
    want, _, _, want_acc = olinear.int8_forward(
        np32(x), module.weight.cpu().numpy(), module.weight_scale.cpu().numpy(), np32(module.bias))
    assert np.array_equal(acc.cpu().numpy().astype(np.int64), want_acc)
    assert np.array_equal(np32(out), want)


@pytest.mark.parametrize("m,n,k,tiles,splits", SHAPES)
def test_fp8_panels_match_oracle(cuda, m, n, k, tiles, splits):
    banner(f"panel fp8 m={m} n={n} k={k}")
    _expect(_native.w8a8_route(m, n, k), tiles, splits)
    module = _fill(Fp8Linear(k, n, True), _gen(n + k)).to(cuda)
    x = torch.randn(m, k, generator=_gen(m)).to(torch.float16)
    check_fp8(module(x.to(cuda)), x, module, label=f"m={m} n={n} k={k}")


@pytest.mark.parametrize("m", [65, 128, 129, 256])
@pytest.mark.parametrize("n,k", [(200, 384), (5000, 256), (17000, 128), (72, 16384)])
def test_block_fp8_panels_match_oracle(cuda, m, n, k):
    banner(f"panel block fp8 m={m} n={n} k={k}")
    module = _fill(BlockFp8Linear(k, n, True), _gen(n + k)).to(cuda)
    x = torch.randn(m, k, generator=_gen(m)).to(torch.bfloat16)
    check_block_fp8(module(x.to(cuda)), x, module, label=f"m={m} n={n} k={k}")


# unsplit and split panels (the reduce pairs the columns), every panel width,
# widths of odd eighths, rows of one and two row tiles per wave; 256 rows of
# 34000 columns are past the panels
@pytest.mark.parametrize("kind,m,width,k,dtype", [
    ("fp8", 65, 1000, 1024, torch.bfloat16), ("fp8", 200, 520, 8320, torch.float16),
    ("fp8", 130, 9000, 272, torch.bfloat16), ("int8", 256, 17000, 256, torch.float16),
    ("int8", 100, 26000, 144, torch.bfloat16), ("fp8", 50, 5004, 400, torch.bfloat16),
    ("int8", 64, 4600, 512, torch.float16), ("int8", 129, 1004, 2048, torch.float16),
    ("fp8", 100, 17000, 144, torch.bfloat16), ("int8", 128, 24500, 272, torch.float16),
    ("fp8", 200, 2200, 6160, torch.bfloat16)])
def test_swiglu_panels_give_the_two_pass_bits(cuda, kind, m, width, k, dtype):
    banner(f"panel swiglu {kind} m={m} I={width} k={k}")
    route = _native.w8a8_route(m, 2 * width, k, swiglu=True)
    forms = {1000: (4, 1), 520: (8, 8), 9000: (8, 1), 26000: (16, 1), 5004: (4, 1), 4600: (4, 1), 1004: (4, 2),
             24500: (12, 1), 2200: (8, 7), 17000: (12, 1) if m == 100 else (None, 1)}
    _expect(route, *forms[width])
    make = Fp8Linear if kind == "fp8" else Int8Linear
    g = _gen(width)
    pack = QuantLinearPack.create([_fill(make(k, width, True), g).to(cuda) for _ in range(2)])
    x = torch.randn(m, k, generator=g).to(dtype).to(cuda)
    fused = pack.swiglu(x)
    packed = torch.cat(pack(x), dim=-1).contiguous()
    two = torch.empty(m, width, device=cuda, dtype=dtype)
    _native.call("kq_swiglu", packed.data_ptr(), packed.stride(0), 0, _native.dtype_code(dtype), two.data_ptr(),
                 m, width, _native.stream_handle(cuda))
    assert np.array_equal(bits(fused), bits(two))


# panels of 2, 4 and 8 tiles (16, 32 and 64 columns), ragged rows and columns,
# the first and last row counts of the launch and the two-pass form past them
@pytest.mark.parametrize("m", [65, 100, 128, 129])
@pytest.mark.parametrize("width,k,bias,dtype", [
    (200, 384, True, torch.bfloat16), (4100, 256, False, torch.float16),
    (8200, 128, True, torch.bfloat16), (72, 16384, False, torch.bfloat16)])
def test_block_fp8_swiglu_panels_give_the_two_pass_bits(cuda, m, width, k, bias, dtype):
    """Each form adds an element's K blocks in one order: the projections'
    outputs through the elementwise pass, bit for bit."""
    banner(f"panel block swiglu m={m} I={width} k={k}")
    mlp = BlockFp8ExpertMlp(128, 128)
    g = _gen(width)
    mlp.gate_proj, mlp.up_proj = (_fill(BlockFp8Linear(k, width, bias), g) for _ in range(2))
    mlp.down_proj = torch.nn.Identity()
    mlp = mlp.to(cuda)
    x = torch.randn(m, k, generator=g).to(dtype).to(cuda)
    packed = torch.cat([mlp.gate_proj(x), mlp.up_proj(x)], dim=-1).contiguous()
    two = torch.empty(m, width, device=cuda, dtype=dtype)
    _native.call("kq_swiglu", packed.data_ptr(), packed.stride(0), 0, _native.dtype_code(dtype), two.data_ptr(),
                 m, width, _native.stream_handle(cuda))
    assert np.array_equal(bits(mlp(x)), bits(two))


# the columns of one round of panels, and a ragged panel more: the tile engine
@pytest.mark.parametrize("m,n,kernel", [(256, 16384, "panel"), (200, 16440, "tile"), (65, 32768, "panel"),
                                        (128, 32776, "tile"), (50, 49152, "stream"), (64, 49160, "tile")])
def test_block_fp8_on_both_sides_of_a_round(cuda, m, n, kernel):
    banner(f"block fp8 round m={m} n={n}")
    k = 256
    assert _native.block_fp8_route(m, n, k).kernel == kernel
    module = _fill(BlockFp8Linear(k, n, True), _gen(n)).to(cuda)
    x = torch.randn(m, k, generator=_gen(m)).to(torch.bfloat16)
    check_block_fp8(module(x.to(cuda)), x, module, label=f"m={m} n={n}")
