"""The weight-streaming GEMM (at most 64 rows) at the edges of its forms: row
tiles of 16, 32, 48 and 64, a weight tile or two per workgroup, 4 to 16 waves,
K blocks fewer than the waves, K tails, ragged columns."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_helpers import assert_moe_close, banner, bits, check_block_fp8, check_fp8, np32
from kairyu_amd._native import w8a8_route
from kairyu_amd.kernels import quant_gemm_hip as hip
from kairyu_amd.moe import BlockFp8ExpertMlp, GroupedBlockFp8Experts
from kairyu_amd.quant.block_fp8 import quantize_block_fp8
from kairyu_amd.quant.fp8 import quantize_fp8
from kairyu_amd.quant.int8 import quantize_int8_weight
from kairyu_amd.quant.linear import BlockFp8Linear, Fp8Linear, Int8Linear
from oracle import linear as olinear
from oracle import moe as omoe

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 15, 16, 17, 32, 33, 48, 49, 64]
# one block, a tail of 16 bytes, 19 blocks for 8 and (one row) 16 waves with a tail;
# 1 to 600 column tiles (one tile, two, many workgroups per CU); long K split
# over workgroups 4 and 8 ways with a tail
SHAPES = [(24, 112), (200, 144), (2600, 2368), (1000, 2368), (4616, 640), (9608, 272), (1000, 8272), (72, 16400)]


def test_the_shapes_reach_every_form():
    reached = {w8a8_route(m, n, k)[1:] for m in ROWS for n, k in SHAPES}
    assert reached >= {(1, 16, 1), (1, 8, 1), (2, 8, 1), (2, 4, 1), (1, 4, 1), (4, 4, 1), (1, 8, 4), (1, 8, 8),
                       (1, 4, 4), (1, 4, 8)}


def _gen(seed):
    return torch.Generator().manual_seed(seed)


def _fill(module, g):
    w = torch.randn(module.out_features, module.in_features, generator=g) * 0.05
    quantize = {Fp8Linear: quantize_fp8, Int8Linear: quantize_int8_weight, BlockFp8Linear: quantize_block_fp8}
    q, s = quantize[type(module)](w)
    module.weight.copy_(q)
    (module.weight_scale_inv if isinstance(module, BlockFp8Linear) else module.weight_scale).copy_(s)
    if module.bias is not None:
        module.bias.data.normal_(generator=g)
    return module


@pytest.mark.parametrize("n,k", SHAPES)
def test_int8_rows_are_exact(cuda, n, k):
    module = _fill(Int8Linear(k, n, True), _gen(n + k)).to(cuda)
    for m in ROWS:
        banner(f"stream int8 m={m} n={n} k={k}")
        x = torch.randn(m, k, generator=_gen(m)).to(torch.bfloat16)
        acc = torch.empty(m, n, dtype=torch.int32, device=cuda)
        out = hip.int8_linear_forward(x.to(cuda), module, accumulators=acc)
        want, _, _, want_acc = olinear.int8_forward(
            np32(x), module.weight.cpu().numpy(), module.weight_scale.cpu().numpy(), np32(module.bias))
        assert np.array_equal(acc.cpu().numpy().astype(np.int64), want_acc)
        assert np.array_equal(np32(out), want)


# rows of a multiple of 4 KB against a tile per CU and more: the waves take K apart
@pytest.mark.parametrize("n,k,tiles,waves", [(4104, 4096, 2, 8), (4096, 4096, 1, 8), (8200, 4096, 2, 4)])
def test_int8_rows_of_aligned_pitch_are_exact(cuda, n, k, tiles, waves):
    module = _fill(Int8Linear(k, n, True), _gen(n + k)).to(cuda)
    for m in (1, 2, 16):
        banner(f"stream int8 apart m={m} n={n} k={k}")
        assert w8a8_route(m, n, k) == ("stream", tiles, waves, 1)
        x = torch.randn(m, k, generator=_gen(m)).to(torch.bfloat16)
        acc = torch.empty(m, n, dtype=torch.int32, device=cuda)
        out = hip.int8_linear_forward(x.to(cuda), module, accumulators=acc)
        want, _, _, want_acc = olinear.int8_forward(
            np32(x), module.weight.cpu().numpy(), module.weight_scale.cpu().numpy(), np32(module.bias))
        assert np.array_equal(acc.cpu().numpy().astype(np.int64), want_acc)
        assert np.array_equal(np32(out), want)


@pytest.mark.parametrize("n,k", SHAPES)
def test_fp8_rows_match_oracle(cuda, n, k):
    module = _fill(Fp8Linear(k, n, True), _gen(n + k)).to(cuda)
    for m in ROWS:
        banner(f"stream fp8 m={m} n={n} k={k}")
        x = torch.randn(m, k, generator=_gen(m)).to(torch.float16)
        check_fp8(module(x.to(cuda)), x, module, label=f"m={m} n={n} k={k}")


# 16 rows quantize in the launch up to K = 8192; 129 blocks would not fit
@pytest.mark.parametrize("n,k", [(24, 128), (200, 384), (2600, 2432), (4616, 640), (9608, 256), (72, 16384)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_block_fp8_rows_match_oracle(cuda, n, k, dtype):
    module = _fill(BlockFp8Linear(k, n, True), _gen(n + k)).to(cuda)
    for m in [1, 8, 9] + ROWS[3:]:
        banner(f"stream block fp8 m={m} n={n} k={k} {dtype}")
        x = torch.randn(m, k, generator=_gen(m)).to(dtype)
        x[0, :k // 2] = 0.0
        check_block_fp8(module(x.to(cuda)), x, module, label=f"m={m} n={n} k={k}")


@pytest.mark.parametrize("m", [1, 8, 16, 40, 64, 65])
@pytest.mark.parametrize("n,k", [(200, 384), (5000, 256)])
@pytest.mark.parametrize("bias", [False, True])
def test_block_fp8_mlp_matches_its_projections(cuda, m, n, k, bias):
    """The expert MLP, whose gate, up and SwiGLU are one launch,
    against down(silu(gate(x)) * up(x)) of the same modules: the sums of a
    gate or up column may be added in another order, so a rounding of the
    activation dtype apart (2^-8 relative in bf16, from both factors)."""
    mlp = BlockFp8ExpertMlp(128, 128)
    g = _gen(m + n)
    mlp.gate_proj, mlp.up_proj = (_fill(BlockFp8Linear(k, n, bias), g) for _ in range(2))
    mlp.down_proj = torch.nn.Identity()
    mlp = mlp.to(cuda)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(cuda)
    banner(f"stream block swiglu m={m} n={n} k={k}")
    out = mlp(x)
    gate, up = mlp.gate_proj(x), mlp.up_proj(x)
    want = torch.nn.functional.silu(gate) * up
    torch.testing.assert_close(out.float(), want.float(), rtol=2.0 ** -6, atol=2.0 ** -9 * float(up.abs().max()))
    if m == 65:  # the panel kernel: the projections' order
        assert np.array_equal(bits(out), bits(want))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_block_fp8_launch_quantizes_as_the_quantizer(cuda, dtype):
    """Edge values through the launch that quantizes and through the quantizer
    and the GEMM: the same bits, NaN and infinite rows included."""
    n, k, m = 200, 512, 8
    module = _fill(BlockFp8Linear(k, n, False), _gen(5)).to(cuda)
    x = torch.randn(m, k, generator=_gen(6)) * 5
    x[0, :128:3] = -0.0
    x[1, :128] = torch.tensor([1.0625, -1.1875, 0.017578125, 240.0]).repeat(32)
    x[1, 127] = 448.0                      # scale 1: exact ties of e4m3
    x[2, 128:256] = torch.randn(128, generator=_gen(7)) * 1e-30
    x[3, 300] = float("inf")
    x[4, 100] = float("nan")
    x[5] = 0.0
    x[6, 0] = 60000.0
    x = x.to(dtype).to(cuda)
    banner(f"stream block fp8 edge values {dtype}")
    out = module(x)
    q, s = hip.quantize_activation_blocks(x)
    want = torch.empty_like(out)
    hip._native.call("kq_block_fp8_gemm", q.data_ptr(), s.data_ptr(), module.weight.data_ptr(),
                     module.weight_scale_inv.data_ptr(), None, hip._native.DTYPE_NONE, want.data_ptr(),
                     hip._native.dtype_code(dtype), m, n, k, hip._native.stream_handle(cuda))
    finite = [0, 1, 2, 5, 6, 7]
    assert np.array_equal(bits(out)[finite], bits(want)[finite])
    assert torch.equal(torch.isnan(out), torch.isnan(want))


# average rows per expert on both sides of each row tile's limit (2, 6 and 16
# rows; then the tile engine), experts with none and with several tiles
@pytest.mark.parametrize("tokens,experts,top_k", [(8, 16, 4), (9, 16, 4), (24, 16, 4), (25, 16, 4),
                                                  (64, 16, 4), (65, 16, 4), (40, 128, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_moe_row_tiles_match_oracle(cuda, tokens, experts, top_k, dtype):
    hidden, inter = 384, 256
    g = _gen(tokens * experts)
    q13, s13 = quantize_block_fp8(torch.randn(experts, 2 * inter, hidden, generator=g) * 0.05)
    q2, s2 = quantize_block_fp8(torch.randn(experts, hidden, inter, generator=g) * 0.05)
    pack = GroupedBlockFp8Experts.from_tensors(*(t.to(cuda) for t in (q13, s13, q2, s2)))
    x = torch.randn(tokens, hidden, generator=g).to(dtype)
    logits = torch.randn(tokens, experts, generator=g)
    logits[:, 0] += 3.0  # one expert holds nearly every token
    logits[:, -1] -= 9.0
    banner(f"moe row tiles tokens={tokens} E={experts} k={top_k} {dtype}")
    out, idx, w = pack.forward_logits(x.to(cuda), logits.to(cuda), top_k)
    name = str(dtype).split(".")[1]
    want = omoe.moe_forward(np32(x), idx.cpu().numpy(), w.cpu().numpy(), bits(q13), s13.numpy(), bits(q2),
                            s2.numpy(), name)
    # the normwise bound of narrow layers (test_gpu_moe.py); a flipped e4m3
    # activation moves an output by the same relative amount whatever its
    # dtype, and 8 ulps of bf16 are 64 of fp16 (oracle.parity.moe_check)
    assert_moe_close(np32(out), want, name, label=f"T={tokens} E={experts}", normwise=2e-2,
                     ulps=8.0 if dtype == torch.bfloat16 else 64.0)


def test_one_row_of_any_pitch_gives_the_contiguous_rows_bits(cuda):
    """One row counts as contiguous at any pitch; the kernels take one of at
    least K."""
    k, n = 256, 64
    module = _fill(Fp8Linear(k, n, True), _gen(1)).to(cuda)
    x = torch.randn(1, k, generator=_gen(2)).to(torch.bfloat16).to(cuda)
    want = module(x)
    banner("one-row pitches")
    narrow = x.reshape(k, 1).t()
    wide = torch.cat([x, x], dim=1)[:, :k]
    assert narrow.is_contiguous() and narrow.stride(0) == 1 and wide.stride(0) == 2 * k
    for row in (narrow, wide, x[0], x[None]):
        assert np.array_equal(bits(module(row)).reshape(-1), bits(want).reshape(-1))


def test_block_fp8_calls_on_two_streams_do_not_meet(cuda):
    """32 rows are quantized into scratch before the GEMM: calls queued on two
    streams, a linear and an MLP's fused gate and up, each give the bits that
    they give alone."""
    n = k = 1024
    module = _fill(BlockFp8Linear(k, n, False), _gen(1)).to(cuda)
    mlp = BlockFp8ExpertMlp(128, 128)
    mlp.gate_proj, mlp.up_proj = (_fill(BlockFp8Linear(k, n, False), _gen(s)) for s in (2, 3))
    mlp.down_proj = torch.nn.Identity()
    mlp = mlp.to(cuda)
    calls = [module, mlp, module]
    xs = [torch.randn(32, k, generator=_gen(10 + i)).to(torch.bfloat16).to(cuda) for i in range(6)]
    want = [[f(x) for f in calls] for x in xs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    banner("block fp8 on two streams")
    got = [[] for _ in xs]
    for _ in range(10):
        for i, x in enumerate(xs):
            with torch.cuda.stream(streams[i % 2]):
                got[i] = [f(x) for f in calls]
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert all(np.array_equal(bits(p), bits(q)) for p, q in zip(a, b))


@pytest.mark.parametrize("k", [112, 144, 256])
def test_a_static_scale_of_zero_gives_one_row_the_bits_of_two(cuda, k):
    """One row is quantized in the launch: past K (112 and 144 end inside a
    block of 128) it holds zeros, also where a scale of zero makes every
    quotient infinite (clamped to 448) or, of a zero, NaN."""
    module = _fill(Fp8Linear(k, 40, True, activation_dynamic=False), _gen(k)).to(cuda)
    module.input_scale.zero_()
    x = torch.randn(1, k, generator=_gen(3)).to(torch.bfloat16).to(cuda)
    banner(f"static scale zero k={k}")
    out = module(x)
    assert torch.isfinite(out).all()
    assert np.array_equal(bits(out), bits(module(x.expand(2, k).contiguous())[:1]))
