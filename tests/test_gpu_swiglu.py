"""silu(gate) * up of the SwiGLU epilogues on every 16-bit gate.

They take a short exponential and quotient where all gates of a wave lie below
80 in magnitude and expf with IEEE division elsewhere; an element must not
depend on its wave's other gates.  ``kq_swiglu`` runs the same code, two
columns a lane: waves of 128 consecutive outputs."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_helpers import banner, bits
from kairyu_amd import _native

pytestmark = pytest.mark.gpu


def _swiglu(gate: torch.Tensor, up: torch.Tensor, cuda) -> torch.Tensor:
    src = torch.cat([gate, up], dim=1).contiguous().to(cuda)
    out = torch.empty(gate.shape, dtype=gate.dtype, device=cuda)
    _native.call("kq_swiglu", src.data_ptr(), src.stride(0), 0, _native.dtype_code(gate.dtype), out.data_ptr(),
                 gate.shape[0], gate.shape[1], _native.stream_handle(cuda))
    return out.cpu()


def _every_gate(dtype) -> torch.Tensor:
    """All 65536 values, the smallest magnitudes first (NaN last)."""
    g = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(dtype)
    return g[torch.argsort(torch.nan_to_num(g.double().abs(), nan=float("inf")), stable=True)]


def _same(a: torch.Tensor, b: torch.Tensor) -> bool:
    nan = torch.isnan(a)
    return torch.equal(nan, torch.isnan(b)) and np.array_equal(bits(a)[~nan.numpy()], bits(b)[~nan.numpy()])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("other", [100.0, float("nan")])
def test_both_routines_give_the_same_bits(cuda, dtype, other):
    banner(f"swiglu every gate {dtype} {other}")
    g = _every_gate(dtype)
    fast = _swiglu(g.view(512, 128), torch.ones(512, 128, dtype=dtype), cuda).reshape(-1)
    # 127 gates a wave, and one that sends the wave to the general routine
    mixed = torch.full((517, 128), other, dtype=dtype)
    padded = torch.cat([g, torch.zeros(517 * 127 - g.numel(), dtype=dtype)]).view(517, 127)
    mixed[:, :127] = padded
    general = _swiglu(mixed, torch.ones(517, 128, dtype=dtype), cuda)[:, :127].reshape(-1)[:g.numel()]
    assert _same(fast, general)
    # against g / (1 + exp(-g)) in fp32 (past 88, where exp(-g) is infinite, a
    # zero), whose exp may be an ulp of fp32 off: the neighbour at worst, and
    # that where the quotient lies within an ulp of fp32 of a tie of the dtype,
    # 2^-15 (bf16) or 2^-12 (fp16) of the values
    f = g.float()
    want = (f / (1.0 + torch.exp(-f))).to(dtype)
    number = ~torch.isnan(want)
    assert torch.equal(torch.isnan(fast), ~number)
    a, b = bits(fast)[number.numpy()].astype(np.int64), bits(want)[number.numpy()].astype(np.int64)
    assert np.abs(a - b).max() <= 1 and np.count_nonzero(a != b) <= (4 if dtype == torch.bfloat16 else 32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("up", [-1.0, 0.0, -0.0, 3.0e-5, -7.5, float("inf")])
def test_the_product_is_rounded_once(cuda, dtype, up):
    """The activation of an up value is torch's product of the rounded silu,
    zeros' signs and subnormal results included."""
    banner(f"swiglu product {dtype} {up}")
    g = _every_gate(dtype).view(512, 128)
    silu = _swiglu(g, torch.ones(512, 128, dtype=dtype), cuda)
    u = torch.full((512, 128), up, dtype=dtype)
    assert _same(_swiglu(g, u, cuda).reshape(-1), (silu.float() * u.float()).to(dtype).reshape(-1))
