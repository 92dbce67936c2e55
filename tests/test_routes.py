"""Which kernel and form a GEMM of a shape takes: the rules of the dispatch,
asked of the library without a GPU (256 CUs are assumed then, as on MI355X)."""

from __future__ import annotations

import pytest
import torch

from kairyu_amd import _native
from kairyu_amd._native import Route, block_fp8_route, w4a16_route, w8a8_route


@pytest.fixture(autouse=True)
def _cus():
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are stated for 256 CUs")


def test_kernels_by_rows():
    assert w8a8_route(8, 4096, 4100).kernel == "generic"        # K % 16
    assert w8a8_route(8, 4096, 4096) == Route("stream", 1, 8, 1)
    assert w8a8_route(8, 28672, 4096) == Route("stream", 2, 4, 1)
    assert w8a8_route(64, 28672, 4096, swiglu=True) == Route("panel", 4, 4, 1)
    assert w8a8_route(128, 28672, 4096) == Route("panel", 8, 8, 1)
    assert w8a8_route(4096, 14336, 4096).kernel == "tile"
    assert block_fp8_route(8, 4096, 4096) == Route("stream", 1, 8, 1)
    assert block_fp8_route(257, 4096, 4096).kernel == "tile"
    assert w4a16_route(torch.float16, False, 16, 4096, 4096, 128).kernel == "generic"
    assert w4a16_route(torch.float16, False, 32, 4096, 4096, 128) == Route("stream", 4, 4, 4)
    assert w4a16_route(torch.float16, False, 32, 4096, 4096, 64).kernel == "generic"
    assert w4a16_route(torch.bfloat16, False, 64, 4096, 4096, 128).kernel == "tile"


def test_bad_shapes_are_refused():
    for call in (lambda: w8a8_route(0, 16, 16), lambda: block_fp8_route(8, 16, 100),
                 lambda: block_fp8_route(129, 256, 256, swiglu=True),
                 lambda: w4a16_route(torch.float16, False, 8, 12, 128, 128)):
        with pytest.raises(ValueError, match="bad shape"):
            call()


@pytest.mark.parametrize("m,most", [(65, 32768), (128, 32768), (129, 16384), (256, 16384), (64, 49152), (49, 49152)])
def test_block_fp8_panels_stay_within_a_round(m, most):
    """Past one round of 128-column panels over the CUs (streamed rows: one and
    a half) the tile engine is the faster one."""
    assert block_fp8_route(m, most, 2048).kernel in ("panel", "stream")
    assert block_fp8_route(m, most + 8, 2048).kernel == "tile"
    assert block_fp8_route(48, 100000, 2048).kernel == "stream"


@pytest.mark.parametrize("m,n,k,tiles,splits", [
    (129, 3456, 5120, 4, 2), (256, 4096, 7168, 4, 2), (65, 8192, 7168, 4, 2),   # at most half the CUs
    (129, 5120, 5120, 8, 6), (190, 6912, 6144, 8, 4), (129, 8192, 8064, 8, 4),  # more, long K
    (190, 6912, 5120, 4, 1), (128, 13824, 5120, 4, 1),
    (256, 8192, 3072, 4, 1), (129, 6144, 4096, 4, 1),                            # more, short K
    (256, 4096, 2048, 4, 1), (256, 4096, 3072, 4, 2), (65, 1024, 4096, 4, 4), (200, 1024, 8192, 8, 8)])
def test_w8a8_panels_leave_no_half_of_the_cus_idle(m, n, k, tiles, splits):
    assert w8a8_route(m, n, k) == Route("panel", tiles, 4 if tiles == 4 else 8, splits)
    assert w8a8_route(m, n, k, swiglu=True) == w8a8_route(m, n, k)


@pytest.mark.parametrize("m,n,k,splits", [
    (16, 512, 16384, 1), (17, 512, 8191, 1), (17, 512, 8192, 4), (32, 512, 16384, 8), (33, 512, 4096, 1), (33, 512, 5120, 4),
    (64, 512, 12288, 8), (64, 1024, 12288, 4), (64, 2048, 8192, 1), (17, 2048, 12288, 2), (64, 2064, 16384, 1),
    (49, 512, 4096, 4), (64, 512, 3968, 1)])
def test_few_rows_of_narrow_long_products_split_k(m, n, k, splits):
    route = w8a8_route(m, n, k)
    assert route.splits == splits and route.kernel == ("generic" if k % 16 else "stream")
    need = _native.library().kq_w8a8_workspace_size(m, n, k)
    assert need == (splits * m * n * 4 if splits > 1 else 0)


@pytest.mark.parametrize("m,n,k,waves", [(1, 1024, 4096, 16), (1, 1024, 2048, 8), (1, 2064, 4096, 8),
                                         (2, 1024, 4096, 8), (16, 512, 16384, 8)])
def test_sixteen_waves_are_for_one_row(m, n, k, waves):
    assert w8a8_route(m, n, k).waves == waves
    assert w8a8_route(m, n, k, swiglu=True) == w8a8_route(m, n, k)


@pytest.mark.parametrize("dtype,gathered,m,width,k,kernel", [
    (torch.float16, False, 32, 14336, 4096, "stream"), (torch.bfloat16, True, 48, 11008, 4096, "stream"),
    (torch.float16, False, 17, 2048, 2048, "stream"), (torch.bfloat16, False, 17, 2048, 2048, "tile"),
    (torch.bfloat16, False, 48, 3072, 1024, "stream"), (torch.float16, False, 48, 2752, 4096, "tile"),
    (torch.bfloat16, False, 17, 3456, 5120, "tile"), (torch.bfloat16, True, 33, 3584, 8192, "tile")])
def test_w4_swiglu_keeps_k_whole_only_where_that_is_short(dtype, gathered, m, width, k, kernel):
    """Else two passes, whose plain product streams with its K split ("tile":
    not this kernel's fused form)."""
    assert w4a16_route(dtype, gathered, m, 2 * width, k, 128, swiglu=True).kernel == kernel
    if kernel == "tile":
        plain = w4a16_route(dtype, gathered, m, 2 * width, k, 128)
        assert plain.kernel == "stream" and plain.splits > 1


@pytest.mark.parametrize("dtype,gathered,m,n,k,kernel", [
    (torch.bfloat16, False, 33, 10240, 8192, "tile"), (torch.bfloat16, False, 32, 10240, 8192, "stream"),
    (torch.float16, False, 48, 10240, 8192, "stream"), (torch.bfloat16, True, 48, 10240, 8192, "tile"),
    (torch.bfloat16, True, 40, 10240, 8192, "stream"), (torch.bfloat16, False, 48, 9472, 3584, "stream"),
    (torch.bfloat16, False, 48, 11008, 8192, "stream")])
def test_w4_rows_leave_the_cus_idle_on_short_k_only(dtype, gathered, m, n, k, kernel):
    assert w4a16_route(dtype, gathered, m, n, k, 128).kernel == kernel
