"""GPU tests of which kernel takes a matrix product, as the diagnostic profile records it."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def rnd(*shape, seed=0, scale=1.0):
    return (torch.randn(*shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed)) * scale).to(BF)


def recorded(call):
    """[(key, M, N, K, launches)] of the products that `call` runs."""
    from olmax_amd import _lib
    L, cap = _lib.load(), 256
    keys, mnk, ms, ln = (ctypes.c_int32 * cap)(), (ctypes.c_int32 * (3 * cap))(), (ctypes.c_double * cap)(), (ctypes.c_int64 * cap)()
    L.olmax_gemm_profile_begin()
    try:
        call()
    finally:
        torch.cuda.synchronize()
        n = L.olmax_gemm_profile_end_shapes(keys, mnk, ms, ln, cap)
    return [(keys[i], *mnk[3 * i:3 * i + 3], ln[i]) for i in range(n)]


def operands(M, N, K, al, bl):
    return rnd(*((M, K) if al == 0 else (K, M)), seed=1), rnd(*((N, K) if bl == 0 else (K, N)), seed=2)


@pytest.mark.parametrize("al,bl", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K", [(4096, 4096, 4096), (4096, 16384, 1024), (2000, 4096, 1024)])
def test_large_products_of_every_layout_run_on_large_tiles(M, N, K, al, bl):
    from olmax_amd import ops
    print(f"[case] choice M{M} N{N} K{K} a{al} b{bl}", flush=True)
    a, b = operands(M, N, K, al, bl)
    got = recorded(lambda: ops.gemm(a, b, a_layout=al, b_layout=bl))
    assert sum(m * n for _, m, n, _, _ in got) == M * N
    assert all((key & 0xfff) >= 128 and (key >> 12 & 3) == (1 - al) + 2 * (1 - bl) for key, *_ in got), got


@pytest.mark.parametrize("al,bl", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K,out_f32", [(77, 2816, 1024, False), (7, 9, 3, True), (512, 256, 512, False)])
def test_products_of_the_64_wide_kernel_are_recorded(M, N, K, out_f32, al, bl):
    from olmax_amd import ops
    print(f"[case] record M{M} N{N} K{K} a{al} b{bl}", flush=True)
    a, b = operands(M, N, K, al, bl)
    assert recorded(lambda: ops.gemm(a, b, a_layout=al, b_layout=bl, out_f32=out_f32)) == [
        (64 | (1 - al) << 12 | (1 - bl) << 13 | out_f32 << 15, M, N, K, 1)]


@pytest.mark.parametrize("al,bl", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (512, 1024, 1024), (264, 1000, 136)])
def test_a_forced_tile_takes_what_the_rule_gives_to_the_64_wide_kernel(M, N, K, tile, al, bl):
    """And the result is the same but for the order of K fp32 additions (2^-24 each) before the rounding to bf16 (2^-9)."""
    from olmax_amd import _lib, ops
    print(f"[case] forced {tile} M{M} N{N} K{K} a{al} b{bl}", flush=True)
    a, b = operands(M, N, K, al, bl)
    want = ops.gemm(a, b, a_layout=al, b_layout=bl).double()
    res = []
    _lib.load().olmax_gemm_set_tile(tile)
    try:
        got = recorded(lambda: res.append(ops.gemm(a, b, a_layout=al, b_layout=bl)))
    finally:
        _lib.load().olmax_gemm_set_tile(0)
    assert [key & 0xfff for key, *_ in got] == [tile], got
    assert (res[0].double() - want).norm() < 2 ** -9 * want.norm()
