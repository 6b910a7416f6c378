"""The k loop of the 256-wide GEMM tiles at its shortest lengths: one k-tile to five, odd and even, whole and ragged, in every layout."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("al,bl", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("M,N", [(256, 256), (520, 768)])
def test_short_reductions_on_large_tiles_are_exact(M, N, al, bl):
    """Whole numbers up to 4: every product and sum (below 2^24) is exact in fp32, so any fragment taken from the wrong place shows."""
    from olmax_amd import _lib, ops
    gen = torch.Generator(device="cuda").manual_seed(5)
    _lib.load().olmax_gemm_set_tile(256)
    try:
        for K in (64, 72, 128, 136, 192, 256, 264, 320):
            print(f"[case] pipeline M{M} N{N} K{K} a{al} b{bl}", flush=True)
            ints = lambda *s: torch.randint(-4, 5, s, device="cuda", generator=gen).bfloat16()  # noqa: E731
            a, b = ints(*((M, K) if al == 0 else (K, M))), ints(*((N, K) if bl == 0 else (K, N)))
            want = (a if al == 0 else a.t()).double() @ (b.t() if bl == 0 else b).double()
            assert torch.equal(ops.gemm(a, b, a_layout=al, b_layout=bl, out_f32=True).double(), want)
    finally:
        _lib.load().olmax_gemm_set_tile(0)
