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


@pytest.mark.parametrize("M,N", [(256, 128), (300, 200), (520, 768)])
def test_short_reductions_on_256_x_128_tiles_are_exact(M, N):
    """Products of -1, 0 and 1: sums and residuals stay below 256, whole numbers that bf16 holds.  One k-tile to seven: the three stages twice over."""
    from olmax_amd import _lib, ops
    gen = torch.Generator(device="cuda").manual_seed(6)
    ints = lambda *s: torch.randint(-1, 2, s, device="cuda", generator=gen).bfloat16()  # noqa: E731
    _lib.load().olmax_gemm_set_tile(384)
    try:
        for K in (64, 72, 128, 136, 192, 256, 264, 320, 384, 448):
            print(f"[case] 256 x 128 tiles M{M} N{N} K{K}", flush=True)
            a, b, r = ints(M, K), ints(N, K), ints(M, N)
            want = a.double() @ b.t().double()
            assert want.abs().max() < 255
            assert torch.equal(ops.gemm(a, b).double(), want)
            assert torch.equal(ops.gemm(a, b, residual=r).double(), want + r.double())
    finally:
        _lib.load().olmax_gemm_set_tile(0)


def test_forward_products_of_few_128_tiles_take_256_x_128_ones():
    from olmax_amd import ops
    from test_gemm_choice_gpu import operands, recorded
    a, b = operands(1500, 4096, 4096, 0, 0)
    print("[case] 256 x 128 tiles chosen", flush=True)
    assert [(key & 0xfff, m, n, k) for key, m, n, k, _ in recorded(lambda: ops.gemm(a, b))] == [(384, 1500, 4096, 4096)]


@pytest.mark.parametrize("M,N,K,tile", [
    (260, 14336, 4096, 384), (4096, 1280, 4096, 384), (8192, 1024, 2816, 384), (1000, 6144, 9216, 384), (448, 9152, 9152, 384), (1500, 2816, 2048, 384),
    (512, 8064, 4096, 384), (768, 5248, 6336, 384), (2048, 2048, 2816, 128), (4096, 1024, 5120, 128), (8192, 512, 11008, 128),
    (1500, 2816, 4104, 128), (768, 5120, 6960, 128), (1064, 5504, 4104, 384), (498, 11896, 2056, 384), (2048, 4096, 1984, 128)])
def test_256_x_128_tiles_take_what_they_are_faster_on(M, N, K, tile):
    """While a tile of 128 has a CU to itself only wide products; part of a k-tile only in wide ones of more; no short reductions.  Against float64: 2^-9 for the rounding to bf16, as much again for the sums."""
    from olmax_amd import ops
    from test_gemm_choice_gpu import operands, recorded
    a, b = operands(M, N, K, 0, 0)
    print(f"[case] 256 x 128 or 128 tiles M{M} N{N} K{K}", flush=True)
    out = []
    assert [(key & 0xfff, m, n, k) for key, m, n, k, _ in recorded(lambda: out.append(ops.gemm(a, b)))] == [(tile, M, N, K)]
    want = a[-300:].double() @ b[-300:].double().t()
    assert (out[0][-300:, -300:].double() - want).norm() < 2 ** -8 * want.norm()


@pytest.mark.parametrize("seq", [8192, 7500])  # whole tiles; ragged rows and a partial k-tile at the end of dW's last part
def test_a_narrow_layers_dw_shares_its_reduction_inside_the_one_launch(seq):
    """Of a block of width 1024 the gate|up projection's dW parks its blocks and the q|k|v projection's comes in parts.  Against the two calls, which
    a forced tile brings back: the products are rounded to bf16 (2^-9 each) and four of them follow one another."""
    import dataclasses

    from olmax_amd import TransformerRecipe, _lib
    from olmax_amd.layer import TransformerBlock
    from test_gemm_choice_gpu import recorded
    print(f"[case] narrow block S{seq}", flush=True)
    cfg = dataclasses.replace(TransformerRecipe.olmo2_7B(), num_layers=1, d_model=1024, hidden_size=2816, n_heads=8, n_kv_heads=8, head_dim=128)
    block = TransformerBlock(cfg, batch_size=1, sequence_length=seq)
    gen = torch.Generator(device="cuda").manual_seed(1)
    for w in (block.wqkv, block.wo, block.wgu, block.wdown):
        w.normal_(0.0, 0.02, generator=gen)
    x, dy = (torch.empty(seq, 1024, device="cuda", dtype=torch.bfloat16).normal_(generator=gen) for _ in range(2))
    block.forward(x)
    dx = []
    got = recorded(lambda: dx.append(block.backward(dy)))
    for out in (3072, 5632):
        assert any(key & 0xfff == (256 if out == 3072 or seq == 8192 else 128) and key >> 19 & 1 and (m, n, k) == (seq, 1024, out) for key, m, n, k, _ in got), got
    res = [dx[0].clone()] + [v.clone() for v in block.grads.values()]
    for v in block.grads.values():
        v.zero_()
    _lib.load().olmax_gemm_set_tile(256)
    try:
        got = recorded(lambda: dx.append(block.backward(dy)))
    finally:
        _lib.load().olmax_gemm_set_tile(0)
    assert not any(key >> 19 & 1 for key, *_ in got), got
    for a, b in zip(res, [dx[1]] + list(block.grads.values())):
        assert ((a.double() - b.double()).norm() / b.double().norm()).item() < 2 ** -7
