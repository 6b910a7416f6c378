"""GPU parity tests of sizes that no tile divides: the ragged forms of the GEMM kernels (edges of the
64, 128 and 256 tiles, partial k-tiles, rows that are not 16-byte aligned) and what is built on them."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu

BF = torch.bfloat16
rt = ref.bf16_round


def rnd(*shape, seed=0, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, device="cuda", generator=g) * scale).to(BF)


def rel(got, want):
    got, want = got.double(), want.double()
    return ((got - want).norm() / (want.norm() + 1e-300)).item()


GEMM_SHAPES = [
    (1, 1, 1), (7, 9, 3), (63, 65, 64), (64, 64, 63), (77, 2816, 1024), (65, 130, 513), (127, 128, 64), (16, 64, 2048),
    (128, 136, 72),      # one 128 tile and 8 columns, k-tile of 8
    (129, 128, 192), (200, 264, 1000), (1024, 1016, 71),
    (300, 3000, 136), (2049, 4104, 200), (4095, 2056, 88), (2500, 4360, 65), (3000, 2816, 1024), (2304, 4352, 128),
    (255, 33000, 128), (33000, 256, 328),
]


@pytest.mark.parametrize("M,N,K", GEMM_SHAPES)
@pytest.mark.parametrize("al,bl", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("pad", [0, 8, 3])
def test_gemm_ragged(M, N, K, al, bl, pad):
    """Every layout at sizes around the tile edges; `pad` widens the row strides (8: rows stay 16-byte
    aligned where they were, 3: they do not).  fp32 output against float64 on the same values:
    products are exact in fp32, so K additions bound the error by K * 2^-24 of the sum of magnitudes
    (taken as sqrt(K) * 2^-24 * 8 in the 2-norm).  Nothing outside the output view is written, the
    bf16 result is the rounded fp32 one and the residual joins it after that rounding."""
    from olmax_amd import ops
    print(f"[case] gemm M{M} N{N} K{K} a{al} b{bl} pad{pad}", flush=True)
    ar, ac = (M, K) if al == 0 else (K, M)
    br, bc = (N, K) if bl == 0 else (K, N)
    a = rnd(ar, ac + pad, seed=1)[:, :ac]
    b = rnd(br, bc + pad, seed=2)[:, :bc]
    r = rnd(M, N + pad, seed=3)[:, :N]
    want = (a.double() if al == 0 else a.double().t()) @ (b.double().t() if bl == 0 else b.double())
    wide = torch.full((M + 1, N + 16), 7.0, device="cuda", dtype=torch.float32)
    ops.gemm(a, b, a_layout=al, b_layout=bl, out=wide[:M, 8:8 + N])
    got = wide[:M, 8:8 + N]
    assert rel(got, want) < max(K, 16) ** 0.5 * 2 ** -24 * 8
    assert (wide[:, :8] == 7).all() and (wide[:, 8 + N:] == 7).all() and (wide[M] == 7).all()
    out = torch.full((M + 1, N + pad), 7.0, device="cuda", dtype=BF)
    ops.gemm(a, b, a_layout=al, b_layout=bl, out=out[:M, :N])
    assert torch.equal(out[:M, :N], got.to(BF))
    assert (out[M] == 7).all() and (out[:, N:] == 7).all()
    res = ops.gemm(a, b, a_layout=al, b_layout=bl, residual=r)
    assert torch.equal(res, (out[:M, :N].float() + r.float()).to(BF))


@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("M,N,K", [(256, 258, 64), (300, 1001, 136), (513, 2050, 128), (257, 3203, 72)])
def test_fp32_results_with_a_residual_at_ragged_edges(M, N, K, tile):
    """Column groups that the previous tile's end cuts, at any 4-byte alignment; bound as above, one addition more."""
    from olmax_amd import _lib, ops
    print(f"[case] fp32 residual M{M} N{N} K{K} tile{tile}", flush=True)
    a, b, r = rnd(M, K, seed=1), rnd(N, K, seed=2), rnd(M, N + 3, seed=3)[:, :N]
    want = a.double() @ b.double().t()
    wide = torch.full((M + 1, N + 16), 7.0, device="cuda", dtype=torch.float32)
    _lib.load().olmax_gemm_set_tile(tile)
    try:
        for res in (None, r):
            ops.gemm(a, b, residual=res, out=wide[:M, 5:5 + N])
            assert rel(wide[:M, 5:5 + N], want if res is None else want + r.double()) < (K + 1) ** 0.5 * 2 ** -24 * 8
    finally:
        _lib.load().olmax_gemm_set_tile(0)
    assert (wide[:, :5] == 7).all() and (wide[:, 5 + N:] == 7).all() and (wide[M] == 7).all()


def test_gemm_ragged_keeps_a_poisoned_neighbour_out():
    """What lies behind the operands' last rows and columns (NaN here) never reaches the result."""
    from olmax_amd import ops
    for M, N, K in ((300, 2824, 200), (2304 + 8, 4096 + 8, 72), (77, 80, 104)):
        for al, bl in ((0, 0), (0, 1), (1, 1)):
            print(f"[case] poisoned M{M} N{N} K{K} a{al} b{bl}", flush=True)
            ar, ac = (M, K) if al == 0 else (K, M)
            br, bc = (N, K) if bl == 0 else (K, N)
            big_a = torch.full((ar + 4, ac + 8), float("nan"), device="cuda", dtype=BF)
            big_b = torch.full((br + 4, bc + 8), float("nan"), device="cuda", dtype=BF)
            a, b = big_a[:ar, :ac], big_b[:br, :bc]
            a.copy_(rnd(ar, ac, seed=4)); b.copy_(rnd(br, bc, seed=5))
            got = ops.gemm(a, b, a_layout=al, b_layout=bl, out_f32=True)
            want = (a.double() if al == 0 else a.double().t()) @ (b.double().t() if bl == 0 else b.double())
            assert rel(got, want) < K ** 0.5 * 2 ** -24 * 8


@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("T,F,d", [(2049, 2048, 128), (4000, 1152, 64), (300, 8320, 128)])
def test_fused_gated_projection_on_ragged_rows(act, T, F, d):
    """Forward and backward form against the plain product followed by the elementwise kernels."""
    from olmax_amd import ops
    print(f"[case] gated projection {act} T{T} F{F} d{d}", flush=True)
    x, w, dact = rnd(T, d, seed=1), rnd(2 * F, d, seed=2, scale=d ** -0.5), rnd(T, F, seed=3)
    gu = ops.gemm(x, w)
    want = ops.glu_fwd(gu[:, :F], gu[:, F:], act)
    got, got_gu = ops.gated_mlp_in(x, w, act)
    only, none = ops.gated_mlp_in(x, w, act, save_gate_up=False)
    assert torch.equal(got, want) and torch.equal(got_gu, gu) and torch.equal(only, want) and none is None
    dg, du = ops.glu_bwd(gu[:, :F], gu[:, F:], dact, act)
    act_b, dgu = ops.gated_mlp_in_bwd(x, w, dact, act)
    assert torch.equal(act_b, want) and torch.equal(dgu[:, :F], dg) and torch.equal(dgu[:, F:], du)


@pytest.mark.parametrize("which", ["x", "w", "out"])
def test_gated_projection_on_ragged_rows_of_unaligned_views(which):
    """Views the fused GEMM cannot take get the two-step path, also when gate|up were not asked for."""
    from olmax_amd import ops
    print(f"[case] gated projection, unaligned {which}", flush=True)
    T, F, d = 2049, 2048, 128
    shift = lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)  # noqa: E731
    x, w, out = rnd(T, d, seed=1), rnd(2 * F, d, seed=2, scale=d ** -0.5), torch.empty(T, F, device="cuda", dtype=BF)
    want, _ = ops.gated_mlp_in(x, w)
    args = {k: shift(t) if k == which else t for k, t in (("x", x), ("w", w), ("out", out))}
    got, _ = ops.gated_mlp_in(args["x"], args["w"], save_gate_up=False, out=args["out"])
    assert rel(got, want) < 2 ** -8


@pytest.mark.parametrize("T,F,d", [(384, 8192, 512), (300, 8192, 576), (900, 9216, 768)])
def test_gated_projection_of_few_ragged_rows_takes_two_steps(T, F, d):
    """Where that is faster; the rows of a whole number of 256 take the fused kernel.  fp32 orders before bf16 roundings."""
    from olmax_amd import _lib, ops
    print(f"[case] gated projection in two steps T{T} F{F} d{d}", flush=True)
    whole = -(-T // 256) * 256
    x, w, dact = rnd(whole, d, seed=1), rnd(2 * F, d, seed=2, scale=d ** -0.5), rnd(whole, F, seed=3)
    args = lambda t: (*map(_lib.ptr, (x, w, dact)), *map(_lib.i32, (t, F, d)), *map(_lib.i64, (d, d, F)))  # noqa: E731
    assert _lib.load().olmax_gemm_glu_fused(*args(T)) == 2 and _lib.load().olmax_gemm_glu_fused(*args(whole)) == 1
    want, want_gu = ops.gated_mlp_in(x, w)
    got, got_gu = ops.gated_mlp_in(x[:T], w)
    only, none = ops.gated_mlp_in(x[:T], w, save_gate_up=False)
    assert rel(got, want[:T]) < 2 ** -8 and rel(got_gu, want_gu[:T]) < 2 ** -8 and torch.equal(only, got) and none is None
    want, want_dgu = ops.gated_mlp_in_bwd(x, w, dact)
    got, got_dgu = ops.gated_mlp_in_bwd(x[:T], w, dact[:T])
    assert rel(got, want[:T]) < 2 ** -8 and rel(got_dgu, want_dgu[:T]) < 2 ** -8


def test_rotary_projection_of_few_ragged_rows_takes_two_steps():
    from olmax_amd import ops
    print("[case] rope projection in two steps", flush=True)
    T, heads, N, d = 640, 64, 12288, 512
    x, w = rnd(768, d, seed=1), rnd(N, d, seed=2, scale=d ** -0.5)
    cos, sin = ops.rope_tables(768, 128, 10000.0, "cuda")
    want = ops.qkv_rope_proj(x, w, cos, sin, rope_heads=heads, seq_len=768)
    got = ops.qkv_rope_proj(x[:T], w, cos, sin, rope_heads=heads, seq_len=768)
    assert rel(got, want[:T]) < 2 ** -8


@pytest.mark.parametrize("T,which,tile", [(2048, "x", 0), (2048, "w", 0), (2048, "out", 0), (2048, "none", 256), (2049, "none", 128)])
def test_gated_projection_gets_scratch_wherever_the_fused_kernel_does_not_run(T, which, tile):
    """Unaligned operands at whole tiles, and a forced tile size; the result differs by fp32 orders before bf16 roundings."""
    from olmax_amd import _lib, ops
    print(f"[case] gated projection T{T}, unaligned {which}, tile {tile}", flush=True)
    F, d = 2048, 128
    shift = lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)  # noqa: E731
    x, w, out = rnd(T, d, seed=1), rnd(2 * F, d, seed=2, scale=d ** -0.5), torch.empty(T, F, device="cuda", dtype=BF)
    want, _ = ops.gated_mlp_in(x, w)
    args = {k: shift(t) if k == which else t for k, t in (("x", x), ("w", w), ("out", out))}
    _lib.load().olmax_gemm_set_tile(tile)
    try:
        got, _ = ops.gated_mlp_in(args["x"], args["w"], save_gate_up=False, out=args["out"])
    finally:
        _lib.load().olmax_gemm_set_tile(0)
    assert rel(got, want) < 2 ** -8


@pytest.mark.parametrize("T", [1000, 1024])
@pytest.mark.parametrize("tile", [0, 128])
def test_forward_of_a_model_whose_weights_are_not_16_byte_aligned(T, tile):
    """The gated projection then takes the two-step path and needs gate|up as scratch although no backward pass follows; so
    it does while a tile size is forced.  The loss differs by fp32 orders before bf16 roundings."""
    from olmax_amd import TransformerConfig, _lib
    print(f"[case] unaligned weights T{T} tile{tile}", flush=True)
    cfg = TransformerConfig(vocab_size=512, d_model=128, hidden_size=4096, num_layers=1, n_heads=1, head_dim=128)
    model = cfg.build(batch_size=1, sequence_length=T, seed=1)
    ids, labels = (torch.randint(0, 512, (T,), device="cuda", dtype=torch.int32) for _ in range(2))
    want = model.forward_loss(ids, labels).item()
    p = model.params_bf16
    model.params_bf16 = torch.cat([p.new_zeros(1), p])[1:]
    assert model.params_bf16.data_ptr() % 16
    _lib.load().olmax_gemm_set_tile(tile)
    try:
        got = [model.forward_loss(ids, labels).item()]
        model.params_bf16 = p
        got.append(model.forward_loss(ids, labels).item())
    finally:
        _lib.load().olmax_gemm_set_tile(0)
    assert all(abs(x - want) < 1e-4 * want for x in got)


@pytest.mark.parametrize("B,S,heads,N,d", [(3, 1000, 24, 3072, 128), (1, 2049, 20, 6144, 64)])
def test_fused_rope_projection_on_ragged_rows(B, S, heads, N, d):
    from olmax_amd import ops
    print(f"[case] rope projection B{B} S{S} heads{heads} N{N} d{d}", flush=True)
    x, w = rnd(B * S, d, seed=1), rnd(N, d, seed=2, scale=d ** -0.5)
    cos, sin = ops.rope_tables(S, 128, 10000.0, "cuda")
    want = ops.gemm(x, w)
    ops.qk_rope_fwd(want[:, :heads * 128], cos, sin, heads=heads, head_dim=128, seq_len=S, out=want[:, :heads * 128])
    assert torch.equal(ops.qkv_rope_proj(x, w, cos, sin, rope_heads=heads, seq_len=S), want)


@pytest.mark.parametrize("T,d,V,cap", [(40, 24, 101, 0.0), (300, 256, 2566, 0.0), (520, 128, 33030, 30.0), (130, 64, 163846, 0.0)])
def test_lm_head_with_a_vocabulary_of_ragged_rows(T, d, V, cap):
    """V % 8 != 0: the logits' row stride is padded inside the workspace; loss and both gradients
    against float64.  Bound: dlogits are rounded to bf16 (2^-9 relative each), and so are dh and dW."""
    from olmax_amd import ops
    print(f"[case] lmhead T{T} d{d} V{V} cap{cap}", flush=True)
    h, W = rnd(T, d, seed=1), rnd(V, d, seed=2, scale=0.1)
    g = torch.Generator().manual_seed(3)
    labels = torch.randint(0, V, (T,), generator=g, dtype=torch.int32)
    labels[0], labels[1], labels[2] = -100, V - 1, V
    loss, dh, dW = ops.lmhead_ce(h, W, labels.cuda(), softcap=cap)
    with torch.device("cuda"):
        wl, wdh, wdw = ref.lm_head_ce(h.double(), W.double(), labels.long().cuda(), softcap=cap, rt=rt)
    assert abs(loss.item() - wl.item()) < 1e-3 * abs(wl.item())
    assert rel(dh, wdh) < 8e-3 and rel(dW, wdw) < 8e-3
