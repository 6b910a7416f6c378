"""GPU parity tests of products in 32 x 32 tiles, and of two gradients in one launch (every size of tile), at the edges of tiles, chunks
and k-tiles."""
import pytest
import torch

from oracle import ref
from test_gemm_choice_gpu import operands, recorded, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("al,bl", [(0, 0), (0, 1), (1, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (31, 33, 63), (32, 32, 64), (33, 40, 65), (40, 96, 1024), (100, 256, 1032), (256, 256, 2048),
                                   (77, 1024, 2816), (520, 264, 1000), (16, 4096, 4096)])
def test_tiles_of_32(M, N, K, al, bl):
    """Against float64: K fp32 additions (2^-24 each) and one rounding to bf16, 2^-9 of the value."""
    from olmax_amd import ops
    print(f"[case] tiles of 32 M{M} N{N} K{K} a{al} b{bl}", flush=True)
    a, b = operands(M, N, K, al, bl)
    r = rnd(M, N, seed=3)
    want = (a if al == 0 else a.t()).double() @ (b.t() if bl == 0 else b).double()
    scale = 2 ** -22 * K ** 0.5 * 6  # of the sum's terms, N(0, 1) products
    for res in (None, r):
        got = ops.gemm(a, b, a_layout=al, b_layout=bl, residual=res).double()
        full = want if res is None else want + res.double()
        # with a residual the product is rounded first, then the sum
        assert ((got - full).abs() <= 2 ** -8 * (want.abs() + full.abs()) + scale).all()
    assert ((ops.gemm(a, b, a_layout=al, b_layout=bl, out_f32=True).double() - want).abs() <= scale).all()


@pytest.mark.parametrize("M,N,bl", [(3000, 8200, 0), (4096, 4096, 1)])
def test_one_k_tile_of_many_outputs(M, N, bl):
    """A single k-tile over many outputs goes to 128 or 256 tiles: thousands of 32 x 32 ones take twice as long.  Bounds as above."""
    from olmax_amd import ops
    print(f"[case] one k-tile M{M} N{N} b{bl}", flush=True)
    a, b = operands(M, N, 64, 0, bl)
    out = []
    got = recorded(lambda: out.append(ops.gemm(a, b, b_layout=bl)))
    assert all(key & 0xfff != 64 for key, *_ in got) and got, got
    want = a.double() @ (b.t() if bl == 0 else b).double()
    assert ((out[0].double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -22 * 48).all()


@pytest.mark.parametrize("T,d,V,pair", [(2048, 256, 4096, True), (64, 1024, 512, True), (100, 264, 520, True), (1001, 64, 2056, True),
                                        (2048, 1024, 256, True), (65, 40, 72, True), (300, 256, 1003, False), (63, 256, 512, False)])
@pytest.mark.parametrize("f32", [False, True])
def test_both_gradients_in_one_launch(T, d, V, pair, f32):
    """dh and dW of the LM head.  The oracle takes the logits as this library rounds them; dlogits and the results are rounded to
    bf16, 2^-9 each, and a handful of logits round the other way: 8e-3 of a row's or column's norm, as two of each."""
    from olmax_amd import ops
    print(f"[case] pair T{T} d{d} V{V} f32{f32}", flush=True)
    h, W = rnd(T, d, seed=1), rnd(V, d, seed=2, scale=0.1)
    labels = torch.arange(T, device="cuda", dtype=torch.int32) * 7 % V
    out = []
    got = recorded(lambda: out.extend(ops.lmhead_ce(h, W, labels, dw_f32=f32)))
    assert any(key >> 19 & 1 for key, *_ in got) == (pair and not f32), got  # (fp32 results keep the kernels with the shorter chains)
    check_gradients(h, W, labels, *out[1:])


def check_gradients(h, W, labels, dh, dW):
    z = (h.double() @ W.double().t()).to(torch.bfloat16).double().cpu()
    dz = ref.cross_entropy_bwd(z, labels.cpu().long()).cuda()
    for g, w in ((dh, dz @ W.double()), (dW, dz.t() @ h.double())):
        for dim in (0, 1):
            e = (g.double() - w).norm(dim=dim) / (w.norm(dim=dim) + 1e-3 * w.norm())
            assert e.max().item() < 8e-3, (dim, e.argmax().item(), e.max().item())


@pytest.mark.parametrize("T,d,V,tile", [
    (4096, 1024, 3072, 128), (4096, 1032, 3072, 128),  # whole tiles; ragged columns in both products
    (3000, 1024, 3072, 128), (3000, 1024, 2880, 128),  # ragged rows and a partial k-tile of dW; dW ragged too
    (4160, 1024, 3072, 128), (4096, 1024, 2880, 128),  # ragged rows, whole k-tiles; only dW ragged
    (2048, 11008, 4096, 256), (2048, 11000, 4096, 256), (2000, 11008, 4096, 256), (2000, 11008, 3904, 256), (1984, 11008, 4096, 256),
    (2048, 11008, 3904, 256),
])
def test_both_gradients_in_one_launch_of_large_tiles(T, d, V, tile):
    """As above; the launch is in tiles of the expected size."""
    from olmax_amd import ops
    print(f"[case] pair T{T} d{d} V{V} tile{tile}", flush=True)
    h, W = rnd(T, d, seed=1), rnd(V, d, seed=2, scale=0.02)
    labels = torch.arange(T, device="cuda", dtype=torch.int32) * 7 % V
    out = []
    got = recorded(lambda: out.extend(ops.lmhead_ce(h, W, labels)))
    assert (tile | 1 << 19, T, d, V, 1) in got, got
    check_gradients(h, W, labels, *out[1:])


@pytest.mark.parametrize("seq,tile,out", [(1500, 0, 0), (2048, 256, 22016), (1000, 128, 22016), (2500, 256, 22016), (3000, 256, 12288)])
def test_a_residual_joins_the_first_product(seq, tile, out):
    """Post-norm blocks add the residual's gradient in dX, in one launch with dW, of whole and of ragged rows and k-tiles; at 1500 tokens
    they are two calls, beside a launch of the products without a residual.  Against the two calls, which a forced tile brings back: the products
    are rounded to bf16 (2^-9 each) and four of them follow one another."""
    from olmax_amd import TransformerRecipe, _lib
    from olmax_amd.layer import TransformerBlock
    import dataclasses
    cfg = dataclasses.replace(TransformerRecipe.olmo2_7B(), num_layers=1)
    block = TransformerBlock(cfg, batch_size=1, sequence_length=seq)
    g = torch.Generator(device="cuda").manual_seed(1)
    for w in (block.wqkv, block.wo, block.wgu, block.wdown):
        w.normal_(0.0, 0.02, generator=g)
    x, dy = rnd(seq, cfg.d_model, seed=2), rnd(seq, cfg.d_model, seed=3)
    block.forward(x)
    res, dx = {}, []
    got = recorded(lambda: dx.append(block.backward(dy)))
    assert any(key >> 19 & 1 for key, *_ in got), got
    assert any(key >> 19 & 1 and key >> 14 & 1 for key, *_ in got) == (tile != 0), got
    assert not tile or (tile | 1 << 14 | 1 << 19, seq, 4096, out, 1) in got, got
    res[0] = [dx[0].clone()] + [v.clone() for v in block.grads.values()]
    for v in block.grads.values():
        v.zero_()
    _lib.load().olmax_gemm_set_tile(256)
    try:
        got = recorded(lambda: dx.append(block.backward(dy)))
    finally:
        _lib.load().olmax_gemm_set_tile(0)
    assert not any(key >> 19 & 1 for key, *_ in got), got
    for a, b in zip(res[0], [dx[1]] + list(block.grads.values())):
        assert ((a.double() - b.double()).norm() / b.double().norm()).item() < 2 ** -7


@pytest.mark.parametrize("T,d,V", [(2048, 256, 4096), (2048, 1024, 256), (4096, 1024, 3072), (2000, 11008, 4096)])
def test_a_weight_gradient_in_the_place_of_the_weights(T, d, V):
    """dh reads the weights first, so dW may overwrite them: the products stay in their order, at sizes where one launch would take
    both.  Bounds as above, which hold for logits of a few units: at a spread of 10 a label's 1 - p may be of the size of the logits' own
    rounding, 2^-9 of 30."""
    from olmax_amd import ops
    print(f"[case] dW over W T{T} d{d} V{V}", flush=True)
    h, W = rnd(T, d, seed=1), rnd(V, d, seed=2, scale=2 * d ** -0.5)
    labels = torch.arange(T, device="cuda", dtype=torch.int32) * 7 % V
    assert any(key >> 19 & 1 for key, *_ in recorded(lambda: ops.lmhead_ce(h, W, labels)))
    kept, out = W.clone(), []
    got = recorded(lambda: out.extend(ops.lmhead_ce(h, W, labels, dW=W)))
    assert not any(key >> 19 & 1 for key, *_ in got), got
    check_gradients(h, kept, labels, *out[1:])


def head_sums(terms_h, terms_W, T, d, V):
    """Gradients of the LM head whose logits are all zero, so that every dlogit but the labels' is one bf16 number c: rows of `terms` sit at
    the first token (vocabulary entry) of their k-tile, and the gradient of the other operand is c times their sum.  Labels name the last
    entry, whose row of W is zero."""
    from olmax_amd import ops
    h, W = (torch.zeros(n, d, device="cuda", dtype=torch.bfloat16) for n in (T, V))
    for x, terms in ((h, terms_h), (W, terms_W)):
        for kt, value in terms:
            x[64 * kt] = value
    labels = torch.full((T,), V - 1, device="cuda", dtype=torch.int32)
    out = []
    got = recorded(lambda: out.extend(ops.lmhead_ce(h, W, labels)))
    c = (torch.tensor(1.0, dtype=torch.float64) / V / T).to(torch.bfloat16)
    return got, out[1], out[2][:-1], c


@pytest.mark.parametrize("T,d,V,waves", [
    (1024, 512, 1024, 8), (1536, 256, 2048, 8),  # every tile finds a CU
    (1024, 256, 1024, 4), (2048, 256, 4096, 4), (2048, 512, 1024, 4)])  # more tiles, of 32 and 64: two chains to a wave
@pytest.mark.parametrize("which", ["dh", "dW"])
def test_one_launch_keeps_eight_chains(T, d, V, waves, which):
    """A tile of the single product has eight waves, and wave w adds the k-tiles w, w + 8, ...: 2^24 and -2^24 meet there and a 1 from a
    k-tile of another wave counts.  One chain for the k-tiles w, w + 4, ... would lose it: 2^24 + 1 = 2^24 in fp32.  Four waves have a chain for the
    first half of these and one for the second: there the 1 comes first."""
    print(f"[case] chains T{T} d{d} V{V} {which}", flush=True)
    n = (V if which == "dh" else T) // 64
    terms = [(w, 2.0 ** 24) for w in range(4)] + [(4 + w, 1.0) for w in range(4)] + [(8 + w, -(2.0 ** 24)) for w in range(4)]
    if waves == 4:
        second = 4 * -(-n // 8)  # wave w's second half
        terms = [(w, 1.0) for w in range(4)] + [(second + w, 2.0 ** 24) for w in range(4)] + [(second + 4 + w, -(2.0 ** 24)) for w in range(4)]
    assert n > 12
    got, dh, dW, c = head_sums(*(([], terms) if which == "dh" else (terms, [])), T, d, V)
    assert (64 | 1 << 19, T, d, V, 1) in got, got
    assert ((dh if which == "dh" else dW).float() == 4 * c.item()).all()


@pytest.mark.parametrize("T,d,V", [(512, 1024, 4096), (2048, 2048, 256)])
def test_one_launch_of_operands_that_only_the_small_kernel_takes(T, d, V):
    """Rows that do not start on 16 bytes: the alternative is the small kernel twice, not the 128 tiles that aligned rows would take."""
    from olmax_amd import ops
    print(f"[case] pair of unaligned rows T{T} d{d} V{V}", flush=True)
    h, W = (torch.empty(n * d + 4, device="cuda", dtype=torch.bfloat16)[4:].view(n, d) for n in (T, V))
    h.copy_(rnd(T, d, seed=1))
    W.copy_(rnd(V, d, seed=2, scale=0.1))
    labels = torch.arange(T, device="cuda", dtype=torch.int32) * 7 % V
    out = []
    got = recorded(lambda: out.extend(ops.lmhead_ce(h, W, labels)))
    assert (64 | 1 << 19, T, d, V, 1) in got, got
    check_gradients(h, W, labels, *out[1:])


@pytest.mark.parametrize("T,d,V,which,block", [
    (8192, 1024, 3072, "dW", 32), (4096, 1024, 3072, "dW", 16), (512, 2816, 1024, "dh", 4), (320, 2816, 320, "dh", 2), (320, 2816, 320, "dW", 2),
    (3000, 1024, 2880, "dh", 12), (3000, 1024, 2880, "dW", 12)])  # partial k-tile and ragged edges
def test_128_tiles_in_one_launch_add_in_blocks(T, d, V, which, block):
    """1 in the first block of k-tiles, 2^24 and -2^24 in the second: one chain over all of them would lose the 1 (2^24 + 1 = 2^24 in fp32).  The
    same in the last whole block.  The blocks are as large as the chains of the two calls allow."""
    print(f"[case] blocks T{T} d{d} V{V} {which}", flush=True)
    K = V if which == "dh" else T
    n, first = -(-K // 64) // block * block, int(K % 64 != 0)  # (a partial k-tile comes before the whole ones)
    for at in (block - first, n - block - first):
        terms = [(0, 1.0), (at, 2.0 ** 24), (at + block - 1, -(2.0 ** 24))]
        got, dh, dW, c = head_sums(*(([], terms) if which == "dh" else (terms, [])), T, d, V)
        assert (128 | 1 << 19, T, d, V, 1) in got, got
        assert ((dh if which == "dh" else dW).float() == c.item()).all()


@pytest.mark.parametrize("seq", [1700, 2048])
def test_one_launch_parks_the_sums_that_the_calls_share(seq, monkeypatch):
    """dX of the q|k|v and the gate|up projections of a post-norm block: 12288 and 22016 long, each half a chain of its own as in the two calls, where
    two workgroups share a reduction.  The calls, which gradients in the place of their weights bring back, add the same two sums: bit-equal."""
    import dataclasses
    from olmax_amd import TransformerRecipe
    from olmax_amd.layer import TransformerBlock
    print(f"[case] parked sums S{seq}", flush=True)
    block = TransformerBlock(dataclasses.replace(TransformerRecipe.olmo2_7B(), num_layers=1), batch_size=1, sequence_length=seq)
    g = torch.Generator(device="cuda").manual_seed(1)
    for w in (block.wqkv, block.wo, block.wgu, block.wdown):
        w.normal_(0.0, 0.02, generator=g)
    block.forward(rnd(seq, 4096, seed=1))
    dy, res = rnd(seq, 4096, seed=2), []

    def backward():
        res.append([block.backward(dy)] + [block.grads[k].clone() for k in ("attention.q_proj.weight", "attention.v_proj.weight", "mlp.up_proj.weight")])
    got = recorded(backward)
    for out in (12288, 22016):
        assert (256 | 1 << 14 | 1 << 19, seq, 4096, out, 1) in got, got
    fresh = torch.empty_like
    monkeypatch.setattr(torch, "empty_like", lambda t: t if t is block.wqkv or t is block.wgu else fresh(t))
    got = recorded(backward)
    for out in (12288, 22016):
        assert any(key >> 18 & 1 and shape[:3] == [seq, 4096, out] for key, *shape in got), got
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("al,bl", [(0, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(900, 1800, 16), (1200, 1200, 40), (1024, 1040, 63), (1040, 1984, 8)])
def test_part_of_a_k_tile_in_one_round_of_64_tiles(M, N, K, al, bl):
    test_tiles_of_32(M, N, K, al, bl)
