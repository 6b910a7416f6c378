"""GPU parity tests of the MFMA attention kernels' head_dim-64 form and of their split forms at the edges of
their 128-row blocks, 64-key and 32-query tiles."""
import math

import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def rnd(*shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, device="cuda", generator=g).to(BF)


def rel(got, want):
    got, want = got.double().cpu(), want.double().cpu()
    return ((got - want).norm() / (want.norm() + 1e-300)).item()


def check(B, S, H, KH, D, window, softcap, strided=False, groups=None):
    """Every output (of the K/V heads `groups` and their query heads only) against the float64 oracle.  P and dS are rounded to
    bf16 (2^-9 each) before the second products and the results once more: 2-norm errors of 0.3 % at most; bounds are three
    times that."""
    from olmax_amd import ops

    print(f"[case] attn B{B} S{S} H{H} KH{KH} D{D} w{window} cap{softcap}", flush=True)
    if strided:  # q | k | v columns of one projection
        qkv = rnd(B * S, (H + 2 * KH) * D, seed=S + D)
        q, k, v = qkv[:, :H * D], qkv[:, H * D:(H + KH) * D], qkv[:, (H + KH) * D:]
    else:
        q, k, v = rnd(B * S, H * D, seed=1), rnd(B * S, KH * D, seed=2), rnd(B * S, KH * D, seed=3)
    do = rnd(B * S, H * D, seed=4)
    kw = dict(B=B, S=S, H=H, KH=KH, D=D, window=window, softcap=softcap)
    guard = torch.full((B * S + 2, H * D), 7.0, device="cuda", dtype=BF)  # nothing outside the output rows is written
    o, lse = ops.attn_fwd(q, k, v, out=guard[1:-1], **kw)
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()
    dq, dk, dv = ops.attn_bwd(q, k, v, o, lse, do, **kw)
    groups = list(range(KH)) if groups is None else groups
    rep = H // KH
    heads = [g * rep + r for g in groups for r in range(rep)]
    cut = lambda t: t.reshape(B, S, -1, D)[:, :, heads if t.shape[1] == H * D else groups].double().cpu()  # noqa: E731
    q4, k4, v4, d4 = (cut(t) for t in (q, k, v, do))
    wo, wlse = ref.attention_fwd(q4, k4, v4, window=window, softcap=softcap)
    assert rel(cut(o), wo) < 1e-2
    assert (lse[:, heads].cpu().double() - wlse).abs().max() < 2e-3
    want = ref.attention_bwd(q4, k4, v4, wo, wlse, d4, window=window, softcap=softcap)
    for name, got, w in zip(("dq", "dk", "dv"), (cut(dq), cut(dk), cut(dv)), want):
        if w.norm() < 1e-12 * math.sqrt(w.numel()):  # S = 1: dS is exactly zero, what remains is rounding
            assert got.double().norm() < 1e-2 * math.sqrt(got.numel()), name
        else:
            assert rel(got, w) < 1e-2, name


@pytest.mark.parametrize("S", [1, 31, 33, 63, 65, 127, 128, 129, 192, 321])
@pytest.mark.parametrize("H,KH,window,softcap", [(4, 4, None, 0.0), (4, 2, 40, 0.0), (2, 1, None, 30.0)])
def test_head_dim_64(S, H, KH, window, softcap):
    check(2, S, H, KH, 64, window, softcap, strided=S % 2 == 1)


@pytest.mark.parametrize("S,H,KH,window,softcap", [(512, 4, 4, None, 0.0), (512, 4, 4, None, 30.0), (512, 4, 2, 128, 50.0), (300, 64, 64, None, 50.0)])
def test_head_dim_64_normaliser_is_exact_to_fp32(S, H, KH, window, softcap):
    """LSE against float64, with few workgroups and with enough for the unsplit form: values of 4 to 8 and two or three
    fp32 roundings of that size (2^-22 each) between the score, the sum's logarithm and their sum: 2^-20 and half of it again."""
    from olmax_amd import ops
    print(f"[case] lse S{S} H{H} KH{KH} w{window} cap{softcap}", flush=True)
    q, k, v = rnd(2 * S, H * 64, seed=1), rnd(2 * S, KH * 64, seed=2), rnd(2 * S, KH * 64, seed=3)
    _, lse = ops.attn_fwd(q, k, v, B=2, S=S, H=H, KH=KH, D=64, window=window, softcap=softcap)
    q4, k4 = q.double().view(2, S, H, 64), k.double().view(2, S, KH, 64)
    i = torch.arange(S, device="cuda")
    hidden = (i[None] > i[:, None]) | (i[None] < i[:, None] - (S if window is None else window))
    for b in range(2):
        for h in range(H):
            s = q4[b, :, h] @ k4[b, :, h * KH // H].t() / 8
            s = softcap * torch.tanh(s / softcap) if softcap else s
            want = torch.logsumexp(s.masked_fill(hidden, -math.inf), -1)
            assert (lse[b, h].double() - want).abs().max() < 1.5 * 2 ** -20, (b, h)


@pytest.mark.parametrize("B,S,H,window,softcap", [(3, 400, 48, None, 0.0), (3, 500, 48, 200, 0.0), (3, 450, 48, None, 30.0), (2, 600, 4, None, 0.0)])
def test_head_dim_64_normaliser_is_as_exact_as_pair_by_pair(B, S, H, window, softcap):
    """Root mean square of LSE's error against float64, on these kernels and on the one-wave-per-query ones (which take views
    that are not 16-byte aligned).  Bound: 1 % for another order of the sums, and three standard deviations of the quotient of two
    root mean squares of N independent samples each, 1 / sqrt(N)."""
    from olmax_amd import ops
    print(f"[case] lse rms B{B} S{S} H{H} w{window} cap{softcap}", flush=True)
    n = B * S
    q, k, v = rnd(n, H * 64, seed=1), rnd(n, H * 64, seed=2), rnd(n, H * 64, seed=3)
    odd = lambda t: torch.cat([t, t.new_zeros(n, 3)], 1)[:, :t.shape[1]]  # noqa: E731
    kw = dict(B=B, S=S, H=H, KH=H, D=64, window=window, softcap=softcap)
    i = torch.arange(S, device="cuda")
    hidden = (i[None] > i[:, None]) | (i[None] < i[:, None] - (S if window is None else window))
    err = []
    for form in (lambda t: t, odd):
        _, lse = ops.attn_fwd(form(q), form(k), form(v), **kw)
        sq = 0.0
        for b in range(B):
            for h in range(H):
                s = q.view(B, S, H, 64)[b, :, h].double() @ k.view(B, S, H, 64)[b, :, h].double().t() / 8
                s = softcap * torch.tanh(s / softcap) if softcap else s
                sq += (lse[b, h].double() - torch.logsumexp(s.masked_fill(hidden, -math.inf), -1)).square().sum().item()
        err.append((sq / (B * H * S)) ** 0.5)
    assert err[0] < (1.01 + 3 / (B * H * S) ** 0.5) * err[1], err


# iterations (query heads x 32-row tiles) that the four query groups share out unevenly, or that some go without
@pytest.mark.parametrize("S,H,KH,window,softcap", [(1, 2, 2, None, 0.0), (32, 3, 1, None, 0.0), (33, 8, 2, None, 0.0), (65, 3, 1, 0, 0.0), (97, 5, 1, 31, 0.0),
                                                   (160, 2, 2, None, 30.0), (257, 4, 1, None, 0.0), (450, 3, 3, 64, 0.0)])
def test_key_gradients_split_over_query_groups(S, H, KH, window, softcap):
    check(2, S, H, KH, 128, window, softcap, strided=S % 2 == 1)


# key tiles that the key groups of the forward and dQ share out unevenly, or that some go without
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,H,KH,window,softcap", [(1, 2, 2, None, 0.0), (64, 2, 1, None, 0.0), (65, 2, 2, 0, 0.0), (130, 3, 1, None, 30.0), (200, 4, 2, 70, 0.0),
                                                   (449, 2, 2, None, 0.0)])
def test_queries_split_over_key_groups(S, H, KH, window, softcap, D):
    check(3, S, H, KH, D, window, softcap, strided=S % 2 == 0)


# chains long enough for the split forward and dQ (from 6 key tiles on at head_dim 128, 2 at 64): ragged ends, windows, soft-caps
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H,KH,window,softcap", [(1, 321, 3, 1, None, 0.0), (2, 385, 2, 2, None, 30.0), (1, 450, 4, 2, 300, 0.0), (2, 641, 2, 1, 257, 50.0), (1, 1100, 2, 2, None, 0.0)])
def test_long_chains_split_over_key_groups(B, S, H, KH, window, softcap, D):
    check(B, S, H, KH, D, window, softcap, strided=S % 2 == 1)


# more workgroups than either rule splits for (n of 128 queries, keys): the forms without a split, over many tiles
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H,KH,window,softcap", [
    (1, 1000, 82, 82, None, 0.0),    # n = 656, 656
    (3, 1000, 28, 28, None, 50.0),   # 672, 672
    (1, 1301, 60, 60, 300, 0.0),     # 660, 660: windows that start inside a tile
    (2, 449, 164, 82, 70, 30.0),     # 1312, 656
    (1, 1000, 132, 33, None, 0.0),   # 1056 plain, 264 split
    (4, 129, 90, 90, None, 0.0),     # 720, 720: a last tile of one row
])
def test_filled_gpus_take_the_forms_without_a_split(B, S, H, KH, window, softcap, D):
    check(B, S, H, KH, D, window, softcap, strided=S % 2 == 1, groups=[0, KH // 2, KH - 1])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,H,KH", [(130, 4, 2), (1, 1, 1)])
def test_a_window_past_the_first_key_hides_nothing(S, H, KH, D):
    """From one that just reaches it to the largest integer: the bits of the global mask."""
    from olmax_amd import ops
    q, do = rnd(2 * S, H * D, seed=1), rnd(2 * S, H * D, seed=4)
    k, v = rnd(2 * S, KH * D, seed=2), rnd(2 * S, KH * D, seed=3)
    kw = dict(B=2, S=S, H=H, KH=KH, D=D)

    def run(window):
        print(f"[case] attn S{S} H{H} KH{KH} D{D} w{window}", flush=True)
        o, lse = ops.attn_fwd(q, k, v, window=window, **kw)
        return (o, lse, *ops.attn_bwd(q, k, v, o, lse, do, window=window, **kw))

    want = run(None)
    for window in (S - 1, S, S + 1, 2 ** 31 - 65, 2 ** 31 - 1):
        assert all(torch.equal(a, b) for a, b in zip(run(window), want)), window


@pytest.mark.parametrize("B,S,H,KH,window,softcap", [(2, 200, 2, 1, None, 0.0), (1, 300, 4, 4, 70, 30.0), (4, 300, 48, 48, None, 0.0), (4, 270, 60, 60, 100, 30.0)])
@pytest.mark.parametrize("value", [math.nan, math.inf, -math.inf])
def test_head_dim_64_keeps_what_a_row_does_not_see_out_of_it(B, S, H, KH, window, softcap, value):
    """Infinities and NaN in one token of an operand reach the rows that see the token and no other: as on the kernels that
    work through visible pairs one by one (which take views that are not 16-byte aligned); few workgroups and enough for the
    unsplit forms.  Finite values: two roundings of P and dS to bf16, bounds as in check()."""
    from olmax_amd import ops
    n, at = B * S, S // 2 + 5
    x = {"q": rnd(n, H * 64, seed=1), "k": rnd(n, KH * 64, seed=2), "v": rnd(n, KH * 64, seed=3), "do": rnd(n, H * 64, seed=4)}
    kw = dict(B=B, S=S, H=H, KH=KH, D=64, window=window, softcap=softcap)
    odd = lambda t: torch.cat([t, t.new_zeros(n, 3)], 1)[:, :t.shape[1]]  # noqa: E731
    for name in x:
        print(f"[case] {value} in {name}, B{B} S{S} H{H} KH{KH} w{window} cap{softcap}", flush=True)
        y = {k: t.clone() for k, t in x.items()}
        y[name][at, 3] = value  # of the first sequence and head
        got, want = [], []
        for form, res in ((lambda t: t, got), (odd, want)):
            q, k, v, do = (form(y[i]) for i in ("q", "k", "v", "do"))
            res += ops.attn_fwd(q, k, v, **kw)
            res += ops.attn_bwd(q, k, v, form(got[0]), got[1], do, **kw)  # (gradients of both from the same forward)
        for a, b in zip(got, want):
            a, b = a.double(), b.double()
            ok = b.isfinite()
            assert torch.equal(ok, a.isfinite()) and torch.equal(a[~ok].nan_to_num(7.0, 8.0, 9.0), b[~ok].nan_to_num(7.0, 8.0, 9.0))
            assert (a[ok] - b[ok]).norm() <= 1e-2 * b[ok].norm()


@pytest.mark.parametrize("B,S,H,KH,window", [(1, 70, 2, 2, None), (2, 200, 4, 2, 0), (4, 300, 48, 48, None)])
def test_head_dim_64_row_whose_only_score_is_minus_infinity(B, S, H, KH, window):
    """Such a softmax is NaN in every column, as on the kernels that work through visible pairs one by one, however many
    waves share the row; few workgroups and enough for the unsplit form."""
    from olmax_amd import ops
    print(f"[case] score of -inf, B{B} S{S} H{H} KH{KH} w{window}", flush=True)
    n = B * S
    q, k, v = rnd(n, H * 64, seed=1), rnd(n, KH * 64, seed=2), rnd(n, KH * 64, seed=3)
    at = 0 if window is None else 37  # a token whose query sees this key only
    q[at, 3], k[at, 3] = 1.0, -math.inf
    kw = dict(B=B, S=S, H=H, KH=KH, D=64, window=window, softcap=0.0)
    odd = lambda t: torch.cat([t, t.new_zeros(n, 3)], 1)[:, :t.shape[1]]  # noqa: E731
    got, want = ops.attn_fwd(q, k, v, **kw), ops.attn_fwd(odd(q), odd(k), odd(v), **kw)
    assert want[0][at, :64].isnan().all() and want[1][0, 0, at].isnan()
    for a, b in zip(got, want):
        ok = b.isfinite()
        assert torch.equal(ok, a.isfinite())
        assert (a[ok].double() - b[ok].double()).norm() <= 1e-2 * b[ok].double().norm()


def test_head_dim_64_gradients_in_place():
    """q | k | v overwritten by their gradients, and dO by dQ; bound as in check()."""
    from olmax_amd import ops
    B, S, H, KH, D = 2, 200, 4, 4, 64
    print("[case] attn in place", flush=True)
    qkv, do = rnd(B * S, (H + 2 * KH) * D, seed=1), rnd(B * S, H * D, seed=2)
    cols = lambda t: (t[:, :H * D], t[:, H * D:(H + KH) * D], t[:, (H + KH) * D:])  # noqa: E731
    kw = dict(B=B, S=S, H=H, KH=KH, D=D)
    o, lse = ops.attn_fwd(*cols(qkv), **kw)
    want = ops.attn_bwd(*cols(qkv), o, lse, do, **kw)
    into_do, fresh = do.clone(), rnd(B * S, 2 * KH * D, seed=3)
    over = [t.clone() for t in (qkv, qkv)]
    ops.attn_bwd(*cols(over[0]), o, lse, do, dq=cols(over[0])[0], dk=cols(over[0])[1], dv=cols(over[0])[2], **kw)
    ops.attn_bwd(*cols(qkv), o, lse, into_do, dq=into_do, dk=fresh[:, :KH * D], dv=fresh[:, KH * D:], **kw)
    q = cols(over[1])[0]
    ops.attn_fwd(*cols(over[1]), out=q, **kw)
    for got in (cols(over[0]), (into_do, fresh[:, :KH * D], fresh[:, KH * D:])):
        assert all(rel(a, b) < 1e-2 for a, b in zip(got, want))
    assert rel(q, o) < 1e-2
