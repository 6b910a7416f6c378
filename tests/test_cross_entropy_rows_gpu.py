"""GPU parity tests of the cross entropy at the row lengths where its kernels change, at the ends of their vectors."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [8, 4096, 4104, 16384, 16392, 51200, 51208, 102400, 102408, 163840, 163848, 163840 + 8 * 4096 + 8])
@pytest.mark.parametrize("cap", [0.0, 20.0])
def test_row_lengths(V, cap):
    """Gradients are rounded to bf16 once: 2^-9 of the value, and fp32 exponentials of |z - lse| < 40 in front of it: 40 * 2^-23.
    Rows with whole vectors of minus infinity (a masked vocabulary) and with the label at either end are among them."""
    from olmax_amd import ops
    print(f"[case] ce rows V{V} cap{cap}", flush=True)
    g = torch.Generator().manual_seed(V)
    z = (torch.randn(6, V, generator=g) * 3).to(torch.bfloat16)
    if V > 64:
        z[3, : V // 2 // 8 * 8] = float("-inf")
        z[4, V // 2 // 8 * 8:] = float("-inf")
    labels = torch.tensor([0, V - 1, V // 2, V - 1, 0, -100], dtype=torch.int32)
    want = ref.cross_entropy_bwd(z.double(), labels.long(), softcap=cap)
    loss, lse = ref.cross_entropy_fwd(z.double(), labels.long(), softcap=cap)[:2]
    for inplace in (False, True):
        got = ops.cross_entropy(z.cuda(), labels.cuda(), softcap=cap, inplace=inplace)
        assert abs(got[0].item() - loss.item()) < 1e-5 * abs(loss.item())
        assert ((got[2].cpu().double() - lse)[:5].abs() < 1e-6 * lse[:5].abs() + 1e-6).all()
        # near the label and under the soft-cap 1 - p and 1 - t^2 cancel: 2^-22 of the row's scale 1/5
        err = (got[1].cpu().double() - want).abs() - (2 ** -8 * want.abs() + 2 ** -22 / 5)
        assert err.max().item() <= 0, (err.argmax().item() // V, err.argmax().item() % V)


@pytest.mark.parametrize("V", [4091, 16379, 51199, 102397, 163835, 163843])
@pytest.mark.parametrize("cap", [0.0, 20.0])
def test_padded_rows(V, cap):
    """The LM head's own logits, rows padded to whole vectors.  A row of one token's dW is its dlogits times h: relative error of two
    bf16 roundings, 2^-8, on top of the logits' own, 2^-9 of |z| < 8 in the exponent."""
    from olmax_amd import ops
    print(f"[case] ce padded V{V} cap{cap}", flush=True)
    g = torch.Generator().manual_seed(V)
    h = torch.randn(2, 64, generator=g).to(torch.bfloat16)
    W = (torch.randn(V, 64, generator=g) * 0.1).to(torch.bfloat16)
    labels = torch.tensor([V - 1, V - 2], dtype=torch.int32)
    loss, dh, dW = ops.lmhead_ce(h.cuda(), W.cuda(), labels.cuda(), softcap=cap, dw_f32=True)
    z = (h.double() @ W.double().t()).to(torch.bfloat16).double()
    assert abs(loss.item() - ref.cross_entropy_fwd(z, labels.long(), softcap=cap)[0].item()) < 1e-4
    d = ref.cross_entropy_bwd(z, labels.long(), softcap=cap)
    for got, want in ((dW, d.t() @ h.double()), (dh, d @ W.double())):
        assert ((got.cpu().double() - want).norm() / want.norm()).item() < 2 ** -8
    assert ((dW.cpu().double() - d.t() @ h.double())[-8:].norm() / (d.t() @ h.double())[-8:].norm()).item() < 2 ** -7


@pytest.mark.parametrize("V", [4096, 51200, 163840, 163848 + 8 * 4096])
def test_rows_far_from_zero(V):
    """Logits whose sum of exponentials lies where half an ulp of lse * log2(e) is not small: rows about 1000 and 1e6, a row of the
    type's lowest value (its lse rounds to the logit: exp(0) each), and one logit above such a mask.  The bound is lse's own
    rounding, 2^-24 of it, and a bf16 store."""
    from olmax_amd import ops
    print(f"[case] ce far V{V}", flush=True)
    low = torch.finfo(torch.bfloat16).min
    z = torch.full((4, V), low)
    z[0] = torch.randint(0, 4, (V,), generator=torch.Generator().manual_seed(V)) * 4.0 + 1000
    z[1] = -1e6
    z[3, 9] = 2.0
    z = z.to(torch.bfloat16)
    labels = torch.tensor([1, 2, 3, 9], dtype=torch.int32)
    loss, dz, lse = ops.cross_entropy(z.cuda(), labels.cuda())
    zd = z.double()
    p = (zd - lse.cpu().double()[:, None]).exp()  # against the lse that the row has in fp32
    assert torch.isfinite(dz).all()
    # sums of up to 2^18 terms, each off by a few 2^-24 for exponents up to 12; then the logarithm is added to the maximum in fp32
    got = lse.cpu().double()
    assert ((got - zd.logsumexp(1)).abs() <= 2 ** -23 * got.abs() + 2 ** -19).all()
    want = (got - zd[torch.arange(4), labels.long()]).mean()
    assert (loss.double().cpu() - want).abs() <= 2 ** -22 * want
    want = p / 4
    want[torch.arange(4), labels.long()] -= 0.25
    err = (dz.cpu().double() - want).abs() - (2 ** -8 * want.abs() + 2 ** -22 / 4)
    assert err.max().item() <= 0, (err.argmax().item() // V, err.argmax().item() % V)


@pytest.mark.parametrize("V", [16392, 51200, 51208, 102400, 51199, 102397])
@pytest.mark.parametrize("cap", [0.0, 20.0])
@pytest.mark.parametrize("T", [256, 257])
def test_number_of_rows(V, cap, T):
    """Up to 256 rows take more threads each.  Bounds as above, the padded ones in the norm of dW and dh."""
    from olmax_amd import ops
    print(f"[case] ce T{T} V{V} cap{cap}", flush=True)
    g = torch.Generator().manual_seed(V)
    labels = torch.arange(T, dtype=torch.int32) * 977 % V
    labels[-1] = V - 1
    if V % 8 == 0:
        few = (torch.randn(4, V, generator=g) * 3).to(torch.bfloat16).cuda()
        z = few.repeat((T + 3) // 4, 1)[:T]
        loss, d, lse = ops.cross_entropy(z, labels.cuda(), softcap=cap)
        rows = [0, 1, 255, T - 1]
        zr = z[rows].cpu()
        want = ref.cross_entropy_bwd(zr.double(), labels[rows].long(), softcap=cap) * (4 / T)
        err = (d[rows].cpu().double() - want).abs() - (2 ** -8 * want.abs() + 2 ** -22 / T)
        assert err.max().item() <= 0
        assert (lse.view(-1)[4:] == lse[:-4]).all()
        return
    h = torch.randn(T, 64, generator=g).to(torch.bfloat16).cuda()
    W = (torch.randn(V, 64, generator=g) * 0.1).to(torch.bfloat16).cuda()
    loss, dh, dW = ops.lmhead_ce(h, W, labels.cuda(), softcap=cap, dw_f32=True)
    z = (h.double() @ W.double().t()).to(torch.bfloat16).double().cpu()
    d = ref.cross_entropy_bwd(z, labels.long(), softcap=cap).cuda()
    for got, want in ((dW, d.t() @ h.double()), (dh, d @ W.double())):
        assert ((got.double() - want).norm() / want.norm()).item() < 2 ** -7


@pytest.mark.parametrize("V", [4096, 16392])
@pytest.mark.parametrize("at", [20, 50, 250])
def test_gradients_round_as_the_exact_ones(V, at):
    """Rows about `at`: gradients that round to another bf16 than the exact ones (against the lse that the row has).  A relative error e of the
    probability flips 185 |e| of them, the mean of p / ulp(p) over a binade: 4e-7, a few fp32 operations of 2^-24 each, 7e-5.  The
    rounding of lse * log2(e), not taken back, would add half an ulp of it, 1e-6 at 20 and 1e-5 at 250."""
    from olmax_amd import ops
    print(f"[case] ce rounding V{V} at{at}", flush=True)
    T = 8192  # a power of two: 1 / T is exact
    g = torch.Generator(device="cuda").manual_seed(V)
    z = (torch.randn(T, V, device="cuda", generator=g) * 4 + at - 12 + torch.rand(T, 1, device="cuda", generator=g) * 4).to(torch.bfloat16)
    labels = torch.full((T,), V - 1, dtype=torch.int32, device="cuda")
    d, lse = ops.cross_entropy(z, labels)[1:]
    wrong = total = 0
    for i in range(0, T, 1024):
        p = (z[i:i + 1024, :-8].double() - lse.view(-1)[i:i + 1024, None].double()).exp() / T
        big = p > 2 ** -100  # (no underflow)
        # to bf16 by fp32 would round twice: half a unit added to the bits of the double, ties have no weight here
        want = ((p.view(torch.int64) + (1 << 44)) >> 45 << 45).view(torch.float64)
        wrong += int(((d[i:i + 1024, :-8].double() != want) & big).sum())
        total += int(big.sum())
    assert wrong / total < 1.25e-4, wrong / total


@pytest.mark.parametrize("T", [512, 513])
@pytest.mark.parametrize("V,cap", [(16392, 0.0), (51200, 20.0), (51199, 0.0)])
def test_number_of_rows_of_two_workgroups_to_a_cu(V, cap, T):
    test_number_of_rows(V, cap, T)
