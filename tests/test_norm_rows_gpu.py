"""GPU parity tests of the RMSNorm backward of narrow rows, at the edges of its choice of workgroups."""
import pytest
import torch

from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [8, 128, 136, 256])
@pytest.mark.parametrize("rows", [1, 512, 513, 4097, 32767, 32768, 40001])
def test_narrow_rows(rows, d):
    """Against float64.  dx: an fp32 row sum of d terms and a rounding to bf16, 2^-9 of the value and of the largest of its two parts.  dw: fp32 sums of
    `rows` terms of unit size, each 2^-22 off, added in any order (2^-24 of a partial sum of sqrt(rows) each, sqrt(rows) of these by chance)."""
    from olmax_amd import ops
    print(f"[case] norm rows{rows} d{d}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows + d)
    x, dy, dres = (torch.randn(rows, d, device="cuda", generator=g).to(torch.bfloat16) for _ in range(3))
    w = (1 + 0.1 * torch.randn(d, device="cuda", generator=g)).to(torch.bfloat16)
    want, wdw = ref.rms_norm_bwd(x.double(), w.double(), dy.double(), 1e-6)
    dx, dw = ops.rms_norm_bwd(x, w, dy, 1e-6)
    assert ((dx.double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -20 * 8).all()
    assert ((dw.double() - wdw).abs() <= 2 ** -22 * 6 * rows ** 0.5 + 2 ** -24 * 6 * rows).all()
    acc = torch.full((d,), 0.5, device="cuda")
    got, _ = ops.rms_norm_bwd(x, w, dy, 1e-6, dres=dres, dw=acc)
    full = want + dres.double()
    assert ((got.double() - full).abs() <= 2 ** -8 * (want.abs() + full.abs()) + 2 ** -20 * 8).all()
    assert ((acc.double() - 0.5 - wdw).abs() <= 2 ** -22 * 6 * rows ** 0.5 + 2 ** -24 * 6 * rows).all()
