"""GPU tests of the rotary embedding's vector kernels (head_dim 64 and 128): strided views, rows that do not fill a workgroup
or give it several, and the one-wave-per-row kernels on unaligned views of the same values."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def rnd(*shape, seed=0):
    return torch.randn(*shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed)).to(BF)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,heads", [(1, 1, 1), (2, 33, 3), (1, 2100, 5), (1, 7000, 5)])
@pytest.mark.parametrize("norm", [False, True])
def test_vector_kernels_equal_the_generic_path(D, B, S, heads, norm):
    """Values differ by the order of a D-term fp32 sum before one bf16 rounding (2^-8 of a value), the weight gradient by
    that of B S heads fp32 terms."""
    from olmax_amd import ops
    print(f"[case] rope D{D} B{B} S{S} heads{heads} norm{norm}", flush=True)
    n, T = heads * D, B * S
    x, dy = rnd(T, n, seed=1), rnd(T, n, seed=2)
    w = (1 + 0.1 * rnd(D, seed=3)) if norm else None
    cos, sin = ops.rope_tables(S, D, 10000.0, "cuda")
    view = lambda t, pad: torch.cat([t, t.new_zeros(T, pad)], 1)[:, :n]  # noqa: E731  (pad 8: vector kernel, 3: generic)
    kw = dict(heads=heads, head_dim=D, seq_len=S)
    res = []
    for pad in (8, 3):
        y = ops.qk_rope_fwd(view(x, pad), cos, sin, w=w, **kw)
        dx, dw = ops.qk_rope_bwd(view(dy, pad), cos, sin, w=w, x=view(x, pad) if norm else None, **kw)
        res.append((y, dx, dw))
    (y, dx, dw), (gy, gdx, gdw) = res
    for a, b in ((y, gy), (dx, gdx)):
        assert (a.float() - b.float()).abs().max() <= 2 ** -7 * b.float().abs().max()
        assert (a.float() - b.float()).norm() <= 2 ** -9 * b.float().norm()
    if norm:
        assert (dw - gdw).norm() <= 1e-4 * gdw.norm()
