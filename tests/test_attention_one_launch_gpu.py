"""dQ and dK/dV in one launch: calls of few workgroups, at the edges of their tiles, in every form, against the float64 oracle."""
import pytest
import torch

from test_attention_choice import ONE, SPLIT_KV, SPLIT_Q, form
from test_attention_forms_gpu import check, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,H,KH,D,window,softcap", [
    (1, 1, 2, 2, 64, None, 0.0), (2, 65, 4, 4, 64, None, 0.0), (1, 321, 4, 2, 64, 100, 30.0), (2, 160, 8, 2, 64, None, 0.0),    # eight waves
    (1, 33, 4, 4, 128, None, 0.0), (1, 129, 4, 2, 128, None, 50.0), (1, 300, 4, 1, 128, None, 0.0), (2, 257, 4, 4, 128, 60, 0.0),
    (1, 2048, 2, 2, 128, None, 0.0), (1, 1024, 4, 2, 128, None, 0.0),  # as many query rows as find room
    (1, 256, 4, 1, 128, None, 0.0), (1, 288, 4, 1, 128, None, 50.0), (2, 97, 16, 2, 128, 40, 0.0), (1, 127, 24, 3, 64, None, 30.0),  # delta of four and eight heads of a group
])
def test_few_workgroups(B, S, H, KH, D, window, softcap):
    # (1 x 300 of 4/1 heads meets 1408 query rows: two launches)
    assert form(B, S, H, KH, D, window) == (SPLIT_KV if (S, KH) == (300, 1) else SPLIT_Q | SPLIT_KV | ONE)
    check(B, S, H, KH, D, window, softcap, strided=True)


@pytest.mark.parametrize("B,S,H,D,softcap", [(16, 130, 8, 128, 0.0), (13, 257, 8, 128, 50.0), (16, 97, 16, 64, 0.0), (11, 385, 8, 64, 0.0)])
def test_as_many_as_the_gpu_holds_at_once(B, S, H, D, softcap):
    """256 to 448 workgroups of 128 queries: four waves each."""
    assert form(B, S, H, H, D) == ONE
    check(B, S, H, H, D, None, softcap, groups=[0, H - 1])


@pytest.mark.parametrize("S", [130, 512])
def test_gradients_in_the_place_of_keys_and_values(S):
    """dK over K and dV over V, which dQ reads: two launches, as ever, and the same numbers but for what the split forms round."""
    from olmax_amd import ops
    B, H, D = 1, 4, 128
    print(f"[case] in place S{S}", flush=True)
    q, k, v, do = (rnd(B * S, H * D, seed=i) for i in range(4))
    kw = dict(B=B, S=S, H=H, KH=H, D=D)
    o, lse = ops.attn_fwd(q, k, v, **kw)
    want = ops.attn_bwd(q, k, v, o, lse, do, **kw)
    got = ops.attn_bwd(q, k, v, o, lse, do, dk=k, dv=v, **kw)
    for a, b in zip(got, want):  # sums of products in another order, rounded to bf16 (2^-9) once
        assert ((a.double() - b.double()).norm() / b.double().norm()).item() < 2 ** -9
