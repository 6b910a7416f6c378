"""dQ and dK/dV in launches of their own, where one hands delta to the other: the split kernels at ragged ends, against the float64 oracle."""
import pytest

from test_attention_choice import ONE, SPLIT_KV, SPLIT_Q, form
from test_attention_forms_gpu import check

pytestmark = pytest.mark.gpu


# several query heads to a K/V head: more query rows than one launch forms delta of
@pytest.mark.parametrize("softcap", [0.0, 30.0])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H,KH,window,want", [
    (1, 449, 8, 2, None, SPLIT_Q | SPLIT_KV), (2, 450, 8, 2, 300, SPLIT_Q | SPLIT_KV), (1, 641, 4, 1, 500, SPLIT_Q | SPLIT_KV), (1, 1000, 16, 4, None, SPLIT_Q | SPLIT_KV),
    (1, 769, 5, 1, None, SPLIT_Q | SPLIT_KV)])
def test_both_split(B, S, H, KH, window, want, D, softcap):
    assert form(B, S, H, KH, D, window) == want
    check(B, S, H, KH, D, window, softcap, strided=S % 2 == 1, groups=[0, KH - 1])


@pytest.mark.parametrize("softcap", [0.0, 30.0])
@pytest.mark.parametrize("B,S,H,KH,D,window", [(1, 300, 4, 1, 128, None), (2, 257, 8, 1, 128, None), (1, 385, 80, 16, 128, 200), (1, 600, 48, 12, 64, None), (1, 577, 48, 8, 64, 500)])
def test_keys_split(B, S, H, KH, D, window, softcap):
    assert form(B, S, H, KH, D, window) == SPLIT_KV
    check(B, S, H, KH, D, window, softcap, strided=S % 2 == 1, groups=[0, KH - 1])


@pytest.mark.parametrize("softcap", [0.0, 30.0])
def test_queries_split(softcap):
    assert form(1, 1650, 39, 39, 128) == SPLIT_Q
    check(1, 1650, 39, 39, 128, None, softcap, groups=[0, 38])


# second rounds of short chains
@pytest.mark.parametrize("B,S,H,KH,D,softcap", [(10, 31, 16, 16, 128, 0.0), (3, 55, 48, 48, 128, 50.0), (8, 113, 32, 16, 128, 0.0), (11, 32, 40, 8, 64, 0.0)])
def test_short_chains(B, S, H, KH, D, softcap):
    assert not form(B, S, H, KH, D) & ONE
    check(B, S, H, KH, D, None, softcap, strided=S % 2 == 1, groups=[0, KH - 1])
