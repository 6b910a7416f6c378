"""Which kernels the attention backward takes (no GPU needed), and that the GPU tests of each form reach it."""
import pytest

SPLIT_Q, SPLIT_KV, ONE = 1, 2, 4


def form(B, S, H, KH, D, window=None):
    from olmax_amd import _lib
    if not _lib.lib_path().exists():
        pytest.skip("libolmax_hip.so not built")
    return _lib.load().olmax_attn_bwd_form(B, S, H, KH, D, -1 if window is None else window)


# second rounds of workgroups with short chains: (B, S, heads, K/V heads, head_dim, window)
SHORT = [(4, 30, 48, 48, 128, None), (9, 30, 16, 16, 128, None), (11, 31, 24, 24, 128, None), (8, 55, 24, 24, 128, None), (11, 43, 24, 24, 128, None), (11, 68, 16, 16, 128, None),
         (8, 113, 32, 16, 128, None), (3, 312, 32, 16, 128, None), (2, 489, 32, 16, 128, 256), (9, 54, 40, 8, 128, None), (11, 59, 32, 8, 128, None), (10, 127, 32, 8, 128, None),
         (11, 32, 40, 8, 64, None), (2, 1590, 8, 4, 128, 64)]
LONG = [(1, 130, 32, 32, 128, None), (4, 30, 16, 16, 128, None), (8, 86, 16, 16, 128, None), (3, 437, 16, 16, 128, None), (9, 34, 32, 16, 128, None), (3, 226, 32, 16, 128, None),
        (8, 28, 40, 8, 128, None), (10, 156, 16, 4, 128, None), (5, 50, 48, 48, 64, None), (9, 151, 16, 4, 64, None), (3, 201, 16, 16, 128, 64)]


@pytest.mark.parametrize("call", SHORT)
def test_a_second_round_of_short_chains_is_not_taken(call):
    assert form(*call) != SPLIT_Q | SPLIT_KV | ONE


@pytest.mark.parametrize("call", LONG)
def test_few_workgroups_and_long_chains_share_a_launch(call):
    assert form(*call) == SPLIT_Q | SPLIT_KV | ONE


@pytest.mark.parametrize("call", [(8, 30, 32, 32, 128, None), (6, 768, 8, 8, 128, None), (4, 709, 16, 16, 64, None), (8, 1024, 8, 8, 128, None)])
def test_plain_forms_share_a_launch(call):
    assert form(*call) == ONE


def test_what_takes_other_kernels_or_is_refused_has_no_form():
    assert form(1, 128, 4, 4, 96) == form(1, 9000, 4, 4, 64) == form(1, 128, 3, 2, 128) == form(0, 128, 4, 4, 128) == -1
    assert form(1, 9000, 4, 4, 128) == SPLIT_Q | SPLIT_KV
    for window in (128, 2 ** 31 - 65, 2 ** 31 - 1):  # past the first key: global
        assert form(1, 128, 4, 4, 128, window) == form(1, 128, 4, 4, 128)
