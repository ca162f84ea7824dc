"""How many workgroups share the keys of latent attention's blocks (a rule on sizes alone; no GPU)."""
from types import SimpleNamespace

import pytest

from llmserve.parts.attention_latent import LatentAttention


def shares(heads, n, max_new, reach, tokens=None, window=None):
    return LatentAttention.key_shares(SimpleNamespace(heads=heads, window=window), n, max_new, reach, 256, tokens)


@pytest.mark.parametrize("heads,n,max_new,reach", [(16, 1, 1, 64), (16, 8, 1, 4000), (16, 4, 448, 900), (128, 3, 7, 300), (1, 300, 1, 500)])
def test_requests_of_one_length_share_as_without_the_number_of_tokens(heads, n, max_new, reach):
    same, counted = shares(heads, n, max_new, reach), shares(heads, n, max_new, reach, n * max_new)
    assert same <= counted <= 2 * same  # (a request's last block may be partly empty)


def test_single_tokens_beside_a_portion_do_not_count_as_portions():
    assert shares(16, 6, 448, 900) == 1
    assert shares(16, 6, 448, 900, 453) == 4


def test_blocks_times_shares_never_pass_the_compute_units():
    for n, tokens in ((1, 1), (2, 300), (7, 1000), (40, 4000)):
        for heads in (1, 16, 128):
            got = shares(heads, n, tokens, 4000, tokens)
            assert 1 <= got <= 16
            assert got == 1 or got * tokens * heads <= 256 * 128


@pytest.mark.parametrize("heads,n,max_new,reach,tokens,expected", [
    (16, 21, 200, 1500, 220, 5), (16, 13, 500, 3000, 512, 3), (32, 21, 200, 1500, 220, 3),  # measured: shared keys are the faster way
    (32, 6, 448, 900, 453, 1), (32, 2, 400, 400, 500, 1), (32, 31, 30, 100, 60, 1),         # adding the shares up costs more
    (128, 4, 100, 300, 103, 1), (128, 5, 40, 200, 44, 1),
    (16, 61, 60, 800, 120, 1),                                                              # mostly single tokens
])
def test_shares_that_cost_more_than_they_spare_are_not_made(heads, n, max_new, reach, tokens, expected):
    assert shares(heads, n, max_new, reach, tokens) == expected


def test_where_the_longest_portion_leaves_compute_units_idle_nothing_changes():
    for heads, n, max_new, reach, tokens in ((32, 8, 16, 4000, 23), (128, 8, 16, 4000, 23), (16, 4, 100, 300, 103), (8, 4, 500, 1000, 802)):
        same = shares(heads, n, max_new, reach)
        assert same > 1 and shares(heads, n, max_new, reach, tokens) == same
