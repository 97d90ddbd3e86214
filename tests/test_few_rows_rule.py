"""When the expert GEMMs for few rows are taken in the place of the tiles (host code: no GPU)."""

import pytest

from minitrain_amd import _lib

BF16, F32 = _lib.MTS_BF16, _lib.MTS_F32


def _in_front(T, K, E, H, I):
    return _lib.load().mts_moe_fwd_few_rows_preferred(BF16, F32, T, T * K, E, H, I)


def _beside(T, K, E, H, I):
    return _lib.load().mts_moe_fwd_few_rows_preferred_to_ride(BF16, T, T * K, E, H, I)


def _rounded(T, K, E, H, I):
    return _lib.load().mts_moe_fwd_few_rows_preferred(BF16, BF16, T, T * K, E, H, I)


@pytest.mark.parametrize("T,K,E,H,I", [(300, 4, 128, 768, 256), (1024, 4, 128, 768, 256), (512, 4, 64, 1024, 512), (96, 2, 8, 768, 1024), (120, 4, 32, 768, 256),
                                       (96, 2, 4, 1024, 2048)])
def test_masters_are_read_where_copies_of_them_are_a_launch_in_front(T, K, E, H, I):
    assert _in_front(T, K, E, H, I)


# us, reading them / with copies: 768/1024, 8 experts, one route a token: 65 tokens 43.9 / 44.7, 80 47.5 / 44.4, 109 48.0 / 44.5, 128 48.2 / 45.0
@pytest.mark.parametrize("T,K,E,H,I,reads", [(80, 1, 8, 768, 1024, False), (109, 1, 8, 768, 1024, False), (128, 1, 8, 768, 1024, False), (128, 2, 8, 768, 1024, False), (120, 4, 32, 768, 256, False), (256, 2, 8, 768, 1024, False), (512, 4, 64, 1024, 512, True),
                                             (65, 1, 8, 768, 1024, True), (128, 1, 64, 1024, 768, True)])
def test_copies_beside_the_head_cost_less(T, K, E, H, I, reads):
    assert bool(_beside(T, K, E, H, I)) == reads


@pytest.mark.parametrize("rule", [_in_front, _beside, _rounded])
@pytest.mark.parametrize("E,H,I", [(8, 768, 1024), (8, 1024, 512), (8, 512, 2048), (16, 768, 1024), (32, 2048, 768), (64, 1024, 512), (128, 768, 256), (3, 712, 680)])
def test_more_rows_never_lead_back(rule, E, H, I):
    taken = [bool(rule(T, 1, E, H, I)) for T in range(1, 80 * E, 7)]
    assert taken == sorted(taken, reverse=True)


@pytest.mark.parametrize("rule", [_in_front, _beside, _rounded])
@pytest.mark.parametrize("E,H", [(8, 768), (8, 2048), (16, 768), (64, 1024)])
def test_the_border_moves_little_from_a_width_to_the_next(rule, E, H):
    """rows an expert up to which it is taken, for widths 16 apart: no steps at single sizes"""
    def border(I):
        return max((T / E for T in range(1, 66 * E, E // 8) if rule(T, 1, E, H, I)), default=0.0)

    borders = [border(I) for I in range(256, 2049, 16)]
    assert all(abs(a - b) <= 6 for a, b in zip(borders, borders[1:])), borders


# us, here / on the tiles, 16 bits: 91 tokens, top-2, 16 experts of 1024/768 54 / 45; 38, top-2, 16 of 2048/1024 57 / 49; 144, top-2, 32 of 1024/1024 64 / 52; 66,
# top-2, 64 of 768/1000 73 / 84; 61, top-2, 4 of 768/1024, uneven 24 / 28; 46, top-2, 4 of 1024/1024 35 / 37
@pytest.mark.parametrize("T,K,E,H,I,taken", [(91, 2, 16, 1024, 768, False), (38, 2, 16, 2048, 1024, False), (144, 2, 32, 1024, 1024, False),
                                             (66, 2, 64, 768, 1000, True), (61, 2, 4, 768, 1024, True), (46, 2, 4, 1024, 1024, True)])
def test_rounded_weights_on_either_side(T, K, E, H, I, taken):
    assert bool(_rounded(T, K, E, H, I)) == taken


@pytest.mark.parametrize("E,H,I", [(8, 768, 1024), (64, 1024, 512), (32, 2048, 768)])
def test_reading_them_beside_the_head_is_never_all_there_is(E, H, I):
    """what is taken in spite of copies beside the head is taken in front of a launch of them: the caller that makes no copies asks a second time"""
    assert all(_in_front(T, 2, E, H, I) for T in range(1, 40 * E, 3) if _beside(T, 2, E, H, I))


# us, two launches / tiles, 16 bits: 29 tokens, top-4, 8 experts of 2048/1536 67 / 71; 15, top-1, 16 of 2048/1024 59 / 62; 1, top-2, 16 of 768/2048 36 / 40
@pytest.mark.parametrize("T,K,E,H,I,weights,taken", [(29, 4, 8, 2048, 1536, BF16, True), (15, 1, 16, 2048, 1024, BF16, True), (1, 2, 16, 768, 2048, BF16, True),
                                                     (32, 2, 8, 1024, 2048, F32, True), (32, 2, 8, 1024, 2056, F32, False), (32, 2, 12, 2048, 2048, BF16, False),
                                                     (33, 2, 8, 768, 1024, BF16, False), (4, 2, 9, 768, 1024, F32, False)])
def test_few_tokens_take_two_launches_up_to_a_size_of_the_weights(T, K, E, H, I, weights, taken):
    assert bool(_lib.load().mts_moe_few_tokens_preferred(BF16, weights, T, K, E, H, I)) == taken
