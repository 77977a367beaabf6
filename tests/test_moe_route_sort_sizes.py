"""Routing and sort in one call: how many workgroups share the tokens (the scratch holds their counts per expert)."""
from nanovllm_amd import _lib


def test_a_wave_has_one_token_beyond_64_experts():
    words = _lib.mixers().nv_moe_route_sort_words
    for E in (65, 128, 512):
        assert words(16, E) == 0                                  # one workgroup of 16 waves
        for T in (17, 32, 128, 512):
            assert words(T, E) == -(-T // 4) * E, (T, E)          # workgroups of four waves
        assert words(8192, E) == 256 * E and words(10 ** 6, E) <= 256 * E
    assert words(128, 64) == 0 and words(129, 64) == 9 * 64       # four tokens of a wave side by side
    assert words(10 ** 6, 513) == 0                               # (two launches of their own)
