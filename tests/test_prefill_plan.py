"""The plan of large prompt launches: query tiles of a workgroup, the cheapest of single tiles and shares."""
import pytest

from nanovllm_amd import _lib


def _tiles(heads, kv_heads, rows, cached=0):
    return _lib.lib().nv_attn_prefill_query_tiles(len(rows), sum(rows), max(rows), max(rows) + cached, heads, kv_heads)


# Measured with one, two and four tiles a workgroup, us
@pytest.mark.parametrize("heads,kv_heads,rows,cached,want", [
    (32, 8, [1066, 900, 800, 700] * 4, 1059, 2),       # 355, 347, 414: four tiles do not pay, two do
    (32, 8, [2794, 2617, 2383, 2340, 741, 423], 0, 2),  # 227, 224, 275
    (16, 8, [4096] + [256] * 16, 0, 1),                 # 101, 94, 173: one long prompt among short ones
    (16, 8, [4096] + [17] * 40, 0, 1),                  # 129, 109, 175
    (32, 8, [4096] + [17] * 40, 0, 2),                  # 218, 191, 177
    (8, 1, [4096] + [17] * 40, 0, 1),                   # 88, 92, 171: the longest workgroup alone
    (64, 8, [2730] * 3, 0, 1),                          # 359, 401, 406
    (32, 8, [3500, 2750, 1999], 0, 1),                  # 200, 218, 217
    (32, 8, [1365] * 6, 0, 1),                          # 114, 140, 145
    (32, 8, [2048] * 4, 0, 2),                          # 147, 141
    (32, 8, [8192], 0, 2),                              # 494, 467
    (64, 8, [1024] * 8, 0, 4),                          # 178, 167, 161
    (16, 8, [2048] * 4, 0, 1),                          # fewer than 512 workgroups of two
    (16, 8, [100] * 4, 0, 0),                           # the other kernel
])
def test_query_tiles_of_a_workgroup(heads, kv_heads, rows, cached, want):
    assert _tiles(heads, kv_heads, rows, cached) == want


@pytest.mark.parametrize("heads,kv_heads", [(8, 1), (16, 8), (32, 8), (64, 8), (32, 32), (48, 8)])
def test_plans_of_any_step(heads, kv_heads):
    """Whatever the step, also where the rows do not add up to what the longest sequence says."""
    for B in (1, 2, 3, 17, 512):
        for most in (1, 63, 64, 65, 1000, 4096, 131072):
            for total in (1, most, most + B, B * most):
                for keys in (most - 1, most, most + 64, most + 30000):
                    assert _lib.lib().nv_attn_prefill_query_tiles(B, total, most, keys, heads, kv_heads) in (0, 1, 2, 4)


def test_single_tiles_only_where_a_grid_can_hold_them():
    assert _lib.lib().nv_attn_prefill_query_tiles(1 << 20, 1 << 28, 8192, 8192, 64, 8) > 1       # (2^31 workgroups of one tile)
