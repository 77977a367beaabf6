"""Rules and index arithmetic of launches, over many launch shapes with a host compiler."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include "launch_order.h"
using namespace nv;
extern "C" int latent(int64_t total, int slots, int last_key, int tile_keys, int nsplit, int fewest, int* share, int* tiles) {
    *share = latent_share(total, slots, fewest);
    *tiles = latent_tiles(last_key, tile_keys, nsplit, fewest);
    return latent_ranges(*tiles, *share);
}
extern "C" int streams(int tile_rows, int64_t pairs, int E, int ff) { return moe_streams(tile_rows, pairs, E, ff); }
extern "C" int few_blocks(int64_t pairs, int E, int n_cols) { return moe_few_blocks(pairs, E, n_cols); }
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch_order")
    src, lib = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "nano-vllm_amd", "csrc"),
                    str(src), "-o", str(lib)], check=True)
    dll = C.CDLL(str(lib))
    dll.latent.argtypes = [C.c_int64] + [C.c_int] * 5 + [C.POINTER(C.c_int)] * 2
    dll.few_blocks.argtypes = [C.c_int64, C.c_int, C.c_int]
    dll.streams.argtypes = [C.c_int, C.c_int64, C.c_int, C.c_int]
    return dll


def test_latent_ranges_stay_within_what_was_stated(order):
    """Whatever a sequence's true length: no state beyond the workspace (none at all where there is one range), no key beyond the stated
    length's ranges, and every key tile within them in one range."""
    share, tiles = C.c_int(), C.c_int()
    for nsplit, fewest in ((1, 1), (1, 7), (1, 40), (2, 8), (3, 9), (7, 8), (32, 8), (32, 30)):
        for last_key in list(range(0, 64 * (nsplit * fewest + 3), 61)) + [10 ** 5, 10 ** 7]:
            for total in (0, 1, 100, 5000, 10 ** 6, 10 ** 12):
                n = order.latent(total, 256, last_key, 64, nsplit, fewest, C.byref(share), C.byref(tiles))
                assert share.value >= fewest and 1 <= n <= nsplit
                assert tiles.value == min(last_key // 64 + 1, nsplit * fewest)
                assert (n - 1) * share.value < tiles.value <= n * share.value


def test_experts_one_workgroup_a_cu(order):
    """Tiles of 128 rows: (pairs an expert, experts, column blocks) on either side of what was measured."""
    for per, E, cols, few in ((40, 16, 8, 1), (96, 16, 8, 1), (96, 32, 8, 1), (100, 32, 8, 1), (112, 32, 8, 0), (192, 16, 8, 1), (256, 16, 8, 0),
                              (256, 16, 4, 1), (512, 16, 4, 0), (40, 64, 8, 0), (1024, 32, 8, 0), (1024, 1, 16, 1)):
        assert order.few_blocks(per * E, E, cols) == few, (per, E, cols)


def test_experts_weights_past_lds(order):
    """The tiles of nv_moe_tile_rows (16 rows, 64 from 32 pairs an expert on) do not read an expert's weights once for each of many tiles."""
    from nanovllm_amd import _lib
    rows = _lib.mixers().nv_moe_tile_rows
    for E, ff, past in ((32, 1024, (1, 8, 12, 32, 36)), (16, 1024, (1, 8, 12, 32, 48, 56)), (32, 512, (8, 32, 56)), (16, 512, (8, 32, 96))):
        for per in past:
            assert order.streams(rows(per * E, E), per * E, E, ff), (E, ff, per)
        for per in (20, 24, 31, 160, 256, 1024, 10 ** 5):
            assert not order.streams(rows(per * E, E), per * E, E, ff), (E, ff, per)
    assert not any(order.streams(64, 64 * E, E, ff) for E, ff in ((32, 1024), (16, 1024), (32, 512)))


def test_experts_tile_rows():
    """Where tiles of 128 rows start, on either side of the lines: blocks of 128 x 128 of the first product, pairs an expert."""
    from nanovllm_amd import _lib
    rows_for = lambda E, W, ff, per: _lib.mixers().nv_moe_tile_rows_for(per * E, E, W, ff, 4096, W, 4096, 4096, 0)
    for E, W, ff, line in ((32, 2048, 1024, 40), (64, 2048, 512, 40), (16, 2048, 1024, 52), (32, 1024, 512, 52), (16, 1024, 512, 84)):
        assert [rows_for(E, W, ff, per) for per in (7, 8, 23, 24, line - 1, line)] == [16, 32, 32, 64, 64, 128], (E, W, ff)
