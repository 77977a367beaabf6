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
extern "C" int alike(int least_in_front, int longest) { return latent_alike(least_in_front, longest); }
extern "C" int turns(int num_seqs, int64_t total_q, int max_q, int max_k) { return latent_turns(num_seqs, total_q, max_q, max_k); }
// where every workgroup of a grid goes: pair and place, -1 for those that leave
extern "C" void scored(int rounds, int slots, int xs_shift, int together, int there_and_back, int pairs, int places, int* pair, int* place) {
    for (int i = 0; i < 8 * rounds * slots; ++i) {
        const PairPlace at = scoremod_order(scoremod_group(i, scoremod_sets(rounds), slots, xs_shift), i, slots, xs_shift, together, there_and_back);
        const bool there = at.pair < pairs && at.place < places;
        pair[i] = there ? at.pair : -1;
        place[i] = there ? at.place : -1;
    }
}
extern "C" int pairs_together(int64_t workgroups, int64_t total_q, int num_seqs, int max_q, int max_k) {
    return prefill_together(workgroups, total_q, num_seqs, max_q, max_k);
}
extern "C" void sets(int rounds, int together, int* least, int* more) {
    const PairSets s = prefill_sets(rounds, together);
    *least = s.least;
    *more = s.more;
}
extern "C" void prompt(int rounds, int slots, int together, int* round, int* place) {
    for (int i = 0; i < rounds * slots; ++i) {
        const RoundPlace at = prefill_order(i, slots, prefill_sets(rounds, together));
        round[i] = at.round;
        place[i] = at.place;
    }
}
extern "C" int even(int64_t keys, int64_t longest, int n, int whole_prompts) { return scoremod_even(keys, longest, n, whole_prompts); }
extern "C" int scored_pairs(int64_t grid_base, int num_seqs, int64_t total_q, int max_q, int max_k) {
    return scoremod_pairs(grid_base, num_seqs, total_q, max_q, max_k);
}
extern "C" int streams(int tile_rows, int64_t pairs, int E, int ff) { return moe_streams(tile_rows, pairs, E, ff); }
extern "C" int outputs_past(int64_t pairs, int width, int E, int ff) { return moe_streams_out(pairs, width, E, ff); }
extern "C" int states_past(int num_seqs, int lead, int rest, int H, int D, int Dv) {
    return recurrence_streams(recurrence_singles(num_seqs, lead, rest != 0), H, D, Dv);
}
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
    dll.even.argtypes = [C.c_int64, C.c_int64, C.c_int, C.c_int]
    dll.scored_pairs.argtypes = [C.c_int64, C.c_int, C.c_int64, C.c_int, C.c_int]
    dll.turns.argtypes = [C.c_int, C.c_int64, C.c_int, C.c_int]
    dll.pairs_together.argtypes = [C.c_int64, C.c_int64] + [C.c_int] * 3
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


def test_experts_tile_rows(order):
    """Where tiles of 128 rows start, on either side of the lines: blocks of 128 x 128 of the first product, pairs an expert."""
    from nanovllm_amd import _lib
    rows_for = lambda E, W, ff, per: _lib.mixers().nv_moe_tile_rows_for(per * E, E, W, ff, 4096, W, 4096, 4096, 0)
    for E, W, ff, line in ((32, 2048, 1024, 40), (64, 2048, 512, 40), (16, 2048, 1024, 52), (32, 1024, 512, 48), (32, 2048, 512, 48), (16, 1024, 512, 84)):
        assert [rows_for(E, W, ff, per) for per in (7, 8, 20, 21, line - 1, line)] == [16, 32, 32, 64, 64, 128], (E, W, ff)
    assert [rows_for(32, 1024, 1024, per) for per in (7, 8, 20, 21, 31, 32, 39, 40)] == [16, 32, 32, 16, 16, 64, 64, 128]
    assert not order.streams(16, 21 * 32, 32, 1024)                   # (those go through LDS)


@pytest.mark.parametrize("there_and_back", [0, 1])
@pytest.mark.parametrize("together", [0, 1])
def test_scored_every_place_once(order, together, there_and_back):
    """Every query tile of every pair of sequence and kv head is one workgroup's, whatever the order; and all pairs of an XCD's group stay there."""
    for pairs in (1, 2, 3, 4, 7, 8, 9, 24, 33, 64, 72):
        for xs_shift in ([0] if pairs > 4 else [0, 1, 2, 3]):
            rounds = -(-pairs // (8 >> xs_shift))
            for places in (1, 2, 5, 8, 20, 31, 32, 33, 64, 97):
                slots = -(-places // (1 << xs_shift))
                n = 8 * rounds * slots
                pair, place = (C.c_int * n)(), (C.c_int * n)()
                order.scored(rounds, slots, xs_shift, together, there_and_back, pairs, places, pair, place)
                got = [(p, w) for p, w in zip(pair, place) if p >= 0]
                assert sorted(got) == [(p, w) for p in range(pairs) for w in range(places)], (pairs, xs_shift, places)
                # a pair's workgroups are on its 1 << xs_shift XCDs (index % 8)
                assert all(i % 8 >> xs_shift == p % (8 >> xs_shift) for i, p in enumerate(pair) if p >= 0)
                if there_and_back and together and rounds == 4 and places == 20 and not xs_shift:
                    plain, at = (C.c_int * n)(), (C.c_int * n)()
                    order.scored(rounds, slots, xs_shift, 1, 0, pairs, places, plain, at)
                    assert list(plain) != list(pair)          # (places 32 .. 63 of the group go back)


def test_scored_pairs_of_about_the_same_length(order):
    """Steps measured on either side (16 / 4 heads of 64: an XCD has every other sequence)."""
    for lengths, whole, even in (((2048, 1957, 1867, 1777), 1, 1), ((1000, 886, 771, 657), 1, 1), ((862, 783, 704, 625, 546, 466), 1, 1),
                                 ((1300, 1100, 900, 700, 500, 300), 1, 0),
                                 ((4000, 4000), 0, 1), ((5000, 4000, 3000), 0, 0), ((4000, 2666), 0, 0), ((3000, 2080, 1160), 0, 0), ((2400, 2300, 2200), 0, 1), ((), 0, 1)):
        assert order.even(sum(lengths), max(lengths, default=0), len(lengths), whole) == even, lengths


def test_scored_pairs_of_a_launch(order):
    """Whole prompts by their rows, whatever the grid; chunks of a small grid one after the other, of a large one by what their groups see."""
    for grid_base, lens, max_k, want in ((160, [230] * 5, 3955, 0), (256, [431] * 2, 4093, 0), (264, [300] * 8, 2696, -1), (160, [600, 590], 600, 1),
                                         (160, [900, 300, 200], 900, 0), (2048, [2048, 1957, 1867, 1777], 2048, 1), (2048, [2048, 300, 300], 2048, 0)):
        assert order.scored_pairs(grid_base, len(lens), sum(lens), max(lens), max_k) == want, (grid_base, lens)


def test_latent_chunks_of_about_the_same_keys(order):
    """Row tiles of about the same length have the host's ranges: steps measured on either side (rows, keys of the sequences)."""
    for rows, shortest, longest, alike in ((290, 2966, 3257, 1), (161, 3708, 3828, 1), (238, 1876, 2009, 1), (256, 3053, 4036, 0), (1024, 3000, 6001, 0), (900, 900, 900, 0)):
        assert order.alike(shortest - rows, longest) == alike, (rows, shortest, longest)


def test_latent_turned_order(order):
    """Launches of more than one round without key ranges, on either side of what was measured."""
    for n_qs, max_k, turned in (([931, 770, 608, 446], 931, 1), ([670 - 50 * i for i in range(8)], 670, 1), ([456] * 4, 865, 1), ([1024, 1000] * 4, 1024, 0),
                                ([164, 103] * 6 + [130], 164, 0), ([805 - 23 * i for i in range(9)], 805, 0), ([542, 309, 425] * 2 + [400], 542, 0), ([900], 4000, 0)):
        assert order.turns(len(n_qs), sum(n_qs), max(n_qs), max_k) == turned, n_qs


@pytest.mark.parametrize("together", [1, 2, 3, 4])
def test_prompt_every_place_once(order, together):
    for rounds in (1, 2, 3, 4, 5, 8, 9, 13, 72):
        least, more = C.c_int(), C.c_int()
        order.sets(rounds, together, C.byref(least), C.byref(more))
        sizes = [least.value + 1] * (more.value // (least.value + 1)) + [least.value] * ((rounds - more.value) // least.value)
        assert sum(sizes) == rounds and least.value >= min(together, rounds) and max(sizes) <= 2 * together       # nothing is left over
        of = [s for s, n in enumerate(sizes) for _ in range(n)]
        for slots in (1, 2, 7, 8, 32, 33):
            n = rounds * slots
            round_, place = (C.c_int * n)(), (C.c_int * n)()
            order.prompt(rounds, slots, together, round_, place)
            assert sorted(zip(round_, place)) == [(r, s) for r in range(rounds) for s in range(slots)], (rounds, slots)
            assert [of[r] for r in round_] == [of[i // slots] for i in range(n)]          # one set after the other
            for s in set(of):                                     # the heaviest tiles of a set first
                at = [p for r, p in zip(round_, place) if of[r] == s]
                assert at == sorted(at)
            if together == 1:
                assert list(zip(round_, place)) == [(i // slots, i % slots) for i in range(n)]


def test_prompt_pairs_together(order):
    # (query tiles of 128 rows of two heads: 2 x 64 rows and, with 4 heads a kv head, 64 of four)
    wgs = lambda lens, H, G: len(lens) * G * -(-max(lens) // (128 if H // G == 2 else 64))
    for H, G, lens, max_k, want in ((16, 8, [2048] * 4, 2048, 2), (16, 8, [1024] * 8, 1024, 4), (16, 8, [1365, 1180, 1000] * 2, 1365, 3), (32, 8, [600, 2048], 2048, 1),
                                    (32, 8, [1100, 850, 600] * 2, 1100, 1), (16, 8, [1000] * 4, 3000, 1), (32, 8, [2048] * 4, 2048, 1)):
        assert order.pairs_together(wgs(lens, H, G), sum(lens), len(lens), max(lens), max_k) == want, (H, lens)


def test_states_past_the_caches(order):
    """From 92 MiB of single-token states on: portions behind them do not count (nor does 32-bit arithmetic)."""
    assert [order.states_past(n, n, 0, 16, 128, 128) for n in (1, 91, 92, 4096)] == [0, 0, 1, 1]
    assert [order.states_past(n, 0, 0, 16, 128, 128) for n in (91, 92)] == [0, 1]            # (not known to lead, but all of one token)
    assert [order.states_past(200, lead, 1, 16, 128, 128) for lead in (0, 91, 92)] == [0, 0, 1]
    assert order.states_past(65535, 65535, 0, 64, 256, 256)


def test_expert_outputs_past_the_caches(order):
    """From 64 MiB of outputs on, where they and the experts' weights come to 224 MiB; in 64 bits."""
    past = lambda tokens, E, top, width, ff: order.outputs_past(C.c_int64(tokens * top), width, E, ff)
    assert past(8192, 32, 4, 2048, 1024) and past(2048, 32, 4, 2048, 1024) and past(4096, 32, 2, 2048, 512) and not past(2047, 32, 4, 2048, 1024)
    assert not past(8000, 16, 2, 1024, 1024) and not past(8192, 16, 2, 1024, 1024) and past(16384, 16, 2, 1024, 1024)
    assert not past(3000, 16, 4, 2048, 512) and past(4096, 16, 4, 2048, 512) and not past(8192, 16, 4, 1024, 512)
    assert past(1 << 20, 256, 8, 8192, 8192) and not past(1, 256, 8, 8192, 8192)
