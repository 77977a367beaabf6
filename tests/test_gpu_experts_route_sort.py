"""GPU: routing and sort of (token, choice) pairs in one call against torch: token counts around the one-launch limit, expert counts
around a wave's 64 and around what the joint launches take."""
import pytest
import torch

from nanovllm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T", [1, 17, 128, 129, 1000, 5000])
@pytest.mark.parametrize("E,top", [(4, 4), (32, 4), (33, 1), (64, 16), (65, 2), (300, 8), (512, 3), (520, 3)])
def test_route_sort(T, E, top):
    g = torch.Generator(device=DEV).manual_seed(T + E)
    logits = torch.randn(T, E, generator=g, device=DEV)
    logits[::3] = logits[::3].round()      # ties: the lowest index first
    dll, rows, i32 = ops._lib.mixers(), 16, torch.int32
    ids, pairs = torch.full((T, top), -1, dtype=i32, device=DEV), torch.full((T * top,), -1, dtype=i32, device=DEV)
    wgt = torch.zeros(T, top, device=DEV)
    tiles = dll.nv_moe_max_tiles(T * top, E, rows)
    meta, counts = torch.zeros(1 + 3 * tiles, dtype=i32, device=DEV), torch.empty(max(dll.nv_moe_route_sort_words(T, E), 1), dtype=i32, device=DEV)
    ops._lib.check(dll.nv_moe_route_sort(logits.data_ptr(), ids.data_ptr(), wgt.data_ptr(), pairs.data_ptr(), meta.data_ptr(), counts.data_ptr(),
                                         T, E, top, rows, torch.cuda.current_stream().cuda_stream), "nv_moe_route_sort", dll)
    val, want = logits.cpu().sort(dim=-1, descending=True, stable=True)
    assert torch.equal(ids.cpu().long(), want[:, :top])
    # (expf and the division on either side: a few roundings of 2^-24)
    torch.testing.assert_close(wgt.cpu(), torch.softmax(val[:, :top], -1), rtol=1e-5, atol=1e-7)
    pairs, flat, m = pairs.cpu().long(), ids.cpu().long().flatten(), meta.cpu()
    assert torch.equal(pairs.sort().values, torch.arange(T * top))
    by_expert, n = flat[pairs], torch.bincount(flat, minlength=E)
    assert torch.equal(by_expert, by_expert.sort().values)
    want_tiles, at = [], 0
    for e in range(E):
        want_tiles += [(e, at + i, min(rows, int(n[e]) - i)) for i in range(0, int(n[e]), rows)]
        at += int(n[e])
    assert int(m[0]) == len(want_tiles) <= tiles
    assert torch.equal(m[1:1 + 3 * len(want_tiles)].view(-1, 3), torch.tensor(want_tiles, dtype=i32).view(-1, 3))


# tokens on either side of one workgroup's (16 beyond 64 experts), a wave with more than one token, more workgroups than one for each 4 tokens
@pytest.mark.parametrize("T", [16, 18, 513, 1025, 3001])
@pytest.mark.parametrize("E,top", [(64, 8), (65, 16), (129, 1), (512, 2), (512, 16)])
def test_route_sort_sizes(T, E, top):
    test_route_sort(T, E, top)


@pytest.mark.parametrize("T", [1, 3, 17, 1000])
@pytest.mark.parametrize("E,top", [(4, 4), (16, 1), (33, 5), (64, 16), (65, 2), (512, 3), (520, 16)])
def test_route(T, E, top):
    """The choice alone (nv_moe_route): ties, equal logits, infinite ones and, in some tokens, logits that are not numbers."""
    g = torch.Generator(device=DEV).manual_seed(T * E)
    logits = torch.randn(T, E, generator=g, device=DEV)
    logits[::3] = logits[::3].round()
    logits[1::5] = 0.0
    logits[2::7, ::2] = float("-inf")
    dll, i32 = ops._lib.mixers(), torch.int32
    ids, wgt = torch.full((T, top), -1, dtype=i32, device=DEV), torch.zeros(T, top, device=DEV)
    run = lambda: ops._lib.check(dll.nv_moe_route(logits.data_ptr(), ids.data_ptr(), wgt.data_ptr(), T, E, top, torch.cuda.current_stream().cuda_stream),
                                 "nv_moe_route", dll)
    run()
    val, want = logits.cpu().sort(dim=-1, descending=True, stable=True)
    assert torch.equal(ids.cpu().long(), want[:, :top])
    torch.testing.assert_close(wgt.cpu(), torch.softmax(val[:, :top], -1), rtol=1e-5, atol=1e-7)
    logits[::2, E // 2] = float("nan")
    run()
    chosen = ids.cpu().long().sort(-1).values
    assert chosen.min() >= 0 and chosen.max() < E and (chosen.diff(dim=-1) > 0).all()       # experts, none of them twice
