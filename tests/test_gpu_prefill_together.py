"""GPU: prompt attention launches whose XCDs take several pairs of sequence and kv head together, against the other kernel: numbers of pairs
that leave the last group short, sequences of unequal length."""
import pytest
import torch

import nanovllm_amd as nv
from nanovllm_amd import _lib, ops
from test_launch_order import order                              # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H,G,lens", [(16, 8, [1024] * 8), (16, 8, [1300, 1299, 1200, 1100, 1000]), (16, 8, [2048, 1900, 1800]), (32, 8, [700, 700, 690, 650])])
def test_together(H, G, lens):
    g = torch.Generator(device=DEV).manual_seed(len(lens))
    T, D, bs = sum(lens), 128, 256
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(DEV)
    need = [-(-n // bs) for n in lens]
    tables, at = torch.full((len(lens), max(need)), -1, dtype=torch.int32), 0
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(1)).to(torch.int32)
    for i, n in enumerate(need):
        tables[i, :n] = order[at:at + n]
        at += n
    mk = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    q, kc, vc = mk(T, H, D), mk(sum(need), bs, G, D), mk(sum(need), bs, G, D)
    assert _lib.lib().nv_attn_prefill_query_tiles(len(lens), T, max(lens), max(lens), H, G) == 1
    call = lambda: ops.attn_prefill_varlen(q, kc, vc, cu, cu, tables.to(DEV), max(lens), max(lens), D ** -0.5)
    got = call()
    try:
        _lib.set_tuning(prefill_kernel=0)
        want = call()
    finally:
        _lib.set_tuning()
    # (both round probabilities and outputs to bf16, 2^-9 each, outputs are at most of order one)
    torch.testing.assert_close(got.float(), want.float(), rtol=2e-2, atol=1e-2)


@pytest.mark.parametrize("H,G,lens,together", [(16, 8, [1024] * 8, 4), (16, 8, [1300, 1299, 1200, 1100, 1000], 3), (16, 8, [2048, 1900, 1800], 2), (32, 8, [700, 700, 690, 650], 4),
                                               (16, 8, [4000, 3900], 1)])
def test_launches_above_take_several_pairs(order, H, G, lens, together):           # noqa: F811
    """The launches of test_together are the ones that they are meant to be: single tiles, several pairs at a time."""
    tiles = -(-max(lens) // (64 * 4 // (H // G)))
    assert order.pairs_together(len(lens) * G * tiles, sum(lens), len(lens), max(lens), max(lens)) == together


# numbers of pairs an XCD that sets of three or four leave a rest of: 5 in one set (the last XCDs have 4), 9 as 5 and 4, 10 as 4, 3 and 3, 5 spread over two XCDs each
@pytest.mark.parametrize("H,G,lens", [(16, 4, [654 - 3 * i for i in range(9)]), (16, 8, [790 - 30 * i for i in range(9)]), (16, 16, [1206, 1100, 990, 880, 771]),
                                      (16, 4, [943, 930, 915, 900, 885])])
def test_uneven_numbers_of_pairs(H, G, lens):
    test_together(H, G, lens)
