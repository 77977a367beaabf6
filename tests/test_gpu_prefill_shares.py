"""GPU: large prompt launches around the line between one and several query tiles a workgroup, against float32 attention."""
import pytest
import torch

from nanovllm_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV, D, BLOCK = "cuda", 128, 256


@pytest.mark.parametrize("H,G,rows", [(32, 8, [1365] * 6), (32, 8, [2048] * 4), (32, 8, [3500, 2750, 1999]), (32, 8, [2047, 1701, 1355, 1009]),
                                      (16, 8, [2048, 1030, 513, 64, 1])])
def test_prompts(H, G, rows):
    _compare(H, G, rows, 0)


def _compare(H, G, rows, cached):
    gen = torch.Generator(device=DEV).manual_seed(sum(rows))
    mk = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)
    keys = [n + cached for n in rows]
    blocks = [-(-n // BLOCK) for n in keys]
    order = torch.randperm(sum(blocks), generator=torch.Generator().manual_seed(1))
    tables = torch.full((len(rows), max(blocks)), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(blocks):
        tables[b, :n] = order[at:at + n].to(torch.int32)
        at += n
    q, k_cache, v_cache = mk(sum(rows), H, D), mk(at, BLOCK, G, D), mk(at, BLOCK, G, D)
    cu, cu_k = (torch.tensor([0] + torch.tensor(x).cumsum(0).tolist(), dtype=torch.int32, device=DEV) for x in (rows, keys))
    out = ops.attn_prefill_varlen(q, k_cache, v_cache, cu, cu_k, tables.to(DEV), max(rows), max(keys), D ** -0.5)
    start = 0
    for b, n in enumerate(rows):
        pages = tables[b, :blocks[b]].long().to(DEV)
        hidden = torch.ones(n, n + cached, dtype=torch.bool, device=DEV).triu(1 + cached)
        for h in (0, H // 2 + 1, H - 1):
            key, val = (c[pages, :, h * G // H].reshape(-1, D)[:n + cached].float() for c in (k_cache, v_cache))
            p = torch.softmax((q[start:start + n, h].float() @ key.t().contiguous() * D ** -0.5).masked_fill(hidden, float("-inf")), -1)
            # one rounding of the weights and one of the output to bf16, on values up to about 4: 2^-9 each
            torch.testing.assert_close(out[start:start + n, h].float(), p @ val, rtol=1e-2, atol=1e-2)
        start += n


@pytest.mark.parametrize("H,G,rows,cached,tiles", [(16, 8, [2048] * 8, 0, 2), (16, 8, [1024] * 16, 700, 2), (64, 8, [2730] * 3, 0, 1), (32, 8, [1066, 900, 800, 700] * 4, 1059, 2),
                                                   (32, 8, [4096] + [64] * 9, 0, 2), (64, 8, [512] * 16, 256, 4)])
def test_plans(H, G, rows, cached, tiles):
    """The other heads, cached keys in front of the rows and a long prompt among short ones, at one, two and four tiles a workgroup."""
    assert _lib.lib().nv_attn_prefill_query_tiles(len(rows), sum(rows), max(rows), max(rows) + cached, H, G) == tiles
    _compare(H, G, rows, cached)
