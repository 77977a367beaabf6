"""GPU: large prompt launches around the line between one and several query tiles a workgroup, against float32 attention."""
import pytest
import torch

from nanovllm_amd import ops

pytestmark = pytest.mark.gpu
DEV, D, BLOCK = "cuda", 128, 256


@pytest.mark.parametrize("H,G,rows", [(32, 8, [1365] * 6), (32, 8, [2048] * 4), (32, 8, [3500, 2750, 1999]), (32, 8, [2047, 1701, 1355, 1009]),
                                      (16, 8, [2048, 1030, 513, 64, 1])])
def test_prompts(H, G, rows):
    gen = torch.Generator(device=DEV).manual_seed(sum(rows))
    mk = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)
    blocks = [-(-n // BLOCK) for n in rows]
    order = torch.randperm(sum(blocks), generator=torch.Generator().manual_seed(1))
    tables = torch.full((len(rows), max(blocks)), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(blocks):
        tables[b, :n] = order[at:at + n].to(torch.int32)
        at += n
    q, k_cache, v_cache = mk(sum(rows), H, D), mk(at, BLOCK, G, D), mk(at, BLOCK, G, D)
    cu = torch.tensor([0] + torch.tensor(rows).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    out = ops.attn_prefill_varlen(q, k_cache, v_cache, cu, cu, tables.to(DEV), max(rows), max(rows), D ** -0.5)
    start = 0
    for b, n in enumerate(rows):
        pages = tables[b, :blocks[b]].long().to(DEV)
        hidden = torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1)
        for h in (0, H // 2 + 1, H - 1):
            key, val = (c[pages, :, h * G // H].reshape(-1, D)[:n].float() for c in (k_cache, v_cache))
            p = torch.softmax((q[start:start + n, h].float() @ key.t().contiguous() * D ** -0.5).masked_fill(hidden, float("-inf")), -1)
            # one rounding of the weights and one of the output to bf16, on values up to about 4: 2^-9 each
            torch.testing.assert_close(out[start:start + n, h].float(), p @ val, rtol=1e-2, atol=1e-2)
        start += n
