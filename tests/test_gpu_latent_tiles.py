"""GPU: latent attention over few key tiles of every remainder: the loop over tiles begins two ahead and ends one behind, a sequence's last tile
may be part of one, waves of a workgroup end on different tiles, and a raised maximum rescales in the middle."""
import pytest
import torch

from nanovllm_amd import ops
from buvalix_util import paged_context
from test_gpu_nekodra_layers import DEV, reference_rows, rn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,Dv", [(256, 256), (160, 160), (96, 96), (64, 64), (32, 32), (128, 128), (192, 128), (320, 320), (576, 512)])
@pytest.mark.parametrize("n_k", [2, 31, 64, 65, 128, 129, 191, 192, 257, 320, 385])
@pytest.mark.parametrize("rows", [2, 70])
def test_few_tiles(D, Dv, n_k, rows):
    rows, H = min(rows, n_k), 4
    n_q, n_ks = [rows, 2], [n_k, 2]
    nb = sum(-(-n // 64) for n in n_ks) + 2
    ctx, _ = paged_context(n_q, n_ks, 64, nb, D, DEV)
    g = torch.Generator().manual_seed(D + n_k)
    q = rn(g, sum(n_q), H, D, std=3.0 / D ** 0.5).to(torch.bfloat16)
    cache = rn(g, nb, 64, 1, D)
    cache *= torch.linspace(0.3, 4.0, nb, device=DEV)[:, None, None, None]        # later blocks raise the maximum (or earlier ones do: any order)
    cache = cache.to(torch.bfloat16)
    got = ops.attn_latent_paged(q, cache, cache[..., :Dv], ctx.cu_seqlens_q, ctx.cu_seqlens_k, ctx.block_tables, 0.9, None, max(n_q), max(n_ks), -1)
    want = reference_rows(q, cache, ctx, 0.9, None, Dv)
    assert torch.isfinite(got).all()
    # (the bound of the other launches' test: probabilities and outputs are rounded to bf16, 2^-9 each)
    err = (got.float() - want).view(sum(n_q), -1).norm(dim=-1) / want.norm(dim=-1)
    assert err.max().item() < 1.2e-2, (int(err.argmax()), err.max().item())


@pytest.mark.parametrize("D,Dv,H", [(32, 32, 4), (96, 96, 33), (160, 160, 16), (160, 128, 16), (192, 192, 16), (256, 256, 16), (256, 192, 40), (320, 320, 8), (512, 512, 16),
                                    (576, 512, 40)])
@pytest.mark.parametrize("softmax", ["flat", "peaked"])
def test_few_tiles_of_single_tokens(D, Dv, H, softmax):
    """Single tokens over few key tiles of every remainder, the four waves of a workgroup with and without tiles of their own, value columns in one group
    and in two, without key ranges."""
    n_ks = [1, 31, 32, 33, 64, 127, 128, 129, 160, 257, 390]
    nb = sum(-(-n // 64) for n in n_ks) + 2
    ctx, _ = paged_context([1] * len(n_ks), n_ks, 64, nb, D, DEV)
    g = torch.Generator().manual_seed(D + H)
    q = rn(g, len(n_ks), H, D, std=(3.0 if softmax == "peaked" else 0.3) / D ** 0.5).to(torch.bfloat16)
    cache = rn(g, nb, 64, 1, D)
    cache *= torch.linspace(0.3, 4.0, nb, device=DEV)[:, None, None, None]
    cache = cache.to(torch.bfloat16)
    sink = rn(g, H)
    got = ops.attn_latent_paged(q, cache, cache[..., :Dv], ctx.cu_seqlens_q, ctx.cu_seqlens_k, ctx.block_tables, 0.9, sink, 1, max(n_ks), 1)
    want = reference_rows(q, cache, ctx, 0.9, sink, Dv)
    assert torch.isfinite(got).all()
    # (the bound of test_few_tiles)
    err = (got.float() - want).view(len(n_ks), -1).norm(dim=-1) / want.norm(dim=-1)
    assert err.max().item() < 1.2e-2, (int(err.argmax()), err.max().item())
