"""GPU: latent attention launches of more workgroups than the chip holds at a time (key ranges by what the step has for every slot, rows of one
range without a state): sequences of very different lengths, single tokens between them, row tiles that are not full, one range alone."""
import pytest
import torch

from nanovllm_amd import ops
from buvalix_util import paged_context
from test_gpu_nekodra_layers import DEV, reference_rows, rn

pytestmark = pytest.mark.gpu

STEPS = {"far_apart": ([150, 1, 150, 150], [2500, 90, 150, 700]), "one_long": ([260, 5], [3000, 64]), "prompts": ([500, 300, 1, 77], [500, 300, 1, 77]),
         "equal": ([200, 200], [1600, 1600])}


@pytest.mark.parametrize("H", [16, 13])
@pytest.mark.parametrize("D,Dv", [(256, 256), (160, 128), (320, 320)])
@pytest.mark.parametrize("step", list(STEPS))
def test_even_shares(D, Dv, H, step):
    n_q, n_k = STEPS[step]
    bs, nb = 64, sum(-(-n // 64) for n in n_k) + 3
    ctx, _ = paged_context(n_q, n_k, bs, nb, D, DEV)
    H *= 4                                 # (rows are tokens times heads)
    g = torch.Generator().manual_seed(D + H)
    q = rn(g, sum(n_q), H, D, std=3.0 / D ** 0.5).to(torch.bfloat16)
    cache = rn(g, nb, bs, 1, D).to(torch.bfloat16)
    sink = torch.linspace(-3.0, 6.0, H, device=DEV)
    got = [ops.attn_latent_paged(q, cache, cache[..., :Dv], ctx.cu_seqlens_q, ctx.cu_seqlens_k, ctx.block_tables, 0.9, sink, max(n_q), max(n_k), -1)
           for _ in range(2)]
    want = reference_rows(q, cache, ctx, 0.9, sink, Dv)
    assert torch.equal(got[0], got[1]) and torch.isfinite(got[0]).all()
    # (the bound of the other launches' test: probabilities and outputs are rounded to bf16, 2^-9 each)
    err = (got[0].float() - want).view(sum(n_q), -1).norm(dim=-1) / want.norm(dim=-1)
    assert err.max().item() < 1.2e-2, (int(err.argmax()), err.max().item())


@pytest.mark.parametrize("step,D,Dv,H,even", [("far_apart", 160, 128, 64, True), ("far_apart", 256, 256, 52, True), ("one_long", 256, 256, 64, True),
                                              ("one_long", 320, 320, 52, True), ("equal", 256, 256, 64, True),
                                              ("one_long", 160, 128, 64, True), ("equal", 160, 128, 64, False), ("one_long", 160, 128, 8, False)])
def test_which_launches_have_even_ranges(step, D, Dv, H, even):
    """The launch writes its share in front of the states in the workspace where ranges are sized on the device, and only there."""
    n_q, n_k = STEPS[step]
    ctx, _ = paged_context(n_q, n_k, 64, sum(-(-n // 64) for n in n_k) + 3, D, DEV)
    g = torch.Generator().manual_seed(D + H)
    q, cache = rn(g, sum(n_q), H, D).to(torch.bfloat16), rn(g, sum(-(-n // 64) for n in n_k) + 3, 64, 1, D).to(torch.bfloat16)
    need = ops._lib.mixers().nv_attn_latent_workspace_bytes(len(n_q), sum(n_q), H, D, Dv, max(n_q), max(n_k))
    assert need > 64
    head = ops._workspace(q.device, need)[:4].view(torch.int32)
    head.fill_(-7)
    ops.attn_latent_paged(q, cache, cache[..., :Dv], ctx.cu_seqlens_q, ctx.cu_seqlens_k, ctx.block_tables, 0.9, None, max(n_q), max(n_k), -1)
    tile, share = 64 if D <= 256 else 32, int(head.item())
    assert (8 <= share <= -(-max(n_k) // tile)) if even else share == -7


@pytest.mark.parametrize("H", [16, 13])
@pytest.mark.parametrize("D,Dv", [(256, 256), (160, 128), (320, 320)])
@pytest.mark.parametrize("step", ["alike"])
def test_alike(D, Dv, H, step, monkeypatch):
    """Chunks behind most of their keys: the host's ranges, in the same launch."""
    monkeypatch.setitem(STEPS, "alike", ([40, 1, 33, 40], [1900, 90, 1800, 1700]))
    test_even_shares(D, Dv, H, step)
