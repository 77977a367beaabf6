"""GPU: routed experts with few rows per expert (weights streamed past LDS, tiles of 16, 32 and 64 rows) against the eager stand-ins."""
import pytest
import torch

from nanovllm_amd import ops
from nanovllm_amd.layers import moe
from oracle import ref_benarax_modules, ref_nekodra_modules, ref_tutedra_modules

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _tol():
    # The stand-ins run in float32 on the same values, so what differs is one rounding of the activations to bf16: relative errors of
    # at most 2^-9 in the summands of an output of order one (activations' root mean square <= 1.3, weights ff^-1/2): a
    # standard deviation of about 0.0015, and 6 of them stay below 0.01.
    return dict(rtol=1e-2, atol=1e-2)


# (experts, tokens, top, width, ff): one pair; a tile and one more row; sizes that fill neither a weight block nor a wave's share
@pytest.mark.parametrize("E,T,top,W,ff,rows", [(4, 1, 1, 64, 64, 16), (32, 32, 4, 256, 128, 16), (2, 17, 1, 128, 576, 32), (4, 65, 2, 192, 320, 64),
                                               (3, 95, 1, 448, 64, 64), (8, 160, 4, 64, 192, 64), (4, 200, 1, 64, 72, 64)])
@pytest.mark.parametrize("form", ["clamped", "relu2", "silu"])
def test_few_rows(form, E, T, top, W, ff, rows):
    g = torch.Generator(device=DEV).manual_seed(E * T + W)
    bf = torch.bfloat16
    mk = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device=DEV) * scale).to(bf)
    f = lambda t: t.float()
    h = mk(T, W + 8)[:, :W]
    up, gate_up, down = mk(E, ff, W, scale=W ** -0.5), mk(E, 2 * ff, W, scale=W ** -0.5), mk(E, W, ff, scale=ff ** -0.5)
    logits = torch.randn(T, E, generator=g, device=DEV)
    logits[: T // 2, E - 1] += 100.0       # an expert with many more rows than the others
    dll = ops._lib.mixers()
    assert dll.nv_moe_tile_rows_for(T * top, E, W, ff, h.data_ptr(), h.stride(0), gate_up.data_ptr(), down.data_ptr(), 0) == rows
    if form == "clamped":
        a, r = moe.MoEExperts(top, 1.5), ref_benarax_modules.MoEExperts(top, 1.5)
        torch.testing.assert_close(a(h, logits, gate_up, down), r(f(h), logits, f(gate_up), f(down)), **_tol())
        return
    ids = logits.topk(top, dim=-1).indices.to(torch.int32)
    weights = torch.rand(T, top, generator=g, device=DEV)
    if form == "relu2":
        a, r = moe.SquaredReluExperts(), ref_tutedra_modules.SquaredReluExperts()
        torch.testing.assert_close(a(h, ids, weights, up, down), r(f(h), ids, weights, f(up), f(down)), **_tol())
        return
    ids[1::7, 0] = E + 1                   # choices that need no product: their rows are not written
    a, r = moe.SiluExperts(), ref_nekodra_modules.SiluExperts()
    got, want = a(h, ids, weights, gate_up, down), r(f(h), ids, weights, f(gate_up), f(down))
    live = (ids < E)[..., None].expand_as(got)
    torch.testing.assert_close(got[live], want[live], **_tol())


# a wave's quarter of the contraction in 4, 5, 8 steps of 64 and, with the last wave short of steps or without any, 5 + 5 + 5 + 2 and 2 + 2 + 1 + 0
@pytest.mark.parametrize("E,T,top,W,ff,rows", [(4, 6, 2, 1024, 1280, 16), (4, 25, 2, 1280, 1088, 32), (4, 60, 2, 1088, 2048, 64), (2, 17, 1, 2048, 320, 32),
                                               (3, 90, 1, 2048, 1024, 64), (32, 40, 4, 1088, 1024, 16)])
@pytest.mark.parametrize("form", ["clamped", "relu2", "silu"])
def test_few_rows_long_contractions(form, E, T, top, W, ff, rows):
    test_few_rows(form, E, T, top, W, ff, rows)
