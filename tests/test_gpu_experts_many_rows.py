"""GPU: routed experts with many rows per expert (tiles of 128 rows and 256 weight rows) against the eager stand-ins: counts around a
tile, experts without any row, sizes that do not fill the weight block, a strided input, choices that need no product."""
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


@pytest.mark.parametrize("E,T,top,W,ff", [(4, 200, 2, 128, 64), (3, 300, 1, 192, 320), (8, 1024, 3, 256, 640), (2, 129, 2, 576, 192)])
@pytest.mark.parametrize("form", ["clamped", "relu2", "silu"])
def test_many_rows(form, E, T, top, W, ff):
    g = torch.Generator(device=DEV).manual_seed(E * T + W)
    bf = torch.bfloat16
    mk = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device=DEV) * scale).to(bf)
    f = lambda t: t.float()
    h = mk(T, W + 8)[:, :W]
    up, gate_up, down = mk(E, ff, W, scale=W ** -0.5), mk(E, 2 * ff, W, scale=W ** -0.5), mk(E, W, ff, scale=ff ** -0.5)
    logits = torch.randn(T, E, generator=g, device=DEV)
    if E > top:
        logits[:, 0] -= 100.0              # an expert that nobody chooses
    assert ops._lib.mixers().nv_moe_tile_rows_for(T * top, E, W, ff, h.data_ptr(), h.stride(0), gate_up.data_ptr(), down.data_ptr(), 0) == 128
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


def test_rows_far_apart():
    """Rows whose byte offsets do not fit 32 bits: another launch takes the same tiles."""
    E, T, top, W, ff = 2, 300, 1, 128, 64
    g = torch.Generator(device=DEV).manual_seed(3)
    h = torch.empty(T, (1 << 31) // T // 8 * 8 + 8, dtype=torch.bfloat16, device=DEV)[:, :W]
    near = torch.randn(T, W, generator=g, device=DEV).to(torch.bfloat16)
    h.copy_(near)
    mk = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device=DEV) * scale).to(torch.bfloat16)
    gate_up, down, logits = mk(E, 2 * ff, W, scale=W ** -0.5), mk(E, W, ff, scale=ff ** -0.5), torch.randn(T, E, generator=g, device=DEV)
    a = moe.MoEExperts(top, 1.5)
    torch.testing.assert_close(a(h, logits, gate_up, down), a(near, logits, gate_up, down), **_tol())


def test_outputs_past_the_caches():
    """Outputs of 64 MiB and more pass by the caches beside 160 MiB of weights: the rows of two calls of half the tokens, whose outputs do not, to the bit."""
    T, E, top, W, ff = 2100, 32, 4, 2048, 448
    assert T * top * W * 4 >= 64 << 20 > T // 2 * top * W * 4 and T * top * W * 4 + 6 * E * ff * W >= 224 << 20
    g = torch.Generator(device="cuda").manual_seed(5)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    h, logits = rn(T, W).to(torch.bfloat16), rn(T, E)
    gate_up, down = (W ** -0.5 * rn(E, 2 * ff, W)).to(torch.bfloat16), (ff ** -0.5 * rn(E, W, ff)).to(torch.bfloat16)
    call = lambda at: ops.moe_experts(h[at].contiguous(), logits[at].contiguous(), gate_up, down, top, 7.0, 1.702)
    assert torch.equal(call(slice(0, T)), torch.cat([call(slice(0, T // 2)), call(slice(T // 2, T))]))
