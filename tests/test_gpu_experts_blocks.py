"""GPU: routed experts in tiles of 128 rows, more blocks than CUs (slices 64 deep; tests of fewer blocks take slices 32 deep), against the eager
stand-ins: one slice and many, weight blocks that are not full, tiles that are not full."""
import pytest
import torch

from nanovllm_amd.layers import moe
from oracle import ref_benarax_modules, ref_nekodra_modules, ref_tutedra_modules
from test_gpu_experts_many_rows import DEV, _tol
from test_launch_order import order                              # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,T,top,W,ff", [(3, 4200, 2, 1088, 1088), (2, 6000, 2, 64, 832)])
@pytest.mark.parametrize("form", ["clamped", "relu2", "silu"])
def test_many_blocks(order, form, E, T, top, W, ff):             # noqa: F811
    assert not order.few_blocks(T * top, E, -(-ff // (256 if form == "relu2" else 128)))
    assert W < 256 or not order.few_blocks(T * top, E, -(-W // 256))
    g = torch.Generator(device=DEV).manual_seed(W)
    mk = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device=DEV) * scale).to(torch.bfloat16)
    f = lambda t: t.float()
    h, logits = mk(T, W), torch.randn(T, E, generator=g, device=DEV)
    up, gate_up, down = mk(E, ff, W, scale=W ** -0.5), mk(E, 2 * ff, W, scale=W ** -0.5), mk(E, W, ff, scale=ff ** -0.5)
    if form == "clamped":
        a, r = moe.MoEExperts(top, 1.5), ref_benarax_modules.MoEExperts(top, 1.5)
        got, want = a(h, logits, gate_up, down), r(f(h), logits, f(gate_up), f(down))
    else:
        ids, weights = logits.topk(top, dim=-1).indices.to(torch.int32), torch.rand(T, top, generator=g, device=DEV)
        a, r = (moe.SquaredReluExperts(), ref_tutedra_modules.SquaredReluExperts()) if form == "relu2" else (moe.SiluExperts(), ref_nekodra_modules.SiluExperts())
        w = up if form == "relu2" else gate_up
        got, want = a(h, ids, weights, w, down), r(f(h), ids, weights, f(w), f(down))
    torch.testing.assert_close(got, want, **_tol())


@pytest.mark.parametrize("form", ["relu2", "silu"])
def test_rows_far_apart(order, form):                            # noqa: F811
    """More blocks than CUs, rows whose byte offsets do not fit 32 bits."""
    E, T, top, W, ff = 2, 4500, 1, 64, 1088
    assert not order.few_blocks(T * top, E, -(-ff // (256 if form == "relu2" else 128))) or form == "relu2"
    g = torch.Generator(device=DEV).manual_seed(3)
    mk = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device=DEV) * scale).to(torch.bfloat16)
    h, near = torch.empty(T, (1 << 31) // T // 8 * 8 + 8, dtype=torch.bfloat16, device=DEV)[:, :W], mk(T, W)
    h.copy_(near)
    w, down, ids = mk(E, (1 if form == "relu2" else 2) * ff, W, scale=W ** -0.5), mk(E, W, ff, scale=ff ** -0.5), torch.arange(T, device=DEV)[:, None].to(torch.int32) % E
    a, weights = moe.SquaredReluExperts() if form == "relu2" else moe.SiluExperts(), torch.rand(T, top, generator=g, device=DEV)
    assert torch.equal(a(h, ids, weights, w, down), a(near, ids, weights, w, down))      # (the sums are in the same order)


def test_experts_of_4_gib():
    """Weight rows whose byte offsets do not fit 32 bits, in both products."""
    T, W, ff = 200, (1 << 20) + 64, 2048
    g = torch.Generator(device=DEV).manual_seed(4)
    mk = lambda *s, scale=1.0: torch.empty(*s, dtype=torch.bfloat16, device=DEV).normal_(0.0, scale, generator=g)
    h, up, down = mk(T, W), mk(1, ff, W, scale=W ** -0.5), mk(1, W, ff, scale=ff ** -0.5)
    ids, weights = torch.zeros(T, 1, dtype=torch.int32, device=DEV), torch.rand(T, 1, generator=g, device=DEV)
    got = moe.SquaredReluExperts()(h, ids, weights, up, down)[:, 0]
    y = torch.zeros(T, ff, device=DEV)
    for c in range(0, W, 1 << 16):
        y += h[:, c:c + (1 << 16)].float() @ up[0, :, c:c + (1 << 16)].float().t().contiguous()
    y = y.clamp(min=0).square()
    for c in range(0, W, 1 << 16):
        want = y @ down[0, c:c + (1 << 16)].float().t().contiguous() * weights
        torch.testing.assert_close(got[:, c:c + (1 << 16)], want, **_tol())
