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
