"""GPU: routed experts whose activations or outputs do not start on 16 bytes, which the suggested tile sizes do not know of."""
import pytest
import torch

from nanovllm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,rows", [(20, 32), (50, 64), (400, 128)])
@pytest.mark.parametrize("y_at,out_at", [(1, 0), (0, 1), (4, 2)])
@pytest.mark.parametrize("form", ["gate_up", "up"])
def test_unaligned_results(form, y_at, out_at, T, rows):
    E, top, W, ff, i32 = 4, 2, 192, 128, torch.int32
    g = torch.Generator(device=DEV).manual_seed(T)
    mk = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device=DEV) * scale).to(torch.bfloat16)
    h, up, down = mk(T, W), mk(E, (2 if form == "gate_up" else 1) * ff, W, scale=W ** -0.5), mk(E, W, ff, scale=ff ** -0.5)
    ids = torch.rand(T, E, generator=g, device=DEV).topk(top, -1).indices.to(i32)
    weights, P = torch.rand(T, top, generator=g, device=DEV), T * top
    dll, s = ops._lib.mixers(), torch.cuda.current_stream().cuda_stream
    assert dll.nv_moe_tile_rows_for(P, E, W, ff, h.data_ptr(), W, up.data_ptr(), down.data_ptr(), 0) == rows
    pairs, meta = torch.empty(P, dtype=i32, device=DEV), torch.empty(1 + 3 * dll.nv_moe_max_tiles(P, E, rows), dtype=i32, device=DEV)
    ops._lib.check(dll.nv_moe_align(ids.data_ptr(), pairs.data_ptr(), meta.data_ptr(), P, E, rows, s), "nv_moe_align", dll)

    def call(y_at, out_at):
        y, out = torch.empty(P * ff + y_at, dtype=h.dtype, device=DEV)[y_at:], torch.empty(P * W + out_at, device=DEV)[out_at:]
        tail = (up.data_ptr(), pairs.data_ptr(), meta.data_ptr(), y.data_ptr(), 0, P, E, top, W, ff)
        if form == "gate_up":
            rc = dll.nv_moe_gate_up(h.data_ptr(), W, *tail, 7.0, 1.702, rows, s)
        else:
            rc = dll.nv_moe_up_relu2(h.data_ptr(), W, *tail, rows, s)
        ops._lib.check(rc, "first product", dll)
        ops._lib.check(dll.nv_moe_down(y.data_ptr(), down.data_ptr(), pairs.data_ptr(), meta.data_ptr(), weights.data_ptr(), out.data_ptr(), 0, P, E,
                                       W, ff, rows, s), "nv_moe_down", dll)
        return out.view(P, W)

    # (the sums in another order in front of the activations' rounding to bf16: a step of 2^-8 in some of the ff summands of order ff^-1/2)
    torch.testing.assert_close(call(y_at, out_at), call(0, 0), rtol=1e-2, atol=1e-2)
