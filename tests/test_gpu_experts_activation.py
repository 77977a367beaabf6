"""GPU: the gated unit of the routed experts, the same from tiles of any number of rows and as exact as float32 gives it."""
import pytest
import torch

from nanovllm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _gate_up(h, gate_up, rows, alpha):
    dll, i32 = ops._lib.mixers(), torch.int32
    T, W = h.shape
    ff = gate_up.shape[1] // 2
    ids, pairs = torch.zeros(T, dtype=i32, device=DEV), torch.empty(T, dtype=i32, device=DEV)
    meta = torch.empty(1 + 3 * dll.nv_moe_max_tiles(T, 1, rows), dtype=i32, device=DEV)
    y, s = torch.empty(T, ff, dtype=h.dtype, device=DEV), torch.cuda.current_stream().cuda_stream
    ops._lib.check(dll.nv_moe_align(ids.data_ptr(), pairs.data_ptr(), meta.data_ptr(), T, 1, rows, s), "nv_moe_align", dll)
    ops._lib.check(dll.nv_moe_gate_up(h.data_ptr(), W, gate_up.data_ptr(), pairs.data_ptr(), meta.data_ptr(), y.data_ptr(), 0, T, 1, 1, W, ff,
                                      float("inf"), alpha, rows, s), "nv_moe_gate_up", dll)
    out = torch.empty_like(y)
    out[pairs.long()] = y
    return out


@pytest.mark.parametrize("alpha", [1.0, 1.702])
def test_gated_unit(alpha):
    # gates that every order of the sums gives exactly: whole numbers from the rows, multiples of 2^-8 from the weights
    whole, part = torch.arange(-128, 128, device=DEV), torch.arange(-255, 257, device=DEV) / 256
    h = torch.zeros(256, 64, device=DEV)
    h[:, 0], h[:, 1] = whole, 1
    gate_up = torch.zeros(1, 1024, 64, device=DEV)
    gate_up[0, :512, 0], gate_up[0, :512, 1], gate_up[0, 512:, 1] = 1, part, 1
    got = {rows: _gate_up(h.to(torch.bfloat16), gate_up.to(torch.bfloat16), rows, alpha) for rows in (16, 32, 64, 128)}
    for rows in (16, 32, 64):
        assert torch.equal(got[rows], got[128])
    g, alpha = (whole[:, None] + part).double(), torch.tensor(alpha).double().item()
    want = g * torch.sigmoid(alpha * g) * 2
    # Where exp(-alpha g) is a float32: its argument is rounded once (a relative error of alpha |g| 2^-24 <= 2^-17 in the exponential), the rest is a
    # few roundings of 2^-24, then one to the eight significant bits of bf16 (at most 2^-8).
    seen = alpha * g > -88
    err = (got[128].double() - want).abs()
    assert (err[seen] <= want.abs()[seen] * (2 ** -8 + 2 ** -16)).all()
    assert (err <= 2e-36).logical_or(seen).all()
