"""GPU: score-modified attention on pages of whole key tiles against the eager stand-in: portions around the 32-row blocks and the 64-key
tiles, every group size's way of sharing a workgroup, key and value sizes 64 / 128, each form of the scores, long portions of one
sequence (cut into key ranges) and single rows beside portions."""
import pytest
import torch

import nanovllm_amd as nv
from nanovllm_amd import ops
from nanovllm_amd.layers import attention
from oracle import ref_mixer_modules as ref
from test_gpu_mixers import DEV, _context

pytestmark = pytest.mark.gpu

STEPS = {"edges": ([1, 31, 32, 33, 64, 65, 2], [64, 31, 96, 161, 64, 129, 66]), "portions": ([200, 1, 130], [200, 77, 600]),
         "ranges": ([40], [2500]), "singles": ([1] * 5, [1500, 63, 64, 65, 1])}
FORMS = {"plain": dict(), "cap_sink": dict(softcap=25.0, use_sink=True, rot_dims=32), "high_cap": dict(softcap=60.0, temp_coef=0.5, temp_every=64),
         "cap_bias_sink": dict(softcap=25.0, use_sink=True, bias=True), "bias": dict(bias=True)}


@pytest.mark.parametrize("step", list(STEPS))
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("shape", [(4, 2, 128, 128, 64), (4, 4, 64, 64, 128), (8, 1, 64, 128, 64), (6, 2, 128, 64, 256)])
def test_portions(shape, form, step):
    H, G, D, Dv, bs = shape
    kw = dict(FORMS[form])
    bias = kw.pop("bias", False)
    n_qs, n_ks = STEPS[step]
    nb = sum(-(-n // bs) for n in n_ks) + 2
    a, r = (m.ScoreModAttention(H, G, D, Dv, D ** -0.5, device=DEV, **kw) for m in (attention, ref))
    g = torch.Generator(device=DEV).manual_seed(H * D + Dv)
    if bias:
        table = torch.randn(H, 90, generator=g, device=DEV)
        a.set_distance_bias(table)
        r.set_distance_bias(table)
    if a.sink is not None:
        with torch.no_grad():
            a.sink.copy_(3 * torch.randn(H, generator=g, device=DEV))
            r.sink.copy_(a.sink)
    ctx, pos = _context(n_qs, n_ks, bs, nb, seed=4)
    ctx.num_decode_seqs = sum(n == 1 for n in n_qs)
    T = sum(n_qs)
    mk = lambda *s: (2 * torch.randn(*s, generator=g, device=DEV)).to(torch.bfloat16)
    q, k, v = mk(T, H, D), mk(T, G, D), mk(T, G, Dv)
    kc, vc = mk(nb, bs, G, D), mk(nb, bs, G, Dv)
    kc_r, vc_r = kc.clone(), vc.clone()
    nv.set_context(ctx)
    o, o_r = a(q, k, v, pos, kc, vc), r(q, k, v, pos, kc_r, vc_r)
    nv.set_context(None)
    torch.testing.assert_close(kc.float(), kc_r.float(), rtol=2e-2, atol=2e-2)
    assert torch.equal(vc, vc_r)
    # probabilities and outputs are rounded to bf16 (2^-9 each) and values are of order two
    torch.testing.assert_close(o.float(), o_r.float(), rtol=2e-2, atol=2e-2)


def _step(H, G, D, Dv, bs, n_qs, n_ks, seed=4, scale=None, spread=1.0, **kw):
    """A layer, its stand-in, the step's rows and caches (bfloat16)."""
    a, r = (m.ScoreModAttention(H, G, D, Dv, scale or D ** -0.5, device=DEV, **kw) for m in (attention, ref))
    g = torch.Generator(device=DEV).manual_seed(H * D + Dv)
    nb = sum(-(-n // bs) for n in n_ks) + 2
    ctx, pos = _context(n_qs, n_ks, bs, nb, seed=seed)
    ctx.num_decode_seqs = sum(n == 1 for n in n_qs)
    mk = lambda *s: (spread * torch.randn(*s, generator=g, device=DEV)).to(torch.bfloat16)
    T = sum(n_qs)
    return a, r, ctx, pos, mk(T, H, D), mk(T, G, D), mk(T, G, Dv), mk(nb, bs, G, D), mk(nb, bs, G, Dv)


@pytest.mark.parametrize("where", ["own", "first"])
@pytest.mark.parametrize("n_qs,n_ks", [([40], [2500]), ([70, 33], [200, 161]), ([1], [1281]), ([1], [1400]), ([1] * 3, [1500, 63, 64])])
@pytest.mark.parametrize("softcap", [0.0, 25.0, 60.0])
def test_a_key_that_is_not_a_number(softcap, n_qs, n_ks, where):
    """Every row that sees such a key is not a number, whatever key ranges there are; the other heads do not notice."""
    H, G, D, bs = 4, 2, 128, 64
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, D, D, bs, n_qs, n_ks, softcap=softcap)
    nv.set_context(ctx)
    clean = a(q, k, v, pos, kc.clone(), vc.clone()).view(-1, H, D)
    if where == "own":
        k[0, 1] = float("nan")             # the first new token's: all rows of the sequence see it
    else:
        kc[ctx.block_tables[0, 0], 0, 1] = float("nan")
    got = a(q, k, v, pos, kc, vc).view(-1, H, D)
    nv.set_context(None)
    n = n_qs[0]
    assert got[:n, 2:].isnan().all()
    assert torch.equal(got[:, :2], clean[:, :2]) and torch.equal(got[n:], clean[n:])


@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("n_qs,n_ks", [([40, 70], [0, 200]), ([3, 33], [1, 50]), ([130], [0])])
def test_rows_without_keys(n_qs, n_ks, sink):
    """Rows that no key precedes are zero (nothing is read for them), whatever stands beside them."""
    H, G, D, bs = 4, 2, 128, 64
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, D, D, bs, n_qs, [max(n, m) for n, m in zip(n_qs, n_ks)], use_sink=True)
    cu_k = torch.tensor([0] + torch.tensor(n_ks).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    call = lambda q, cu_q, cu_k, bt, most: ops.attn_scoremod_paged(q, kc, vc, cu_q, cu_k, bt, D ** -0.5, 0.0, a.sink if sink else None, None,
                                                                  max(n_qs), most, 0)
    got = call(q, ctx.cu_seqlens_q, cu_k, ctx.block_tables, max(n_ks))
    assert got[:n_qs[0] - n_ks[0]].eq(0).all()
    if len(n_qs) > 1:
        n = n_qs[0]
        alone = call(q[n:], torch.tensor([0, n_qs[1]], dtype=torch.int32, device=DEV),
                     torch.tensor([0, n_ks[1]], dtype=torch.int32, device=DEV), ctx.block_tables[1:], n_ks[1])
        torch.testing.assert_close(got[n:], alone, rtol=1e-2, atol=1e-2)     # (key ranges may differ)


@pytest.mark.parametrize("n_qs,n_ks", [([64, 40], [190, 170]), ([40], [2500])])
def test_denominators_of_portions(n_qs, n_ks):
    """The denominator is a sum of float32 weights: all but one weight are just below one, where bfloat16 rounds them up."""
    H, G, D, bs = 4, 2, 128, 64
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, D, D, bs, n_qs, n_ks, scale=1.0)
    q.zero_()[..., 0] = 1.0
    for t in (k, kc):
        t.zero_()[..., 0] = -0.0017013549  # exp of it is 0.9983: 1 in bfloat16
    v.zero_()
    vc.zero_()
    first = ctx.block_tables[:, 0].long()
    kc[first, 0] = 0.0                     # the largest weight, and the only one with values
    vc[first, 0] = (1 + torch.rand(G, D, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)).to(torch.bfloat16)
    nv.set_context(ctx)
    o = a(q, k, v, pos, kc, vc)
    nv.set_context(None)
    w = torch.tensor(-0.0017013549, dtype=torch.bfloat16).double().exp().item()
    at = 0
    for b, (n, m) in enumerate(zip(n_qs, n_ks)):
        seen = torch.arange(m - n, m, dtype=torch.float64, device=DEV)   # keys in front of each row, with its own
        want = vc[first[b], 0].double().repeat_interleave(H // G, 0).flatten()[None] / (1 + seen * w)[:, None]
        # one rounding of the outputs, unbiased over rows * H * D of them; rounded weights would give 1.7e-3
        assert abs((o[at:at + n].double() / want - 1).mean().item()) < 4e-4
        at += n


@pytest.mark.parametrize("softcap", [1.0, 25.0, 60.0, 1000.0, 1e6])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("sign", [1, -1])
def test_single_rows_any_soft_cap(sign, softcap, bias):
    """Scores small against the soft cap: the error is one of the score, not of the cap."""
    H, G, D, bs = 8, 4, 64, 64
    n_ks = [700, 64, 130]
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, D, 128, bs, [1] * 3, n_ks, scale=sign * D ** -0.5, softcap=softcap)
    if bias:
        table = torch.randn(H, 90, generator=torch.Generator(device=DEV).manual_seed(2), device=DEV)
        a.set_distance_bias(table)
        r.set_distance_bias(table)
    nv.set_context(ctx)
    o, o_r = a(q, k, v, pos, kc, vc), r(q, k, v, pos, kc, vc)
    nv.set_context(None)
    # fp32 throughout and one rounding of the output (2^-9) on both sides
    torch.testing.assert_close(o.float(), o_r.float(), rtol=2 ** -7, atol=1e-3)


@pytest.mark.parametrize("step", list(STEPS))
@pytest.mark.parametrize("softcap", [0.0, 25.0])
@pytest.mark.parametrize("D,Dv,at", [(128, 64, 0), (128, 64, 64), (128, 64, 8), (128, 128, 0), (64, 64, 0)])
def test_values_as_columns_of_the_keys(D, Dv, at, softcap, step):
    """Value rows with a stride of their own, as a column range of the key rows: what a dense copy of them gives, bit for bit."""
    H, G, bs = 4, 2, 64
    n_qs, n_ks = STEPS[step]
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, D, Dv, bs, n_qs, n_ks)
    values = kc[..., at:at + Dv]
    got, want = (ops.attn_scoremod_paged(q, kc, x, ctx.cu_seqlens_q, ctx.cu_seqlens_k, ctx.block_tables, D ** -0.5, softcap, None, None,
                                         max(n_qs), max(n_ks)) for x in (values, values.contiguous()))
    assert got.isfinite().all() and torch.equal(got, want)


@pytest.mark.parametrize("H,G,n_qs", [(16, 16, [700] * 11 + [90]), (8, 8, [300, 40, 129, 257, 300, 2, 64, 299, 31]), (4, 1, [1500, 700, 900]), (8, 4, [640])])
def test_every_row_whatever_the_order(H, G, n_qs):
    """Launches of more and of fewer workgroups than the chip holds, numbers of sequences and kv heads that leave the last group of an XCD's
    pairs short, pairs spread over XCDs: every row is written once, by the workgroup that has its keys."""
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, 64, 64, 64, n_qs, n_qs, softcap=25.0)
    kc_r, vc_r = kc.clone(), vc.clone()
    nv.set_context(ctx)
    o, o_r = a(q, k, v, pos, kc, vc), r(q, k, v, pos, kc_r, vc_r)
    nv.set_context(None)
    # (as in test_portions)
    torch.testing.assert_close(o.float(), o_r.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("H,G,n_qs,n_ks", [
    (8, 8, [2500] * 4, None),                         # all resident, 4 rounds of 20: workgroups 32 .. 63 of an XCD's group go back
    (16, 8, [900] * 9, None),                         # more than are resident, 9 rounds: sets of five and four pairs that turn
    (16, 4, [400] * 6, [410, 430, 450, 440, 420, 400]),   # chunks of about the same length, a set of three pairs
    (16, 4, [400] * 6, [2000, 430, 1200, 440, 700, 400]),  # and of very different ones: one after the other
    (16, 4, [300] * 6, [310, 330, 350, 340, 320, 300]),   # too few workgroups to look at their lengths
    (16, 4, [430, 1, 430, 40, 1], [1000, 3000, 980, 990, 64]),     # single rows between them
    (16, 8, [200] * 13, [201 + i for i in range(13)]),    # sets of five, four and four
    (16, 8, [700, 90, 350, 300, 410], None)])         # prompts of very different lengths
def test_orders_of_pairs(H, G, n_qs, n_ks):
    """Every order that the launch chooses from: every row is written once, by the workgroup that has its keys."""
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, 64, 64, 64, n_qs, n_ks or n_qs, softcap=25.0)
    kc_r, vc_r = kc.clone(), vc.clone()
    nv.set_context(ctx)
    o, o_r = a(q, k, v, pos, kc, vc), r(q, k, v, pos, kc_r, vc_r)
    nv.set_context(None)
    # (as in test_portions)
    torch.testing.assert_close(o.float(), o_r.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("H,G,D,Dv", [(4, 2, 128, 128), (8, 2, 64, 64), (4, 2, 64, 128)])
@pytest.mark.parametrize("softcap,spread", [(30.0, 0.5), (30.0, 1.0), (8.0, 1.0), (2.0, 1.0), (0.5, 1.0), (30.0, 6.0), (1e-3, 1.0), (1e4, 1.0)])
def test_caps_far_above_and_below_the_scores(H, G, D, Dv, softcap, spread):
    """Scores from a hundredth of the cap to far beyond it.  Tiles whose rows see all of them, and edges."""
    n_qs, n_ks = [150, 64, 33], [700, 64, 290]
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, D, Dv, 64, n_qs, n_ks, spread=spread, softcap=softcap, use_sink=True)
    nv.set_context(ctx)
    o, o_r = a(q, k, v, pos, kc.clone(), vc.clone()), r(q, k, v, pos, kc.clone(), vc.clone())
    nv.set_context(None)
    # probabilities and outputs are rounded to bf16 (2^-9 each), values are of order `spread`
    torch.testing.assert_close(o.float(), o_r.float(), rtol=2e-2, atol=1e-2 * spread)


@pytest.mark.parametrize("D,Dv", [(128, 128), (64, 64), (64, 128), (128, 64)])
@pytest.mark.parametrize("softcap,spread", [(30.0, 1.0), (8.0, 0.5), (300.0, 3.0), (0.0, 1.0)])
def test_a_row_in_portions_that_begin_elsewhere(D, Dv, softcap, spread):
    """A row's bits do not depend on the other rows of its portion: a tile that all rows of its wave see in one portion is at the diagonal of a row of its
    wave in another, and one in which no row's maximum rises in one may raise another row's."""
    H, G, bs, n_k = 4, 2, 64, 704
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, D, Dv, bs, [n_k], [n_k], spread=spread, softcap=softcap, use_sink=True)
    cu = lambda n: torch.tensor([0, n], dtype=torch.int32, device=DEV)
    got = {n: ops.attn_scoremod_paged(q[n_k - n:], kc, vc, cu(n), cu(n_k), ctx.block_tables, D ** -0.5, softcap, a.sink, None, n, n_k, 0).view(n, -1)
           for n in (144, 140, 128, 97)}
    for n, o in got.items():
        assert torch.equal(o, got[144][144 - n:]), n


@pytest.mark.parametrize("D,Dv", [(128, 128), (64, 64)])
@pytest.mark.parametrize("softcap,rows,keys", [(1e-9, 0.0, 1.0), (1e-12, 0.0, 1.0), (1e24, 1e12, 1e10), (1e30, 1e10, 1e10)])
def test_caps_beyond_all_measure(D, Dv, softcap, rows, keys):
    """Scores of zero under a cap near zero weigh all keys alike; products far beyond 2^64 under a cap still larger leave finite outputs."""
    H, G, bs, n_q, n_k = 4, 2, 64, 70, 330
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, D, Dv, bs, [n_q], [n_k], softcap=softcap)
    got = ops.attn_scoremod_paged(q * rows, kc * keys, vc, ctx.cu_seqlens_q, ctx.cu_seqlens_k, ctx.block_tables, D ** -0.5, softcap, None, None, n_q, n_k, 0)
    assert torch.isfinite(got.float()).all()
    if rows == 0.0:
        vals = vc[ctx.block_tables[0].long()].flatten(0, 1)[:n_k].float().repeat_interleave(H // G, dim=1)
        seen = torch.arange(n_k - n_q, n_k, device=DEV) + 1
        want = vals.cumsum(0)[seen - 1] / seen[:, None, None]
        # (the mean of hundreds of values of order one, about 0.06, rounded to bf16)
        torch.testing.assert_close(got.view(n_q, H, Dv).float(), want, rtol=2 ** -8, atol=1e-4)


@pytest.mark.parametrize("D,Dv", [(128, 128), (64, 64), (64, 128), (128, 64)])
@pytest.mark.parametrize("form", ["plain", "cap", "bias", "cap_bias"])
def test_short_and_long_launches(D, Dv, form):
    """Launches of up to three key tiles take another loop than longer ones (without a bias): the same rows with a longer sequence behind them have the
    same bits; prompts and portions that end around the tiles' edges."""
    H, G, bs = 4, 2, 64
    n_qs, n_ks = [1, 2, 33, 64, 100, 128, 70, 192, 200], [1, 2, 33, 64, 129, 128, 190, 192, 700]
    cap = 25.0 if "cap" in form else 0.0
    a, r, ctx, pos, q, k, v, kc, vc = _step(H, G, D, Dv, bs, n_qs, n_ks, softcap=cap, use_sink=True, spread=2.0)
    bias = torch.randn(H, 90, device=DEV) if "bias" in form else None
    call = lambda n, T: ops.attn_scoremod_paged(q[:T], kc, vc, ctx.cu_seqlens_q[:n + 1], ctx.cu_seqlens_k[:n + 1], ctx.block_tables[:n].contiguous(), D ** -0.5, cap,
                                                a.sink, bias, max(n_qs[:n]), max(n_ks[:n]), -1)
    T = sum(n_qs[:-1])
    assert max(n_ks[:-1]) <= 192 < n_ks[-1]
    assert torch.equal(call(len(n_qs) - 1, T), call(len(n_qs), sum(n_qs))[:T])
