"""GPU: the recurrences with a decay per head and key channel against the eager stand-ins of the same layers, at the sizes where
their launches change: around the chunks of 8 and of 16 tokens, single tokens in front of, between and beside longer portions, fresh and
carried states, every built number of key channels, value columns that do not fill a workgroup, decays from none to total."""
import pytest
import torch

import nanovllm_amd as nv
from nanovllm_amd import ops
from nanovllm_amd.layers import delta_rule, gated_memory, general_delta
from oracle import ref_benarax_modules, ref_mixer_modules, ref_tutedra_modules

pytestmark = pytest.mark.gpu
DEV = "cuda"

STEPS = {   # rows of the sequences; keys in front of them
    "chunk_edges": ([2, 7, 8, 9, 16, 17], [0, 3, 0, 5, 1, 0]),
    "mixed": ([1, 1, 30, 1, 0, 65], [4, 0, 7, 2, 3, 0]),
    "singles": ([1, 1, 1], [0, 9, 1]),
    "long": ([300], [0]),
}


def _context(rows, before, hints):
    cu = lambda xs: torch.tensor([0] + torch.tensor(xs).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    lead = 0
    while lead < len(rows) and rows[lead] == 1:
        lead += 1
    known = dict(max_seqlen_q=max(rows), num_leading_decode=lead, portion_kinds=ops.portion_kinds(rows[lead:])) if hints else {}
    slots = [(3 * i + 1) % (len(rows) + 2) if (len(rows) + 2) % 3 else i for i in range(len(rows))]
    return nv.CacheContext(cu_seqlens_q=cu(rows), cu_seqlens_k=cu([r + n for r, n in zip(rows, before)]),
                           state_slots=torch.tensor(slots, dtype=torch.int32, device=DEV), **known)


def _layers(form, H, D, Dv, mk):
    if form == "gated":
        a, r = (m.GatedDeltaRule(H, H // 2, D, Dv, 1e-5, device=DEV) for m in (delta_rule, ref_mixer_modules))
    elif form == "general":
        a, r = (m.GeneralDeltaRule(H, D, 1e-5, device=DEV) for m in (general_delta, ref_benarax_modules))
    else:
        a, r = (m.GatedWriteMemory(H, D, Dv, 1e-5, device=DEV) for m in (gated_memory, ref_tutedra_modules))
    spread = torch.linspace(-6, 8, H * D, device=DEV)[torch.randperm(H * D, generator=torch.Generator().manual_seed(1)).to(DEV)]
    with torch.no_grad():
        a.norm_weight.copy_(1 + 0.3 * mk(a.norm_weight.numel()))
        if form == "gated":            # decays from exp(-0.02) to exp(-22) per token
            a.A_log.copy_(torch.linspace(-1, 1, H, device=DEV))
            a.dt_bias.copy_(spread)
        elif form == "general":
            a.w_bias.copy_(spread)
            a.a_bias.copy_(0.5 * mk(H * D))
        else:                          # forget gates from 0.997 to 4e-6
            a.f_bias.copy_(-2 * spread + 4)
            a.lower.copy_(torch.where(spread > 3, 0.0, 0.3) * torch.rand(H * D, device=DEV))
    r.load_state_dict(a.state_dict())
    return a, r


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("step", list(STEPS))
@pytest.mark.parametrize("form,D,Dv", [("gated", 128, 128), ("gated", 64, 80), ("gated", 96, 16), ("general", 128, 128),
                                       ("general", 64, 64), ("general", 32, 32), ("write", 128, 128), ("write", 32, 144),
                                       ("write", 40, 24)])
def test_portions(form, D, Dv, step, dtype):
    rows, before = STEPS[step]
    H, T = 4, sum(rows)
    g = torch.Generator(device=DEV).manual_seed(7 * D + Dv)
    mk = lambda *s: torch.randn(*s, generator=g, device=DEV)
    a, r = _layers(form, H, D, Dv, mk)
    G = H // 2 if form == "gated" else H
    q, k, v = mk(T, G, D).to(dtype), mk(T, H if form == "write" else G, D).to(dtype), mk(T, H, Dv + 8)[:, :, :Dv].contiguous().to(dtype)
    wide = mk(T, H * Dv + 1).to(dtype)
    gate = wide[:, 1:] if Dv == 80 else wide[:, :-1].contiguous()      # rows that do not start on 16 bytes
    w, rate, b = mk(T, H * D).to(dtype), mk(T, H * D).to(dtype), mk(T, H).to(dtype)
    if D == 64:                            # rows that start on any element
        w = mk(T, H * D + 1).to(dtype)[:, 1:]
    state = mk(len(rows) + 2, H, D, Dv)
    call = {"gated": lambda m, s: m(q, k, v, w, b, gate, s), "general": lambda m, s: m(q, k, v, w, rate, gate, s),
            "write": lambda m, s: m(q, k, v, {"state": s})}[form]
    nv.set_context(_context(rows, before, False))
    want_state = state.clone()
    want = call(r, want_state)
    # float32: sums of up to 128 products of order one taken in another order, read-outs divided by their root mean square;
    # bfloat16: one rounding of the output (2^-9 of values up to 8)
    tol = dict(rtol=5e-5, atol=5e-5) if dtype == torch.float32 else dict(rtol=1e-2, atol=2e-2)
    scale = want_state.abs().max().item()
    for hints in (True, False):
        nv.set_context(_context(rows, before, hints))
        got_state = state.clone()
        got = call(a, got_state)
        torch.cuda.synchronize()
        torch.testing.assert_close(got.float(), want.float(), **tol)
        torch.testing.assert_close(got_state, want_state, rtol=2e-5, atol=2e-6 * scale)
    nv.set_context(None)


def _operands(form, rows, before, H, D, Dv, dtype, seed, extra=0):
    """A layer, its eager stand-in, the raw projections by name and the states."""
    T = sum(rows)
    g = torch.Generator(device=DEV).manual_seed(seed)
    mk = lambda *s: torch.randn(*s, generator=g, device=DEV)
    a, r = _layers(form, H, D, Dv, mk)
    G = H // 2 if form == "gated" else H
    x = dict(q=mk(T, G, D), k=mk(T, G, D), v=mk(T, H, Dv), w=mk(T, H * D), a=mk(T, H * D), b=mk(T, H), gate=mk(T, H * Dv))
    return a, r, {n: t.to(dtype) for n, t in x.items()}, mk(len(rows) + 2, H, D, Dv)


def _forward(form, m, x, state):
    if form == "gated":
        return m(x["q"], x["k"], x["v"], x["w"], x["b"], x["gate"], state)
    if form == "general":
        return m(x["q"], x["k"], x["v"], x["w"], x["a"], x["gate"], state)
    return m(x["q"], x["k"], x["v"], {"state": state})


@pytest.mark.parametrize("entry", ["plain", "no_workspace", "no_rows"])
@pytest.mark.parametrize("form", ["gated", "general", "write"])
def test_entries_without_workspace(form, entry):
    """The C entries without portions, and those with portions but no workspace or an unknown number of rows, go token by token at
    sizes that have a launch in chunks too."""
    from nanovllm_amd import _lib
    rows, before = [1, 9, 30, 1], [4, 0, 7, 0]
    H, D, T = 4, 128, sum(rows)
    a, r, x, state = _operands(form, rows, before, H, D, D, torch.float32, 5)
    ctx = _context(rows, before, True)
    nv.set_context(ctx)
    want_state, got_state = state.clone(), state.clone()
    want = _forward(form, r, x, want_state)
    nv.set_context(None)
    out = torch.full((T, H * D), float("nan"), device=DEV)
    dll, p = _lib.mixers(), lambda t: t.data_ptr()
    q, k, v = (x[n] for n in "qkv")
    seqs = [p(ctx.cu_seqlens_q), p(ctx.cu_seqlens_k), p(ctx.state_slots), len(rows)]
    sizes = {"gated": [H, H // 2, D, D, 1e-5], "general": [H, D, 1e-5, getattr(a, "decay_rate", 0.0), getattr(a, "key_eps", 0.0)],
             "write": [H, D, D, 1e-5]}[form]
    head = [p(q), p(k), p(v), q.stride(0), k.stride(0), v.stride(0)]
    if form == "gated":
        head += [p(x["w"]), H * D, p(x["b"]), H, p(x["gate"]), H * D, p(a.A_log), p(a.dt_bias), p(a.norm_weight)]
    elif form == "general":
        head += [p(x["w"]), H * D, p(x["a"]), H * D, p(x["gate"]), H * D, p(a.w_bias), p(a.a_bias), p(a.norm_weight)]
    else:
        head += [p(a.f_bias), p(a.lower), p(a.norm_weight)]
    head += [p(got_state), p(out), H * D] + seqs
    name = {"gated": "nv_gated_delta_rule", "general": "nv_general_delta_rule", "write": "nv_gated_write_memory"}[form]
    dt, stream = ops._dt(q, "q"), ops._stream(q)
    if entry == "plain":
        rc = getattr(dll, name)(*head, *sizes, dt, stream)
    else:                                  # a workspace without the number of rows is not used
        ws = torch.empty(1 << 24, dtype=torch.uint8, device=DEV) if entry == "no_rows" else None
        rc = getattr(dll, name + "_portions")(*head, 0 if entry == "no_rows" else T, *sizes, 1, ops.portion_kinds(rows[1:]), dt,
                                              p(ws) if ws is not None else None, ws.numel() if ws is not None else 0, stream)
    _lib.check(rc, name, dll)
    torch.cuda.synchronize()
    torch.testing.assert_close(out, want, rtol=5e-5, atol=5e-5)          # (the bounds of test_portions)
    torch.testing.assert_close(got_state, want_state, rtol=2e-5, atol=2e-6 * want_state.abs().max().item())


@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("form,name", [("gated", "q"), ("gated", "k"), ("gated", "v"), ("gated", "w"), ("gated", "b"), ("gated", "gate"),
                                       ("general", "q"), ("general", "k"), ("general", "v"), ("general", "w"), ("general", "a"),
                                       ("write", "q"), ("write", "k"), ("write", "v")])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Dv", [16, 128])                               # two waves for a state's columns and one
def test_values_that_are_not_finite(form, name, value, dtype, Dv):
    """What is not finite in one token's row reaches that row and what comes after it, as token by token: no row in front of it,
    no other head, no other sequence; and what it makes finite (a gate fully open or closed) is finite."""
    Dv = 128 if form == "general" else Dv
    rows, before = [21, 9, 13], [0, 5, 0]
    if Dv == 128:
        rows, before = rows * 16, before * 16
    _strike(form, name, value, dtype, Dv, rows, before, 11)              # token 3 of the second chunk of 8 of the first sequence


@pytest.mark.parametrize("at", [0, 3, 7, 8, 15, 16])
@pytest.mark.parametrize("value", [float("nan"), float("-inf")])
@pytest.mark.parametrize("form,name", [("gated", "q"), ("gated", "k"), ("gated", "v"), ("gated", "w"), ("gated", "b"), ("general", "q"),
                                       ("general", "k"), ("general", "v"), ("general", "w"), ("general", "a"), ("write", "q"),
                                       ("write", "k"), ("write", "v")])
def test_values_that_are_not_finite_in_chunks_of_16(form, name, value, at):
    """The same in both halves of a chunk, at its ends and in front of the next one, for portions that run in chunks of 16."""
    _strike(form, name, value, torch.float32, 128, [130, 129, 128], [0, 5, 0], at)


@pytest.mark.parametrize("form,name,rows", [("gated", "k", 257), ("gated", "w", 257), ("write", "k", 130), ("write", "v", 130)])
def test_values_that_are_not_finite_in_chunks_of_16_one_wave(form, name, rows):
    _strike(form, name, float("nan"), torch.bfloat16, 128, [rows] * 17, [0, 5] * 8 + [0], 8)


def _strike(form, name, value, dtype, Dv, rows, before, at):
    H, D = 4, 128
    n, ctx = rows[0], _context(rows, before, True)
    a, r, x, state = _operands(form, rows, before, H, D, Dv, dtype, 9)
    nv.set_context(ctx)
    clean_state = state.clone()
    clean = _forward(form, a, x, clean_state)
    x[name] = x[name].clone()
    if x[name].dim() == 3:
        x[name][at, 0, 3] = value
    else:
        x[name][at, 3 if name != "b" else 0] = value                     # (b: one value per head)
    got_state = state.clone()
    got = _forward(form, a, x, got_state)
    slot = int(ctx.state_slots[0])
    others = [s for s in range(state.shape[0]) if s != slot]
    one = state[slot:slot + 1].clone()     # the first sequence alone through the stand-in
    ctx = _context(rows[:1], before[:1], True)
    ctx.state_slots = torch.zeros(1, dtype=torch.int32, device=DEV)
    nv.set_context(ctx)
    want = _forward(form, r, {k: t[:n] for k, t in x.items()}, one).detach()
    nv.set_context(None)
    heads = lambda t: t[:n].float().view(n, H, Dv)
    hit = 2 if form == "gated" and name in "qk" else 1                   # heads that share the row
    tol = dict(rtol=5e-5, atol=5e-5) if dtype == torch.float32 else dict(rtol=1e-2, atol=2e-2)       # (the bounds of test_portions)
    # (rows in front of it up to rounding: its decay is a factor of both sides of its chunk's pair products)
    torch.testing.assert_close(got[:at].float(), clean[:at].float(), **tol)
    assert torch.equal(got[n:], clean[n:])
    assert torch.equal(heads(got)[:, hit:], heads(clean)[:, hit:])
    assert torch.equal(got_state[others], clean_state[others])
    if name == "v" and abs(value) == float("inf"):
        # Its column of the state holds infinities of both signs: a read-out as a sum over them is NaN and its norm takes the row
        # along, one from the write's own product is infinite and leaves zeros beside it.  Only its own column counts.
        assert not heads(got)[at:, 0, 3].isfinite().any() and not heads(want)[at:, 0, 3].isfinite().any()
        got[at:n, :Dv] = want[at:, :Dv] = 0
    for g, w, tol in ((heads(got), heads(want), tol),
                      (got_state[slot], one[0], dict(rtol=2e-5, atol=2e-6 * clean_state.abs().max().item()))):
        ok = w.isfinite()
        assert torch.equal(g.isfinite(), ok)
        torch.testing.assert_close(g[ok], w[ok], **tol)


@pytest.mark.parametrize("rows,B", [(1, 32), (8, 32), (100, 2), (257, 32)])    # (the last two: chunks of 16, two waves and one)
def test_decays_keep_their_precision(rows, B):
    """A state that nothing is written to is its decays' product.  Against 64 bits the launches for known portions are no further off
    than the token-by-token entry: each decay is the rounding of its exponent's two sums and products, and of the exponential, on
    both sides, so their root-mean-square errors over 65536 channels agree within a few percent (softplus and exponential of
    single instructions: 1.35 and 1.24 times as far off)."""
    from nanovllm_amd import _lib
    H, D, Dv = 16, 128, 16
    T = B * rows
    g = torch.Generator(device=DEV).manual_seed(3)
    zero, v = torch.zeros(T, H, D, device=DEV), torch.zeros(T, H, Dv, device=DEV)
    raw, b, gate = 0.5 * torch.randn(T, H * D, generator=g, device=DEV), torch.zeros(T, H, device=DEV), torch.zeros(T, H * Dv, device=DEV)
    m = delta_rule.GatedDeltaRule(H, H, D, Dv, 1e-5, device=DEV)
    m.A_log.data.copy_(torch.linspace(1, 16, H, device=DEV).log())
    m.dt_bias.data.copy_(torch.linspace(-7, -2, H * D, device=DEV))
    log_w = -(m.A_log.double().exp()[:, None] * torch.log1p(torch.exp((raw.double() + m.dt_bias.double()).view(T, H, D))))
    want = torch.exp(log_w.view(B, rows, H, D).sum(1))
    ctx = _context([rows] * B, [1] * B, True)
    ctx.state_slots = torch.arange(B, dtype=torch.int32, device=DEV)
    off = []
    for known in (True, False):
        got = torch.ones(B, H, D, Dv, device=DEV)
        if known:
            nv.set_context(ctx)
            m(zero, zero, v, raw, b, gate, got)
            nv.set_context(None)
        else:
            p, dll = lambda t: t.data_ptr(), _lib.mixers()
            out = torch.empty(T, H * Dv, device=DEV)
            rc = dll.nv_gated_delta_rule(p(zero), p(zero), p(v), H * D, H * D, H * Dv, p(raw), H * D, p(b), H, p(gate), H * Dv, p(m.A_log),
                                         p(m.dt_bias), p(m.norm_weight), p(got), p(out), H * Dv, p(ctx.cu_seqlens_q),
                                         p(ctx.cu_seqlens_k), p(ctx.state_slots), B, H, H, D, Dv, 1e-5, ops._dt(v, "v"), ops._stream(v))
            _lib.check(rc, "nv_gated_delta_rule", dll)
        torch.cuda.synchronize()
        assert torch.equal(got, got[..., :1].expand_as(got))
        big = want > 1e-30
        off.append((((got[..., 0].double() - want) / want)[big] ** 2).mean().sqrt().item())
    assert off[0] <= 1.1 * off[1], off


@pytest.mark.parametrize("at", range(8, 16))
@pytest.mark.parametrize("form", ["gated", "general", "write"])
def test_total_decay_behind_large_values(form, at):
    """A token whose decays forget everything sees nothing of what was written before it, also within its chunk and however large
    that was: its factors are below any that the pair products could divide by."""
    _forget(form, at, [24, 13])


@pytest.mark.parametrize("at", [3, 7, 8, 15, 16, 17])
@pytest.mark.parametrize("form", ["gated", "general", "write"])
def test_total_decay_behind_large_values_in_chunks_of_16(form, at):
    _forget(form, at, [130, 129])


def _forget(form, at, rows):
    H, D, before = 4, 128, [0, 3]
    a, r, x, state = _operands(form, rows, before, H, D, D, torch.float32, 13)
    for m in (a, r):
        if form == "gated":
            m.A_log.data.zero_()
            m.dt_bias.data.fill_(-8.0)
        elif form == "general":
            m.decay_rate = 60.0
            m.w_bias.data.zero_()
        else:
            m.lower.data.zero_()
            m.f_bias.data.zero_()
    keep, forget = {"gated": (0.0, 60.0), "general": (-12.0, 12.0), "write": (1.0, -60.0)}[form]
    decay = x["k"] if form == "write" else x["w"]
    decay.mul_(0.1).add_(keep)
    decay[at] = forget
    x["a"][at] = -60.0                             # (general: nothing of the old state is moved either)
    x["v"][:at] *= 1e6
    got_state, want_state = state.clone(), state.clone()
    nv.set_context(_context(rows, before, True))
    want, got = _forward(form, r, x, want_state), _forward(form, a, x, got_state)
    nv.set_context(None)
    torch.testing.assert_close(got, want, rtol=5e-5, atol=5e-5)          # (the bounds of test_portions)
    # (about 110 writes behind it add up to more than the states before: each is rounded at the sum's size, as in test_portions)
    scale = max(state.abs().max().item(), want_state.abs().max().item() if max(rows) > 100 else 0.0)
    torch.testing.assert_close(got_state, want_state, rtol=2e-5, atol=2e-6 * scale)


def test_read_outs_keep_their_precision():
    """Read-outs of float32 rows against 64 bits, in a portion of one chunk: both launches sum 128 products with about 32 roundings
    one after the other, so the chunk's error is that of the token-by-token entry and of the few sums over its tokens (measured:
    1.11 times; with one sum over all key channels 1.62 times)."""
    from nanovllm_amd import _lib
    B, rows, H, D, Dv = 16, 8, 16, 128, 128
    T = B * rows
    g = torch.Generator(device=DEV).manual_seed(11)
    mk = lambda *s: torch.randn(*s, generator=g, device=DEV)
    m = delta_rule.GatedDeltaRule(H, H, D, Dv, 1e-5, device=DEV)
    m.A_log.data.copy_(torch.linspace(1, 16, H, device=DEV).log())
    m.dt_bias.data.copy_(torch.linspace(-7, -2, H * D, device=DEV))
    q, k, v, raw, b, gate = mk(T, H, D), mk(T, H, D), mk(T, H, Dv), 0.5 * mk(T, H * D), mk(T, H), mk(T, H * Dv)
    state = 0.3 * mk(B, H, D, Dv)
    # the same in 64 bits
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
    seqs = lambda t, *s: t.double().view(B, rows, H, *s)
    w = torch.exp(-m.A_log.double().exp()[:, None] * torch.log1p(torch.exp(seqs(raw, D) + m.dt_bias.double().view(H, D))))
    k64, q64, v64, beta = unit(seqs(k, D)), unit(seqs(q, D)) * D ** -0.5, seqs(v, Dv), torch.sigmoid(seqs(b))
    S, o = state.double(), []
    for t in range(rows):
        S = S * w[:, t, :, :, None]
        u = (v64[:, t] - (S * k64[:, t, :, :, None]).sum(2)) * beta[:, t, :, None]
        S = S + k64[:, t, :, :, None] * u[:, :, None]
        o.append((S * q64[:, t, :, :, None]).sum(2))
    o = torch.stack(o, 1)
    want = (o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5) * torch.sigmoid(seqs(gate, Dv))).view(T, H * Dv)
    ctx = _context([rows] * B, [1] * B, True)
    ctx.state_slots = torch.arange(B, dtype=torch.int32, device=DEV)
    nv.set_context(ctx)
    got = m(q, k, v, raw, b, gate, state.clone()).detach()
    nv.set_context(None)
    p, dll, tokens, st = lambda t: t.data_ptr(), _lib.mixers(), torch.empty(T, H * Dv, device=DEV), state.clone()
    rc = dll.nv_gated_delta_rule(p(q), p(k), p(v), H * D, H * D, H * Dv, p(raw), H * D, p(b), H, p(gate), H * Dv, p(m.A_log), p(m.dt_bias),
                                 p(m.norm_weight), p(st), p(tokens), H * Dv, p(ctx.cu_seqlens_q), p(ctx.cu_seqlens_k), p(ctx.state_slots),
                                 B, H, H, D, Dv, 1e-5, ops._dt(v, "v"), ops._stream(v))
    _lib.check(rc, "nv_gated_delta_rule", dll)
    torch.cuda.synchronize()
    off = [((x.double() - want).norm() / want.norm()).item() for x in (got, tokens)]
    assert off[0] <= 1.35 * off[1], off


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form,D,Dv", [("gated", 128, 128), ("gated", 96, 48), ("gated", 32, 80), ("general", 128, 128), ("general", 96, 96),
                                       ("write", 96, 144), ("write", 64, 16)])
@pytest.mark.parametrize("rows", [[900, 15, 16, 17, 31, 32, 33, 48], [15, 16, 17, 31, 32, 33, 48], [24] * 40], ids=["edges", "edges_of_8", "many"])
def test_chunks_of_16(form, D, Dv, rows, dtype):
    """Around the chunk of 16 tokens and its halves (edges; the long portion makes it the step's chunk), and at the same rows in chunks of
    8, carried and fresh states.  The bounds are those of test_portions: the same sums, of up to 128 products and 16 tokens, in another
    order."""
    _compare_portions(form, D, Dv, rows, 2 if rows[0] == 900 else 4, dtype)


@pytest.mark.parametrize("form,D,Dv,rows", [("gated", 128, 128, [300, 220] * 10), ("gated", 96, 48, [400, 300] * 18), ("write", 128, 128, [150, 129] * 9),
                                            ("write", 64, 16, [150, 129] * 33)])
def test_chunks_of_16_one_wave(form, D, Dv, rows):
    """Steps that fill the chip: one wave for a state's columns."""
    _compare_portions(form, D, Dv, rows, 4, torch.bfloat16)


def _compare_portions(form, D, Dv, rows, H, dtype):
    before = [5 * (i % 3) for i in range(len(rows))]
    a, r, x, state = _operands(form, rows, before, H, D, Dv, dtype, 11)
    nv.set_context(_context(rows, before, False))
    want_state = state.clone()
    want = _forward(form, r, x, want_state)
    nv.set_context(_context(rows, before, True))
    got = _forward(form, a, x, state)
    nv.set_context(None)
    tol = dict(rtol=5e-5, atol=5e-5) if dtype == torch.float32 else dict(rtol=1e-2, atol=2e-2)
    torch.testing.assert_close(got.float(), want.float(), **tol)
    torch.testing.assert_close(state, want_state, rtol=2e-5, atol=2e-6 * want_state.abs().max().item())


def _in_64_bits(form, m, x, state, B, rows):
    """The same call in 64 bits: B sequences of `rows` rows each that continue the first B states."""
    H, D, Dv = state.shape[1:]
    seqs = lambda t: t.double().view(B, rows, H, -1)
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
    heads = lambda t: t.repeat_interleave(H // t.shape[1], 1)
    q, k, v, S, o, gate = seqs(heads(x["q"])), seqs(heads(x["k"])), seqs(x["v"]), state[:B].double(), [], torch.sigmoid(seqs(x["gate"]))
    raw = seqs(x["w"])
    read = lambda S, t: (S * t[..., None]).sum(2)
    if form == "gated":
        q, k, beta = unit(q) * D ** -0.5, unit(k), torch.sigmoid(seqs(x["b"]))
        w = torch.exp(-m.A_log.double().exp()[:, None] * torch.nn.functional.softplus(raw + m.dt_bias.double().view(H, D)))
    elif form == "general":
        u = unit(k)
        w = torch.exp(-m.decay_rate * torch.sigmoid(raw + m.w_bias.double().view(H, D)))
        a = torch.sigmoid(seqs(x["a"]) + m.a_bias.double().view(H, D)) * u
    else:
        lower, gate = m.lower.double().view(H, D), 1.0
        w = lower + (1 - lower) * torch.sigmoid(k + m.f_bias.double().view(H, D))
        q, k = torch.nn.functional.silu(q), 1 - w
    for t in range(rows):
        old, S = S, S * w[:, t, :, :, None]
        if form == "gated":
            S = S + k[:, t, :, :, None] * (beta[:, t] * (v[:, t] - read(S, k[:, t])))[:, :, None]
        else:
            S = S + k[:, t, :, :, None] * v[:, t, :, None]
        if form == "general":
            S = S - a[:, t, :, :, None] * read(old, u[:, t])[:, :, None]
        o.append(read(S, q[:, t]))
    o = torch.stack(o, 1)
    weight = m.norm_weight.double().view(-1, Dv)
    return (o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5) * weight * gate).view(B * rows, H * Dv), S


# Bounds of (read-outs, states).  Measured at 33 .. 257 rows: 0.95 to 1.03 and 0.89 to 0.96 (gated), 0.98 to 1.02 and 0.90 to 0.95 (general),
# 0.99 to 1.02 and 0.99 (write); at 33 and 70 rows with decays multiplied in 32 bits, pair products in four sums and removals on top of the
# state: up to 1.09 and 0.97, 1.16 and 1.30, 1.05 and 1.005.
OFF = {"gated": (1.05, 1.0), "general": (1.05, 1.0), "write": (1.035, 1.0)}


@pytest.mark.parametrize("form,B,rows", [("gated", 2, 97), ("gated", 16, 257), ("general", 2, 129), ("general", 2, 144), ("write", 2, 33),
                                         ("write", 16, 129)])          # two waves for a state's columns and (B = 16) one
def test_long_portions_keep_their_precision(monkeypatch, form, B, rows):
    """Float32 rows over carried states against 64 bits, relative to the token-by-token launch: a chunk takes the same sums in another
    order."""
    H, D, before = 8, 128, [1] * B
    a, _, x, state = _operands(form, [rows] * B, before, H, D, D, torch.float32, 21)
    with torch.no_grad():                  # decays of trained layers: exp(-0.001) .. exp(-1.6) a token
        if form == "gated":
            a.A_log.copy_(torch.linspace(1, 16, H, device=DEV).log())
            a.dt_bias.copy_(torch.linspace(-7, -2, H * D, device=DEV))
        elif form == "general":
            a.w_bias.copy_(torch.linspace(-4, 0, H * D, device=DEV))
            a.a_bias.mul_(0.5)
            x["k"].mul_(0.5)
        else:
            a.f_bias.copy_(torch.linspace(0, 4, H * D, device=DEV))
            a.lower.copy_(torch.linspace(0, 0.9, H * D, device=DEV))
    x["w"].mul_(0.5)
    state.mul_(0.3)
    ctx = _context([rows] * B, before, True)
    ctx.state_slots = torch.arange(B, dtype=torch.int32, device=DEV)
    want = _in_64_bits(form, a, x, state, B, rows)
    nv.set_context(ctx)
    off = []
    for tokens in (False, True):
        if tokens:
            monkeypatch.setattr(ops, "_portions", lambda *args: (0, 7, None))
        got = state.clone()
        out = _forward(form, a, x, got)
        off.append([((g.double() - w).norm() / w.norm()).item() for g, w in ((out, want[0]), (got[:B], want[1]))])
    nv.set_context(None)
    ratio = [c / t for c, t in zip(*off)]
    assert all(r <= bound for r, bound in zip(ratio, OFF[form])), (ratio, off)


@pytest.mark.parametrize("rate", [6.5, 7.5, 13.0, 14.5])
@pytest.mark.parametrize("rows", [[130, 129], [17, 8]], ids=["chunks_of_16", "chunks_of_8"])
@pytest.mark.parametrize("form", ["gated", "general", "write"])
def test_fast_decays(form, rows, rate):
    """Channels that decay by about exp(-rate) a token beside slow ones, on both sides of where eight (6.9) and four (13.9) factors
    multiply to 2^-80 and the chunk's pairs are taken in more sets."""
    H, D, before = 4, 128, [0, 3]
    a, r, x, state = _operands(form, rows, before, H, D, D, torch.float32, 17)
    fast = (torch.arange(H * D, device=DEV) % 5 == 0).float() * rate
    for m in (a, r):
        if form == "gated":
            m.A_log.data.zero_()
            m.dt_bias.data.copy_(torch.expm1(fast + 0.02).log())
        elif form == "general":
            m.decay_rate = rate
            m.w_bias.data.copy_(torch.where(fast > 0, 20.0, -8.0))
        else:
            m.lower.data.zero_()
            m.f_bias.data.copy_(3.0 - fast)
    x["k" if form == "write" else "w"].mul_(0.02)
    got_state, want_state = state.clone(), state.clone()
    nv.set_context(_context(rows, before, True))
    want, got = _forward(form, r, x, want_state), _forward(form, a, x, got_state)
    nv.set_context(None)
    torch.testing.assert_close(got, want, rtol=5e-5, atol=5e-5)          # (the bounds of test_portions)
    torch.testing.assert_close(got_state, want_state, rtol=2e-5, atol=2e-6 * want_state.abs().max().item())


@pytest.mark.parametrize("form,H,D,Dv,seqs", [("gated", 16, 128, 128, 96), ("general", 16, 128, 128, 93), ("write", 16, 64, 64, 400),
                                              ("gated", 8, 96, 80, 400), ("write", 4, 32, 32, 6000)])
def test_single_tokens_of_more_states_than_the_cache_keeps(form, H, D, Dv, seqs):
    """Launches of single tokens whose states pass by the caches against the same sequences in launches of half as many, whose states do not:
    the same bits, fresh states among carried ones, and no other state is touched."""
    assert seqs * H * D * Dv * 4 >= 92 << 20 > seqs // 2 * H * D * Dv * 4
    g = torch.Generator(device=DEV).manual_seed(D + seqs)
    mk = lambda *s: torch.randn(*s, generator=g, device=DEV)
    a, _ = _layers(form, H, D, Dv, mk)
    G = H // 2 if form == "gated" else H
    q, k, v = (x.to(torch.bfloat16) for x in (mk(seqs, G, D), mk(seqs, H if form == "write" else G, D), mk(seqs, H, Dv)))
    gate, w, rate, b = (x.to(torch.bfloat16) for x in (mk(seqs, H * Dv), mk(seqs, H * D), mk(seqs, H * D), mk(seqs, H)))
    state = mk(seqs + 3, H, D, Dv)
    slots = torch.randperm(seqs + 3, generator=g, device=DEV)[:seqs].to(torch.int32)

    def run(lo, hi, state):
        n = hi - lo
        cu = torch.arange(n + 1, dtype=torch.int32, device=DEV)
        before = torch.tensor([0 if i % 7 == 3 else 5 for i in range(lo, hi)])
        cu_k = torch.tensor([0] + (1 + before).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
        nv.set_context(nv.CacheContext(cu_seqlens_q=cu, cu_seqlens_k=cu_k, state_slots=slots[lo:hi].contiguous(), max_seqlen_q=1, num_leading_decode=n,
                                       portion_kinds=ops.portion_kinds([])))
        at = slice(lo, hi)
        if form == "gated":
            out = a(q[at], k[at], v[at], w[at], b[at], gate[at], state)
        elif form == "general":
            out = a(q[at], k[at], v[at], w[at], rate[at], gate[at], state)
        else:
            out = a(q[at], k[at], v[at], {"state": state})
        nv.set_context(None)
        return out

    one, two = state.clone(), state.clone()
    out = run(0, seqs, one)
    parts = torch.cat([run(0, seqs // 2, two), run(seqs // 2, seqs, two)])
    assert torch.equal(out, parts) and torch.equal(one, two) and not torch.equal(one, state)
