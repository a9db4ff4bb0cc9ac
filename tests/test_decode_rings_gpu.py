"""Single tokens' attention with keys and values on their way to LDS: contexts at the edges of steps, waves and rings, keys that are
split or not, a block or more a CU, masks, and the gate behind the heads, against the plain operation."""
from types import SimpleNamespace

import pytest
import torch

from emu_ops import EmuOps
from test_kernels_gpu import DEV, _attention_case, _ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,d,page", [(6, 2, 128, 16), (8, 1, 64, 64), (34, 2, 64, 16), (3, 3, 32, 32), (4, 4, 128, 128)])
@pytest.mark.parametrize("ctx", [[1, 31, 32, 33], [255, 256, 257], [511, 512, 64, 481], [513, 2049, 17], [1500]])
def test_edges(heads, kv, d, page, ctx):
    """Waves with no step, one, or one more than their neighbours; the last key alone in its step, its half or its page; what lies
    behind the last key is not finite."""
    for window in (0, 13, 300):
        got = _attention_case(torch.bfloat16, heads, kv, d, page, [1] * len(ctx), ctx, window, seed=len(ctx) + d, poison=True)
        assert bool(torch.isfinite(got.float()).all())


@pytest.mark.parametrize("heads,kv,n,longest", [(16, 8, 12, 900), (16, 8, 12, 2100), (16, 8, 30, 700), (8, 8, 45, 400)])
def test_many_requests(heads, kv, n, longest):
    """65 to 128, 129 to 256 and more blocks a split, contexts from a few keys on; beside a portion as well."""
    ctx = [1 + i * (longest - 1) // (n - 1) for i in range(n)]
    _attention_case(torch.bfloat16, heads, kv, 64, 16, [1] * n, ctx, 0, seed=n, poison=True)
    _attention_case(torch.bfloat16, heads, kv, 64, 16, [1] * (n - 1) + [40], ctx, 0, seed=n, poison=True)


@pytest.mark.parametrize("ctx,page", [(300, 16), (1500, 16), (300, 8)])
@pytest.mark.parametrize("per", [1, 64])
def test_gate_behind_the_heads(ctx, page, per):
    """The gate by the kernel that writes a row (keys split or not, ring or registers): the bits of its own kernel."""
    ops = _ops()
    g = torch.Generator().manual_seed(ctx + per)
    heads, kv, d, n = 4, 2, 64, 3
    pages = -(-ctx // page)
    bt = torch.randperm(n * pages, generator=g).to(torch.int32).view(n, pages).to(DEV)
    k = torch.randn(n * pages, kv, page, d, generator=g).to(DEV).bfloat16()
    v = torch.randn(n * pages, kv, d, page, generator=g).to(DEV).bfloat16()
    q = torch.randn(n, heads, d, generator=g).to(DEV).bfloat16()
    cu = torch.arange(n + 1, dtype=torch.int32, device=DEV)
    cl = torch.tensor([ctx, ctx - 40, 7], dtype=torch.int32, device=DEV)
    rows = torch.randn(n, 5 + heads * d, generator=g).to(DEV)
    args = (q, k, v, bt, cu, cl, cu[:n], d ** -0.5, 0, 1, ctx, n)
    plain = ops.paged_attention(*args)
    for gate in (rows, None):
        want, got = (torch.zeros(n, heads * d + 8, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        ops.sigmoid_gate(plain, gate, 5, 0.75, want, 8, per)
        assert ops.paged_attention(*args, into=(gate, 5, 0.75, got, 8, per)) is None
        assert torch.equal(got, want)


def _step(ctx_lens, kv, d, page, g):
    """A step of one token for each request: what the parts read of it, and caches with every earlier key in place."""
    n, width = len(ctx_lens), -(-max(ctx_lens) // page) + 1
    tables = torch.randperm(n * width, generator=g).to(torch.int32).view(n, width)
    cl = torch.tensor(ctx_lens, dtype=torch.int32)
    slots = torch.stack([tables[i, (c - 1) // page] * page + (c - 1) % page for i, c in enumerate(ctx_lens)]).to(torch.int32)
    ctx = SimpleNamespace(num_tokens=n, num_requests=n, num_single=n, max_q_len=1, max_context_len=max(ctx_lens), positions=(cl - 1).to(DEV),
                          context_lens=cl.to(DEV), cu_seqlens=torch.arange(n + 1, dtype=torch.int32, device=DEV), block_tables=[tables.to(DEV)],
                          slot_mapping=[slots.to(DEV)], state_slots=torch.randperm(n + 2, generator=g)[:n].to(torch.int32).to(DEV))
    ctx.token_req = ctx.cu_seqlens[:n]
    k = torch.randn(n * width, kv, page, d, generator=g).to(DEV).bfloat16()
    v = torch.randn(n * width, kv, d, page, generator=g).to(DEV).bfloat16()
    return ctx, k, v


@pytest.mark.parametrize("heads,kv,d,page", [(6, 2, 128, 16), (8, 8, 64, 32), (16, 1, 64, 16)])
@pytest.mark.parametrize("ctx_lens", [[1, 2, 31, 32, 33, 64, 65], [257, 16, 17, 300], [2000, 700, 1]])
@pytest.mark.parametrize("how", ["plain", "partials", "conv", "norms", "gate", "half"])
def test_attention_from_the_projections_rows(heads, kv, d, page, ctx_lens, how):
    """One launch against the kernels it stands for: the same cache, carried inputs and outputs, bit for bit; a norm per head sums its
    squares in another order, which may move a rounding to bfloat16."""
    ops = _ops()
    g = torch.Generator().manual_seed(heads + d + len(ctx_lens))
    ctx, k, v = _step(ctx_lens, kv, d, page, g)
    n, width, col0 = len(ctx_lens), (heads + 2 * kv) * d, 0 if how == "partials" else 6
    rows = torch.randn(3 if how == "partials" else 1, n, width + col0, generator=g).to(DEV)
    freq = (10000.0 ** -torch.arange(0, 1, 2.0 / d, dtype=torch.float64)).to(DEV)
    rotary = d // 2 if how == "half" else d
    freq = freq[: rotary // 2].contiguous()
    table = ops.rope_table(ctx.positions, freq, rotary, 1.25) if how == "conv" else None
    taps, norms = 3, tuple(torch.rand(d, generator=g).add(0.5).to(DEV) for _ in "qk") if how == "norms" else None
    conv_w = torch.randn(taps, width, generator=g).to(DEV)
    state = torch.randn(n + 2, 4 + (taps - 1) * width, generator=g).to(DEV)
    gate = torch.randn(n, heads * d, generator=g).to(DEV)
    if not ops.attention_rows_ok(rows[0], ctx, heads, kv, d, d, k, taps if how == "conv" else 0):
        assert how == "conv" and max(ctx_lens) > 1024
        pytest.skip("keys that are split keep the convolution's own launch")
    k2, v2, state2 = k.clone(), v.clone(), state.clone()
    if how == "partials":
        given = ops.Partials(rows)
        plain = ops.Partials(rows.clone())
    else:
        given, plain = rows[0], rows[0, :, col0:].contiguous()
    if how == "conv":
        plain = ops.causal_conv(plain, 0, width, conv_w, None, state2, ctx.cu_seqlens, ctx.token_req, ctx.state_slots, n, state_off=4, act=False, max_run=1)
    if how == "norms":
        ops.head_rmsnorm(plain, 0, heads, norms[0], heads * d, kv, norms[1], d, 1e-6)
    q = ops.rope_kv_write(plain, ctx.positions, ctx.slot_mapping[0], freq, rotary, 1.25, heads, kv, d, k2, v2, torch.bfloat16, table)
    window, scale = (40 if how == "half" else 0), d ** -0.5
    args = (q, k2, v2, ctx.block_tables[0], ctx.cu_seqlens, ctx.context_lens, ctx.token_req, scale, window, 1, ctx.max_context_len, n)
    into = [torch.zeros(n, heads * d, dtype=torch.bfloat16, device=DEV) for _ in "ab"]
    want = ops.paged_attention(*args, into=(gate, 0, 0.5, into[0], 0, 1) if how == "gate" else None)
    got = ops.attention_rows(given, col0, ctx, 0, heads, kv, d, k, v, scale, freq, rotary, 1.25, table, window, norms=norms, norm_eps=1e-6,
                             conv=(conv_w, state, 4) if how == "conv" else None, into=(gate, 0, 0.5, into[1], 0, 1) if how == "gate" else None)
    if how == "gate":
        want, got = into
    assert torch.equal(v, v2) and torch.equal(state, state2)
    if how == "norms":
        assert float((k.float() - k2.float()).abs().max()) <= 2.0 ** -8 * float(k2.float().abs().max())
        assert float((got.float() - want.float()).norm()) <= 2.0 ** -8 * float(want.float().norm())
    else:
        assert torch.equal(k, k2) and torch.equal(got, want)


@pytest.mark.parametrize("d,kv", [(64, 2), (128, 4)])
@pytest.mark.parametrize("ctx_lens", [[3, 200], [1, 700, 900, 33], [2500]])
@pytest.mark.parametrize("kind,n_step,dim,vdim", [("delta", 3, 64, 64), ("delta", 2, 128, 100), ("linear", 3, 64, 128), ("linear", 2, 100, 72)])
def test_a_step_beside_the_attention(d, kv, ctx_lens, kind, n_step, dim, vdim):
    """A recurrent mixer's step in the attention's launch: the bits of both launches, outputs and states alike."""
    ops = _ops()
    g = torch.Generator().manual_seed(d + dim + len(ctx_lens))
    ctx, k, v = _step(ctx_lens, kv, d, 16, g)
    n, heads, width = len(ctx_lens), 2 * kv, 4 * kv * d
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)
    rows, (hd, hv), rank, taps = rnd(n, width), (n_step * dim, n_step * vdim), 33, 4
    channels = 2 * hd + hv
    proj = rnd(n, (2 * channels + 2 * rank + 3) // 4 * 4)
    off = (taps - 1) * channels
    state = rnd(n + 2, (off + hd * vdim + 3) // 4 * 4)
    w2, b, nw, a_log, cw = rnd(rank, hd) * 0.3, rnd(hd) - 2.0, rnd(vdim), rnd(n_step), rnd(taps, channels)
    g2, out_col0 = rnd(rank, hv), heads * d

    def step(state, out, prepared=None):
        where = (state, 0, off) if kind == "delta" else (state, off)
        if kind == "delta":
            ops.delta_step(proj, 0, channels, channels + n_step, channels + n_step + rank, cw, w2, g2, a_log, b, nw, *where, ctx.token_req, ctx.state_slots,
                           n_step, dim, vdim, dim ** -0.5, 1e-6, 1e-6, 1.3, out, out_col0, prepared)
        else:
            ops.linear_step((proj, 0), (proj, hd), (proj, 2 * hd), (proj, 2 * hd + 2 * hv), w2, "root_sigmoid", b, 0.06, None, None, 0.3,
                            (proj, 2 * hd + hv), nw, 1e-6, 1.3, *where, ctx.token_req, ctx.state_slots, n_step, dim, vdim, out, out_col0, prepared)

    def attend(out, beside=None):
        kk, vv = k.clone(), v.clone()
        ops.attention_rows(rows, 0, ctx, 0, heads, kv, d, kk, vv, d ** -0.5, None, 0, 1.0, None, into=(None, 0, 0.75, out, 0, 1), beside=beside)
        return kk, vv
    assert ops.attention_beside_ok(ctx, heads, kv, 0, 0, n_step)
    outs, states, caches = [torch.zeros(n, heads * d + hv, dtype=torch.bfloat16, device=DEV) for _ in "ab"], [state.clone(), state.clone()], []
    force = ops.decode_force_splits
    try:
        ops.decode_force_splits = ops._rows_splits(ctx, heads, kv, 0, 0, 0, False, True)      # (the same parts of the keys both ways)
        step(states[0], outs[0])
        caches.append(attend(outs[0]))
        ops.decode_force_splits = 2 * ops.decode_force_splits if ops.decode_force_splits > 1 else 1
        buffer = ops.step_buffer()
        step(states[1], outs[1], buffer)
        caches.append(attend(outs[1], buffer))
    finally:
        ops.decode_force_splits = force
    assert torch.equal(outs[0][:, out_col0:], outs[1][:, out_col0:]) and torch.equal(states[0], states[1])
    assert all(torch.equal(a, c) for a, c in zip(*caches))
    # (the attention's sums by eight waves here and by four there where the keys are split)
    assert float((outs[0][:, :out_col0].float() - outs[1][:, :out_col0].float()).norm()) <= 2.0 ** -8 * float(outs[0][:, :out_col0].float().norm())


def _from_rows_and_apart(ops, ctx, rows, heads, kv, d, k, v, g, conv_state=None, norms=None, rotary=0, **mask):
    """(launches apart, one launch): outputs and caches of ``attention_rows`` and of the kernels that it stands for."""
    width, n = (heads + 2 * kv) * d, ctx.num_tokens
    freq = (10000.0 ** -torch.arange(0, 1, 2.0 / max(2, rotary), dtype=torch.float64))[: rotary // 2].contiguous().to(DEV)
    k2, v2, plain, conv = k.clone(), v.clone(), rows.clone(), None
    if conv_state is not None:
        state, off, taps = conv_state
        conv_w, state2 = torch.randn(taps, width, generator=g).to(DEV), state.clone()
        plain = ops.causal_conv(plain, 0, width, conv_w, None, state2, ctx.cu_seqlens, ctx.token_req, ctx.state_slots, n, state_off=off, act=False, max_run=1)
        conv = (conv_w, state, off)
    if norms is not None:
        ops.head_rmsnorm(plain, 0, heads, norms[0], heads * d, kv, norms[1], d, 1e-6)
    q = ops.rope_kv_write(plain, ctx.positions, ctx.slot_mapping[0], freq if rotary else None, rotary, 1.0, heads, kv, d, k2, v2, torch.bfloat16)
    want = ops.paged_attention(q, k2, v2, ctx.block_tables[0], ctx.cu_seqlens, ctx.context_lens, ctx.token_req, d ** -0.5, mask.get("window", 0), 1,
                               ctx.max_context_len, n, sink=mask.get("sink"), keep_first=mask.get("keep_first", 0), chunk=mask.get("chunk", 0))
    got = ops.attention_rows(rows, 0, ctx, 0, heads, kv, d, k, v, d ** -0.5, freq if rotary else None, rotary, 1.0, None, norms=norms, norm_eps=1e-6,
                             conv=conv, **mask)
    if conv is not None:
        assert torch.equal(state, state2)
    return (want, k2, v2), (got, k, v)


@pytest.mark.parametrize("heads,kv,d", [(6, 2, 128), (8, 8, 64)])
@pytest.mark.parametrize("ctx_lens", [[1, 33, 40, 47, 300], [2000, 700, 64, 1]])
@pytest.mark.parametrize("mask", [{"sink": True}, {"window": 40, "keep_first": 7}, {"window": 700, "keep_first": 40, "sink": True}, {"chunk": 48}, {"chunk": 1},
                                  {"chunk": 700, "sink": True}])
def test_masks_from_the_projections_rows(heads, kv, d, ctx_lens, mask):
    """A sink, kept first keys and chunks, keys split or not: bit for bit."""
    ops = _ops()
    g = torch.Generator().manual_seed(heads + d + len(ctx_lens))
    ctx, k, v = _step(ctx_lens, kv, d, 16, g)
    rows = torch.randn(len(ctx_lens), (heads + 2 * kv) * d, generator=g).to(DEV)
    assert ops.attention_rows_ok(rows, ctx, heads, kv, d, d, k)
    more = {**mask, **({"sink": torch.randn(heads, generator=g).to(DEV)} if "sink" in mask else {})}
    for want, got in zip(*_from_rows_and_apart(ops, ctx, rows, heads, kv, d, k, v, g, rotary=d, **more)):
        assert torch.equal(want, got)


@pytest.mark.parametrize("n,heads,kv", [(9, 8, 8), (70, 2, 1)])
def test_a_convolution_in_front_of_many_long_requests(n, heads, kv):
    """More than 64 blocks and more than 1,024 keys: the keys stay whole, in blocks of eight waves and of four."""
    ops = _ops()
    g = torch.Generator().manual_seed(n)
    d, taps = 64, 4
    ctx, k, v = _step([1 + i * 1500 // (n - 1) for i in range(n)], kv, d, 16, g)
    width = (heads + 2 * kv) * d
    rows = torch.randn(n, width, generator=g).to(DEV)
    state = torch.randn(n + 2, 6 + (taps - 1) * width, generator=g).to(DEV)
    assert ops.attention_rows_ok(rows, ctx, heads, kv, d, d, k, taps, 0, 0, state, 6)
    one = _from_rows_and_apart(ops, ctx, rows, heads, kv, d, k, v, g, conv_state=(state, 6, taps), rotary=32)
    assert torch.equal(one[0][1], one[1][1]) and torch.equal(one[0][2], one[1][2])
    # (apart the keys are cut into splits: sums of float32 in another order, then a rounding to bfloat16)
    assert float((one[0][0].float() - one[1][0].float()).norm()) <= 2.0 ** -8 * float(one[0][0].float().norm())


@pytest.mark.parametrize("kind,n_step,dim,vdim", [("delta", 3, 64, 64), ("linear", 2, 100, 72)])
@pytest.mark.parametrize("how", ["convolution", "norms and rotation"])
def test_a_step_beside_what_an_attention_brings(kind, n_step, dim, vdim, how):
    """Beside an attention with a convolution, whose carried inputs lie in the state rows of the step, and beside one with a norm per head and
    a rotation: outputs, states and caches bit for bit those of two launches."""
    ops = _ops()
    d, kv, ctx_lens = 64, 2, [1, 700, 900, 33]
    g = torch.Generator().manual_seed(dim + len(how))
    ctx, k, v = _step(ctx_lens, kv, d, 16, g)
    n, heads, width = len(ctx_lens), 2 * kv, 4 * kv * d
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)
    rows, (hd, hv), rank, taps = rnd(n, width), (n_step * dim, n_step * vdim), 33, 4
    channels, front = 2 * hd + hv, 3 * width
    proj = rnd(n, (2 * channels + 2 * rank + 3) // 4 * 4)
    off = front + (taps - 1) * channels
    state0 = rnd(n + 2, (off + hd * vdim + 3) // 4 * 4)
    w2, b, nw, a_log, cw, g2 = rnd(rank, hd) * 0.3, rnd(hd) - 2.0, rnd(vdim), rnd(n_step), rnd(taps, channels), rnd(rank, hv)
    conv_w, norms = rnd(4, width), tuple(torch.rand(d, generator=g).add(0.5).to(DEV) for _ in "qk")
    freq = (10000.0 ** -torch.arange(0, 1, 2.0 / d, dtype=torch.float64)).to(DEV)

    def step(state, out, prepared=None):
        if kind == "delta":
            ops.delta_step(proj, 0, channels, channels + n_step, channels + n_step + rank, cw, w2, g2, a_log, b, nw, state, front, off, ctx.token_req,
                           ctx.state_slots, n_step, dim, vdim, dim ** -0.5, 1e-6, 1e-6, 1.3, out, heads * d, prepared)
        else:
            ops.linear_step((proj, 0), (proj, hd), (proj, 2 * hd), (proj, 2 * hd + 2 * hv), w2, "root_sigmoid", b, 0.06, None, None, 0.3,
                            (proj, 2 * hd + hv), nw, 1e-6, 1.3, state, off, ctx.token_req, ctx.state_slots, n_step, dim, vdim, out, heads * d, prepared)
    results = []
    force = ops.decode_force_splits
    for beside in (False, True):
        state, out, kk, vv = state0.clone(), torch.zeros(n, heads * d + hv, dtype=torch.bfloat16, device=DEV), k.clone(), v.clone()
        buffer = ops.step_buffer() if beside else None
        step(state, out, buffer)
        conv = (conv_w, state, 0) if how == "convolution" else None
        try:
            ops.decode_force_splits = 1      # (whole keys and eight waves both ways)
            ops.attention_rows(rows, 0, ctx, 0, heads, kv, d, kk, vv, d ** -0.5, freq, d, 1.0, None, norms=None if conv else norms, norm_eps=1e-6, conv=conv,
                               into=(None, 0, 0.75, out, 0, 1), beside=buffer)
        finally:
            ops.decode_force_splits = force
        results.append((out, state, kk, vv))
    assert not torch.equal(results[0][1], state0)
    assert all(torch.equal(a, c) for a, c in zip(*results))


@pytest.mark.parametrize("heads,kv,d,vd,page", [(6, 2, 128, 128, 16), (3, 3, 64, 64, 32), (8, 4, 128, 64, 16), (34, 2, 32, 32, 16), (10, 2, 64, 64, 16)])
@pytest.mark.parametrize("q_lens,ctx_lens", [([1, 40, 1], [700, 40, 33]), ([2, 1], [2, 1]), ([1] * 70 + [17] + [1] * 3 + [130, 1], [50] * 70 + [400] + [9] * 3 + [131, 2000]),
                                             ([300, 1, 1, 16], [300, 900, 1100, 64])])
@pytest.mark.parametrize("mask", [{}, {"window": 37}, {"window": 24, "keep_first": 9}, {"chunk": 48, "sink": True}, {"softcap": 4.0}])
def test_portions_and_single_tokens_in_one_launch(heads, kv, d, vd, page, q_lens, ctx_lens, mask):
    """Portions anywhere among single tokens, more requests than a wave has lanes, keys split or not, more and fewer than 256 blocks of single
    tokens: the portions' rows are bit for bit those of a launch of their own, the single tokens' differ by what the sums of four waves
    instead of eight move a rounding to bfloat16 (2^-8), and both are what the plain operation gives within that rounding (twice: q k and the result)."""
    ops = _ops()
    R, n = len(q_lens), sum(q_lens)
    g = torch.Generator().manual_seed(n + heads)
    width = max(-(-c // page) for c in ctx_lens)
    pages = sum(-(-c // page) for c in ctx_lens)
    order, bt, at = torch.randperm(pages, generator=g), torch.zeros(R, width, dtype=torch.int32), 0
    for r, c in enumerate(ctx_lens):
        used = -(-c // page)
        bt[r, :used] = order[at: at + used]
        at += used
    k = torch.randn(pages, kv, page, d, generator=g).bfloat16()
    v = torch.randn(pages, kv, vd, page, generator=g).bfloat16()
    q = torch.randn(n, heads, d, generator=g).bfloat16()
    cu = torch.tensor([0] + list(torch.tensor(q_lens).cumsum(0)), dtype=torch.int32)
    cl, tr = torch.tensor(ctx_lens, dtype=torch.int32), torch.repeat_interleave(torch.arange(R, dtype=torch.int32), torch.tensor(q_lens))
    more = dict(mask)
    window = more.pop("window", 0)
    if more.get("sink"):
        more["sink"] = torch.randn(heads, generator=g)
    args = (d ** -0.5, window, max(q_lens), max(ctx_lens), q_lens.count(1))
    dev = {a: b.to(DEV) if torch.is_tensor(b) else b for a, b in more.items()}
    place = [t.to(DEV) for t in (q, k, v, bt, cu, cl, tr)]
    got = ops.paged_attention(*place, *args, **dev)
    lib = ops.library()
    lib.tp_attention_tune(4)      # (no choice of a kernel's variant, and one launch for each kind)
    try:
        apart = ops.paged_attention(*place, *args, **dev)
    finally:
        lib.tp_attention_tune(0)
    single = torch.tensor([q_lens[r] == 1 for r in tr.tolist()])
    assert torch.equal(got.cpu()[~single], apart.cpu()[~single])
    want = EmuOps().paged_attention(q, k, v, bt, cu, cl, tr, *args, **more)
    for a, b in ((got, apart), (got, want)):
        a, b = a.double().cpu(), b.double().cpu()
        assert float((a - b)[single].norm() / b[single].norm()) < 2.0 ** -8
        assert float((a - b).abs().max() / b.abs().max()) < 2.0 ** -6


@pytest.mark.parametrize("n,places", [(33, 32), (48, 32), (64, 32), (65, 32), (130, 64), (2, 1), (512, 8)])
def test_order_of_requests_among_blocks(n, places):
    """Every request once; up to two a place: the longest alone, the others in pairs (place p and p + places), the longest with the shortest; else longest first."""
    ops = _ops()
    g = torch.Generator().manual_seed(n)
    lens = torch.randint(1, 900, (n,), generator=g).to(torch.int32)
    shared, kvh = {}, 256 // places
    got = ops.decode_order(shared, lens.to(DEV), n, kvh, kvh, 1, 0, 0, 0).cpu().tolist()
    assert len(shared) == 1 and sorted(got) == list(range(n))
    rank = sorted(range(n), key=lambda i: (-((int(lens[i]) + 31) // 32), i))
    if n > 2 * places:
        assert got == rank
        return
    alone = 2 * places - n
    assert got[n - places: places] == rank[:alone]
    assert [(got[p], got[p + places]) for p in range(n - places)] == [(rank[alone + i], rank[n - 1 - i]) for i in range(n - places)]


@pytest.mark.parametrize("heads,kv,d,n,longest", [(16, 8, 64, 33, 700), (16, 8, 128, 48, 1300), (5, 5, 128, 110, 300)])
@pytest.mark.parametrize("mask", [{}, {"window": 100}, {"sink": True, "chunk": 200}])
def test_ordered_requests_give_the_same_bits(heads, kv, d, n, longest, mask):
    """With an order among the blocks and without: outputs and caches, from rows and from q."""
    ops = _ops()
    g = torch.Generator().manual_seed(n + d)
    ctx, k, v = _step([1 + (i * 37 % n) * (longest - 1) // (n - 1) for i in range(n)], kv, d, 16, g)
    rows = torch.randn(n, (heads + 2 * kv) * d, generator=g).to(DEV)
    q = torch.randn(n, heads, d, generator=g).to(DEV).bfloat16()
    if "sink" in mask:
        mask = {**mask, "sink": torch.randn(heads, generator=g).to(DEV)}
    outs = []
    for shared in (None, {}):
        ctx.shared, kk, vv = shared, k.clone(), v.clone()
        a = ops.attention_rows(rows, 0, ctx, 0, heads, kv, d, kk, vv, d ** -0.5, None, 0, 1.0, None, **mask)
        b = ops.paged_attention(q, kk, vv, ctx.block_tables[0], ctx.cu_seqlens, ctx.context_lens, ctx.token_req, d ** -0.5, mask.get("window", 0), 1,
                                ctx.max_context_len, n, sink=mask.get("sink"), chunk=mask.get("chunk", 0), shared=shared)
        outs.append((a, b, kk, vv))
    assert len(ctx.shared) == 1 and all(torch.equal(x, y) for x, y in zip(*outs))
