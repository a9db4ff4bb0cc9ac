"""Single tokens' attention with keys and values on their way to LDS: contexts at the edges of steps, waves and rings, keys that are
split or not, a block or more a CU, masks, and the gate behind the heads, against the plain operation."""
from types import SimpleNamespace

import pytest
import torch

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
