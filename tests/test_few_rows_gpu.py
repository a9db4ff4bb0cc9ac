"""Row kernels that read their rows once in 16-byte pieces, against the plain operations and against the kernels that take any size
and place (reached by columns that start off a 16-byte place); single-token steps against the general ones."""
import pytest
import torch

from emu_ops import EmuOps

pytestmark = pytest.mark.gpu
emu = EmuOps()
DEV = "cuda:0"


def _close(got, ref, tol):
    got, ref = got.double().cpu(), ref.double().cpu()
    assert float((got - ref).abs().max()) <= tol * float(ref.abs().max())


def _runs(lens, g):
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    req = torch.repeat_interleave(torch.arange(len(lens), dtype=torch.int32), torch.tensor(lens))
    slots = torch.randperm(len(lens) + 2, generator=g)[: len(lens)].to(torch.int32)
    return cu.to(DEV), req.to(DEV), slots.to(DEV)


@pytest.mark.parametrize("channels,taps", [(4, 2), (1024, 4), (2052, 3), (6144, 4)])
@pytest.mark.parametrize("lens", [[1, 1, 1], [70], [1, 2, 3, 60, 1, 17], [8, 56, 64]])
def test_causal_conv_paths_agree(channels, taps, lens):
    """Every path forms a channel's sum in the same order: the same bits, outputs and states alike."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(channels + len(lens))
    n = sum(lens)
    proj = torch.randn(n, channels + 8, generator=g).to(DEV)
    off = torch.cat([torch.zeros(n, 1, device=DEV), proj], dim=1).contiguous()         # rows off the 16-byte places
    w, b = torch.randn(taps, channels, generator=g).to(DEV), torch.randn(channels, generator=g).to(DEV)
    cu, req, slots = _runs(lens, g)
    state = torch.randn(len(lens) + 2, 5 + (taps - 1) * channels, generator=g).to(DEV)
    for act in (True, False):
        s0, s1, s2 = state.clone(), state.clone(), state.clone()
        want = ops.causal_conv(off, 5, channels, w, b, s0, cu, req, slots, len(lens), 5, act)
        got = ops.causal_conv(proj, 4, channels, w, b, s1, cu, req, slots, len(lens), 5, act)
        assert torch.equal(got, want) and torch.equal(s1, s0)
        got = ops.causal_conv(proj, 4, channels, w, b, s2, cu, req, slots, len(lens), 5, act, max_run=max(lens))
        assert torch.equal(got, want) and torch.equal(s2, s0)


@pytest.mark.parametrize("channels,taps,lens", [(20480, 4, [70]), (10244, 4, [1, 2, 3, 60, 1, 70]), (2052, 3, [8, 56, 64, 1, 700]),
                                                (1028, 2, [1600]), (12, 4, [100003, 9])])
def test_causal_conv_of_steps_large_enough_for_runs(channels, taps, lens):
    """Steps of some more than a million inputs go by runs of tokens a thread: the same bits as by single tokens."""
    test_causal_conv_paths_agree(channels, taps, lens)


@pytest.mark.parametrize("width,subs,taps", [(8, 1, 2), (1024, 2, 4), (4100, 3, 3)])
def test_residual_conv_of_single_tokens(width, subs, taps):
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(width)
    lens = [1, 1, 1, 1]
    cu, req, slots = _runs(lens, g)
    x, w = torch.randn(4, width, generator=g).to(DEV), torch.randn(subs, taps, width, generator=g).to(DEV)
    state = torch.randn(6, 3 + (taps - 1) * width, generator=g).to(DEV)
    s0, s1 = state.clone(), state.clone()
    want = ops.residual_conv(x, w, s0, 3, cu, req, slots, 4, torch.bfloat16)
    got = ops.residual_conv(x, w, s1, 3, cu, req, slots, 4, torch.bfloat16, max_run=1)
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and torch.equal(s0, s1)
    if ops.few_rows_ok(4, width, torch.bfloat16):
        got = ops.residual_conv(x, w, state.clone(), 3, cu, req, slots, 4, torch.bfloat16, max_run=1, blocked=[subs - 1])
        assert torch.equal(got[-1].data.permute(1, 0, 2).reshape(4, width), want[-1])
        assert subs == 1 or torch.equal(got[0], want[0])


@pytest.mark.parametrize("streams", [2, 4])
@pytest.mark.parametrize("width", [4, 260, 4096, 4100, 8192])
def test_stream_step_in_registers(streams, width):
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(width + streams)
    n = 3
    h, y = torch.randn(n, streams * width, generator=g), torch.randn(n, width, generator=g)
    mix, oc, ic, w = torch.randn(streams, streams, generator=g), torch.randn(streams, generator=g), torch.randn(streams, generator=g), torch.randn(width, generator=g)
    for kw in (dict(y=y, mix=mix, out_coef=oc, in_coef=ic, norm_weight=w, eps=1e-6, out_dtype=torch.float32),
               dict(y=y, mix=mix, out_coef=oc), dict(out_dtype=torch.float32, write_back=False),
               dict(norm_weight=w, eps=1e-6, out_dtype=torch.bfloat16, rows=torch.tensor([2, 0], dtype=torch.int32), write_back=False)):
        h0, h1 = h.clone(), h.to(DEV)
        want = emu.stream_step(h0, streams, **kw)
        got = ops.stream_step(h1, streams, **{k: v.to(DEV) if torch.is_tensor(v) else v for k, v in kw.items()})
        _close(h1, h0, 1e-6)
        if want is not None:
            _close(got, want, 2e-6 if want.dtype == torch.float32 else 8e-3)


@pytest.mark.parametrize("width,groups", [(256, 1), (1024, 4), (2048, 4), (4096, 8), (1028, 1), (4100, 1), (8192, 1), (24, 6)])
def test_group_rmsnorm_in_registers(width, groups):
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(width)
    x, w = torch.randn(5, width + 8, generator=g) * 3, torch.randn(width, generator=g)
    for dt, tol in ((torch.float32, 2e-6), (torch.bfloat16, 8e-3)):
        want = emu.rmsnorm_cols(x, 4, width, w, 1e-6, dt, groups)
        _close(ops.rmsnorm_cols(x.to(DEV), 4, width, w.to(DEV), 1e-6, dt, groups), want, tol)


@pytest.mark.parametrize("hidden", [4, 1028, 4096, 4100])
@pytest.mark.parametrize("lens", [[1, 1, 1], [5, 1, 9]])
def test_embed_bigram_leaves_the_last_tokens(hidden, lens):
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(hidden)
    n, vocab, buckets = sum(lens), 50, 37
    cu, req, slots = _runs(lens, g)
    toks = torch.randint(0, vocab, (n,), generator=g, dtype=torch.int32)
    pos = torch.arange(n, dtype=torch.int32)                     # (the first run begins its request, the others go on)
    table, bigram, ptab = torch.randn(vocab, hidden, generator=g), torch.randn(buckets + 1, hidden, generator=g), torch.randn(n, hidden, generator=g)
    prev = torch.randint(0, vocab, (len(lens) + 2, 1), generator=g, dtype=torch.int32)
    for dt in (torch.float32, torch.bfloat16):
        a, b, p = (t.to(dt) for t in (table, bigram, ptab))
        p0, p1 = prev.clone(), prev.to(DEV)
        want = emu.embed_bigram(toks, a, b, pos, req.cpu(), cu.cpu(), slots.cpu(), p0, len(lens), 31, 7, buckets, 0.5, p)
        got = ops.embed_bigram(toks.to(DEV), a.to(DEV), b.to(DEV), pos.to(DEV), req, cu, slots, p1, len(lens), 31, 7, buckets, 0.5, p.to(DEV))
        _close(got, want, 1e-6)
        assert torch.equal(p1.cpu(), p0)


@pytest.mark.parametrize("dims", [(32, 96, 32, 128), (3, 8, 4, 12), (2, 6, 2, 5)])
def test_latent_rows_in_pieces(dims):
    from tempura_amd.kernels import ops
    heads, dim, rot, vdim = dims
    g = torch.Generator().manual_seed(heads)
    proj, up = torch.randn(3, 4 + heads * (rot + dim) + rot + 4, generator=g), torch.randn(3, heads * (dim + vdim), generator=g)
    want = emu.latent_rows(proj, 4, 4 + heads * (rot + dim), up, heads, dim, rot, vdim)
    assert torch.equal(ops.latent_rows(proj.to(DEV), 4, 4 + heads * (rot + dim), up.to(DEV), heads, dim, rot, vdim).cpu(), want)


@pytest.mark.parametrize("experts,groups,keep", [(8, 4, 2), (64, 1, 1), (65, 1, 1), (128, 8, 3), (130, 2, 1)])
def test_moe_route_by_experts_a_lane(experts, groups, keep):
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(experts)
    logits = torch.randn(9, experts, generator=g)
    want = emu.moe_route(logits, None, experts, 2, groups, keep)
    got = ops.moe_route(logits.to(DEV), None, experts, 2, groups, keep)
    assert torch.equal(got[1].cpu(), want[1])
    _close(got[0], want[0], 2e-6)


@pytest.mark.parametrize("width", [4, 6, 1028, 4096])
def test_moe_rows_there_and_back(width):
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(width)
    n, experts, top = 33, 5, 2
    x, ids = torch.randn(n, width, generator=g), torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(n)]).to(torch.int32)
    wts, y = torch.randn(n, top, generator=g), torch.randn(n, width, generator=g)
    counts, offsets, rank = ops.moe_plan(ids.to(DEV), experts)
    xg, row_of = ops.moe_gather(x.to(DEV), ids.to(DEV), rank, offsets)
    order = sorted(range(n * top), key=lambda p: (int(ids.view(-1)[p]), p))
    assert torch.equal(xg.cpu(), x[torch.tensor(order) // top])
    want = (x.double()[:, None] * wts.double()[:, :, None]).sum(1)
    _close(ops.moe_scatter(xg, row_of, wts.to(DEV)), want, 1e-6)
    _close(ops.moe_scatter(xg, row_of, wts.to(DEV), y.to(DEV)), want + y.double(), 1e-6)


@pytest.mark.parametrize("counts,n,k", [([0, 5, 0, 300, 128, 1], 256, 64), ([129, 127, 255, 257], 400, 192), ([1], 128, 320), ([0, 0, 3], 16, 64)])
@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("output", ["float32", "swiglu", "relu2"])
def test_moe_linear(counts, n, k, tiled, output):
    """Rows of several experts in one launch: experts without rows, tiles that end inside an expert, weights whose columns are no whole
    tile; float64 of the bfloat16 operands, float32 sums of k products within 2^-24 k of their magnitudes (2e-6 of the largest here)."""
    from tempura_amd.kernels import ops
    if output == "relu2" and n % 128:
        pytest.skip("whole tiles of activated columns only")
    g = torch.Generator().manual_seed(sum(counts) + n)
    E, pairs = len(counts), sum(counts)
    x, w = torch.randn(pairs, k, generator=g).to(torch.bfloat16), (torch.randn(E * n, k, generator=g) * 0.2).to(torch.bfloat16)
    offsets = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32)
    want = torch.cat([x[offsets[e]: offsets[e + 1]].double() @ w[e * n: (e + 1) * n].double().T for e in range(E)])
    wd = ops.tile_weight(w.to(DEV)) if tiled else w.to(DEV)
    assert isinstance(wd, ops.TiledWeight) == tiled and ops.moe_linear_ok(E, n, k, wd)
    got = ops.moe_linear(x.to(DEV), wd, offsets.to(DEV), E, output)
    if output == "float32":
        _close(got, want, 2e-6)
    elif output == "relu2":
        _close(got, want.clamp(min=0.0) ** 2, 8e-3)
    else:
        pair = want.view(pairs, -1, 2, 8)
        gate, up = pair[:, :, 0].reshape(pairs, -1), pair[:, :, 1].reshape(pairs, -1)
        _close(got, gate * torch.sigmoid(gate) * up, 8e-3)
    assert torch.equal(got, ops.moe_linear(x.to(DEV), wd, offsets.to(DEV), E, output))


@pytest.mark.parametrize("m", [1, 2, 7, 16])
@pytest.mark.parametrize("act_cols,side,k", [(128, 0, 64), (256, 16, 2048), (384, 48, 8192)])
@pytest.mark.parametrize("kind", ["gelu_tanh", "silu", "gelu_erf"])
def test_up_products_of_a_few_rows_leave_activated(m, act_cols, side, k, kind):
    """The activation in the product's epilogue and the activation's own kernel see the same float32 sums: the same bits."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = ops.tile_weight((torch.randn(act_cols + side, k, generator=g) * 2 * k ** -0.5).to(torch.bfloat16).to(DEV))
    assert ops.linear_act_ok(m, act_cols, k, torch.bfloat16) and not ops.linear_act_ok(17, act_cols, k, torch.bfloat16)
    sums = ops.linear(x, w, torch.float32)
    want = ops.activation(sums, kind, torch.bfloat16, 0, act_cols)
    got, beside = ops.linear_relu2(x, w, act_cols, kind=kind)
    assert torch.equal(got, want) and torch.equal(beside, sums[:, act_cols:])
    blocked, _ = ops.linear_relu2(x, w, act_cols, blocked_out=True, kind=kind)
    assert torch.equal(blocked.data.permute(1, 0, 2).reshape(m, act_cols), want)


@pytest.mark.parametrize("m", [1, 3, 16])
@pytest.mark.parametrize("n,k", [(16, 64), (272, 2048), (528, 8192)])
@pytest.mark.parametrize("slope,limit,offset", [(1.702, 7.0, 1.0), (1.0, 0.5, 0.0), (1.0, 0.0, 0.5)])
def test_gated_products_of_a_few_rows_take_the_gates_constants(m, n, k, slope, limit, offset):
    """Against the activation of the same float32 sums (a rounding to bfloat16 and the hardware's exponential and reciprocal: 2^-8)."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + n)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = ops.tile_weight((torch.randn(n, k, generator=g) * 3 * k ** -0.5).to(torch.bfloat16).to(DEV))
    want = ops.gated_act(ops.linear(x, w, torch.float32), torch.float32, slope, limit, offset, interleaved=True)
    got = ops.linear_swiglu(x, w, slope=slope, limit=limit, up_offset=offset)
    assert float((got.float() - want).abs().max()) <= 2.0 ** -8 * float(want.abs().max())
    blocked = ops.linear_swiglu(x, w, True, slope, limit, offset)
    if isinstance(blocked, ops.KBlocked):
        blocked = blocked.data.permute(1, 0, 2).reshape(m, n // 2)
    assert torch.equal(blocked, got)


@pytest.mark.parametrize("m,n,k", [(1, 16, 64), (3, 528, 8192), (16, 272, 2048), (16, 65536, 64)])
@pytest.mark.parametrize("slope,limit,offset", [(1.702, 7.0, 1.0), (0.3, 0.0, 0.0), (3.0, 0.5, 0.5)])
def test_gates_with_constants_have_the_bits_of_the_activations_kernel(m, n, k, slope, limit, offset):
    """What a decoded row's gate is as a kernel of its own: float32 exponential and division, not the hardware's short forms (which round
    one bfloat16 in some ten thousand the other way)."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + n)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    w = ops.tile_weight((torch.randn(n, k, generator=g) * 3 * k ** -0.5).to(torch.bfloat16).to(DEV))
    want = ops.gated_act(ops.linear(x, w, torch.float32), torch.bfloat16, slope, limit, offset, interleaved=True)
    assert torch.equal(ops.linear_swiglu(x, w, slope=slope, limit=limit, up_offset=offset), want)


def test_layout_bits_of_an_activation_belong_to_its_epilogue():
    """Refused, as every unknown bit is, by a product that has no such epilogue (nothing is launched)."""
    import ctypes
    from tempura_amd.kernels import ops
    x, w, out = (torch.zeros(16, 64, dtype=torch.bfloat16, device=DEV) for _ in range(3))
    none, zero, ptr = ctypes.c_void_p(None), ctypes.c_float(0.0), lambda t: ctypes.c_void_p(t.data_ptr())
    def call(layout, accumulate):
        splits = ctypes.c_int(1)
        return ops.library().tp_linear_fused(ptr(x), ptr(w), 1, ptr(out), 1, accumulate, 16, 16, 64, 1, none, ctypes.c_size_t(0), none, 0, zero,
                                             none, none, none, layout, 0, ctypes.byref(splits), ctypes.c_float(1.0), zero, zero, 0, none, none)
    for layout in (256, 1024, 1 << 12):
        for accumulate in (0, 2):
            assert call(layout, accumulate) == 1 and b"layout" in ops.library().tp_last_error()
    assert call(0, 0) == 0


def test_a_closed_gate_leaves_zero_of_a_huge_value():
    """gate -200, up 2^121: their product overflows, the gated value does not."""
    from tempura_amd.kernels import ops
    x, w = torch.zeros(1, 64), torch.zeros(16, 64)
    x[0, 0], x[0, 1], w[:8, 0], w[8:, 1] = 1.0, 2.0 ** 60, -200.0, 2.0 ** 61
    got = ops.linear_swiglu(x.to(torch.bfloat16).to(DEV), w.to(torch.bfloat16).to(DEV), slope=1.0, limit=0.0, up_offset=0.5)
    assert torch.equal(got, torch.zeros_like(got))


@pytest.mark.parametrize("heads,kv,d,vd", [(4, 2, 64, 64), (3, 1, 96, 96), (8, 8, 32, 32), (16, 1, 576, 512), (2, 2, 160, 96)])
@pytest.mark.parametrize("ctx", [[700], [1, 40, 1500], [3, 260]])
@pytest.mark.parametrize("how", ["columns", "heads", "scale", "sink", "portions"])
def test_attention_gates_what_it_combines(heads, kv, d, vd, ctx, how):
    """The kernel that adds the splits of single tokens gates them in the order of the gate's own kernel: the same bits, also where
    keys are not split or a portion is among the requests (the two kernels then)."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(heads + ctx[-1])
    page, r = 16, len(ctx)
    q_lens = [1] * r if how != "portions" else [min(3, ctx[0])] + [1] * (r - 1)
    n, width, per = sum(q_lens), -(-max(ctx) // page), vd if how == "heads" else 1
    kc = (torch.randn(r * width, kv, page, d, generator=g)).to(torch.bfloat16).to(DEV)
    vc = (torch.randn(r * width, kv, vd, page, generator=g)).to(torch.bfloat16).to(DEV)
    tables = torch.randperm(r * width, generator=g).to(torch.int32).view(r, width).to(DEV)
    q = torch.randn(n, heads, d, generator=g).to(torch.bfloat16).to(DEV)
    cu, req, _ = _runs(q_lens, g)
    args = (q, kc, vc, tables, cu, torch.tensor(ctx, dtype=torch.int32, device=DEV), req, d ** -0.5, 0, max(q_lens), max(ctx), q_lens.count(1))
    sink = torch.randn(heads, generator=g).to(DEV) if how == "sink" else None
    rows = None if how == "scale" else torch.randn(n, 5 + heads * vd // per + 2, generator=g).to(DEV)
    want, got = (torch.full((n, heads * vd + 9), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.sigmoid_gate(ops.paged_attention(*args, sink=sink), rows, 5, 0.75, want, 4, per)
    assert ops.paged_attention(*args, sink=sink, into=(rows, 5, 0.75, got, 4, per)) is None
    assert torch.isfinite(got.float()).all() and torch.equal(got, want)


@pytest.mark.parametrize("m", [17, 40, 64])
@pytest.mark.parametrize("n,k", [(8256, 2048), (16384, 2112), (9216, 2624)])
def test_products_of_one_deep_block_a_cu(m, n, k):
    """17 to 64 rows onto 129 to 256 blocks of 64 columns, 32 steps of K and more: eight stages of LDS, the last of them
    drained one by one.  Float32 sums of k products against float32 sums in another order: an error of sqrt(k) roundings."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(DEV).bfloat16()
    w = torch.randn(n, k, generator=g).to(DEV).bfloat16()
    want = x.float() @ w.float().t()
    for weight in (w, ops.tile_weight(w)):
        got = ops.linear(x, weight, torch.float32)
        assert float((got - want).norm()) <= 4 * k ** 0.5 * 2.0 ** -24 * float(want.norm())
        h = torch.ones(m, n, device=DEV)
        ops.linear(x, weight, torch.float32, residual=h)
        assert torch.equal(h, got + 1.0)


@pytest.mark.parametrize("m,experts,top,groups,keep", [(1, 8, 2, 1, 1), (3, 8, 2, 4, 2), (9, 20, 4, 5, 2), (16, 64, 6, 1, 1)])
@pytest.mark.parametrize("k,ff,size,gated", [(64, 64, 64, True), (1152, 128, 192, False), (2048, 64, 0, False)])
def test_router_beside_the_shared_expert(m, experts, top, groups, keep, k, ff, size, gated):
    """Choice, shared up product and down product in the routed experts' launches: the choice and the routed sum bit for bit those of
    the kernels by themselves, the shared expert's sum with its gate behind the down product instead of in front of it."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m * 100 + k + experts)
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.1).to(DEV).bfloat16()
    n, pad = 96, -experts % 16
    x = rnd(m, k) * 10
    w_router = torch.cat([rnd(experts, k), torch.zeros(pad, k, dtype=torch.bfloat16, device=DEV)])
    w_up, w_down = ops.tile_weight(rnd(experts * ff, k)), rnd(experts, n, ff)
    w_down = ops.TiledWeight(torch.cat([ops.tile_weight(w).data for w in w_down]), experts * n, ff)
    correction, bias = torch.rand(experts, generator=g).to(DEV) * 0.1, torch.randn(experts, generator=g).to(DEV) * 0.1
    rest = dict(score="sigmoid" if gated else "softmax", group_best=2 if groups > 1 else 1, normalize=gated, sum_eps=1e-6, scale=1.5, bias=bias)
    router, rows = ops.tile_weight(w_router), ops.block_rows(x)
    shared = down = None
    if size:
        w_su, w_sd = rnd(size + 16, k), rnd(n, size)
        shared = (ops.tile_weight(w_su), size, "relu2" if not gated else "silu", gated)
    assert ops.moe_open_ok(experts, router, k, *([shared[0], ops.tile_weight(w_sd), size] if size else []))
    want = ops.moe_route(ops.linear(rows, router, torch.float32), correction, experts, top, groups, keep, **rest)
    *got, opened = ops.moe_open(rows, router, correction, experts, top, groups, keep, shared=shared, **rest)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    plain = ops.moe_few(rows, w_up, w_down, want[0], ff, "silu")
    if not size:
        assert opened is None
        return
    y = ops.moe_few(rows, w_up, w_down, got[0], ff, "silu", torch.ones(m, n, device=DEV), (ops.tile_weight(w_sd),) + opened)
    u = x.double() @ w_su.double().t()
    act = torch.relu(u[:, :size]) ** 2 if not gated else torch.nn.functional.silu(u[:, :size])
    add = act @ w_sd.double().t() * (torch.sigmoid(u[:, size:size + 1]) if gated else 1.0)
    # (the activations are rounded to bfloat16: 2^-9 of each term, whose sum over `size` of them is off by that much of its norm)
    assert float((y.double() - 1.0 - plain.double() - add).norm()) <= 2.0 ** -8 * float(add.norm()) + 1e-5 * float(plain.norm())


@pytest.mark.parametrize("m", [1, 3, 16])
@pytest.mark.parametrize("n,k,parts", [(16, 4096, 4), (2048, 4096, 2), (1024, 8192, 4), (4096, 8192, 1), (2064, 8192, 1), (272, 6144, 2)])
@pytest.mark.parametrize("blocked", [True, False])
def test_few_column_blocks_leave_parts(m, n, k, parts, blocked):
    """Products of few column blocks against float64, and the norm that adds their parts against the norm of the added rows."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=g).to(DEV).bfloat16(), (torch.randn(n, k, generator=g) * 0.05).to(DEV).bfloat16()
    assert ops.few_splits(m, n, k) == parts and ops.few_splits(17, n, k) == 1
    y = ops.linear(ops.block_rows(x), ops.tile_weight(w), torch.float32, partial_ok=True)
    assert isinstance(y, ops.Partials) == (parts > 1)
    total = y
    if parts > 1:
        total = y.data[0].clone()
        for p in range(1, parts):
            total += y.data[p]
    ref = x.double() @ w.double().t()
    # (k products of float32 sums: rounding of the running sum, 2^-24 of it each, as a random walk)
    assert float((total.double() - ref).abs().max()) <= 2.0 ** -24 * k ** 0.5 * 4 * float(ref.abs().max())
    wide = torch.randn(m, n + 8, generator=g).to(DEV)
    nw, bias = torch.rand(n, generator=g).to(DEV), torch.rand(n, generator=g).to(DEV)
    for gate in (None, wide):
        for normed in (True, False):
            h0 = torch.randn(m, n, generator=g).to(DEV)
            h1 = h0.clone()
            more = dict(gate=gate, gate_col0=4, gate_bias=bias) if gate is not None else {}
            a = ops.norm_add(h0, y, nw, 1e-5, bias, 1e-6, torch.bfloat16, normed=normed, blocked=blocked and n % 64 == 0, **more)
            b = ops.norm_add(h1, total, nw, 1e-5, bias, 1e-6, torch.bfloat16, normed=normed, blocked=blocked and n % 64 == 0, **more)
            assert torch.equal(h0, h1) and torch.equal(getattr(a, "data", a), getattr(b, "data", b))


@pytest.mark.parametrize("width", [6, 1028, 20484])
def test_norm_of_partial_sums(width):
    """The norm kernels' other widths (no whole vectors, more than the registers hold) with three parts."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(width)
    y, h0, w = torch.randn(3, 5, width, generator=g).to(DEV), torch.randn(5, width, generator=g).to(DEV), torch.rand(width, generator=g).to(DEV)
    h1 = h0.clone()
    a = ops.norm_add(h0, ops.Partials(y), w, 1e-5, w, 1e-5, torch.bfloat16)
    b = ops.norm_add(h1, y[0] + y[1] + y[2], w, 1e-5, w, 1e-5, torch.bfloat16)
    assert torch.equal(h0, h1) and torch.equal(a, b)


@pytest.mark.parametrize("n, width, parts", [(1025, 1028, 1), (1025, 2048, 1), (513, 2052, 1), (513, 2052, 5), (513, 3000, 1), (513, 4096, 1), (513, 4096, 5),
                                             (2049, 1028, 1), (2049, 2048, 1), (1025, 2052, 1), (1025, 4096, 1), (513, 4100, 1), (513, 6144, 1), (513, 6144, 3),
                                             (513, 6148, 1), (513, 8192, 1), (513, 1028, 1), (513, 2048, 1), (2049, 2044, 1), (301, 2052, 1), (301, 4096, 1),
                                             (769, 2052, 1), (769, 4096, 1), (301, 4100, 1), (301, 8192, 1)])
def test_norm_of_many_rows(n, width, parts):
    """Many rows (half as many threads a row, the gate and the next weight late) against the same rows a few at a time, bit by bit, and against float64."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(width + parts)
    y, h, w = torch.randn(parts, n, width, generator=g).to(DEV), torch.randn(n, width, generator=g).to(DEV), torch.rand(width, generator=g).to(DEV)
    gates = torch.randn(n, width, generator=g).to(DEV)
    for gate in (None, gates):
        def run(lo, hi, out):
            data = y[:, lo:hi].contiguous()
            more = dict(gate=gate[lo:hi], gate_col0=0, gate_bias=w) if gate is not None else {}
            return ops.norm_add(out, ops.Partials(data) if parts > 1 else data[0], w, 1e-5, w, 1e-6, torch.float32, **more)
        h0, h1, h2 = h.clone(), h[:300].clone(), h[300:].clone()
        a, b, c = run(0, n, h0), run(0, 300, h1), run(300, n, h2)
        assert torch.equal(h0, torch.cat([h1, h2])) and torch.equal(a, torch.cat([b, c]))
        v = y.double().sum(0) * (1 if gate is None else torch.sigmoid(gate.double() + w.double()))
        t = h.double() + v * torch.rsqrt(v.square().mean(1, keepdim=True) + 1e-5) * w.double()
        ref = t * torch.rsqrt(t.square().mean(1, keepdim=True) + 1e-6) * w.double()
        # (a value's own roundings, under twenty of 2^-24, of the largest value; the sums' relative error is smaller)
        assert float((h0.double() - t).abs().max()) <= 2.0 ** -24 * 20 * float(t.abs().max())
        assert float((a.double() - ref).abs().max()) <= 2.0 ** -24 * 20 * float(ref.abs().max())


@pytest.mark.parametrize("m,experts", [(1, 8), (4, 8), (16, 3)])
@pytest.mark.parametrize("ff,n,parts", [(2048, 96, 2), (4096, 1024, 4), (2112, 96, 1), (2048, 2064, 1)])
@pytest.mark.parametrize("size", [0, 512])
def test_experts_down_products_in_parts(m, experts, ff, n, parts, size):
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + ff + n)
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.1).to(DEV).bfloat16()
    x, w_up, w_down = ops.block_rows(rnd(m, 64)), ops.tile_weight(rnd(experts * ff, 64)), rnd(experts, n, ff)
    w_down = ops.TiledWeight(torch.cat([ops.tile_weight(w).data for w in w_down]), experts * n, ff)
    dense = torch.rand(m, experts, generator=g) * (torch.rand(m, experts, generator=g) < 0.5)
    shared = (ops.tile_weight(rnd(n, size)), ops.block_rows(rnd(m, size)).data, torch.randn(m, generator=g).to(DEV)) if size else None
    args = (x, w_up, w_down, dense.to(DEV), ff, "silu", None, shared)
    want, got = ops.moe_few(*args), ops.moe_few(*args, partial_ok=True)
    assert isinstance(got, ops.Partials) == (parts > 1)
    if parts > 1:
        assert got.data.shape == (parts, m, n)
        got = got.data.double().sum(0)
    # (the same products added in another order: 2^-24 of the sum of magnitudes at each of some hundred additions, as a random walk)
    assert float((got - want.double()).abs().max()) <= 2.0 ** -24 * 64 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("m", [1, 3, 16])
@pytest.mark.parametrize("streams,n,k", [(4, 32, 64), (4, 1024, 4160), (4, 4096, 1024), (4, 288, 14336)])
@pytest.mark.parametrize("coefs", [True, False])
def test_product_closes_streams(m, streams, n, k, coefs):
    """The product that closes a sublayer over the copies, and a product behind it that finishes the norm, against float64."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + n + k)
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)
    x, w, w2 = rnd(m, k).bfloat16(), (rnd(n, k) * k ** -0.5).bfloat16(), (rnd(48, n) * 0.1).bfloat16()
    mix, out, inc = (rnd(streams, streams), rnd(streams), rnd(streams)) if coefs else (None, None, None)
    weight, h0 = rnd(n), rnd(m, streams * n)
    y = x.double() @ w.double().t()
    mixed = h0.double().view(m, streams, n)
    if coefs:
        mixed = torch.einsum("ab,man->mbn", mix.double(), mixed)
    ref = mixed + (out.double() if coefs else torch.ones(streams, device=DEV).double())[None, :, None] * y[:, None]
    u = (ref * inc.double()[None, :, None]).sum(1) if coefs else ref.sum(1)
    normed = u / torch.sqrt((u * u).mean(1, keepdim=True) + 1e-5) * weight.double()
    assert ops.stream_linear_ok(m, n, streams, torch.bfloat16) and not ops.stream_linear_ok(17, n, streams, torch.bfloat16) and not ops.stream_linear_ok(m, n, 2, torch.bfloat16)
    got = {}
    for rows in (x, ops.block_rows(x)):
        for opening in (None, (inc, weight, 1e-5)):
            h = h0.clone()
            x2 = ops.linear(rows, ops.tile_weight(w), torch.float32, residual=ops.StreamClose(h, streams, mix, out, opening))
            # (y: k products in float32, 2^-24 each as a random walk; then a sum of streams + 1 terms)
            assert float((h.double().view_as(ref) - ref).norm()) <= (4 * k ** 0.5 + 16) * 2.0 ** -24 * float(ref.norm())
            assert torch.equal(got.setdefault("h", h), h)
            if opening is None:
                assert x2 is None
                continue
            z = ops.linear(x2, ops.tile_weight(w2), torch.float32)
            # (rows and weights in bfloat16: the rows' rounding, 2^-9 of each term of a sum)
            assert float((z.double() - normed @ w2.double().t()).norm()) <= 2.0 ** -8 * float(z.norm()) + 1e-6
            assert torch.equal(got.setdefault("z", z), z)


@pytest.mark.parametrize("n", [1, 5, 64])
@pytest.mark.parametrize("width,groups,taps,subs", [(8, 2, 2, 1), (264, 11, 4, 2), (4096, 8, 4, 2), (1024, 8, 3, 1), (2048, 2, 4, 2), (8192, 2, 2, 2), (3072, 2, 4, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_norm_in_the_residual_convolution(n, width, groups, taps, subs, dtype):
    """The norm and the convolution behind it in one launch: the bits of the two kernels, rows and states alike."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(n + width + taps)
    h, nw, w = torch.randn(n, width, generator=g).to(DEV), torch.randn(width, generator=g).to(DEV), torch.randn(subs, taps, width, generator=g).to(DEV)
    cu, req, slots = _runs([1] * n, g)
    for off in (0, 3):
        s0 = torch.randn(n + 2, off + (taps - 1) * width + 5, generator=g).to(DEV)
        s1 = s0.clone()
        blocked = [subs - 1] if dtype == torch.bfloat16 and n <= 16 and ops.few_rows_ok(n, width, dtype) else []
        want = ops.residual_conv(ops.rmsnorm(h, nw, 1e-5, torch.float32, groups=groups), w, s0, off, cu, req, slots, n, dtype, max_run=1, blocked=blocked)
        assert ops.norm_residual_conv_ok(n, width, groups, taps, subs, 1) and not ops.norm_residual_conv_ok(n, width, groups, taps, subs, 2)
        got = ops.norm_residual_conv(h, nw, 1e-5, groups, w, s1, off, req, slots, dtype, blocked)
        assert torch.equal(s0, s1)
        assert all(torch.equal(getattr(a, "data", a), getattr(b, "data", b)) for a, b in zip(got, want))


@pytest.mark.parametrize("n", [1, 15, 17, 300])
@pytest.mark.parametrize("experts,top,groups,keep,group_best", [(1, 1, 1, 1, 1), (8, 2, 4, 2, 1), (12, 5, 3, 2, 3), (16, 16, 1, 1, 1), (16, 3, 8, 3, 2), (15, 4, 5, 4, 1)])
@pytest.mark.parametrize("sigmoid,normalize,scale", [(False, False, 1.0), (True, True, 2.5), (False, True, 1.0)])
def test_choice_of_few_experts(n, experts, top, groups, keep, group_best, sigmoid, normalize, scale):
    """Up to 16 experts against the choice one by one of float64 scores, with equal scores, infinite corrections and rows of NaN."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(n + experts + top)
    logits = torch.randn(n, experts + 3, generator=g).mul(4).round().div(4)          # (many equal ones)
    if n > 2:
        logits[1] = float("nan")
    bias, correction = torch.randn(experts, generator=g).round(), torch.randn(experts, generator=g).mul(2).round().div(2)
    if experts > 8:
        correction[3], correction[5] = float("inf"), -float("inf")
    dense, ids, weights = ops.moe_route(logits.to(DEV), correction.to(DEV), experts, top, groups, keep, score="sigmoid" if sigmoid else "softmax",
                                        group_best=group_best, normalize=normalize, sum_eps=1e-6, scale=scale, bias=bias.to(DEV))
    dense, ids, weights = dense.cpu(), ids.cpu(), weights.cpu()
    for t in range(n):
        z = logits[t, :experts] + bias
        s = torch.sigmoid(z) if sigmoid else torch.softmax(z, 0)
        # (equal logits give equal scores in any precision, so the order of float32 scores is theirs)
        ch = (s + correction).tolist()
        if groups > 1:
            per, total = experts // groups, []
            for q in range(groups):
                best = sorted((c for c in ch[q * per: (q + 1) * per] if c == c), reverse=True)[:group_best]
                v = torch.tensor(0.0)
                for i, c in enumerate(best):
                    v = torch.tensor(c) if i == 0 else v + torch.tensor(c)
                total.append(float(v))
            kept = [q for q in range(groups) if total[q] == float("inf")]
            kept += sorted((q for q in range(groups) if total[q] < float("inf")), key=lambda q: (-total[q], q))[:keep]
            ch = [c if i // per in kept else -float("inf") for i, c in enumerate(ch)]
        order = sorted((i for i in range(experts) if ch[i] > -float("inf")), key=lambda i: (-ch[i], i))[:top]
        near = any(abs(a - b) < 1e-6 and a != b for i, a in enumerate(ch) for b in ch[:i])
        want = torch.zeros(experts)
        chosen = sum(float(s[i]) for i in order)
        for i in order:
            want[i] = float(s[i]) * (scale / (chosen + 1e-6) if normalize else scale)
        if near:
            continue
        assert ids[t, : len(order)].tolist() == order, t
        assert torch.allclose(dense[t], want, rtol=1e-5, atol=1e-7) and torch.equal(dense[t][order], weights[t, : len(order)]), t


@pytest.mark.parametrize("n", [1, 5, 64])
@pytest.mark.parametrize("q_dim,c_dim", [(8, 8), (512, 256), (1024, 128), (520, 516), (4096, 4096), (72, 1032)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_latent_norms_and_store(n, q_dim, c_dim, dtype):
    """Both norms and the cache write in one launch: the bits of the three."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(n + q_dim + c_dim)
    c_dim -= c_dim % (16 // dtype.itemsize)
    rows, qw, cw = torch.randn(n, 4 + q_dim + c_dim + 8, generator=g).to(DEV), torch.randn(q_dim, generator=g).to(DEV), torch.randn(c_dim, generator=g).to(DEV)
    slots = torch.randperm(80, generator=g)[:n].to(torch.int32).to(DEV)
    k0, v0 = torch.randn(5, 1, 16, c_dim, generator=g).to(dtype).to(DEV), torch.randn(5, 1, c_dim, 16, generator=g).to(dtype).to(DEV)
    k1, v1 = k0.clone(), v0.clone()
    ops.vector_store(ops.rmsnorm_cols(rows, 4 + q_dim, c_dim, cw, 1e-5, dtype), slots, k0, v0)
    want = ops.rmsnorm_cols(rows, 4, q_dim, qw, 1e-5, dtype)
    assert ops.latent_norms_ok(rows, 4, q_dim, 4 + q_dim, c_dim, dtype, dtype) and not ops.latent_norms_ok(rows, 2, q_dim, 4, c_dim, dtype, dtype)
    got = ops.latent_norms(rows, 4, q_dim, qw, 4 + q_dim, c_dim, cw, 1e-5, slots, k1, v1)
    assert torch.equal(got, want) and torch.equal(k0, k1) and torch.equal(v0, v1)


@pytest.mark.parametrize("m,k,n", [(1, 64, 16), (1, 192, 4128), (1, 4096, 4128), (1, 4160, 8192), (1, 8256, 4112), (1, 16448, 4128), (2, 4160, 64), (3, 960, 544),
                                   (4, 4096, 48), (5, 4160, 96), (8, 1024, 8224), (9, 320, 288), (16, 2112, 272), (16, 1088, 8192)])
@pytest.mark.parametrize("tiled", [True, False])
def test_products_of_few_rows_at_the_edges_of_their_variants(m, k, n, tiled):
    """Rows through LDS (one to four pieces a thread, one and several rows) and straight from memory, whole and partial runs of K, waves without
    a run, more column blocks than CUs; sums that are stored, or added into the stream with the next norm prepared, and a product that finishes it (all other
    ends: ``test_row_major_rows`` and ``test_one_row_through_lds``).  Bounds: k products of exact bfloat16 factors summed in float32 are within k * 2^-24 of
    the sum of their magnitudes; a result in bfloat16 within 2^-8 of itself besides; the norm's scale adds 2^-22 (its own sum and root)."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + k + n)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(torch.bfloat16)
    ref, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    slack = k * 2.0 ** -24 * mag
    wd = ops.tile_weight(w.to(DEV)) if tiled else w.to(DEV)
    assert not tiled or isinstance(wd, ops.TiledWeight)
    blocked = ops.KBlocked(x.view(m, k // 8, 8).transpose(0, 1).contiguous().to(DEV), m, k)
    for given in (x.to(DEV), blocked):
        assert bool(((ops.linear(given, wd, torch.float32).cpu().double() - ref).abs() <= slack).all())
    low = ops.linear(x.to(DEV), wd, torch.bfloat16).cpu().double()
    assert bool(((low - ref).abs() <= slack + 2.0 ** -8 * ref.abs() + 1e-30).all())
    # added into the stream, the next norm prepared, and a product that finishes it
    h = torch.randn(m, n, generator=g)
    nw = torch.rand(n, generator=g) + 0.5
    hd = h.to(DEV)
    out, pre = ops.linear(x.to(DEV), wd, torch.float32, residual=hd, next_norm=(nw.to(DEV), 1e-6))
    assert out is hd and bool(((hd.cpu().double() - h.double() - ref).abs() <= slack + 2.0 ** -23 * (h.double() + ref).abs()).all())
    if pre is None:
        assert n % 32 != 0
        return
    assert torch.equal(pre.rows().cpu(), (hd.cpu() * nw).to(torch.bfloat16))
    sums = (hd.cpu().double() ** 2).sum(1)
    assert bool(((pre.ss.cpu().double().sum(0)[:m] - sums).abs() <= n * 2.0 ** -24 * sums).all())
    w2 = (torch.randn(32, n, generator=g) * n ** -0.5).to(torch.bfloat16)
    rows = pre.rows().cpu().double()
    rstd = torch.rsqrt(sums / n + 1e-6)[:, None]
    want, most = rows @ w2.double().T * rstd, rows.abs() @ w2.double().abs().T * rstd
    for weight in (ops.tile_weight(w2.to(DEV)), w2.to(DEV)) if n % 64 == 0 else (w2.to(DEV),) if n % 32 == 0 else ():
        got = ops.linear(pre, weight, torch.float32).cpu().double()
        assert bool(((got - want).abs() <= (n * 2.0 ** -24 + 2.0 ** -22) * most + n * 2.0 ** -25 * want.abs()).all())


@pytest.mark.parametrize("counts,n,k", [([0, 5, 1121, 300, 128, 641], 2048, 64), ([129, 1850, 0, 127], 2048, 128), ([1, 2047, 255, 257, 0, 0], 1792, 320),
                                        ([4097], 1024, 192)])
@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("output", ["float32", "swiglu", "relu2"])
def test_moe_linear_of_256_columns(counts, n, k, tiled, output):
    """Blocks of 128 x 256: fewer steps of K than stages and more, experts without rows, tiles that end inside an expert.  Bounds as of
    ``test_moe_linear``; a product for each expert alone, in blocks of 128 x 128, gives the same bits."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(sum(counts) + n + k)
    E, pairs = len(counts), sum(counts)
    assert ops.library().tp_moe_linear_columns(pairs, E, n) == 256
    x, w = torch.randn(pairs, k, generator=g).to(torch.bfloat16), (torch.randn(E * n, k, generator=g) * 0.2).to(torch.bfloat16)
    offsets = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32)
    wd = ops.tile_weight(w.to(DEV)) if tiled else w.to(DEV)
    got = ops.moe_linear(x.to(DEV), wd, offsets.to(DEV), E, output)
    want = torch.cat([x[offsets[e]: offsets[e + 1]].double() @ w[e * n: (e + 1) * n].double().T for e in range(E)])
    if output == "float32":
        _close(got, want, 2e-6)
    elif output == "relu2":
        _close(got, want.clamp(min=0.0) ** 2, 8e-3)
    else:
        pair = want.view(pairs, -1, 2, 8)
        gate, up = pair[:, :, 0].reshape(pairs, -1), pair[:, :, 1].reshape(pairs, -1)
        _close(got, gate * torch.sigmoid(gate) * up, 8e-3)
    for e in range(E):
        for a in range(int(offsets[e]), int(offsets[e + 1]), 512):
            b = min(a + 512, int(offsets[e + 1]))
            assert ops.library().tp_moe_linear_columns(b - a, 1, n) == 128
            we = w[e * n: (e + 1) * n].to(DEV).contiguous()
            one = ops.moe_linear(x[a:b].to(DEV), ops.tile_weight(we) if tiled else we, torch.tensor([0, b - a], dtype=torch.int32, device=DEV), 1, output)
            assert torch.equal(got[a:b], one)


def _in_order(values, group):
    """float32 sums of ``group`` neighbours along the last axis, added in ascending order."""
    v = values.reshape(*values.shape[:-1], -1, group)
    total = torch.zeros_like(v[..., 0])
    for i in range(group):
        total = total + v[..., i]
    return total


@pytest.mark.parametrize("m,k", [(1, 1024), (2, 3072), (8, 4096), (9, 4128), (16, 5120), (1, 16384)])
def test_handed_over_norms_add_in_a_stated_order(m, k):
    """The order in which a norm's sums of squares are added is part of the result.  A block's sum: neighbours, fours, then the fours in ascending
    order; a row's: 32 sums of every 32nd block, then those in ascending order.  The same bits as these additions in float32."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + k)
    h = torch.randn(m, k, generator=g)
    nw = torch.rand(k, generator=g) + 0.5
    x, w = torch.zeros(m, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(k, 64, dtype=torch.bfloat16, device=DEV)
    hd = h.to(DEV)
    _, pre = ops.linear(x, ops.tile_weight(w), torch.float32, residual=hd, next_norm=(nw.to(DEV), 1e-5))
    fours = _in_order(_in_order(h * h, 2), 2)
    assert torch.equal(hd.cpu(), h) and torch.equal(pre.ss.t().cpu(), _in_order(fours, 4))
    # the same scale as of sums that are the expected total and zeros
    ss = torch.rand(m, k // 16, generator=g) ** 8 * 64.0
    lanes = torch.zeros(m, 32)
    for at in torch.cat([ss, torch.zeros(m, -ss.shape[1] % 32)], 1).view(m, -1, 32).unbind(1):
        lanes = lanes + at
    alone = torch.zeros_like(ss)
    alone[:, 0] = _in_order(lanes, 32)[:, 0]
    w2 = torch.randn(64, k, generator=g).to(torch.bfloat16)
    for weight in (ops.tile_weight(w2.to(DEV)), w2.to(DEV)) if k % 64 == 0 else (w2.to(DEV),):
        got, want = (ops.linear(ops.Prenormed(pre.x, t.to(DEV).t(), 1e-5, pre.blocked), weight, torch.float32) for t in (ss, alone))
        assert torch.equal(got, want)


def _every_end(ops, plain, normed, w, g):
    """What a product of these rows (plain ones, and ones whose norm it finishes) gives at every kind of end."""
    m, n = plain.shape[0], w.shape[0]
    slots = torch.randperm(32, generator=g)[:m].to(torch.int32).to(DEV)
    positions = torch.randint(0, 4000, (m,), generator=g).to(torch.int32).to(DEV)
    freq = (10000.0 ** (-torch.arange(0, 16, 2, dtype=torch.float64) / 16)).to(DEV)
    h, nw = torch.randn(m, n, generator=g).to(DEV), (torch.rand(n, generator=g) + 0.5).to(DEV)
    out = []
    for x in (plain, normed):
        out += [ops.linear(x, w, torch.float32), ops.linear(x, w, torch.bfloat16)]
        stream = h.clone()
        _, handed = ops.linear(x, w, torch.float32, residual=stream, next_norm=(nw, 1e-6))
        out += [stream] + ([] if handed is None else [handed.x, handed.ss])
    out += [ops.linear_swiglu(normed, w), ops.linear_swiglu(normed, w, slope=1.5, limit=4.0, up_offset=1.0)]
    if n > 128 and w.shape[1] % 64 == 0:
        out += ops.linear_relu2(plain, w, 128)
    for table in (None, ops.rope_table(positions, freq, 16, 1.0)):
        k_cache, v_cache = (torch.zeros(2, 1, *s, dtype=torch.bfloat16, device=DEV) for s in ((16, 16), (16, 16)))
        out += [ops.linear_rope_kv(normed, w, positions, slots, freq, 16, 1.0, n // 16 - 2, 1, 16, k_cache, v_cache, table), k_cache, v_cache]
    return out


@pytest.mark.parametrize("m,k,n,tiled", [(2, 2048, 65536, True), (16, 4160, 16384, True), (15, 8192, 16400, True), (14, 8192, 16400, True), (12, 4096, 65536, True), (11, 4096, 65536, True),
                                         (2, 2048, 48, False), (16, 3104, 64, False), (9, 4128, 160, False), (8, 8192, 48, False), (7, 8192, 48, False), (16, 8224, 48, False),
                                         (2, 1024, 64, True), (16, 512, 4128, True), (3, 2112, 48, True), (4, 4096, 160, True), (5, 4096, 160, True), (16, 2048, 4096, True),
                                         (15, 2048, 4112, True), (14, 8192, 8192, True), (14, 8192, 8208, True), (13, 8192, 4112, True), (13, 3136, 14336, True), (13, 3136, 14320, True), (12, 3072, 14336, True), (12, 3136, 14336, True)])
def test_row_major_rows(m, k, n, tiled):
    """Rows through LDS in chunks of K, whole and partial ones, rows that go there whole (one to four pieces a thread), and sizes beside theirs: the bits of
    k-blocked rows at every end."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + k + n)
    x, ss = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV), torch.rand(m, k // 16, generator=g).to(DEV).t()
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(torch.bfloat16).to(DEV)
    w = ops.tile_weight(w) if tiled else w
    assert isinstance(w, ops.TiledWeight) == tiled
    xb = x.view(m, k // 8, 8).transpose(0, 1).contiguous()
    got = _every_end(ops, x, ops.Prenormed(x, ss, 1e-6), w, torch.Generator().manual_seed(n))
    want = _every_end(ops, ops.KBlocked(xb, m, k), ops.Prenormed(xb, ss, 1e-6, (m, k)), w, torch.Generator().manual_seed(n))
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("k,n", [(1024, 4112), (4096, 5120), (4160, 8192), (8256, 4128), (16384, 4112), (4032, 8208), (4096, 8208), (4160, 32784), (5184, 8208),
                                 (9280, 8208), (16448, 4112), (32768, 4112), (32832, 4112)])
def test_one_row_through_lds(k, n):
    """One row of more column blocks than CUs with a tiled weight, one to eight pieces a thread, one run of K on its way and two, up to
    2,052 sums of a norm: the bits of the row-major
    weight, whose product reads the row from memory, at every end."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(k + n)
    x, ss = torch.randn(1, k, generator=g).to(torch.bfloat16).to(DEV), torch.rand(1, k // 16, generator=g).to(DEV).t()
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(torch.bfloat16).to(DEV)
    got, want = (_every_end(ops, x, ops.Prenormed(x, ss, 1e-6), weight, torch.Generator().manual_seed(n)) for weight in (ops.tile_weight(w), w))
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))


def test_moe_linear_of_256_columns_keeps_within_its_offsets():
    """A block of 256 columns reaches 255 rows of its weight by offsets into 2 GiB: longer rows, which blocks of 128 columns take, are left to those."""
    from tempura_amd.kernels import ops
    longest = (2 ** 31 - 129) // 510 // 64 * 64
    columns = lambda k: ops.library().tp_moe_tile_columns(20, 2048, k)
    assert columns(64) == columns(longest) == 256 and columns(longest + 64) == columns((2 ** 31 - 129) // 254 // 64 * 64) == 128


def test_moe_linear_chooses_its_blocks_by_the_rows_there_are():
    """Blocks of 256 columns where they need clearly fewer rounds of 256 CUs, by the blocks of rows that the routing makes: as many pairs of rows need one
    round or two.  (Blocks of rows and columns, and rounds of 128 / 256 columns.)"""
    from tempura_amd.kernels import ops
    for row_blocks, n, wide in ((16, 2048, False), (17, 2048, True), (8, 4096, False), (9, 4096, True), (16, 4096, True), (17, 4096, False), (24, 4096, False),
                                (25, 4096, True), (1, 2048, False), (300, 128, False), (300, 384, False), (300, 256, False), (500, 256, True), (4000, 8192, True), (7, 7168, True),
                                (10, 7168, False), (4, 7168, False)):
        rounds = lambda columns: -(-row_blocks * (n // columns) // 256)
        assert wide == (n % 256 == 0 and 8 * rounds(256) < 5 * rounds(128)), (row_blocks, n)
        assert ops.library().tp_moe_tile_columns(row_blocks, n, 64) == (256 if wide else 128), (row_blocks, n)


@pytest.mark.parametrize("counts", [[256] * 8, [2048] + [0] * 7, [0, 1024, 0, 0, 1024, 0, 0, 0], [300, 212, 129, 383, 255, 257, 1, 511], [2049, 0, 0, 0, 0, 0, 0, 0],
                                    [512] * 8, [4096, 0, 0, 0, 0, 0, 0, 0], [1] * 7 + [8000]])
@pytest.mark.parametrize("output", ["float32", "swiglu", "relu2"])
def test_moe_linear_of_any_routing(counts, output):
    """As many rows in one, two and eight experts, which take blocks of 128 and of 256 columns, and rows that always take those of 256: the bits of a product
    for each expert alone."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(counts[0] + len(output))
    E, pairs, n, k = len(counts), sum(counts), 2048, 192
    row_blocks = sum(-(-c // 128) for c in counts)
    assert ops.library().tp_moe_tile_columns(row_blocks, n, k) == (128 if row_blocks == 16 else 256)
    x, w = torch.randn(pairs, k, generator=g).to(torch.bfloat16).to(DEV), (torch.randn(E * n, k, generator=g) * 0.2).to(torch.bfloat16).to(DEV)
    first = [0] + torch.tensor(counts).cumsum(0).tolist()
    got = ops.moe_linear(x, ops.tile_weight(w), torch.tensor(first, dtype=torch.int32, device=DEV), E, output)
    for e in range(E):
        for a in range(first[e], first[e + 1], 512):
            b = min(a + 512, first[e + 1])
            we = ops.tile_weight(w[e * n: (e + 1) * n].contiguous())
            one = ops.moe_linear(x[a:b], we, torch.tensor([0, b - a], dtype=torch.int32, device=DEV), 1, output)
            assert torch.equal(got[a:b], one)


@pytest.mark.parametrize("k,n", [(4096, 4128), (4096, 4096), (4032, 4128), (4160, 4128), (8192, 4128)])
def test_one_and_two_rows_with_two_runs_on_their_way(k, n):
    """Products in groups, that close a sublayer over four copies, and of routed experts: one and two rows, long K and more blocks than CUs, and sizes
    beside these, have the bits that they have among three rows (whose products are within k * 2^-24 of the sum of their magnitudes)."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(k + n)
    draw = lambda *s: (torch.randn(*s, generator=g) * k ** -0.5).to(torch.bfloat16).to(DEV)
    plain, experts = draw(n, k), 3
    w = ops.tile_weight(plain)
    w_up, w_down = ops.tile_weight(draw(experts * 2 * k, 1024)), ops.tile_weight(draw(experts * n, k))
    w_up_long, w_down_short = ops.tile_weight(draw(experts * 2816, k)), ops.tile_weight(draw(experts * 64, 1408))
    rows, inner = draw(3, k), draw(3, 1024)
    h = torch.randn(3, 4 * n, generator=g).to(DEV)
    mix, coef, nw = torch.randn(4, 4, generator=g).to(DEV), torch.randn(4, generator=g).to(DEV), torch.ones(n, device=DEV)
    dense = torch.tensor([[0.3, 0.0, 0.7], [0.0, 1.0, 0.0], [0.5, 0.5, 0.0]], device=DEV)

    def results(m):
        x, y, d, copies = ops.block_rows(rows[:m].contiguous()), ops.block_rows(inner[:m].contiguous()), dense[:m].contiguous(), h[:m].clone()
        out = [ops.group_linear(torch.stack([x.data, x.data]), w, [16, n])]
        handed = ops.linear(x, w, torch.float32, residual=ops.StreamClose(copies, 4, mix, coef, (coef, nw, 1e-6)))
        out += [copies, handed.rows(), handed.ss.t()]
        return out + [ops.moe_few(y, w_up, w_down, d, k, None), ops.moe_few(x, w_up_long, w_down_short, d, 1408, None)]
    want = results(3)
    ref, mag = rows.double() @ plain.double().T, rows.double().abs() @ plain.double().abs().T
    assert bool(((want[0].double() - ref).abs() <= k * 2.0 ** -24 * mag).all())
    for m in (1, 2):
        for got, all_rows in zip(results(m), want):
            assert torch.equal(got, all_rows[:m])
