"""Long runs of the recurrences as products over chunks of tokens, against float64 and against the kernels that walk token by token
(reached by rows that start off a 16-byte place): chunks, pieces and tiles that are not full, states that are not zero, values that are
not finite."""
import pytest
import torch

from emu_ops import EmuOps

pytestmark = pytest.mark.gpu
emu = EmuOps()
DEV = "cuda:0"


def _off(t):
    """The same rows from a place that is no multiple of 16 bytes."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    flat[1:] = t.flatten()
    return flat[1:].view(t.shape)


def _error(got, want):
    return float((got.double().cpu() - want.double()).norm() / want.double().norm())


def _scan_inputs(lens, H, P, N, G, seed):
    g = torch.Generator().manual_seed(seed)
    n, ch = sum(lens), H * P + 2 * G * N
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    slots = torch.randperm(len(lens) + 2, generator=g)[: len(lens)].to(torch.int32)
    state = torch.randn(len(lens) + 2, 7 + H * N * P, generator=g) * 0.5
    xbc, proj = torch.randn(n, ch, generator=g) * 0.7, torch.randn(n, H + 3, generator=g)
    consts = torch.randn(H, generator=g) - 1.5, torch.log(torch.rand(H, generator=g) * 0.5 + 0.05), torch.randn(H, generator=g)
    return xbc, proj, consts, state, cu, slots


@pytest.mark.parametrize("H,P,N,G", [(4, 16, 16, 2), (2, 48, 32, 1), (3, 64, 64, 3), (8, 64, 128, 4), (2, 80, 128, 1)])
@pytest.mark.parametrize("lens", [[257], [31, 300, 1, 160], [513, 32, 33, 128, 129]])
def test_selective_scan_in_chunks(H, P, N, G, lens):
    from tempura_amd.kernels import ops
    xbc, proj, consts, state, cu, slots = _scan_inputs(lens, H, P, N, G, H * N + len(lens))
    s_ref = state.clone()
    want = emu.ssm_scan(xbc, proj, 2, *consts, s_ref, 7, cu, slots, len(lens), H, P, N, G)
    dev, dc = [t.to(DEV) for t in (xbc, proj, cu, slots)], [c.to(DEV) for c in consts]
    out = []
    for x in (dev[0], _off(dev[0])):
        s = state.to(DEV)
        y = ops.ssm_scan(x, dev[1], 2, *dc, s, 7, dev[2], dev[3], len(lens), H, P, N, G, max_run=max(lens))
        assert torch.equal(s.cpu()[:, :7], state[:, :7])
        spare = [i for i in range(len(lens) + 2) if i not in slots.tolist()]
        assert torch.equal(s.cpu()[spare], state[spare])
        out.append((y, s))
    for i, ref in enumerate((want, s_ref)):
        chunks, walk = _error(out[0][i], ref), _error(out[1][i], ref)
        # (root mean squares over all results.  The sums of the two are chains of about as many roundings; which one is the nearer changes
        # from one set of inputs to the next, by up to a sixth over those few results, and over all sizes here the chunks are)
        assert chunks <= 1.25 * walk and chunks <= 1e-6, (i, chunks, walk)


def _selective_scan_64(xbc, proj, c0, dt_bias, a_log, d_skip, state, off, H, P, N, G):
    """One run from the state rows' first slot on, in float64 and not rounded: outputs and the state."""
    n, X = xbc.shape[0], xbc.double()
    x = X[:, : H * P].view(n, H, P)
    B, C = (X[:, H * P + i * G * N: H * P + (i + 1) * G * N].view(n, G, N).repeat_interleave(H // G, dim=1) for i in (0, 1))
    dt = torch.nn.functional.softplus(proj.double()[:, c0: c0 + H] + dt_bias.double())
    decay, S, y = torch.exp(-torch.exp(a_log.double()) * dt), state[0, off: off + H * N * P].double().view(H, N, P), []
    for t in range(n):
        S = decay[t, :, None, None] * S + dt[t, :, None, None] * B[t, :, :, None] * x[t, :, None, :]
        y.append((S * C[t, :, :, None]).sum(1) + d_skip.double()[:, None] * x[t])
    return torch.stack(y).view(n, H * P), S.reshape(-1)


@pytest.mark.parametrize("H,P,N,G", [(4, 16, 16, 2), (2, 48, 32, 1), (3, 64, 64, 3), (8, 64, 128, 4)])
def test_selective_scan_in_chunks_rounds_no_more_than_the_walk(H, P, N, G):
    """Against float64 with weak decays, strong ones, and strong ones of small steps: the mean (of logarithms) over inputs of the error's
    ratio to that of the token-by-token walk.  A single ratio scatters by some percent, the mean over 16 by one (states of few heads, the
    sum of a few tokens where decays are strong, by three)."""
    from tempura_amd.kernels import ops
    for bias, rate in ((0.0, 0.0), (2.5, 2.0), (0.0, 4.0)):
        ratios = []
        for seed in range(16):
            xbc, proj, consts, state, cu, slots = _scan_inputs([270 + 17 * seed], H, P, N, G, 1000 * seed + H * N)
            xbc, proj, state, cu, slots = (t.to(DEV) for t in (xbc, proj, state, cu, slots))
            consts = [c.to(DEV) for c in (consts[0] + bias, consts[1] + rate, consts[2])]
            y64, s64 = _selective_scan_64(xbc, proj, 2, *consts, state[int(slots[0]):], 7, H, P, N, G)
            err = []
            for x in (xbc, _off(xbc)):
                s = state.clone()
                y = ops.ssm_scan(x, proj, 2, *consts, s, 7, cu, slots, 1, H, P, N, G, max_run=xbc.shape[0])
                err.append(((y - y64).norm(), (s[int(slots[0]), 7: 7 + s64.numel()] - s64).norm()))
            ratios.append([float(torch.log(a / b)) for a, b in zip(*err)])
        y, s = torch.tensor(ratios).mean(0).exp().tolist()
        assert y <= 1.01 and s <= 1.03, (bias, rate, y, s)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("where", ["x", "b", "c", "dt"])
def test_selective_scan_keeps_what_is_not_finite_where_it_belongs(bad, where):
    """A value that is not finite reaches the tokens from its own on, and of these only those that the token-by-token walk gives one."""
    from tempura_amd.kernels import ops
    H, P, N, G, lens, t = 4, 32, 64, 2, [300], 141
    xbc, proj, consts, state, cu, slots = _scan_inputs(lens, H, P, N, G, 3)
    if where == "dt":
        proj[t, 2 + 1] = bad
    else:
        xbc[t, {"x": 1 * P + 5, "b": H * P + 9, "c": H * P + G * N + 9}[where]] = bad
    dev, dc = [v.to(DEV) for v in (xbc, proj, cu, slots)], [c.to(DEV) for c in consts]
    res = [ops.ssm_scan(x, dev[1], 2, *dc, state.to(DEV), 7, dev[2], dev[3], 1, H, P, N, G, max_run=300).cpu() for x in (dev[0], _off(dev[0]))]
    finite = [torch.isfinite(y) for y in res]
    assert not finite[0].all() and torch.equal(finite[0][:t], torch.ones_like(finite[0][:t])) and torch.equal(finite[0], finite[1])
    assert float((res[0] - res[1])[finite[0]].abs().max()) <= 2e-5 * float(res[1][finite[0]].abs().max())


def _delta_inputs(lens, H, G, D, Dv, seed, low):
    g = torch.Generator().manual_seed(seed)
    n = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    slots = torch.randperm(len(lens) + 2, generator=g)[: len(lens)].to(torch.int32)
    state = torch.randn(len(lens) + 2, 5 + H * D * Dv, generator=g) * 0.3
    qkv = torch.randn(n, 2 * G * D + H * Dv, generator=g)
    qkv[:, G * D: 2 * G * D] += 0.8 * torch.randn(1, G * D, generator=g)      # (keys that share a direction: the system is not near the identity)
    decay, proj = low + (1.0 - low) * torch.rand(n, H * D, generator=g), torch.randn(n, H + 3, generator=g) * 2
    return qkv, decay, proj, state, cu, slots


@pytest.mark.parametrize("H,G,D,Dv", [(2, 2, 64, 16), (4, 2, 128, 48), (3, 1, 64, 128), (2, 2, 128, 128)])
@pytest.mark.parametrize("lens,low", [([97], 0.9), ([300, 1, 15, 16, 17], 0.99), ([65, 129], 0.0), ([1000], 0.98)])
def test_delta_rule_by_groups_of_tokens(H, G, D, Dv, lens, low):
    from tempura_amd.kernels import ops
    qkv, decay, proj, state, cu, slots = _delta_inputs(lens, H, G, D, Dv, H * D + len(lens), low)
    s_ref = state.clone()
    want = emu.delta_scan(qkv, decay, proj, 2, s_ref, 5, cu, slots, len(lens), H, G, D, Dv, D ** -0.5, 1e-6)
    dev = [t.to(DEV) for t in (decay, proj, cu, slots)]
    out = []
    for max_run in (max(lens), 0):
        s = state.to(DEV)
        y = ops.delta_scan(qkv.to(DEV), dev[0], dev[1], 2, s, 5, dev[2], dev[3], len(lens), H, G, D, Dv, D ** -0.5, 1e-6, max_run=max_run)
        spare = [i for i in range(len(lens) + 2) if i not in slots.tolist()]
        assert torch.equal(s.cpu()[:, :5], state[:, :5]) and torch.equal(s.cpu()[spare], state[spare])
        out.append((y, s))
    for i, ref in enumerate((want, s_ref)):
        groups, walk = _error(out[0][i], ref), _error(out[1][i], ref)
        # (root mean squares; a group's sums are no longer chains of roundings than the same tokens' one after the other)
        assert groups <= 1.25 * walk and groups <= 2e-6, (i, groups, walk)


def _delta_rule_64(qkv, decay, proj, b0, state, off, H, G, D, Dv, q_scale, eps):
    """One run from the state rows' first slot on, in float64 and not rounded: outputs and the state."""
    x, n, unit = qkv.double(), qkv.shape[0], lambda v: v / torch.sqrt((v * v).sum(-1, keepdim=True) + eps)
    q, k = ((unit(x[:, i * G * D: (i + 1) * G * D].view(n, G, D)) * f).repeat_interleave(H // G, dim=1) for i, f in ((0, q_scale), (1, 1.0)))
    v, g, beta = x[:, 2 * G * D:].view(n, H, Dv), decay.double().view(n, H, D), torch.sigmoid(proj.double()[:, b0: b0 + H])
    S, y = state[0, off: off + H * D * Dv].double().view(H, Dv, D), []
    for t in range(n):
        S = g[t][:, None, :] * S
        S = S + (beta[t][:, None] * (v[t] - (S * k[t][:, None, :]).sum(-1)))[:, :, None] * k[t][:, None, :]
        y.append((S * q[t][:, None, :]).sum(-1))
    return torch.stack(y).view(n, H * Dv), S.reshape(-1)


@pytest.mark.parametrize("low", [0.0, 0.5, 0.8, 0.9, 0.99])
def test_delta_rule_by_groups_rounds_no_more_than_token_by_token(low):
    """Against float64 from strong decays to weak ones, the mean (of logarithms) over sizes and inputs of the error's ratio to that of the
    chain of single tokens: a single ratio scatters by some percent, the mean over 24 by one (states by two)."""
    from tempura_amd.kernels import ops
    ratios = []
    for H, G, D, Dv in ((2, 2, 64, 16), (3, 1, 64, 128), (4, 2, 128, 48), (2, 2, 128, 128)):
        for seed in range(6):
            qkv, decay, proj, state, cu, slots = (t.to(DEV) for t in _delta_inputs([97 + 31 * seed], H, G, D, Dv, 100 * seed + H * D, low))
            y64, s64 = _delta_rule_64(qkv, decay, proj, 2, state[int(slots[0]):], 5, H, G, D, Dv, D ** -0.5, 1e-6)
            err = []
            for max_run in (qkv.shape[0], 0):
                s = state.clone()
                y = ops.delta_scan(qkv.clone(), decay, proj, 2, s, 5, cu, slots, 1, H, G, D, Dv, D ** -0.5, 1e-6, max_run=max_run)
                err.append(((y - y64).norm(), (s[int(slots[0]), 5: 5 + s64.numel()] - s64).norm()))
            ratios.append([float(torch.log(a / b)) for a, b in zip(*err)])
    y, s = torch.tensor(ratios).mean(0).exp().tolist()
    assert y <= 1.01 and s <= 1.02, (y, s)


@pytest.mark.parametrize("H,G,D,Dv,lens", [(4, 2, 64, 16, [300, 1, 63, 0, 20, 64] + [1] * 70 + [50, 257]), (2, 2, 128, 128, [300, 1, 63, 0, 20, 64, 50, 257]),
                                           (16, 8, 128, 128, [20, 1, 0, 64, 63] + [1] * 40), (8, 8, 64, 32, [1] * 300 + [64, 63])])
def test_delta_rule_of_a_run_does_not_depend_on_its_neighbours(H, G, D, Dv, lens):
    """Decoded tokens and short portions beside long ones, in their launches or (many blocks of short runs) behind them: the bits, outputs
    and states, that every run has alone."""
    from tempura_amd.kernels import ops
    qkv, decay, proj, state, cu, slots = (t.to(DEV) for t in _delta_inputs(lens, H, G, D, Dv, 31, 0.8))
    together = state.clone()
    y = ops.delta_scan(qkv.clone(), decay, proj, 2, together, 5, cu, slots, len(lens), H, G, D, Dv, D ** -0.5, 1e-6, max_run=max(lens))
    for i, n in enumerate(lens):
        rows, alone = slice(int(cu[i]), int(cu[i + 1])), state.clone()
        if n:
            one = torch.tensor([0, n], dtype=torch.int32, device=DEV)
            got = ops.delta_scan(qkv[rows].clone(), decay[rows].contiguous(), proj[rows].contiguous(), 2, alone, 5, one, slots[i: i + 1], 1, H, G, D, Dv,
                                 D ** -0.5, 1e-6, max_run=n)
            assert torch.equal(y[rows], got), n
        assert torch.equal(together[int(slots[i])], alone[int(slots[i])]), n
        if n in (20, 63):      # (and those that its tokens have one a step)
            alone, one = state.clone(), torch.tensor([0, 1], dtype=torch.int32, device=DEV)
            for t in range(int(cu[i]), int(cu[i + 1])):
                got = ops.delta_scan(qkv[t: t + 1].clone(), decay[t: t + 1].contiguous(), proj[t: t + 1].contiguous(), 2, alone, 5, one, slots[i: i + 1],
                                     1, H, G, D, Dv, D ** -0.5, 1e-6, max_run=1)
                assert torch.equal(y[t: t + 1], got), (n, t)
            assert torch.equal(together[int(slots[i])], alone[int(slots[i])]), n


def _held_groups(lens, H, D, Dv):
    """Groups of 16 tokens that the scratch holds for these runs."""
    from tempura_amd.kernels import ops
    floats = ops.library().tp_delta_scan_scratch(sum(lens), len(lens), max(lens), H, D, Dv)
    assert floats <= 64 << 20 and floats % (H * (49 * D + 528)) == 0
    return floats // (H * (49 * D + 528))


@pytest.mark.parametrize("lens", [[1200, 700, 3] + [1] * 21, [1] * 70 + [64, 450, 63] + [1, 0] * 70 + [520, 100]])
def test_delta_rule_in_several_pairs_of_launches(lens):
    """More tokens and heads than the scratch holds at a time: each pair of launches goes on from the states that the one before left, also
    in the middle of a run; runs whose groups begin behind those of more than 64 others."""
    from tempura_amd.kernels import ops
    H, D, Dv = 160, 128, 16
    assert 1 <= _held_groups(lens, H, D, Dv) < sum(-(-n // 16) for n in lens if n > 63)
    qkv, decay, proj, state, cu, slots = _delta_inputs(lens, H, H, D, Dv, 5, 0.9)
    dev = [t.to(DEV) for t in (decay, proj, cu, slots)]
    out = []
    for max_run in (max(lens), 0):
        s = state.to(DEV)
        out.append((ops.delta_scan(qkv.to(DEV), dev[0], dev[1], 2, s, 5, dev[2], dev[3], len(lens), H, H, D, Dv, D ** -0.5, 1e-6, max_run=max_run), s))
    assert _error(out[0][0], out[1][0].cpu()) <= 1e-6 and _error(out[0][1], out[1][1].cpu()) <= 1e-6


@pytest.mark.parametrize("lens", [[1800] + [1] * 63, [1800] + [1] * 299, [64] * 11, [2000]])
def test_delta_rule_scratch_is_sized_by_tokens(lens):
    """A long run beside many single tokens needs the room of its own groups, and one more a run that could be long."""
    need = sum(-(-n // 16) for n in lens if n > 63)
    assert need <= _held_groups(lens, 16, 128, 128) <= sum(lens) // 16 + sum(lens) // 64


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("where", ["q", "k", "v", "beta"])
def test_delta_rule_keeps_what_is_not_finite_where_it_belongs(bad, where):
    from tempura_amd.kernels import ops
    H, D, Dv, t = 2, 64, 32, 77
    qkv, decay, proj, state, cu, slots = _delta_inputs([200], H, H, D, Dv, 9, 0.9)
    if where == "beta":
        proj[t, 2 + 1] = float("nan")
    else:
        qkv[t, {"q": D + 3, "k": 3 * D + 3, "v": 4 * D + Dv + 3}[where]] = bad
    dev = [v.to(DEV) for v in (decay, proj, cu, slots)]
    res = [ops.delta_scan(qkv.to(DEV), dev[0], dev[1], 2, state.to(DEV), 5, dev[2], dev[3], 1, H, H, D, Dv, D ** -0.5, 1e-6, max_run=m).cpu()
           for m in (200, 0)]
    finite = [torch.isfinite(y) for y in res]
    assert not finite[0].all() and finite[0][:t].all() and torch.equal(finite[0], finite[1])
    assert float((res[0] - res[1])[finite[0]].abs().max()) <= 2e-6 * float(res[1][finite[0]].abs().max())


@pytest.mark.parametrize("H,P,N,G", [(4, 8, 16, 2), (2, 24, 5, 1), (6, 40, 56, 2), (3, 64, 128, 3), (1, 41, 600, 1), (2, 16, 1100, 1), (8, 16, 30, 1)])
@pytest.mark.parametrize("off", [7, 8])
def test_selective_scan_of_single_tokens(H, P, N, G, off):
    """A kernel of its own, with the sums of the one that walks runs: the same bits, outputs and states; a request without a token is left alone."""
    from tempura_amd.kernels import ops
    xbc, proj, consts, state, _, slots = _scan_inputs([1, 1, 1], H, P, N, G, H + N)
    cu = torch.tensor([0, 1, 1, 2, 3], dtype=torch.int32)
    slots, state = torch.tensor([2, 0, 4, 1], dtype=torch.int32), torch.cat([torch.zeros(5, off - 7), state], dim=1).contiguous()
    dev, dc, out = [t.to(DEV) for t in (xbc, proj, cu, slots)], [c.to(DEV) for c in consts], []
    for max_run in (1, 2):
        s = state.to(DEV)
        out.append((ops.ssm_scan(dev[0], dev[1], 2, *dc, s, off, dev[2], dev[3], 4, H, P, N, G, max_run=max_run), s))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert torch.equal(out[0][1][0].cpu(), state[0]) and not torch.equal(out[0][1][2].cpu(), state[2])
