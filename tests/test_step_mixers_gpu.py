"""Recurrent mixers of one token a request in one launch, against the separate kernels: the same bits, outputs and states alike.
Key and value sizes around the kernel's edges (33 to 128, lanes that hold no channel), ranks that are no whole run of 32."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SIZES = [(3, 2, 36, 4, 5), (2, 3, 64, 64, 64), (1, 2, 64, 128, 33), (5, 2, 100, 72, 100), (16, 4, 128, 128, 64), (1, 1, 128, 128, 128)]


def _case(n, heads, dim, vdim, rank, columns, state_floats):
    g = torch.Generator().manual_seed(n * 1000 + dim + vdim + rank)
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)
    slots = torch.randperm(n + 2, generator=g)[:n].to(torch.int32).to(DEV)
    cu, req = torch.arange(n + 1, dtype=torch.int32, device=DEV), torch.arange(n, dtype=torch.int32, device=DEV)
    return rnd, slots, cu, req, rnd(n, columns), rnd(n + 2, state_floats + (-state_floats) % 4)


def _outs(n, heads, vdim):
    return [[torch.full((n, heads * vdim + 8), 7.0, dtype=dt, device=DEV) for _ in range(2)] for dt in (torch.float32, torch.bfloat16)]


@pytest.mark.parametrize("n,heads,dim,vdim,rank", SIZES)
@pytest.mark.parametrize("taps", [1, 4])
def test_delta_step(n, heads, dim, vdim, rank, taps):
    from tempura_amd.kernels import ops
    channels, g_rank = heads * (2 * dim + vdim), max(1, rank - 3)
    conv = (taps - 1) * channels
    off = conv + (-conv) % 4
    rnd, slots, cu, req, proj, state = _case(n, heads, dim, vdim, rank, 1 + channels + heads + rank + g_rank, off + heads * dim * vdim)
    beta, a1, g1 = 1 + channels, 1 + channels + heads, 1 + channels + heads + rank
    cw, a2, g2 = rnd(taps, channels), rnd(rank, heads * dim) * 0.3, rnd(g_rank, heads * vdim)
    a_log, dt, nw = rnd(heads), rnd(heads * dim), rnd(vdim)
    for plain, fused in _outs(n, heads, vdim):
        s0, s1 = state.clone(), state.clone()
        qkv = ops.causal_conv(proj, 1, channels, cw, None, s0, cu, req, slots, n, 0, True, max_run=1)
        decay = ops.lowrank_up(proj, a1, a2, "decay", a_log, dt, dim)
        gate = ops.lowrank_up(proj, g1, g2, "sigmoid")
        o = ops.delta_scan(qkv, decay, proj, beta, s0, off, cu, slots, n, heads, heads, dim, vdim, dim ** -0.5, 1e-6)
        ops.head_norm_gate(o, nw, gate, 1e-6, 1.3, heads, plain, 4)
        assert ops.mixer_step_ok(n, 1, heads, dim, vdim, (rank, g_rank), s1, off, fused, 4)
        ops.delta_step(proj, 1, beta, a1, g1, cw, a2, g2, a_log, dt, nw, s1, 0, off, req, slots, heads, dim, vdim, dim ** -0.5, 1e-6, 1e-6,
                       1.3, fused, 4)
        assert torch.equal(plain, fused) and torch.equal(s0, s1)


@pytest.mark.parametrize("n,heads,dim,vdim,rank", [s for s in SIZES if s[2] == s[3]] + [(3, 2, 40, 40, 7)])
def test_general_delta_step(n, heads, dim, vdim, rank):
    from tempura_amd.kernels import ops
    hd = heads * dim
    rnd, slots, cu, req, proj, state = _case(n, heads, dim, vdim, rank, (5 * hd + rank + 3) // 4 * 4, 4 + hd * dim)
    w2, w0, ab, nw = rnd(rank, hd), rnd(hd), rnd(hd), rnd(hd)
    for plain, fused in _outs(n, heads, dim):
        s0, s1 = state.clone(), state.clone()
        decay = ops.lowrank_up(proj, 5 * hd, w2, "rate_sigmoid", bias=w0, rate=0.6, in_act="tanh")
        o = ops.general_delta_scan(proj, 0, decay, ab, s0, 4, cu, slots, n, heads, dim, 1e-6)
        ops.head_norm_gate(o, nw, None, 1e-6, 0.7, heads, plain, 4, gate_rows=proj, gate_col0=4 * hd)
        assert ops.mixer_step_ok(n, 1, heads, dim, dim, (rank,), s1, 4, fused, 4, 4 * hd, proj.shape[1])
        ops.general_delta_step(proj, 0, 4 * hd, 5 * hd, w2, w0, 0.6, ab, nw, s1, 4, req, slots, heads, dim, 1e-6, 1e-6, 0.7, fused, 4)
        assert torch.equal(plain, fused) and torch.equal(s0, s1)


@pytest.mark.parametrize("n,heads,dim,vdim,rank", SIZES)
@pytest.mark.parametrize("bonus", [False, True])
def test_linear_step(n, heads, dim, vdim, rank, bonus):
    from tempura_amd.kernels import ops
    hd, hv = heads * dim, heads * vdim
    rnd, slots, cu, req, proj, state = _case(n, heads, dim, vdim, rank, (2 * hd + 2 * hv + rank + 3) // 4 * 4, 8 + hd * vdim)
    w2, b, u = rnd(rank, hd) * 0.3, rnd(hd) - 2.0, rnd(hd) if bonus else None
    nw, mode, act = (rnd(hv), "exp_exp", "tanh") if bonus else (rnd(vdim), "root_sigmoid", None)
    q, k, v, gate, x = (proj, 0), (proj, hd), (proj, 2 * hd), (proj, 2 * hd + hv), (proj, 2 * hd + 2 * hv)
    for plain, fused in _outs(n, heads, vdim):
        s0, s1 = state.clone(), state.clone()
        decay = ops.lowrank_up(proj, x[1], w2, mode, bias=b, rate=0.06, in_act=act)
        o = ops.linear_scan(q, k, v, decay, s0, 8, cu, slots, n, heads, dim, vdim, bonus=u, q_scale=0.3, max_run=1)
        ops.head_norm_gate(o, nw, None, 1e-6, 1.0, heads, plain, 0, gate_rows=proj, gate_col0=gate[1], gate_act="silu")
        assert ops.mixer_step_ok(n, 1, heads, dim, vdim, (rank,), s1, 8, fused, 0, gate[1], proj.shape[1])
        ops.linear_step(q, k, v, x, w2, mode, b, 0.06, act, u, 0.3, gate, nw, 1e-6, 1.0, s1, 8, req, slots, heads, dim, vdim, fused, 0)
        assert torch.equal(plain, fused) and torch.equal(s0, s1)


@pytest.mark.parametrize("taps", [2, 3, 5, 6])
@pytest.mark.parametrize("n,heads,dim,vdim,rank", SIZES[:2])
def test_delta_step_of_other_convolutions(n, heads, dim, vdim, rank, taps):
    """Fewer taps than are requested in front, and more: the same bits as the separate kernels."""
    test_delta_step(n, heads, dim, vdim, rank, taps)
