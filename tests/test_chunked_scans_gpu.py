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
