"""Single tokens' attention with keys and values on their way to LDS: contexts at the edges of steps, waves and rings, keys that are
split or not, a block or more a CU, masks, and the gate behind the heads, against the plain operation."""
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
