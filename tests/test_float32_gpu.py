"""The float32 products and the float32 attention on the matrix cores against float64 and against the general kernels."""
import math

import pytest
import torch

from emu_ops import EmuOps

pytestmark = pytest.mark.gpu
emu = EmuOps()
DEV = "cuda:0"


def _rel(got, ref):
    got, ref = got.double().cpu(), ref.double().cpu()
    return float((got - ref).norm() / ref.norm())


# rows: the edges of the few-row kernels (1, 2, 4, 8, 16) and of the 64- and 128-row blocks; K: no whole 256, 32 or 8; N: no whole
# block, and few enough columns that K is cut into parts
@pytest.mark.parametrize("m,n,k", [(1, 5, 4), (2, 130, 1028), (3, 64, 260), (5, 67, 2052), (9, 12, 96), (16, 1030, 516), (17, 100, 36),
                                   (40, 200, 4100), (64, 384, 96), (65, 130, 2048), (129, 257, 132), (300, 1000, 68), (611, 3072, 256)])
def test_float32_products(m, n, k):
    """Against float64: a sum of k products, each rounded once and added in float32, is off by at most about k / 2 units of 2^-24 of
    the sum of magnitudes, and by the root of that in the mean: 2^-24 sqrt(k) of the norm is four times what is seen."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + n + k)
    x, w, res = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g), torch.randn(m, n, generator=g)
    ref = x.double() @ w.double().T
    xd, wd = x.to(DEV), w.to(DEV)
    got = ops.linear(xd, wd, torch.float32)
    tol = 2.0 ** -24 * max(2.0, math.sqrt(k))
    assert _rel(got, ref) < tol
    assert _rel(ops.linear(xd, wd, torch.float32, residual=res.to(DEV)), ref + res.double()) < tol + 2.0 ** -23
    assert torch.equal(got, ops.linear(xd, wd, torch.float32))
    ops.allow_mfma = False
    try:
        general = ops.linear(xd, wd, torch.float32)
    finally:
        ops.allow_mfma = True
    assert _rel(got, ref) <= max(_rel(general, ref), 2.0 ** -24 * 2)
    # a row's bits do not depend on the rows beside it, up to 16 rows
    if m <= 16:
        assert torch.equal(ops.linear(xd[: m // 2 + 1].contiguous(), wd, torch.float32), got[: m // 2 + 1])
    # rows that are no whole 16-byte pieces (an odd K, an operand that starts off such a place) run the general kernel
    flat = torch.zeros(m * k + 1, device=DEV)
    off = flat[1:].view(m, k).copy_(xd)
    assert off.data_ptr() % 16 != 0 and _rel(ops.linear(off, wd, torch.float32), ref) < tol


@pytest.mark.parametrize("small,large,n,k,parts", [(385, 449, 6150, 68, 1), (257, 383, 8198, 132, 1), (513, 577, 4100, 1028, 3)])
def test_float32_products_in_blocks_of_128_and_64(small, large, n, k, parts):
    """Rows, columns and k that fill no block, with and without K in parts, plain and added into rows: against float64 with the bound above,
    and the bits of a row are the same in either block."""
    from tempura_amd.kernels import ops
    lib = ops.library()
    assert lib.tp_linear_f32_block(large, n, k) == 128 and lib.tp_linear_f32_block(small, n, k) == 64
    assert [lib.tp_linear_f32_scratch(m, n, k) for m in (small, large)] == [parts * m * n if parts > 1 else 0 for m in (small, large)]
    g = torch.Generator().manual_seed(large + n + k)
    x, w, res = (torch.randn(*s, generator=g).to(DEV) for s in ((large, k), (n, k), (large, n)))
    ref, tol = x.double() @ w.double().T, 2.0 ** -24 * math.sqrt(k)
    got, added = ops.linear(x, w, torch.float32), ops.linear(x, w, torch.float32, residual=res.clone())
    assert _rel(got, ref) < tol and _rel(added, ref + res.double()) < tol + 2.0 ** -23
    worst = ((got.double() - ref).abs() / (x.double().abs() @ w.double().abs().T)).max()      # (no result of a wrong place among the others)
    assert float(worst) < 2.0 ** -24 * k / 2
    few = x[:small].contiguous()
    assert torch.equal(ops.linear(few, w, torch.float32), got[:small])
    assert torch.equal(ops.linear(few, w, torch.float32, residual=res[:small].clone()), added[:small])


# rows and columns at the edges of the blocks, K: whole stages of 32, an odd number of them, a part of one
@pytest.mark.parametrize("m,n,k", [(17, 70, 132), (64, 512, 2048), (65, 4097, 1536), (129, 2050, 1572), (300, 3072, 3072), (700, 5200, 1536)])
def test_float32_products_keep_every_bit(m, n, k):
    """A sum of one term is the correctly rounded product, whatever the operands' size: ordinary ones, small ones (down to those below the
    smallest normal number) beside large ones, infinity beside the smallest weights.  (Nothing but that term is rounded: added zeros are exact.)"""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + n + k)
    rows, at = torch.arange(m), torch.randint(0, k, (m,), generator=g)
    value, w = torch.randn(m, generator=g), torch.randn(n, k, generator=g)
    value = torch.copysign(value.abs().clamp(2.0 ** -3, 4.0), value)
    w = torch.copysign(w.abs().clamp(2.0 ** -6, 8.0), w)
    for low, high in ((0, 0), (-60, 40), (-112, 90), (-118, 110), (-123, 110)):
        for ex, ew in ((low, high), (high, low)):
            x, b = torch.zeros(m, k), w * 2.0 ** ew
            x[rows, at] = value * 2.0 ** ex
            want = (x[rows, at].double()[:, None] * b[:, at].double().T).float()
            assert torch.isfinite(want).all() and torch.equal(ops.linear(x.to(DEV), b.to(DEV), torch.float32).cpu(), want)
    x = torch.zeros(m, k)
    x[rows, at] = math.inf * torch.sign(value)
    b = torch.sign(w) * 2.0 ** -140
    got = ops.linear(x.to(DEV), b.to(DEV), torch.float32).cpu()
    assert torch.equal(got, math.inf * torch.sign(value)[:, None] * torch.sign(b[:, at].T))


@pytest.mark.parametrize("m,n,k", [(65, 4097, 1536), (128, 4100, 1540), (129, 2050, 1572), (255, 4096, 1568), (300, 3072, 3072), (640, 6500, 1600),
                                   (700, 5200, 1536)])
def test_float32_products_of_many_kinds(m, n, k):
    """Plain and added into rows, against float64 with the bound of the products above: of normal operands, of operands over twelve orders of magnitude,
    of positive ones, and of tiny ones; the same call gives the same bits; a row's bits are the same when rows are added up to the next whole
    block of 128."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + n + k)
    x, w, res = (torch.randn(*s, generator=g).to(DEV) for s in ((m, k), (n, k), (m, n)))
    tol = 2.0 ** -24 * math.sqrt(k)
    for a, b in ((x, w), (x * torch.exp(3 * torch.randn(m, k, generator=g)).to(DEV), w * torch.exp(2 * torch.randn(n, k, generator=g)).to(DEV)),
                 (x.abs(), w.abs()), (x * 2.0 ** -60, w * 2.0 ** -40)):
        ref, got = a.double() @ b.double().T, ops.linear(a, b, torch.float32)
        assert _rel(got, ref) < tol
        assert float(((got.double() - ref).abs() / (a.double().abs() @ b.double().abs().T)).max()) < 2.0 ** -24 * k / 2
        assert torch.equal(got, ops.linear(a, b, torch.float32))
    ref, got = x.double() @ w.double().T, ops.linear(x, w, torch.float32)
    assert _rel(ops.linear(x, w, torch.float32, residual=res.clone()), ref + res.double()) < tol + 2.0 ** -23
    padded = torch.cat([x, torch.randn((-m) % 128, k, generator=g).to(DEV)])
    assert torch.equal(ops.linear(padded, w, torch.float32)[:m], got)


def test_float32_products_of_extreme_values():
    """Infinity, NaN and the largest finite values: infinity of the sign of the factor beside it, NaN for infinity times zero, and finite
    results of values that bfloat16 would round to infinity."""
    from tempura_amd.kernels import ops
    m, n, k = 256, 4096, 1536
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)
    top = torch.finfo(torch.float32).max
    x[0, 7], x[1, 100], x[2, 1535], x[3, 0] = math.inf, -math.inf, math.nan, math.inf
    w[5, 7], w[6, 100] = 0.0, 1000.0 + 1.0 / 3.0
    w[9, 3] = -math.inf
    x[4], x[5] = 0.0, 0.0
    x[4, 11], x[5, 12] = top, -top
    w[:, 11], w[:, 12] = 0.25, 0.5
    got = ops.linear(x.to(DEV), w.to(DEV), torch.float32).cpu()
    ref = x.double() @ w.double().T
    odd = ~torch.isfinite(ref)
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
    assert torch.equal(got[torch.isinf(ref)].double(), ref[torch.isinf(ref)])
    got, ref = torch.where(odd, 0.0, got.double()), torch.where(odd, 0.0, ref)
    assert float(((got[4:6] - ref[4:6]).abs() / ref[4:6].abs().clamp_min(1.0)).max()) < 2.0 ** -22
    assert _rel(got[6:], ref[6:]) < 2.0 ** -24 * math.sqrt(k)


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(3, 4), (130, 260), (1026, 3072)])
def test_float32_products_norm_and_gate_their_rows(m, n, k):
    """Rows before their norm and gate/up sums of a few rows: against float64 with the bound above (the norm and the gate add a few
    roundings), no further from it than the separate kernels, and a row's bits the same whatever rows stand beside it."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(m + n + k)
    x, w, wn = torch.randn(m, k, generator=g) * 3, torch.randn(2 * n, k, generator=g) * k ** -0.5, torch.rand(k, generator=g) + 0.5
    xd, wd, nd = x.to(DEV), w.to(DEV), wn.to(DEV)
    normed = x.double() / (x.double().pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * wn.double()
    rows = ops.Unnormed(xd, nd, 1e-5)
    assert ops.norm_in_product_ok(xd, torch.float32) and ops.linear_gate_f32_ok(rows, wd) and ops.linear_gate_f32_ok(xd, wd)
    tol = 2.0 ** -24 * max(8.0, math.sqrt(k))      # (a silu of a gate's sum, their product and the norm: up to eight roundings at few k)

    def gated(v):
        return torch.nn.functional.silu(v[:, :n]) * v[:, n:]

    apart = ops.linear(ops.rmsnorm(xd, nd, 1e-5, torch.float32), wd, torch.float32)
    for got, ref, old in ((ops.linear(rows, wd, torch.float32), normed @ w.double().T, apart),
                          (ops.linear_gate_f32(rows, wd), gated(normed @ w.double().T), ops.swiglu(apart, torch.float32))):
        assert _rel(got, ref) < tol
        if k > 4:      # (a few results of four terms, which share their row's scale, say little about which way is nearer)
            assert _rel(got, ref) <= 1.2 * _rel(old, ref) + 2.0 ** -25
    assert torch.equal(ops.linear_gate_f32(xd, wd), ops.swiglu(ops.linear(xd, wd, torch.float32), torch.float32))
    few = ops.Unnormed(xd[: m // 2 + 1].contiguous(), nd, 1e-5)
    assert torch.equal(ops.linear(few, wd, torch.float32), ops.linear(rows, wd, torch.float32)[: m // 2 + 1])
    assert torch.equal(ops.linear_gate_f32(few, wd), ops.linear_gate_f32(rows, wd)[: m // 2 + 1])


@pytest.mark.parametrize("what", ["plain", "window", "kept", "chunk", "cap", "bias", "sink"])
@pytest.mark.parametrize("heads,kv,d,page,q_lens,ctx_lens", [
    (6, 2, 64, 16, [37, 1, 20], [37, 90, 200]),                    # portions beside a single token
    (4, 4, 32, 32, [1, 1, 1], [1, 16, 17]),                        # single tokens at the edges of a tile
    (24, 8, 128, 16, [1, 1], [700, 300]),                          # keys split over blocks
    (3, 1, 96, 48, [5], [260]),
])
def test_float32_attention(heads, kv, d, page, q_lens, ctx_lens, what):
    """Every form against float64 (2e-6: sums of a few hundred float32 terms) and against the general kernel; every cache place that
    holds no key of its request is NaN."""
    from tempura_amd.kernels import ops
    g = torch.Generator().manual_seed(heads * 1000 + d)
    R, n = len(q_lens), sum(q_lens)
    pages = sum((c + page - 1) // page for c in ctx_lens) + 2
    perm = torch.randperm(pages, generator=g).tolist()
    width = max((c + page - 1) // page for c in ctx_lens) + 1
    bt = torch.full((R, width), perm[-1], dtype=torch.int32)
    it = iter(perm)
    used = torch.zeros(pages, page, dtype=torch.bool)
    for r, c in enumerate(ctx_lens):
        for i in range((c + page - 1) // page):
            bt[r, i] = next(it)
        for i in range(c):
            used[bt[r, i // page], i % page] = True
    kc, vc = torch.randn(pages, kv, page, d, generator=g) * 1.5, torch.randn(pages, kv, d, page, generator=g)
    q = torch.randn(n, heads, d, generator=g) * 1.5
    cu = torch.tensor([0] + list(torch.tensor(q_lens).cumsum(0)), dtype=torch.int32)
    cl, tr = torch.tensor(ctx_lens, dtype=torch.int32), torch.repeat_interleave(torch.arange(R, dtype=torch.int32), torch.tensor(q_lens))
    scale, window, more = d ** -0.5, 0, {}
    if what == "window":
        window = 19
    elif what == "kept":
        window, more = 33, {"keep_first": 21}
    elif what == "chunk":
        more = {"chunk": 50}
    elif what == "cap":
        more = {"softcap": 3.0}
    elif what == "bias":
        more = {"dist_bias": torch.randn(heads, 40, generator=g)}
    elif what == "sink":
        more = {"sink": torch.randn(heads, generator=g) * 3}
    ref = emu.paged_attention(q.double(), kc.double(), vc.double(), bt, cu, cl, tr, scale, window, max(q_lens), max(ctx_lens),
                              **{a: b.double() if torch.is_tensor(b) else b for a, b in more.items()})
    bad = ~used[:, None, :].expand(pages, kv, page)
    kc, vc = kc.clone(), vc.clone()
    kc[bad] = float("nan")
    vc.transpose(2, 3)[bad] = float("nan")
    more = {a: b.to(DEV) if torch.is_tensor(b) else b for a, b in more.items()}

    def run(values):
        return ops.paged_attention(q.to(DEV), kc.to(DEV), values.to(DEV), bt.to(DEV), cu.to(DEV), cl.to(DEV), tr.to(DEV), scale, window,
                                   max(q_lens), max(ctx_lens), **more)
    got = run(vc)
    assert _rel(got, ref) < 2e-6
    ops.allow_fast_attention = False
    try:
        general = run(vc)
    finally:
        ops.allow_fast_attention = True
    assert _rel(got, ref) <= max(2.0 * _rel(general, ref), 3e-7)
    # a last key whose values are infinite is its own token's matter: rows in front of it keep their bits
    if q_lens[0] > 1 and what == "plain":
        inf = vc.clone()
        last = ctx_lens[0] - 1
        inf[bt[0, last // page], :, :, last % page] = float("inf")
        other = run(inf)
        assert torch.equal(other[: q_lens[0] - 1], got[: q_lens[0] - 1])
        assert not torch.isfinite(other[q_lens[0] - 1]).any()


@pytest.mark.parametrize("d", [32, 64, 96, 128])
@pytest.mark.parametrize("ctx_lens", [[130, 1, 256], [600, 77], [1000], [1300]])
def test_float32_attention_of_split_keys(d, ctx_lens):
    """Single tokens whose keys are cut into two, four, eight and more splits, some of them without a key, heads that fill no whole
    wave: against float64 (2e-6, as above), with and without a sink."""
    from tempura_amd.kernels import ops
    heads, kv, page, R = 6, 2, 16, len(ctx_lens)
    g = torch.Generator().manual_seed(d + sum(ctx_lens))
    width = -(-max(ctx_lens) // page)
    bt = torch.randperm(R * width, generator=g).to(torch.int32).view(R, width)
    kc, vc = torch.randn(R * width, kv, page, d, generator=g), torch.randn(R * width, kv, d, page, generator=g)
    q, sink = torch.randn(R, heads, d, generator=g), torch.randn(heads, generator=g)
    cu, cl = torch.arange(R + 1, dtype=torch.int32), torch.tensor(ctx_lens, dtype=torch.int32)
    for more in ({}, {"sink": sink}):
        want = emu.paged_attention(q.double(), kc, vc, bt, cu, cl, cu[:R], d ** -0.5, 0, 1, max(ctx_lens), **more)
        got = ops.paged_attention(*(t.to(DEV) for t in (q, kc, vc, bt, cu, cl, cu[:R].contiguous())), d ** -0.5, 0, 1, max(ctx_lens),
                                  **{k: v.to(DEV) for k, v in more.items()})
        assert float((got.double().cpu() - want).abs().max() / want.abs().max()) < 2e-6
