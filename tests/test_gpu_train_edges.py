"""The training path's fused edge functions (second_order): the first-order value aggregation, the softmax attention
weights and the sum with two gathered tensors, their values, gradients and second-order gradients against float64
compositions of plain torch, on ragged lists with isolated rows and columns, single-edge rows, rows longer than a
workgroup's pass and logits with exact ties at the row maximum.

Bounds: relative 2-norm error 2e-5 per tensor (fp32 sums of up to a few hundred products, second order through two
such sums)."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 2e-5
H, C = 128, 256


def _edges(n, seed, cuda, max_deg=40):
    from ubio_molfm_amd import second_order as so
    g = torch.Generator().manual_seed(seed)
    deg = torch.randint(0, max_deg, (n,), generator=g)
    if n > 3:
        deg[0], deg[1], deg[2] = 0, 1, 90
    row = torch.repeat_interleave(torch.arange(n), deg)
    E = row.numel()
    col = torch.randint(0, max(1, n - 1), (E,), generator=g)          # the last atom is no edge's source
    ptr = torch.cat([torch.zeros(1, dtype=torch.long), deg.cumsum(0)])
    eid = torch.argsort(col, stable=True)
    kptr = torch.cat([torch.zeros(1, dtype=torch.long), torch.bincount(col, minlength=n).cumsum(0)])
    dev = [t.to(cuda, torch.int32) for t in (ptr, col, row, kptr, eid)]
    e = so.TrainEdges.__new__(so.TrainEdges)
    e.N, e.E, e.row32, e.col32 = n, E, dev[2], dev[1]
    e.nl = types.SimpleNamespace(row_ptr=dev[0], key_ptr=dev[3])
    ids = torch.arange(E, dtype=torch.int32, device=cuda)
    e.md = (dev[0], dev[1], ids, dev[3], dev[2][eid.to(cuda)], dev[4])
    return e, row, col, g


def ref_aggregation(w, u, v, row, col):
    out = []
    for k in range(3):
        t = (w * u[:, k:k + 1]).repeat(1, 2) * v[:, col]
        out.append(torch.zeros(v.shape, dtype=v.dtype).index_add(1, row, t))
    return torch.stack(out)


def ref_alpha(ga, i, q, pp, row, n):
    a = ga * q
    idx = row.unsqueeze(1).expand(-1, H)
    m = torch.full((n, H), -float("inf"), dtype=a.dtype).scatter_reduce(0, idx, a.detach(), "amax")
    tie = (a.detach() == m[row]).to(a.dtype)
    cnt = torch.zeros(n, H, dtype=a.dtype).index_add(0, row, tie).clamp_min(1)
    # the maximum as the mean of the edges that attain it: its value, and its gradient split over them
    top = torch.zeros(n, H, dtype=a.dtype).index_add(0, row, torch.where(tie > 0, a, torch.zeros_like(a))) / cnt
    ex = torch.exp(a - top[row]) * pp.unsqueeze(1)
    s = torch.zeros(n, H, dtype=a.dtype).index_add(0, row, ex)
    return ex * i / (s + 1e-3)[row]


def _compare(fn, ref, ins, g, cuda):
    """Values, gradients and second-order gradients (through a random cotangent of every gradient)."""
    a = [t.to(cuda, torch.float32).requires_grad_(True) for t in ins]
    b = [t.clone().double().requires_grad_(True) for t in ins]
    y, z = fn(*a), ref(*b)
    go = torch.randn(z.shape, generator=g, dtype=torch.float64)
    gy = go.to(cuda, torch.float32).requires_grad_(True)
    gz = go.clone().requires_grad_(True)
    da = torch.autograd.grad(y, a, gy, create_graph=True)
    db = torch.autograd.grad(z, b, gz, create_graph=True)
    cot = [torch.randn(t.shape, generator=g, dtype=torch.float64) for t in db]
    sa = sum((x * c.to(cuda, torch.float32)).sum() for x, c in zip(da, cot))
    sb = sum((x * c).sum() for x, c in zip(db, cot))
    d2a = torch.autograd.grad(sa, [*a, gy], allow_unused=True)
    d2b = torch.autograd.grad(sb, [*b, gz], allow_unused=True)
    for name, got, want in (("value", [y], [z]), ("gradient", da, db), ("second order", d2a, d2b)):
        for i, (p, q) in enumerate(zip(got, want)):
            if q is None or p is None:
                assert q is None or float(q.abs().max()) == 0 if p is None else float(p.abs().max()) == 0
                continue
            d = p.detach().double().cpu() - q.detach()
            err = float(d.norm() / q.detach().norm().clamp_min(1e-30))
            print(f"{name} {i}: {err:.1e}", flush=True)
            assert err < TOL, (name, i, err)


@pytest.mark.parametrize("n", [1, 5, 61])
def test_value_aggregation(pkg, cuda, n):
    from ubio_molfm_amd import second_order as so
    e, row, col, g = _edges(n, n, cuda)
    E = e.E
    ins = [torch.randn(*s, generator=g, dtype=torch.float64) for s in ((E, H), (E, 3), (9, n, C))]

    _compare(lambda w, u, v: so._So2AggFn.apply(w, u, v, e), lambda w, u, v: ref_aggregation(w, u, v, row, col), ins, g,
             cuda)


# (a lone edge's weight does not depend on its logit: all of those gradients are exactly zero, which a relative
# error cannot judge, so the lists here hold such rows among others)
@pytest.mark.parametrize("n", [5, 61, 200])
@pytest.mark.parametrize("separate", [False, True])
def test_attention_weights(pkg, cuda, n, separate):
    from ubio_molfm_amd import second_order as so
    e, row, col, g = _edges(n, 10 + n, cuda)
    E = e.E
    gate, ih, qk = (torch.randn(E, H, generator=g, dtype=torch.float64).float().double() for _ in range(3))
    gate[E // 2:, :7] = 1.0
    qk[E // 2:, :7] = 0.75                         # rows whose maximum is attained by several edges
    p = torch.rand(E, generator=g, dtype=torch.float64).float().double()
    p[::11] = 0.0

    if separate:
        _compare(lambda i, ga, q, pp: so._AttnWeightsFn.apply(i, ga, q, pp, e),
                 lambda i, ga, q, pp: ref_alpha(ga, i, q, pp, row, n), [ih, gate, qk, p], g, cuda)
    else:
        _compare(lambda eg, q, pp: so._AttnWeightsFn.apply(eg, None, q, pp, e),
                 lambda eg, q, pp: ref_alpha(eg[:, :H], eg[:, H:], q, pp, row, n),
                 [torch.cat([gate, ih], 1), qk, p], g, cuda)


@pytest.mark.parametrize("through", ["function", "dispatch"])
def test_attention_weights_of_strided_operands(pkg, cuda, through):
    """Operands that are halves of wider tensors (QKdotS_alpha's inputhead) or transposed: their gradients of both
    orders reach the tensors they are views of."""
    from ubio_molfm_amd import second_order as so
    n = 61
    e, row, col, g = _edges(n, 71, cuda)
    E = e.E
    ins = [torch.randn(*s, generator=g, dtype=torch.float64).float().double() for s in ((E, 2 * H), (H, E), (2, E, H))]
    p = torch.rand(E, 2, generator=g, dtype=torch.float64).float().double()

    def views(wide, gate, both, pp):
        return wide.tanh().split(H, 1)[0], gate.tanh().t(), both.tanh()[1], pp.sqrt()[:, 1]

    def fn(*t):
        i, ga, q, pp = views(*t)
        return so._AttnWeightsFn.apply(i, ga, q, pp, e) if through == "function" else \
            so.attention_weights(i, ga, q, pp, e, "softmax")

    def ref(*t):
        i, ga, q, pp = views(*t)
        return ref_alpha(ga, i, q, pp, row, n)
    _compare(fn, ref, [*ins, p + 0.05], g, cuda)


@pytest.mark.parametrize("value", [float("-inf"), float("inf"), float("nan")])
@pytest.mark.parametrize("where", ["first", "last", "one_group", "all"])
def test_attention_weights_of_logits_that_are_not_finite(pkg, cuda, value, where):
    """Rows holding infinite or NaN logits: NaN where the composition has NaN, its values elsewhere (also on the
    other edges of such a row, and of a wavefront's share of the row that holds nothing else)."""
    from ubio_molfm_amd import second_order as so
    e, row, _, g = _edges(12, 3, cuda)
    e.qi = row.to(cuda)
    eg, qk = torch.randn(e.E, 2 * H, generator=g), torch.randn(e.E, H, generator=g)
    p = torch.rand(e.E, generator=g)
    for r, heads in ((1, slice(0, 5)), (2, slice(64, 128)), (4, slice(0, 128))):
        ids = torch.nonzero(row == r).flatten()
        ids = {"first": ids[:1], "last": ids[-1:], "one_group": ids[3::8], "all": ids}[where]
        for x in ids.tolist():
            eg[x, :H][heads], qk[x, heads] = value, 1.0
    eg, qk, p = (t.to(cuda) for t in (eg, qk, p))
    got, want = so._AttnWeightsFn.apply(eg, None, qk, p, e), so._softmax_weights(eg, None, qk, p, e)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    got, want = got[~nan].double(), want[~nan].double()
    assert float((got - want).norm()) <= TOL * float(want.norm())


@pytest.mark.parametrize("n,F", [(1, 4), (61, 128), (61, 100), (5, 1024)])
def test_sum_with_gathered_rows(pkg, cuda, n, F):
    from ubio_molfm_amd import second_order as so
    e, row, col, g = _edges(n, 20 + n, cuda)
    ins = [torch.randn(*s, generator=g, dtype=torch.float64) for s in ((e.E, F), (n, F), (n, F))]
    # (a quadratic of the sum, so that second-order gradients are not all zero)
    _compare(lambda y, a, b: so._AddGathersFn.apply(y, a, b, e).pow(2), lambda y, a, b: (y + a[row] + b[col]).pow(2),
             ins, g, cuda)


def test_third_order(pkg, cuda):
    """The gradient of the second-order pass: where a third order is asked for the fused kernels give way to
    differentiable compositions."""
    from ubio_molfm_amd import second_order as so
    e, row, col, g = _edges(5, 3, cuda)
    E, n = e.E, e.N
    e.qi = row.to(cuda)
    w, u, v = (torch.randn(*s, generator=g, dtype=torch.float64) for s in ((E, H), (E, 3), (9, n, C)))
    eg, qk, p = (0.5 * torch.randn(*s, generator=g, dtype=torch.float64) for s in ((E, 2 * H), (E, H), (E,)))
    p = p.abs() + 0.1

    def third(fn, x):
        x = x.clone().requires_grad_(True)
        d, = torch.autograd.grad(fn(x).pow(2).sum(), x, create_graph=True)
        d2, = torch.autograd.grad(d.pow(2).sum(), x, create_graph=True)
        return torch.autograd.grad(d2.pow(2).sum(), x)[0]
    dev = [t.to(cuda, torch.float32) for t in (u, v, eg, p)]
    for got, want in ((third(lambda t: so._So2AggFn.apply(t, dev[0], dev[1], e), w.to(cuda, torch.float32)),
                       third(lambda t: ref_aggregation(t, u, v, row, col), w)),
                      (third(lambda t: so._AttnWeightsFn.apply(dev[2], None, t, dev[3], e), qk.to(cuda, torch.float32)),
                       third(lambda t: ref_alpha(eg[:, :H], eg[:, H:], t, p, row, n), qk))):
        assert float((got.double().cpu() - want).norm() / want.norm()) < 10 * TOL


def test_third_order_of_a_strided_gradient(pkg, cuda):
    """The same with gradients that reach the functions as transposed tensors: the copies that the kernels read
    belong to no graph."""
    from ubio_molfm_amd import second_order as so
    e, row, col, g = _edges(5, 4, cuda)
    E, n = e.E, e.N
    e.qi = row.to(cuda)
    eg, qk, p = (0.5 * torch.randn(*s, generator=g, dtype=torch.float64) for s in ((E, 2 * H), (E, H), (E,)))
    p = p.abs() + 0.1

    def third(fn, x):
        x = x.clone().requires_grad_(True)
        y = fn(x).t().clone(memory_format=torch.contiguous_format).sin()      # (its gradient comes back transposed)
        d, = torch.autograd.grad(y.sum(), x, create_graph=True)
        d2, = torch.autograd.grad(d.pow(2).sum(), x, create_graph=True)
        return torch.autograd.grad(d2.pow(2).sum(), x)[0]
    dev = [t.to(cuda, torch.float32) for t in (eg, p, qk)]
    got = third(lambda t: so._AttnWeightsFn.apply(dev[0], None, t, dev[1], e), dev[2])
    want = third(lambda t: ref_alpha(eg[:, :H], eg[:, H:], t, p, row, n), qk)
    assert float((got.double().cpu() - want).norm() / want.norm()) < 10 * TOL


def test_value_aggregation_of_strided_operands_to_third_order(pkg, cuda):
    from ubio_molfm_amd import second_order as so
    e, row, col, g = _edges(5, 6, cuda)
    E, n = e.E, e.N
    ins = [0.5 * torch.randn(*s, generator=g, dtype=torch.float64) for s in ((H, E), (E, 4), (n, 9, C))]

    def chain(fn, ins):
        x = [t.clone().requires_grad_(True) for t in ins]
        y = fn(x[0].tanh().t(), x[1].tanh()[:, 1:], x[2].tanh().permute(1, 0, 2))
        z = y.transpose(-1, -2).clone(memory_format=torch.contiguous_format).sin()
        d1 = torch.autograd.grad(z.sum(), x, create_graph=True)
        d2 = torch.autograd.grad(sum(t.pow(2).sum() for t in d1), x, create_graph=True)
        return [t.detach() for t in (y, *d1, *d2, *torch.autograd.grad(sum(t.pow(2).sum() for t in d2), x))]
    got = chain(lambda w, u, v: so._So2AggFn.apply(w, u, v, e), [t.to(cuda, torch.float32) for t in ins])
    for i, (a, b) in enumerate(zip(got, chain(lambda w, u, v: ref_aggregation(w, u, v, row, col), ins))):
        rel = float((a.double().cpu() - b).norm() / b.norm())
        print(i, f"{rel:.2e}", flush=True)
        assert rel < 10 * TOL


def test_value_aggregation_rule(pkg, cuda, monkeypatch):
    """fp32 at the kernels' sizes takes them; half precision and 64 heads the composition, with the same values."""
    from ubio_molfm_amd import second_order as so
    n = 61
    e, row, col, g = _edges(n, 31, cuda)
    e.qi = row.to(cuda)
    calls = []
    real = so._lib.call
    monkeypatch.setattr(so._lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    u = torch.randn(e.E, 3, generator=g)
    for heads, dtype in ((128, torch.float32), (64, torch.float32), (128, torch.bfloat16)):
        w, v = (torch.randn(*s, generator=g).to(dtype) for s in ((e.E, heads), (9, n, C)))
        calls.clear()
        got = so.value_aggregation(w.to(cuda), u.to(cuda, dtype), v.to(cuda), e)
        assert ("e2v2_so2_agg" in calls) == (heads == 128 and dtype == torch.float32)
        ref = ref_aggregation(w.double().repeat(1, 128 // heads), u.to(dtype).double(), v.double(), row, col)
        assert float((got.double().cpu() - ref).norm() / ref.norm()) < (TOL if dtype == torch.float32 else 1e-2)


def test_other_shapes_do_not_reach_the_kernels(pkg, cuda, monkeypatch):
    """Operands that the list's sizes do not fit are refused by the composition's own checks."""
    from ubio_molfm_amd import second_order as so
    e, row, _, g = _edges(5, 33, cuda)
    e.qi = row.to(cuda)
    E, n = e.E, e.N

    def never(name, *a):
        assert not name.startswith(("e2v2_attn_weights", "e2v2_add_gather2")), name
        return real(name, *a)
    real = so._lib.call
    monkeypatch.setattr(so._lib, "call", never)
    qk, p = torch.randn(E, H, device=cuda), torch.rand(E, device=cuda)
    for eg, gate in ((torch.randn(E, 192, device=cuda), None), (torch.randn(E, H, device=cuda), None),
                     (torch.randn(E, 192, device=cuda), qk)):
        with pytest.raises(RuntimeError):
            so.attention_weights(eg, gate, qk, p, e, "softmax")
    for xq in (torch.randn(n, 64, device=cuda), torch.randn(n - 1, H, device=cuda)):
        with pytest.raises((RuntimeError, ValueError)):
            e.add_gathers(qk, xq, xq)
