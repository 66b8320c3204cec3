"""The training path's weight-gradient kernel (dW per degree, summed over its m-rows and the nodes) and the sums of
per-block partial rows, at the edges of their chunks and tiles, against float64; and the SO(3) linear built on them
to the third order.

Weight gradient: sums of K = (2 l + 1) n fp32 products in chunks, error over sum |a| |b| at most 8 units of 2^-24
times max(sqrt(K), 4), the bound of the GEMM tests.  Partial sums: at most rows / 128 + 8 additions in a chain,
each one rounding of a partial sum that sum |x| bounds."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


@pytest.mark.parametrize("n,m,k", [(1, 64, 64), (24, 256, 256), (63, 128, 64), (65, 64, 192), (412, 512, 256),
                                   (1501, 256, 512), (9000, 64, 64)])
@pytest.mark.parametrize("bounds", [(0, 1, 4, 9), (0, 1)])
def test_wgrad_against_float64(pkg, cuda, n, m, k, bounds):
    from ubio_molfm_amd import _lib
    g = torch.Generator().manual_seed(n + m)
    B = bounds[-1]
    wide = torch.randn(B, n, m + 6, generator=g).to(cuda)
    a, b = wide[:, :, 2:2 + m], torch.randn(B, n, k, generator=g).to(cuda)
    chunks = int(_lib.load().e2v2_wgrad_chunks(n, B, m, k))
    part = torch.full((B * chunks, m, k), float("nan"), device=cuda)
    out = torch.full((len(bounds) - 1, m, k), float("nan"), device=cuda)
    print(f"n={n} m={m} k={k} batches={B} chunks={chunks}", flush=True)
    _lib.call("e2v2_wgrad", _lib.vp(a.data_ptr()), _lib.i64(m + 6), _lib.i64(n * (m + 6)), _lib.vp(b.data_ptr()),
              _lib.i64(k), _lib.i64(n * k), _lib.i32(n), _lib.i32(B), _lib.i32(m), _lib.i32(k),
              (C.c_int32 * len(bounds))(*bounds), _lib.i32(len(bounds) - 1), _lib.vp(part.data_ptr()),
              _lib.vp(out.data_ptr()), _lib.stream(cuda))
    for i, (p, q) in enumerate(zip(bounds, bounds[1:])):
        A, Bm = a[p:q].double().reshape(-1, m), b[p:q].double().reshape(-1, k)
        scale = A.abs().t().contiguous() @ Bm.abs()
        err = float(((out[i].double() - A.t().contiguous() @ Bm).abs() / scale).max())
        print(f"  group {i}: {err / U:.2f} u", flush=True)
        assert err <= 8 * U * max(A.shape[0] ** 0.5, 4.0)


def test_wgrad_infinities_stay_in_their_columns(pkg, cuda):
    from ubio_molfm_amd import second_order as so
    a, b = torch.randn(9, 40, 64, device=cuda), torch.rand(9, 40, 64, device=cuda) + 0.5
    a[5, 7, 3], a[0, 1, 2] = float("inf"), float("nan")
    d = so._DegreeWGradFn.apply(a, b)
    assert bool((d[2, 3] == float("inf")).all()) and bool(d[0, 2].isnan().all())
    d[2, 3] = 0
    d[0, 2] = 0
    assert bool(d.isfinite().all())


@pytest.mark.parametrize("rows,w", [(1, 4), (3, 128), (64, 256), (65, 36), (129, 512), (2048, 128), (1024, 1024)])
@pytest.mark.parametrize("groups", [1, 2])
def test_sum_parts(pkg, cuda, rows, w, groups):
    from ubio_molfm_amd import second_order as so
    x = torch.randn(groups, rows, w, generator=torch.Generator().manual_seed(rows)).to(cuda)
    out, x64 = so._sum_parts(x), x.double()
    assert bool(((out.double() - x64.sum(1)).abs() <= (rows / 128 + 8) * U * x64.abs().sum(1) + 1e-300).all())


@pytest.mark.parametrize("n,hid", [(1, 4), (33, 12), (130, 512)])
def test_m_contraction_to_third_order(pkg, cuda, n, hid):
    """Each value is at most five products and sums per order (relative 2^-24 each of sum |a| |b|)."""
    from ubio_molfm_amd import second_order as so
    g = torch.Generator().manual_seed(n)
    a, b, r = (torch.randn(s, generator=g).to(cuda) for s in ((9, n, hid), (9, n, hid), (n, 3 * hid)))

    def compose(a, b):
        return torch.cat([p.sum(0) for p in (a * b).split([1, 3, 5])], dim=-1)

    def chain(f, a, b, r):
        a, b = a.clone().requires_grad_(True), b.clone().requires_grad_(True)
        h = f(a, b)
        d1 = torch.autograd.grad((h * h * r).sum(), (a, b), create_graph=True)
        d2 = torch.autograd.grad(sum((t * t).sum() for t in d1), (a, b), create_graph=True)
        return [t.detach() for t in (h, *d1, *d2, *torch.autograd.grad(sum((t * t).sum() for t in d2), (a, b)))]

    for i, (x, y) in enumerate(zip(chain(so._MDotFn.apply, a, b, r), chain(compose, a.double(), b.double(), r.double()))):
        rel = float((x.double() - y).norm() / y.norm())
        print(n, hid, i, f"{rel:.2e}", flush=True)
        assert rel < 1e-5


@pytest.mark.parametrize("n", [1, 37])
def test_so3_linear_to_third_order(pkg, cuda, n):
    """y, its gradients, and the gradients of scalar functions of these, twice over, against float64."""
    from ubio_molfm_amd import second_order as so
    from ubio_molfm_amd.modules import SO3_Linear_e2former
    torch.manual_seed(n)
    lin = SO3_Linear_e2former(64, 128, lmax=2).to(cuda)
    torch.nn.init.normal_(lin.bias)
    x, r = torch.randn(9, n, 64, device=cuda), torch.randn(9, n, 128, device=cuda)

    def chain(lin, x, r):
        x = x.clone().requires_grad_(True)
        ps = [x, lin.weight, lin.bias]
        y = so.so3_linear(lin, x)
        out = [y]
        d1 = torch.autograd.grad((y * y * r).sum(), ps, create_graph=True)
        d2 = torch.autograd.grad(sum((t * t).sum() for t in d1), ps, create_graph=True)
        d3 = torch.autograd.grad(sum((t * t).sum() for t in d2), ps)
        return [t.detach() for t in (*out, *d1, *d2, *d3)]

    got = chain(lin, x, r)
    ref = chain(lin.double(), x.double(), r.double())
    for i, (a, b) in enumerate(zip(got, ref)):
        rel = float((a.double() - b).norm() / b.norm())
        print(n, i, f"{rel:.2e}", flush=True)
        # relative error of a sum of at most 9 n x 128 products per order, orders chained three deep
        assert rel < 1e-5


@pytest.mark.parametrize("name", ["m_contraction", "m_expansion", "weight_gradient"])
def test_third_order_of_strided_operands(pkg, cuda, name):
    """Operands that are views, and incoming gradients that are transposed: the copies that the kernels read belong
    to no graph.  Bound as above."""
    from ubio_molfm_amd import second_order as so
    g = torch.Generator().manual_seed(7)
    n, w = 13, 64
    shapes = {"m_contraction": ((n, 9, w), (n, 9, w)), "m_expansion": ((3 * w, n), (n, 9, w)),
              "weight_gradient": ((n, 9, w), (n, 9, w))}[name]
    ins = [0.3 * torch.randn(s, generator=g) for s in shapes]

    def of(t):
        return t.tanh().t() if t.dim() == 2 else t.tanh().permute(1, 0, 2)

    def compose(a, b):
        if name == "m_contraction":
            return torch.cat([p.sum(0) for p in (a * b).split([1, 3, 5])], dim=-1)
        if name == "m_expansion":
            return torch.cat([a.view(n, 3, w)[:, l].unsqueeze(0) * b[l * l:(l + 1) ** 2] for l in range(3)])
        return torch.stack([(a[p:q].reshape(-1, w).t().contiguous() @ b[p:q].reshape(-1, w).contiguous())
                            for p, q in ((0, 1), (1, 4), (4, 9))])
    fn = {"m_contraction": so._MDotFn, "m_expansion": so._MExpandFn, "weight_gradient": so._DegreeWGradFn}[name].apply

    def chain(f, ins):
        x = [t.clone().requires_grad_(True) for t in ins]
        y = f(*map(of, x))
        z = y.transpose(-1, -2).clone(memory_format=torch.contiguous_format).sin()    # (its gradient: transposed)
        d1 = torch.autograd.grad(z.sum(), x, create_graph=True)
        d2 = torch.autograd.grad(sum(t.pow(2).sum() for t in d1), x, create_graph=True)
        return [t.detach() for t in (y, *d1, *d2, *torch.autograd.grad(sum(t.pow(2).sum() for t in d2), x))]

    got = chain(fn, [t.to(cuda) for t in ins])
    for i, (a, b) in enumerate(zip(got, chain(compose, [t.double() for t in ins]))):
        rel = float((a.double().cpu() - b).norm() / b.norm())
        print(name, i, f"{rel:.2e}", flush=True)
        assert rel < 1e-5
