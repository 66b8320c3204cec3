"""Host-side pieces of the training path that are plain PyTorch compositions
(no HIP call), checked on the CPU in float64 against the modules they stand in
for: the per-edge Linear with the split-K weight gradient (values, forces-style
first differentiation with create_graph=True, and the second differentiation to
the inputs and parameters, including a first differentiation that skips the
weight gradient), the split-K product with rows left over, and run_seq over a
RadialProfile net (on the CPU every LayerNorm + SiLU pair runs as the modules)."""
import pytest
import torch

from ubio_molfm_amd import modules
from ubio_molfm_amd import second_order as so


def _rel(a, b):
    return float((a - b).norm() / b.norm().clamp_min(1e-300))


def test_splitk_matches_plain_product():
    g = torch.Generator().manual_seed(1)
    for E in (5, 2048 * 3, 2048 * 32 + 7, 2048 * 40 + 1):
        a = torch.randn(E, 9, generator=g, dtype=torch.float64)
        b = torch.randn(E, 5, generator=g, dtype=torch.float64)
        assert _rel(so._splitk_tn(a, b), a.t() @ b) < 1e-13, E


def test_edge_linear_second_order_matches_linear():
    torch.manual_seed(0)
    E, k, n = 2048 * 4 + 37, 24, 16
    lin = torch.nn.Linear(k, n).double()
    p = torch.randn(E, k, dtype=torch.float64, requires_grad=True)
    R = torch.randn(E, k, dtype=torch.float64)

    def run(f):
        x = torch.sin(p) * 1.3
        y = f(x)
        e = (torch.tanh(y) ** 2).sum()
        gp, = torch.autograd.grad(e, p, create_graph=True)     # the weight gradient is not asked for
        L = (gp * R).sum() + e
        return [y, gp] + list(torch.autograd.grad(L, [p, lin.weight, lin.bias]))

    got = run(lambda x: so.edge_linear(lin, x))
    ref = run(lin)
    for a, b in zip(got, ref):
        assert _rel(a, b) < 1e-12


def test_run_seq_matches_radial_profile_on_cpu():
    torch.manual_seed(2)
    prof = modules.RadialProfile([32, 64, 64, 16]).double()
    h = torch.randn(300, 64, dtype=torch.float64)
    assert not so.ln_silu_fusable(prof.net[1], h)
    assert torch.equal(so.run_seq(prof.net[1:], h), prof.net[1:](h))


class _HostEdges:
    """The value aggregation of an edge list in plain PyTorch."""

    def __init__(self, row, col, n):
        self.row, self.col, self.N, self.E = row, col, n, row.numel()

    def v_agg(self, value, alpha):
        out = torch.zeros(self.N, *value.shape[1:], dtype=value.dtype)
        return out.index_add(0, self.row, value[self.col] * alpha.unsqueeze(1).to(value.dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,channels,heads", [(9, 256, 128), (9, 128, 128), (9, 256, 64), (4, 256, 128)])
def test_value_aggregation_of_other_types_and_sizes(monkeypatch, dtype, rows, channels, heads):
    """The fused kernels take raw pointers and fixed sizes: operands of another type, size or device never reach
    them and run the composition."""
    def never(*a):
        raise AssertionError("the kernel was called")
    monkeypatch.setattr(so._lib, "call", never)
    g = torch.Generator().manual_seed(5)
    n, E = 7, 30
    row, col = torch.randint(0, n, (2, E), generator=g)
    w, u, v = (torch.randn(*s, generator=g).to(dtype) for s in ((E, heads), (E, 3), (rows, n, channels)))
    got = so.value_aggregation(w, u, v, _HostEdges(row, col, n))
    assert got.shape == (3, rows, n, channels) and got.dtype == dtype
    t = w.double().repeat(1, channels // heads).unsqueeze(0) * v.double()[:, col]
    ref = torch.stack([torch.zeros(rows, n, channels, dtype=torch.float64).index_add(1, row, t * u.double()[:, k:k + 1])
                       for k in range(3)])
    # up to 30 terms of three factors, each product and sum rounded once in the type
    assert _rel(got.double(), ref) < 40 * torch.finfo(dtype).eps
