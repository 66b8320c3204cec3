"""The 16-byte forms of the segment kernels against float64 at the sizes where they change form: head counts that
do and do not divide the workgroup, one or many d per lane, rows longer than the staged chunk, isolated rows,
skipped slots whose clamped partner row holds infinities, and operands off the 16-byte grid (one value per lane).

Bound: a sum of n products in any order errs by at most n 2^-24 times the sum of magnitudes; n <= 700 here, and the
error of such random sums stays far below, so 64 units of 2^-24 of that scale."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 64 * 2.0 ** -24


def _layout(rows, cols, seed, long_row=True):
    g = torch.Generator().manual_seed(seed)
    deg = torch.randint(0, 40, (rows,), generator=g)
    deg[1] = 0
    if long_row:
        deg[2] = 700                              # longer than a staged chunk
    row = torch.repeat_interleave(torch.arange(rows), deg)
    E = row.numel()
    col = torch.randint(1, cols, (E,), generator=g)   # partner row 0 is only reached by skipped slots
    eid = torch.randperm(E, generator=g)
    ptr = torch.cat([torch.zeros(1, dtype=torch.long), deg.cumsum(0)])
    return ptr, row, col, eid, E


def _segments(so, ptr, col, eid, rows, cols, E, cuda):
    keep = [t.to(cuda, torch.int32) for t in (ptr, col, eid)]
    from ubio_molfm_amd import _lib
    return keep, _lib.Segments(*[so._vp(t) for t in keep], rows, cols, eid.numel(), E)


def _check(got, ref, scale):
    assert float(((got.double().cpu() - ref).abs() / (scale + 1e-30)).max()) <= TOL


@pytest.mark.parametrize("H,D,fast,shift", [(128, 18, "h", 0), (128, 8, "d", 0), (64, 9, "h", 0), (100, 7, "h", 0),
                                            (100, 4, "d", 0), (8, 33, "h", 0), (8, 32, "d", 0), (4, 1, "h", 0),
                                            (132, 24, "h", 0), (1028, 3, "h", 0), (300, 8, "d", 0), (6, 5, "h", 0),
                                            (128, 18, "h", 1), (128, 8, "d", 1)])
def test_segment_dot_and_reduce(pkg, cuda, H, D, fast, shift):
    from ubio_molfm_amd import _lib, sparse_ops as so
    rows, cols = 23, 31
    ptr, row, col, eid, E = _layout(rows, cols, H + D)
    bad = torch.zeros(E, dtype=torch.bool)
    bad[::17] = True                               # these slots name no partner row
    cmeta = torch.where(bad, torch.tensor(-1), col)
    keep, S = _segments(so, ptr, cmeta, eid, rows, cols, E, cuda)
    g = torch.Generator().manual_seed(7)

    def operand(n):
        shape = (n, D, H) if fast == "h" else (n, H, D)
        flat = torch.randn(n * H * D + shift, generator=g, dtype=torch.float32)
        t = flat.to(cuda)[shift:].view(shape)      # shift: off the 16-byte grid
        return t, (t.permute(0, 2, 1) if fast == "h" else t)
    A, a = operand(rows)
    B, b = operand(cols)
    b[0] = float("inf")
    a64, b64 = a.double().cpu(), b.double().cpu()
    ok = ~bad
    out = torch.zeros(E, H, device=cuda)
    st = _lib.vp(torch.cuda.current_stream().cuda_stream)
    _lib.call("e2v2_seg_dot", C.byref(S), so._vp(a), so._strides(a), so._vp(b), so._strides(b), _lib.i32(H),
              _lib.i32(D), so._vp(out), (C.c_int64 * 3)(H, 1, 0), st)
    ref, scale = torch.zeros(E, H, dtype=torch.float64), torch.zeros(E, H, dtype=torch.float64)
    ref[eid[ok]] = (a64[row[ok]] * b64[col[ok]]).sum(-1)
    scale[eid[ok]] = (a64[row[ok]] * b64[col[ok]]).abs().sum(-1)
    _check(out, ref, scale)
    W = torch.randn(E, H, generator=g).to(cuda)
    red = torch.full((rows, D, H) if fast == "h" else (rows, H, D), float("nan"), device=cuda)
    r = red.permute(0, 2, 1) if fast == "h" else red
    _lib.call("e2v2_seg_reduce", C.byref(S), so._vp(W), (C.c_int64 * 3)(H, 1, 0), so._vp(b), so._strides(b),
              _lib.i32(H), _lib.i32(D), so._vp(r), so._strides(r), st)
    w64 = W.double().cpu()
    terms = w64[eid[ok]].unsqueeze(-1) * b64[col[ok]]
    z = torch.zeros(rows, H, D, dtype=torch.float64)
    _check(r, z.index_add(0, row[ok], terms), z.index_add(0, row[ok], terms.abs()))
    plain = torch.full((rows, H), float("nan"), device=cuda)
    _lib.call("e2v2_seg_reduce", C.byref(S), so._vp(W), (C.c_int64 * 3)(H, 1, 0), None, None, _lib.i32(H),
              _lib.i32(1), so._vp(plain), (C.c_int64 * 3)(H, 1, 0), st)
    z = torch.zeros(rows, H, dtype=torch.float64)
    _check(plain, z.index_add(0, row, w64[eid]), z.index_add(0, row, w64[eid].abs()))


@pytest.mark.parametrize("L,H", [(1, 256), (3, 128), (5, 256), (9, 100), (4, 64), (7, 20), (2, 12), (5, 30), (10, 64)])
def test_outer_product_and_gradient(pkg, cuda, L, H):
    from ubio_molfm_amd import sparse_ops as so
    rows = 23
    ptr, row, _, eid, E = _layout(rows, 31, L * H)
    q = torch.empty(E, dtype=torch.long)
    q[eid] = row                                   # query row of each edge, not sorted
    g = torch.Generator().manual_seed(3)
    sh, fea, G = (torch.randn(*s, generator=g) for s in ((E, L), (E, H), (rows, L, H)))
    a = [t.to(cuda).requires_grad_(True) for t in (sh, fea)]
    out = so.edge_degree_outer_triton(a[0], a[1], q.to(cuda), rows)
    ds, df = torch.autograd.grad(out, a, G.to(cuda), retain_graph=True)
    s64, f64, g64 = sh.double(), fea.double(), G.double()
    terms = s64.unsqueeze(2) * f64.unsqueeze(1)
    z = torch.zeros(rows, L, H, dtype=torch.float64)
    _check(out.detach(), z.index_add(0, q, terms), z.index_add(0, q, terms.abs()))
    _check(ds, (g64[q] * f64.unsqueeze(1)).sum(2), (g64[q] * f64.unsqueeze(1)).abs().sum(2))
    _check(df, (g64[q] * s64.unsqueeze(2)).sum(1), (g64[q] * s64.unsqueeze(2)).abs().sum(1))
    only = torch.autograd.grad(out, a[1], G.to(cuda))[0]
    assert torch.equal(only, df)


@pytest.mark.parametrize("F", [4, 100, 128, 1024, 1028, 7])
def test_gather_rows(pkg, cuda, F):
    from ubio_molfm_amd import _lib, sparse_ops as so
    x = torch.randn(50, F, device=cuda)
    idx = torch.randint(0, 50, (1003,), device=cuda, dtype=torch.int32)
    idx[5], idx[1002] = -1, 50                      # outside: zero rows
    out = torch.full((1003, F), float("nan"), device=cuda)
    _lib.call("e2v2_gather_rows", so._vp(x), _lib.i64(50), so._vp(idx), _lib.i64(1003), _lib.i32(F), so._vp(out),
              so._stream(cuda))
    ref = x[idx.long().clamp(0, 49)]
    ref[5] = ref[1002] = 0
    assert torch.equal(out, ref)
