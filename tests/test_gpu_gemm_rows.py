"""The few-row tiles of the split GEMMs at their edges: row counts around the 32-row tile and around the switch to
the 128 x 128 tiles, K from one 16-k stage (three of the four wavefronts that split it idle) over stage counts
that do not divide by four, every operand form; and the Q/K projection likewise.  The one-piece forms, which do
not split K, bitwise between few and many rows.

Error over the GEMM's own scale sum_k |a| |b|, as in test_gpu_gemm.py: at most 8 units of 2^-24 times
max(sqrt(k), 4) (the sums are of at least six fp32-rounded terms per 16 k); one-piece (bf16) operands against
float64 products of the rounded operands under the same bound."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
L_OF_M = [0, 1, 1, 1, 2, 2, 2, 2, 2]


def _err(c, a64, w64):
    scale = a64.abs() @ w64.abs().transpose(-1, -2)
    return float(((c.double() - a64 @ w64.transpose(-1, -2)).abs() / (scale + 1e-300)).max())


@pytest.mark.parametrize("m,n,k,batch", [(1, 128, 16, 1), (31, 128, 32, 3), (32, 256, 48, 2), (33, 256, 144, 9),
                                         (65, 384, 256, 9), (700, 128, 1536, 2), (2560, 128, 80, 2),
                                         (2561, 128, 80, 2)])
@pytest.mark.parametrize("form", ["fp32", "one piece", "bf16 A"])
def test_few_rows_against_float64(pkg, cuda, m, n, k, batch, form):
    from ubio_molfm_amd import gemm
    g = torch.Generator().manual_seed(m + k)
    a = torch.randn(batch, m, k, generator=g).to(cuda)
    w = (torch.randn(2, n, k, generator=g) / math.sqrt(k)).to(cuda)
    widx = [b % 2 for b in range(batch)]
    pw = gemm.pack(w, pieces=3 if form == "fp32" else 1)
    if form == "bf16 A":
        a = a.bfloat16()
    out = torch.full((batch, m, n), float("nan"), device=cuda)
    gemm.gemm(a, pw, out, widx)
    if form != "fp32":
        a, w = a.bfloat16(), w.bfloat16()
    err = _err(out, a.double(), w.double()[widx])
    print(f"{form} m={m} k={k}: {err / U:.2f} u", flush=True)
    assert err <= 8 * U * max(math.sqrt(k), 4.0)


@pytest.mark.parametrize("m", [1, 33, 300])
def test_few_rows_strided_bias_residual_and_mixed_group(pkg, cuda, m):
    """Rows of a wider matrix, a bias on the first batch, the residual read from the output, a bf16 output;
    and a group whose members straddle the switch, bitwise equal to their own launches."""
    from ubio_molfm_amd import gemm
    g = torch.Generator().manual_seed(m)
    n, k, batch = 256, 144, 3
    wide = torch.randn(batch, m, k + 48, generator=g).to(cuda)
    a = wide[:, :, 16:16 + k]
    w = (torch.randn(2, n, k, generator=g) / 12).to(cuda)
    bias, res = torch.randn(n, generator=g).to(cuda), torch.randn(batch, m, n, generator=g).to(cuda)
    out = res.clone()
    gemm.gemm(a, gemm.pack(w), out, [1, 0, 1], bias=bias, bias_batches=1, res=out)
    ref = a.double() @ w.double()[[1, 0, 1]].transpose(1, 2).contiguous() + res.double()
    ref[0] += bias.double()
    scale = a.double().abs() @ w.double()[[1, 0, 1]].abs().transpose(1, 2).contiguous() + res.double().abs() + 4
    assert float(((out.double() - ref).abs() / scale).max()) <= 8 * U * math.sqrt(k)
    big = torch.randn(2600, k, generator=g).to(cuda)
    p1 = gemm.pack(w[0], pieces=3)
    outs, refs = [], []
    problems = []
    for t in (a[0], big, a[1]):
        o = torch.empty(t.shape[0], n, device=cuda)
        r = torch.empty_like(o)
        gemm.gemm(t, p1, r, bias=bias)
        problems.append(dict(a=t, pw=p1, out=o, bias=bias))
        outs.append(o)
        refs.append(r)
    gemm.gemm_grouped(problems)
    assert all(torch.equal(o, r) for o, r in zip(outs, refs))
    ob = torch.empty(m, n, dtype=torch.bfloat16, device=cuda)
    gemm.gemm(a[0], p1, ob, bias=bias)
    assert torch.equal(ob, refs[0].bfloat16())


@pytest.mark.parametrize("n,hid", [(1, 512), (33, 64), (300, 512), (1024, 128), (1025, 128)])
@pytest.mark.parametrize("with_v", [True, False])
def test_qk_projection_few_rows(pkg, cuda, n, hid, with_v):
    """y, hq, hk and the input gradient against float64, on both sides of the switch."""
    from ubio_molfm_amd import gemm
    torch.manual_seed(n + hid)
    C, Cv = 256, 256
    W = torch.randn(3, 4 * hid, C, device=cuda) / 16
    b = torch.randn(4 * hid, device=cuda)
    Wv = torch.randn(3, Cv, C, device=cuda) / 16
    P = gemm.pack_qk(W, b, Wv)
    x = torch.randn(9, n, C, device=cuda)
    hq, hk, y = gemm.qk_forward(x, P)
    _, order = gemm.qk_orders(hid)
    ym = torch.empty(9, n, 4 * hid, device=cuda)
    ym[:, :, torch.as_tensor(order, device=cuda)] = y
    y64 = x.double() @ W.double()[L_OF_M].transpose(1, 2).contiguous()
    y64[0] += b.double()
    assert float((ym.double() - y64).norm() / y64.norm()) < 2e-6
    for got, o in ((hq, 0), (hk, 2 * hid)):
        p = y64[:, :, o:o + hid] * y64[:, :, o + hid:o + 2 * hid]
        ref = torch.cat([p[:1].sum(0), p[1:4].sum(0), p[4:].sum(0)], 1)
        assert float((got.double() - ref).norm() / ref.norm()) < 4e-6
    ghq, ghk = torch.randn(n, 3 * hid, device=cuda), torch.randn(n, 3 * hid, device=cuda)
    gv = torch.randn(9, n, Cv, device=cuda) if with_v else None
    gx = gemm.qk_backward(y, ghq, ghk, gv, P)
    gq = torch.stack([ghq[:, l * hid:(l + 1) * hid] for l in L_OF_M]).double()
    gk = torch.stack([ghk[:, l * hid:(l + 1) * hid] for l in L_OF_M]).double()
    qa, qb, ka, kb = y64.split(hid, dim=2)
    ref = torch.cat([qb * gq, qa * gq, kb * gk, ka * gk], dim=2) @ W.double()[L_OF_M]
    if with_v:
        ref = ref + gv.double() @ Wv.double()[L_OF_M]
    assert float((gx.double() - ref).norm() / ref.norm()) < 4e-6


def _same_rows(few, many, at, m):
    assert torch.equal(few, many[..., at:at + m, :])


@pytest.mark.parametrize("m,n,k", [(1, 128, 16), (33, 256, 144), (700, 512, 256), (2500, 256, 512),
                                   (768, 128, 48), (1024, 128, 48), (1536, 128, 48)])
@pytest.mark.parametrize("form", ["fp32 A", "bf16 A", "gated"])
def test_one_piece_rows_do_not_depend_on_the_call(pkg, cuda, m, n, k, form):
    """bf16 mode: a row's result is bitwise the same among few rows as among many, alone and in a group (a sum in
    another order would be rounded to another bf16 further on)."""
    from ubio_molfm_amd import gemm
    g = torch.Generator().manual_seed(m + n)
    batch, many, at = 3, 6000, 3211
    a = torch.randn(batch, many, k, generator=g).to(cuda)
    w = (torch.randn(2, n, k, generator=g) / math.sqrt(k)).to(cuda)
    bias, res = torch.randn(n, generator=g).to(cuda), torch.randn(batch, many, n, generator=g).to(cuda)
    pw, widx = gemm.pack(w, pieces=1), [0, 1, 0]
    logits = torch.randn(many, 2 * k, generator=g).to(cuda)
    if form == "bf16 A":
        a = a.bfloat16()

    def run(rows, dtype, grouped=False):
        x, r = a[:, rows].contiguous(), res[:, rows].contiguous()
        out = torch.empty(batch, x.shape[1], n, device=cuda, dtype=dtype)
        if grouped:
            gemm.gemm_grouped([dict(a=x, pw=pw, out=out, widx=widx, bias=bias, res=r),
                               dict(a=a[0], pw=pw, out=torch.empty(many, n, device=cuda), widx=[1])])
        else:
            gate = (logits[rows].contiguous(), 1.5, 0.75) if form == "gated" else None
            gemm.gemm(x, pw, out, widx, bias=bias, bias_batches=1, res=r, gate=gate)
        return out
    some = slice(at, at + m)
    for dtype in (torch.float32, torch.bfloat16):
        _same_rows(run(some, dtype), run(slice(None), dtype), at, m)
    if form != "gated":
        assert torch.equal(run(some, torch.float32, True), run(slice(None), torch.float32, True)[:, some])


@pytest.mark.parametrize("n,hid", [(1, 512), (33, 64), (300, 192), (1024, 512)])
@pytest.mark.parametrize("y_bf16", [True, False])
def test_one_piece_qk_projection_does_not_depend_on_the_call(pkg, cuda, n, hid, y_bf16):
    from ubio_molfm_amd import gemm
    torch.manual_seed(n + hid)
    C, Cv, many, at = 256, 256, 2100, 1007
    W, b = torch.randn(3, 4 * hid, C, device=cuda) / 16, torch.randn(4 * hid, device=cuda)
    P = gemm.pack_qk(W, b, torch.randn(3, Cv, C, device=cuda) / 16, pieces=1)
    x = torch.randn(9, many, C, device=cuda)
    ghq, ghk = torch.randn(many, 3 * hid, device=cuda), torch.randn(many, 3 * hid, device=cuda)
    gv = torch.randn(9, many, Cv, device=cuda)
    some = slice(at, at + n)
    out = []
    for rows in (slice(None), some):
        hq, hk, y = gemm.qk_forward(x[:, rows].contiguous(), P, y_bf16=y_bf16)
        out.append([hq, hk, y])
        for v in (gv[:, rows].contiguous(), None):
            out[-1].append(gemm.qk_backward(y, ghq[rows].contiguous(), ghk[rows].contiguous(), v, P))
    for all_rows, few in zip(*out):
        _same_rows(few, all_rows, at, n)


def test_bf16_layers_do_not_depend_on_the_batch(pkg, cuda):
    """Degree embedding, attention layer and feed-forward block of the bf16 mode: a molecule among copies of itself
    has bitwise the features and gradients that it has alone."""
    import numpy as np
    from ubio_molfm_amd import modules, neighbors, ops
    from ubio_molfm_amd.model import MolfmAtomic, default_args
    torch.manual_seed(2)
    m = MolfmAtomic(default_args(num_layers=1)).to(cuda).eval().requires_grad_(False)
    dec, rng, n = m.decoder.decoder, np.random.default_rng(4), 33
    one = torch.as_tensor(rng.random((n, 3)) * 6.0, dtype=torch.float32)
    Z1 = torch.as_tensor(rng.choice([1, 6, 8], n))
    x1, g1 = torch.randn(9, n, 256), torch.randn(9, n, 256)
    out = []
    for copies in (1, 130):
        ptr = np.arange(copies + 1) * n
        pos = one.repeat(copies, 1).to(cuda)
        Z = Z1.repeat(copies).to(cuda)
        nl = neighbors.build_neighbors(pos, ptr, np.zeros((copies, 3, 3)), np.zeros((copies, 3), bool), 6.0)
        type_z, type_key, slot = modules.atom_type_slots(Z, ptr)
        pos.requires_grad_(True)
        x, g = (t.repeat(1, copies, 1).to(cuda) for t in (x1, g1))
        x.requires_grad_(True)
        dvec, dist = ops.EdgeGeometryFn.apply(pos, nl)
        ctx = modules.EdgeContext(nl, dvec, dist, slot, type_z, type_key, dec.rbf, 6.0, True)
        d = dec.edge_deg_embed_dense(ctx)
        y = dec.blocks[0].ga(x, ctx)
        z = dec.blocks[0].ffn(y, bf16=True)
        grads = torch.autograd.grad([d, y, z], [x, pos], [g, g, g])
        out.append([t[..., :n, :] for t in (d.detach(), y.detach(), z.detach(), *grads)])
    for alone, among in zip(*out):
        assert torch.equal(alone, among)
