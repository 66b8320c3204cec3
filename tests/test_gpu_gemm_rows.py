"""The K-split tiles of the split GEMMs (matrices of few rows) at their edges: row counts around the 32-row
tile and around the switch to the 128 x 128 tiles, K from one 16-k stage (three of the four wavefronts idle)
over stage counts that do not divide by four, every operand form; and the Q/K projection likewise.

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
