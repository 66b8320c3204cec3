"""Attention layers and feed-forward blocks enqueued by one native call each way against the same layers launched
one kernel at a time from Python: the launches are the same, so energies, forces and node features are bitwise
equal, for every attention type, gate and weight form, in both compute modes."""
import copy
import pickle

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

VARIANTS = [dict(), dict(attn_type="zero-order"), dict(attn_type="so2-first-order+zero-order"),
            dict(tp_type="QKdot_alpha"), dict(tp_type="QKdotS_alpha+sigmoid"), dict(tp_type="QK_alpha+softplus")]


def _model(cuda, over):
    from ubio_molfm_amd.model import MolfmAtomic, default_args
    args = default_args(num_layers=2)
    args.backbone_config.update(over)
    torch.manual_seed(5)
    return MolfmAtomic(args).to(cuda).eval()


@pytest.mark.parametrize("over", VARIANTS, ids=[str(sorted(v.values())) for v in VARIANTS])
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_layer_calls_bitwise(pkg, cuda, monkeypatch, over, dtype):
    from ubio_molfm_amd import modules
    m = _model(cuda, over)
    m.decoder.set_compute_dtype(dtype)
    rng = np.random.default_rng(3)
    for counts, box in (([2], 2.0), ([2, 5, 1], 3.0), ([70, 61], 9.0)):         # the lone atom: a row without edges
        ptr = np.concatenate([[0], np.cumsum(counts)])
        n = int(ptr[-1])
        pos = torch.as_tensor(rng.random((n, 3)) * box, dtype=torch.float32, device=cuda)
        Z = torch.as_tensor(rng.choice([1, 6, 8], n), device=cuda)
        cell, pbc = np.zeros((len(counts), 3, 3)), np.zeros((len(counts), 3), bool)
        out = {}
        for rows in (8192, 0):
            monkeypatch.setattr(modules, "LAYER_ROWS", rows)
            calls = []
            real = modules._lib.call
            monkeypatch.setattr(modules._lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
            e, f, _ = m.energy_forces_flat(pos, Z, ptr, cell, pbc)
            monkeypatch.setattr(modules._lib, "call", real)
            assert ("e2v2_attn_layer_bwd" in calls) == ("e2v2_ffn_layer_bwd" in calls) == (rows > 0), calls
            out[rows] = (e, f)
        print(over, dtype, n, float(out[0][0][0]), flush=True)
        assert torch.equal(out[0][0], out[8192][0]) and torch.equal(out[0][1], out[8192][1])


def test_layer_call_follows_the_weights(pkg, cuda):
    """A weight changed in place, or replaced, is the one the next call uses."""
    m = _model(cuda, {})
    ffn = next(x for x in m.modules() if type(x).__name__ == "FeedForwardNetwork_s3")
    x = torch.randn(9, 7, 256, device=cuda)
    y0 = ffn(x, res=x)
    with torch.no_grad():
        ffn.slinear_2.weight.mul_(2.0)
        ffn.slinear_2.bias.add_(1.0)
    y1 = ffn(x, res=x)
    ffn.slinear_2.weight = torch.nn.Parameter(ffn.slinear_2.weight.detach() / 2)
    ffn.slinear_2.bias = torch.nn.Parameter(ffn.slinear_2.bias.detach() - 1)
    y2 = ffn(x, res=x)
    assert not torch.equal(y0, y1)
    torch.testing.assert_close(y1 - x, 2 * (y0 - x) + torch.eye(9, device=cuda)[0].view(9, 1, 1), rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(y2, y0, rtol=0, atol=1e-6)


def test_layer_saved_state_survives_a_saved_tensor_hook(pkg, cuda):
    m = _model(cuda, {})
    ffn = next(x for x in m.modules() if type(x).__name__ == "FeedForwardNetwork_s3")
    x = torch.randn(9, 33, 256, device=cuda, requires_grad=True)
    g = torch.randn(9, 33, 256, device=cuda)
    a = torch.autograd.grad(ffn(x), x, g)[0]
    with torch.autograd.graph.save_on_cpu():
        y = ffn(x)
    assert torch.equal(a, torch.autograd.grad(y, x, g)[0])


def test_layer_copies_and_pickles_with_its_module(pkg, cuda):
    m = _model(cuda, {})
    ffn = next(x for x in m.modules() if type(x).__name__ == "FeedForwardNetwork_s3")
    x = torch.randn(9, 5, 256, device=cuda)
    y = ffn(x)
    twin, back = copy.deepcopy(ffn), pickle.loads(pickle.dumps(ffn))
    with torch.no_grad():
        twin.slinear_2.weight.mul_(2.0)
    assert torch.equal(ffn(x), y) and torch.equal(back(x), y) and not torch.equal(twin(x), y)


@pytest.mark.parametrize("rows", [8192, 0], ids=["layer_call", "single_calls"])
def test_ffn_gradient_is_not_differentiated_again_silently(pkg, cuda, monkeypatch, rows):
    """The fused blocks leave no graph of their gradient: with create_graph=True they raise, as the fused attention
    does, where a second differentiation would have lost their terms."""
    from ubio_molfm_amd import modules
    monkeypatch.setattr(modules, "LAYER_ROWS", rows)
    m = _model(cuda, {})
    ffn = next(x for x in m.modules() if type(x).__name__ == "FeedForwardNetwork_s3")
    x = torch.randn(9, 5, 256, device=cuda, requires_grad=True)
    g = torch.randn(9, 5, 256, device=cuda)
    for res, bf16 in ((None, False), (x, False), (None, True)):
        torch.autograd.grad(ffn(x, res=res, bf16=bf16), x, g)
        with pytest.raises(NotImplementedError, match="first-order"):
            torch.autograd.grad(ffn(x, res=res, bf16=bf16), x, g, create_graph=True)
