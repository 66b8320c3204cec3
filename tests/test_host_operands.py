"""Operands in host memory: entry points refuse them with an error before their pointers reach a kernel, and the
host-side helpers that take them (bounding boxes, a neighbour plan of one graph) go on doing so.  No GPU needed."""
import numpy as np
import pytest
import torch

from ubio_molfm_amd import _lib, model, neighbors


@pytest.mark.parametrize("device", ["cpu", torch.device("cpu"), "meta"])
def test_stream_of_a_device_without_streams(device):
    with pytest.raises(ValueError, match="Expected a cuda device"):
        _lib.stream(device)


@pytest.mark.parametrize("call", [
    lambda p: model.spatial_order(p, [0, 5]),
    lambda p: model.spatial_order(p, [0, 2, 5]),
    lambda p: neighbors.coordinate_bounds(p),
    lambda p: neighbors.cluster_slots(torch.tensor([0, 1], dtype=torch.int32), 1, torch.zeros(1, dtype=torch.int32),
                                      None, 4),
], ids=["order_one_graph", "order_two_graphs", "bounds", "cluster_slots"])
def test_host_operands_are_refused(call, monkeypatch):
    def launched(name, *args):
        raise AssertionError(f"{name} was called with host pointers")
    monkeypatch.setattr(_lib, "call", launched)
    with pytest.raises(ValueError, match="Expected a cuda device"):
        call(torch.rand(5, 3))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_bounds_and_plan_of_one_graph_in_host_memory(dtype):
    pos = torch.rand(7, 3, generator=torch.Generator().manual_seed(0), dtype=torch.float64).to(dtype) * 20
    lo, hi = model.graph_bounds(pos, torch.tensor([7]))
    assert lo.dtype == dtype and torch.equal(lo[0], pos.amin(0)) and torch.equal(hi[0], pos.amax(0))
    args = ([0, 7], np.eye(3)[None] * 20, [[False] * 3], 5.0)
    plan = neighbors.make_plan(pos, *args, workspace=False)[0]
    box = np.stack([pos.amin(0).numpy(), pos.amax(0).numpy()])[:, None]
    want = neighbors.make_plan(pos, *args, workspace=False, grid_box=box)[0]
    assert plan.n_bins == want.n_bins and plan.n_bins > 1
