"""The attention backward's workspace: 384 bytes per edge are enough for any list (one sized for a longer list serves a
shorter one), more of it lets the head groups run at once, and the results are bitwise the same."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_longer_lists_ask_for_enough(pkg):
    from ubio_molfm_amd import _lib
    size = _lib.load().e2v2_attn_bwd_workspace
    for n in (0, 1, 98304, 98305, 120000, 10 ** 7):
        assert size(n) >= 384 * n


@pytest.mark.parametrize("tp", ["QK_alpha", "QKdot_alpha"])
@pytest.mark.parametrize("rows", [8192, 0], ids=["layer_call", "single_calls"])
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_smaller_workspaces_give_the_same_bits(pkg, cuda, monkeypatch, rows, dtype, tp):
    from ubio_molfm_amd import _lib, modules, systems
    from ubio_molfm_amd.model import MolfmAtomic, default_args
    torch.manual_seed(1)
    args = default_args(num_layers=1)
    args.backbone_config.update(tp_type=tp)
    m = MolfmAtomic(args).to(cuda).eval()
    m.decoder.set_compute_dtype(dtype)
    monkeypatch.setattr(modules, "LAYER_ROWS", rows)
    s = systems.water_box(200, 18.2, 3)
    pos, Z = torch.as_tensor(s["pos"], device=cuda), torch.as_tensor(s["Z"], device=cuda)
    lib = _lib.load()
    size = lib.e2v2_attn_bwd_workspace

    def forces():
        e, f, nl = m.energy_forces_flat(pos, Z, s["graph_ptr"], s["cell"], s["pbc"])
        return f, nl.n_edges
    want, E = forces()
    print(f"E={E}: {size(E)} bytes, a list of 98,305 edges {size(98305)}", flush=True)
    assert 32769 < E < 98304                  # (the longer list's workspace is below this one's)
    for nb in (384 * E, 384 * E + 16, size(98305), 1152 * E - 16, 1152 * E, size(98304)):
        monkeypatch.setattr(lib, "e2v2_attn_bwd_workspace", lambda n: nb)
        assert torch.equal(forces()[0], want), nb
    monkeypatch.setattr(lib, "e2v2_attn_bwd_workspace", lambda n: 384 * E - 16)
    with pytest.raises(RuntimeError, match="workspace"):
        forces()
