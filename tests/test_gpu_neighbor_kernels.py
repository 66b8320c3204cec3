"""The neighbour build's helper kernels at the sizes where they change form: the multi-workgroup exclusive scan,
and column clusters around the merge kernel's item limit and with segments out of order (left to the sort)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 63, 1023, 1024, 1025, 262144, 262145, 500001])
def test_exclusive_scan(pkg, cuda, n):
    from ubio_molfm_amd import _lib
    rng = np.random.default_rng(n)
    a = rng.integers(0, 200, n).astype(np.int32)
    d = torch.as_tensor(a, device=cuda)
    out = torch.full((n + 1,), -1, dtype=torch.int32, device=cuda)
    stats = torch.full((2,), -1, dtype=torch.int32, device=cuda)
    _lib.call("e2v2_scan_i32", _lib.vp(d.data_ptr() if n else 0), _lib.i32(n), _lib.vp(out.data_ptr()),
              _lib.vp(stats.data_ptr()), _lib.vp(torch.cuda.current_stream().cuda_stream))
    ref = np.concatenate([[0], np.cumsum(a.astype(np.int64))])
    assert np.array_equal(out.cpu().numpy(), ref)
    assert stats.tolist() == [int(ref[-1]), int(a.max()) if n else 0]


@pytest.mark.parametrize("per_segment", [1, 255, 256, 257, 300])
@pytest.mark.parametrize("shuffled", [False, True])
def test_cluster_slots_at_the_merge_limit(pkg, cuda, per_segment, shuffled):
    """Clusters of four segments of 4 to 1,200 items (the merge holds 1,024), members repeated within and across
    segments; with one segment of every other cluster out of order.  Slots equal those of the definition: one per
    (member, occurrence) in order, the edge of each segment or -1."""
    from ubio_molfm_amd import neighbors
    rng = np.random.default_rng(per_segment)
    n_seg, span = 19, 4                              # the last cluster has three segments
    sizes = rng.integers(max(0, per_segment - 2), per_segment + 1, n_seg)
    sizes[5] = 0
    ptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    member = np.concatenate([np.sort(rng.integers(0, 2 * per_segment, k)) for k in sizes]).astype(np.int32)
    if shuffled:
        for seg in (2, 9, 17):
            member[ptr[seg]:ptr[seg + 1]] = member[ptr[seg]:ptr[seg + 1]][::-1]
    E = len(member)
    eid = rng.permutation(E).astype(np.int32)        # item -> edge id; member is indexed by edge id
    by_edge = np.empty(E, np.int32)
    by_edge[eid] = member
    t = [torch.as_tensor(x, device=cuda) for x in (ptr, by_edge, eid)]
    sm, se, ns = neighbors.cluster_slots(t[0], n_seg, t[1], t[2], span)
    sm, se, ns = sm.cpu().numpy(), se.cpu().numpy(), ns.cpu().numpy()
    for c in range((n_seg + span - 1) // span):
        want = {}
        for r, seg in enumerate(range(c * span, min(c * span + span, n_seg))):
            seen = {}
            for q in range(ptr[seg], ptr[seg + 1]):
                m = int(member[q])
                k = seen.get(m, 0)
                seen[m] = k + 1
                want.setdefault((m, k), [-1] * span)[r] = int(eid[q])
        b, keys = ptr[c * span], sorted(want)
        assert ns[c] == len(keys)
        assert [int(x) for x in sm[b:b + len(keys)]] == [k[0] for k in keys]
        assert se[b:b + len(keys)].tolist() == [want[k] for k in keys]


@pytest.mark.parametrize("n", [1, 2, 63, 256, 257, 65536, 99999])
def test_coordinate_bounds(pkg, cuda, n):
    """Exactly the smallest and largest coordinates; NaN where one is, infinities kept."""
    from ubio_molfm_amd.neighbors import coordinate_bounds
    pos = (torch.randn(n, 3, generator=torch.Generator().manual_seed(n)) * 50).to(cuda)
    b = coordinate_bounds(pos)
    assert torch.equal(b[0], pos.amin(0)) and torch.equal(b[1], pos.amax(0))
    pos[n // 2, 1], pos[n - 1, 2] = float("nan"), float("-inf")
    b = coordinate_bounds(pos)
    assert bool(b[:, 1].isnan().all()) and float(b[0, 2]) == float("-inf")
    assert torch.equal(b[:, 0], torch.stack([pos[:, 0].amin(), pos[:, 0].amax()]))
