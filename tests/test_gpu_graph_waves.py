"""Graph replays at every workgroup size, on units whose masks go to the per-wave
global scratch: the captured launch has the workgroups that its blocks and its
scratch were sized for.  Enough units that every resident wave has one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block_waves", [0, 4, 2, 1])
@pytest.mark.parametrize("dim, qb", [(3, 8), (12, 8), (6, 4)])
def test_graph_at_every_workgroup_size(oracle, dim, qb, block_waves):
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    rng = np.random.default_rng(dim)
    n, eps = 24000, 0.04
    pts = rng.random((n, dim))
    pts[:, 0] = 0.5 + 0.01 * pts[:, 0]  # k = 1: one cell, every point a candidate
    total, want = oracle.join_stats(pts, 1, eps)
    print("case", dim, qb, block_waves, total, flush=True)
    with H.GridIndex(pts, eps, indexed_dims=1) as ix:
        for _ in range(3):
            t = ix.selfjoin(refine="fp64", use_graph=True, queries_per_unit=qb, block_waves=block_waves)
            info = t.info
            off, nb = t.csr()
            t.close()
            assert (info["total_neighbors"], info["pair_hash"]) == (total, want)
            assert oracle.csr_hash(off, nb) == want and info["graph_replay"] == 1
