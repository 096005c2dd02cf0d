"""Unit distribution and output chunks of the grid joins: static first grabs,
per-XCD queues and stealing for every split, from fewer units than waves to
many grabs per wave; and estimates far below the result, so chunks run into
the end of the batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    return H


@pytest.mark.parametrize("n", [1, 70, 3000, 60000])
@pytest.mark.parametrize("dim", [2, 3, 6])
def test_unit_distribution(H, oracle, n, dim):
    pts = oracle.generate_expo(n, dim, seed=n + dim)
    eps = {2: 0.0008, 3: 0.003, 6: 0.012}[dim]
    eoff, enb = oracle.join(pts, dim, eps)
    print("case", n, dim, len(enb), flush=True)
    with H.GridIndex(pts, eps) as ix:
        for parts in (1, 3, 8):
            for grab in (0, 1, 3, 64):
                for waves in (1, 2, 4):
                    for by_block in (0, 1):
                        t = ix.selfjoin(xcd_parts=parts, units_per_grab=grab, block_waves=waves,
                                        part_by_block=by_block)
                        info = t.info
                        t.close()
                        assert info["total_neighbors"] == len(enb), (parts, grab, waves, by_block)
                        assert info["pair_hash"] == oracle.csr_hash(eoff, enb)


def test_skewed_units(H, oracle):
    """A few dense cells among many sparse ones: unit sizes three orders of
    magnitude apart, small and large reservations mixed, sampled by an
    estimate that sees few of the dense ones."""
    rng = np.random.default_rng(1)
    sparse = rng.random((60000, 2))
    dense = 0.5 + rng.random((6000, 2)) * 0.004
    pts = np.concatenate([sparse, dense])
    eps = 0.002
    eoff, enb = oracle.join(pts, 2, eps)
    with H.GridIndex(pts, eps) as ix:
        for qb in (4, 8, 16):
            for refine in ("fp64", "f32"):
                t = ix.selfjoin(queries_per_unit=qb, refine=refine, xcd_parts=8)
                off, nb = t.csr()
                t.close()
                assert np.array_equal(off, eoff) and np.array_equal(nb, enb)
