"""GPU test of the serving loop's admission: a client that collects results in
the order it submitted them is served however the counts end, also when later
and quicker requests could take all of the result-buffer pool.  No reference
counterpart."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [2, 4])
def test_collecting_in_submission_order(oracle, slots):
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    base = oracle.generate_expo(30000, 6, seed=101)
    slow = oracle.generate_expo(20000, 6, seed=102)  # many queries, ~3M pairs
    quick = 0.2 * oracle.generate_expo(60, 6, seed=103)  # few, near most points
    q_off, q_nb = oracle.range_join(base, quick, 0.079)
    s_off, s_nb = oracle.range_join(base, slow, 0.02)
    one, first = 4 * len(q_nb) + 1024, 4 * len(s_nb) + 8 * len(s_off) + 1024
    pool = 2 * max(first, 2 * one) + 4096
    with H.Server(base, [0.02 * 1.0001, 0.08], slots=slots, result_bytes=pool, max_queries=20000) as S:
        for _ in range(3):
            tickets = [S.submit(slow, 0.02)] + [S.submit(quick, 0.079) for _ in range(12)]
            got = [S.result(t) for t in tickets]
            assert np.array_equal(got[0][0], s_off) and len(got[0][1]) == len(s_nb)
            for off, nb in got[1:]:
                assert np.array_equal(off, q_off) and len(nb) == len(q_nb)
        assert S.stats()["pool_peak"] <= pool
