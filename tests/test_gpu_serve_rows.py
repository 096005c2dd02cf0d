"""Rows of requests that share the result pool, whole: many results of several
sizes held at once, in the order of submission and out of it, with a pool that
has room for about half of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows(off, nb):
    return np.concatenate([np.sort(nb[off[i]:off[i + 1]]) for i in range(len(off) - 1)] or [nb])


@pytest.mark.parametrize("slots", [1, 2, 4])
def test_rows_of_a_crowded_pool(oracle, slots):
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    base = oracle.generate_expo(30000, 6, seed=111)
    requests = []
    for i, (nq, eps) in enumerate([(9000, 0.02), (60, 0.079), (1, 0.05), (2500, 0.03), (700, 0.019), (64, 0.079)]):
        q = oracle.generate_expo(nq, 6, seed=120 + i) * (0.2 if nq < 100 else 1.0)
        off, nb = oracle.range_join(base, q, eps)
        requests.append((q, eps, off, nb))
    size = [4 * len(nb) + 8 * len(off) + 1024 for _, _, off, nb in requests]
    pool = max(2 * max(size), sum(size)) + 4096
    with H.Server(base, [0.02 * 1.0001, 0.04, 0.08], slots=slots, result_bytes=pool, max_queries=9000) as S:
        for seed in range(3):
            order = np.random.default_rng(seed).permutation(2 * len(requests)) % len(requests)
            tickets = [S.submit(*requests[i][:2]) for i in order]
            for i, t in zip(order, tickets):
                _, _, eoff, enb = requests[i]
                info = S.wait(t)
                off, nb = S.result(t)
                assert np.array_equal(off, eoff) and np.array_equal(rows(off, nb), enb)
                assert info["pair_hash"] == oracle.csr_hash(eoff, enb)
