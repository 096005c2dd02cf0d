"""GPU tests of a request's plan: its three-launch form for few queries, the
split of heavy units into segments, and the general form, at the sizes where
one gives way to the other.  The oracle is oracle.range_join; rows have to be
the same, in the same order, whichever form planned them.  No reference
counterpart."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 0.04


@pytest.fixture(scope="module")
def H():
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    return H


def data(oracle, dim):
    """A dense spot (heavy units) in a thin spread, and queries of both kinds,
    some of them outside every cell."""
    base = oracle.generate_expo(6000, dim, seed=71)
    base[:4000] = 0.3 + 0.05 * base[:4000]
    q = oracle.generate_expo(4200, dim, seed=72)
    q[::3] = 0.3 + 0.05 * q[::3]
    q[5::50] += 3.0
    return base, q


@pytest.mark.parametrize("dim", [2, 6, 3])
def test_rows_at_the_edges_of_the_plans(H, oracle, dim):
    base, q = data(oracle, dim)
    off, nb = oracle.range_join(base, q, EPS)
    big = np.tile(q, (12, 1))  # 50400 queries: no unit is split
    with H.Server(base, [0.05], slots=1, result_bytes=1 << 30, max_queries=len(big)) as S:
        t = S.submit(big, EPS)
        assert S.wait(t)["pairs"] == 12 * len(nb)
        boff, bnb = S.result(t)
        assert np.array_equal(boff[:len(off)], off)
        whole = bnb[:len(nb)]
        rows = whole.copy()
        for i in range(len(q)):
            rows[off[i]:off[i + 1]].sort()
        assert np.array_equal(rows, nb)
        for nq in (1, 2, 63, 64, 65, 513, 1023, 1025, 3072, 4095, 4096, 4097, 4200):
            print("dim", dim, "nq", nq, flush=True)
            t = S.submit(q[:nq], EPS)
            info = S.wait(t)
            o, b = S.result(t)
            assert np.array_equal(o, off[:nq + 1])
            assert np.array_equal(b, whole[:off[nq]])
            assert info["pair_hash"] == oracle.csr_hash(off[:nq + 1], nb[:off[nq]])


def test_only_dead_queries(H, oracle):
    base, q = data(oracle, 6)
    with H.Server(base, [0.05], slots=1, result_bytes=1 << 20, max_queries=5000) as S:
        for nq in (1, 100, 4200):
            t = S.submit(q[:nq] + 5.0, EPS)
            assert S.wait(t)["pairs"] == 0
            o, b = S.result(t)
            assert not o.any() and len(o) == nq + 1 and len(b) == 0
