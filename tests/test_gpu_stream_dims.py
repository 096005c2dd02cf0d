"""The grid joins whose coordinates are streamed (every dimensionality without an
instance of its own): each remainder of their groups of 4 and tiles of 8 or 16
dims, units of 1 to 16 queries, FP64 and DTYPE=float, exact against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIMS = [1, 3, 4, 5, 7, 8, 9, 10, 11, 12, 13, 15, 16, 17, 19, 20, 23, 24, 25, 31, 32, 33, 47, 48, 49, 64, 65, 90]


@pytest.fixture(scope="module")
def H():
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    return H


def points(dim, dtype):
    """A dense blob (full units), pairs (short ones) and single points, so
    every number of queries occurs; eps with some 5% of the blob in range."""
    rng = np.random.default_rng(100 + dim)
    blob = 0.3 + 0.1 * rng.random((600, dim))
    eps = float(np.quantile(np.linalg.norm(blob[:100, None] - blob[None, 100:200], axis=2), 0.05))
    eps = min(max(eps, 1e-3), 1.0)
    lone = rng.random((300, dim))
    pts = np.concatenate([blob, lone, lone + 0.3 * eps / np.sqrt(dim) * rng.random((300, dim))])
    if dtype == "f32":
        return pts.astype(np.float32).astype(np.float64), float(np.float32(eps))
    return pts, eps


@pytest.mark.parametrize("dim", DIMS)
@pytest.mark.parametrize("qb", [4, 8, 16])
def test_fp64(H, oracle, dim, qb):
    if qb * dim * 32 > 36 << 10:
        pytest.skip("more coordinates than the LDS share of a unit")
    pts, eps = points(dim, "f64")
    k = min(dim, 6)
    eoff, enb = oracle.join(pts, k, eps)
    print("case", dim, qb, len(enb), flush=True)
    with H.GridIndex(pts, eps, indexed_dims=k) as ix:
        t = ix.selfjoin(refine="fp64", queries_per_unit=qb)
        off, nb = t.csr(sort_rows=True)
        t.close()
    assert np.array_equal(off, eoff) and np.array_equal(nb, enb)


@pytest.mark.parametrize("dim", DIMS)
def test_not_finite(H, oracle, dim):
    """Coordinates that are inf or NaN in the last dim (next to the padding)."""
    pts, eps = points(dim, "f64")
    k = max(1, min(dim - 1, 6))
    if dim > 1:
        pts[5, -1], pts[6, -1], pts[7, -1] = np.inf, np.nan, -np.inf
    eoff, enb = oracle.join(pts, k, eps)
    print("case", dim, len(enb), flush=True)
    with H.GridIndex(pts, eps, indexed_dims=k) as ix:
        t = ix.selfjoin(refine="fp64", queries_per_unit=4)
        off, nb = t.csr(sort_rows=True)
        t.close()
    assert np.array_equal(off, eoff) and np.array_equal(nb, enb)


@pytest.mark.parametrize("dim", [d for d in DIMS if d != 90])
@pytest.mark.parametrize("qb", [4, 8])
def test_float(H, oracle, dim, qb):
    """DTYPE=float: d = fl32(c - q), acc = fmaf(d, d, acc), sqrtf(acc) <= eps,
    by the oracle's float join."""
    pts, eps = points(dim, "f32")
    k = min(dim, 6)
    eoff, enb = oracle.join(pts, k, eps, f32=True)
    with H.GridIndex(pts, eps, indexed_dims=k, dtype="f32") as ix:
        print("case", dim, qb, len(enb), flush=True)
        t = ix.selfjoin(refine="fp64", queries_per_unit=qb)
        off, nb = t.csr(sort_rows=True)
        t.close()
    assert np.array_equal(off, eoff) and np.array_equal(nb, enb)


def test_masks_that_fit_nowhere(H, oracle):
    """Units of more masks than the scratch holds: one query at a time in the
    write pass, streamed too."""
    rng = np.random.default_rng(9)
    pts = rng.random((70000, 7))
    pts[:, 0] = 0.5 + 0.004 * pts[:, 0]
    total, want = oracle.join_stats(pts, 1, 0.05)
    with H.GridIndex(pts, 0.05, indexed_dims=1) as ix:
        print("case masks", total, flush=True)
        t = ix.selfjoin(refine="fp64", queries_per_unit=8)
        info = t.info
        t.close()
    assert (info["total_neighbors"], info["pair_hash"]) == (total, want)
