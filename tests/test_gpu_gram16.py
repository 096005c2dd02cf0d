"""The FP16 Gram join (MFMA refine) where it can go wrong: K-block edges,
unit and tile remainders, candidates of silenced queries, and data its
operands cannot serve (those take the split-BF16 join).  The pair set is
defined bit for bit, so every comparison with the oracle is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    return H


def check(H, oracle, pts, eps, k, emulate=True, **kw):
    print("case", pts.shape, "eps", eps, "k", k, "emulate", emulate, flush=True)
    eoff, enb = oracle.join(pts, k, eps, emulate_cell0=emulate)
    with H.GridIndex(pts, eps, indexed_dims=k, emulate_cell0=emulate) as ix:
        for _ in range(2):  # the second call reuses the operands
            t = ix.selfjoin(refine="mfma", **kw)
            off, nb = t.csr(sort_rows=True)
            raw_off, raw = t.csr(sort_rows=False)
            ila = ix.copy_grid()[2]
            info = t.info
            t.close()
            assert info["refine_used"] == "mfma"
            assert np.array_equal(off, eoff) and np.array_equal(nb, enb)
            assert info["pair_hash"] == oracle.csr_hash(eoff, enb)
            # unsorted rows come in cell order
            pos = np.empty(len(pts), np.int64)
            pos[ila] = np.arange(len(pts))
            p = pos[raw]
            inner = np.ones(max(len(p) - 1, 0), bool)
            ends = raw_off[1:-1].astype(np.int64) - 1
            inner[ends[(ends >= 0) & (ends < len(inner))]] = False
            assert np.all(np.diff(p)[inner] > 0)
    return info


@pytest.mark.parametrize("dim", [16, 28, 29, 60, 61, 92, 93, 124, 125])
def test_k_block_edges(H, oracle, dim):
    """The last dimension of each K-block count and the first of the next
    (125: past the FP16 kernels), dense enough for hits in every tile."""
    rng = np.random.default_rng(dim)
    pts = rng.exponential(1 / 40, (1300, dim))
    eps = float(np.quantile(np.linalg.norm(pts[:200, None] - pts[None, 200:400], axis=2), 0.02))
    check(H, oracle, pts, eps, 6)


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 511, 512, 513, 1025, 2500])
def test_unit_and_tile_remainders(H, oracle, n):
    """n points in one cell (one query block of 512, its 16-query tiles, the
    candidate chunks): most pairs are hits, so the survivor list's blocks
    fill and close too."""
    rng = np.random.default_rng(n)
    eps = 0.1
    pts = 0.5 + rng.random((n, 18)) * (1.45 * eps / np.sqrt(18))
    check(H, oracle, np.ascontiguousarray(pts), eps, 6)


@pytest.mark.parametrize("emulate", [True, False])
def test_silenced_queries_stay_candidates(H, oracle, emulate):
    """A point in grid cell 0 is no query (cell-0 wrap) but a candidate of
    its neighbours: pairs are then not symmetric."""
    rng = np.random.default_rng(5)
    base, eps = rng.exponential(1 / 40, (1500, 18)), 0.06
    for v in np.linspace(0.02, 0.7, 2000):
        if np.floor((v - (v - eps)) / eps) == 0:
            break
    pts = base.copy()
    pts[:, 2] += v
    order = np.argsort(pts[:, 2])
    pts[order[:40], 2] = v
    pts[order[0]] = pts[order[40]]  # a silenced point with a live neighbour
    pts[order[0], 2] = v
    assert oracle.count_cell0(pts, 6, eps) > 0
    info = check(H, oracle, pts, eps, 6, emulate=emulate)
    assert info["total_neighbors"] > 0


def test_survivor_list_overflow(H, oracle):
    """A first list far too small for the survivors and the pairs."""
    pts = oracle.generate_expo(3000, 18, seed=22)
    check(H, oracle, pts, 0.15, 6, result_capacity=1)


@pytest.mark.parametrize("kind", ["outlier", "far outlier", "tiny", "huge eps", "nan", "inf", "constant"])
def test_ranges(H, oracle, kind):
    """Scales: one outlier (its pairs in the band), one so far that FP16
    cannot hold the rest, near-denormal coordinates, eps beyond the data,
    coordinates that are not finite, and a single repeated point."""
    rng = np.random.default_rng(3)
    pts, eps = rng.random((900, 24)) * 0.1, 0.15
    if kind == "outlier":
        pts[7, 20:] = 30.0
    elif kind == "far outlier":
        pts[7, 20:] = 1e7
    elif kind == "tiny":
        pts, eps = pts * 1e-6, 0.15e-6
    elif kind == "huge eps":
        eps = 1.0
    elif kind == "nan":
        pts[11, 15] = np.nan
    elif kind == "inf":
        pts[11, 15] = np.inf
    else:
        pts[:] = pts[0]
    check(H, oracle, pts, eps, 6)


@pytest.mark.parametrize("dim", [18, 40, 90])
def test_pairs_on_the_threshold(H, oracle, dim):
    """Pairs at eps (1 + r), |r| from 1e-15 to 1e-3: on both sides of both
    guards, decided exactly."""
    rng = np.random.default_rng(dim)
    eps, m = 0.05, 300
    base = 0.3 + 0.2 * rng.random((m, dim))
    parts = [base]
    for rel in (-1e-3, -1e-4, -1e-9, -1e-15, 0.0, 1e-15, 1e-9, 1e-4, 1e-3):
        d = rng.standard_normal((m, dim))
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        parts.append(base + d * eps * (1 + rel))
    info = check(H, oracle, np.ascontiguousarray(np.concatenate(parts)), eps, 6)
    assert info["band_rechecks"] >= m
