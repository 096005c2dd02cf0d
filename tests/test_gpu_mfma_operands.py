"""Which of the two MFMA joins ran, and the split-BF16 one on its own ground:
data whose spread FP16 cannot hold, or more than 124 dimensions.  The pair set
is defined bit for bit, so every comparison with the oracle is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    return H


def join(H, oracle, pts, eps, operands, **kw):
    print("case", pts.shape, "eps", eps, kw, flush=True)
    eoff, enb = oracle.join(pts, 6, eps)
    with H.GridIndex(pts, eps, indexed_dims=6) as ix:
        t = ix.selfjoin(refine="mfma", **kw)
        off, nb = t.csr(sort_rows=True)
        info = t.info
        t.close()
    assert info["refine_used"] == "mfma" and info["mfma_operands"] == operands
    assert np.array_equal(off, eoff) and np.array_equal(nb, enb)
    assert info["pair_hash"] == oracle.csr_hash(eoff, enb)
    return info


def cloud(rng, n, dim, far, both=True):
    """Points with an eps of about 2% of their distances, and one or (so that
    the mean stays among the rest) two outliers in the last coordinates, which
    are not indexed."""
    pts = rng.exponential(1 / 40, (n, dim))
    eps = float(np.quantile(np.linalg.norm(pts[:200, None] - pts[None, 200:400], axis=2), 0.02))
    if far:
        pts[7, -4:] = far
        if both:
            pts[8, -4:] = -far
    return pts, eps


@pytest.mark.parametrize("dim", [16, 28, 29, 60, 61, 92, 93, 124])
def test_ordinary_data_take_fp16(H, oracle, dim):
    pts, eps = cloud(np.random.default_rng(dim), 700, dim, 0)
    join(H, oracle, pts, eps, "f16")


# the first and last dimension of each K-block count that is built (2, 3, 4, 6, 8, 9, 12)
@pytest.mark.parametrize("dim", [16, 19, 20, 30, 31, 40, 41, 62, 63, 83, 84, 94, 95, 126])
def test_split_bf16_of_every_size(H, oracle, dim):
    """Tiles that decide (a band of a few per cent), unit and chunk remainders."""
    pts, eps = cloud(np.random.default_rng(dim), 1100 + dim, dim, 1e8)
    info = join(H, oracle, pts, eps, "bf16")
    assert info["total_neighbors"] > 2 * len(pts) and info["band_rechecks"] < info["total_neighbors"]


@pytest.mark.parametrize("dim", [18, 40, 90])
def test_split_bf16_pairs_on_the_threshold(H, oracle, dim):
    """Pairs at eps (1 + r), |r| from 1e-15 to 1e-3, on both sides of both guards."""
    rng = np.random.default_rng(dim)
    eps, m = 0.05, 200
    base = 0.3 + 0.02 * rng.random((m, dim))
    parts = [base]
    for rel in (-1e-3, -1e-9, -1e-15, 0.0, 1e-15, 1e-9, 1e-3):
        d = rng.standard_normal((m, dim))
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        parts.append(base + d * eps * (1 + rel))
    far = np.full((2, dim), 0.31)
    far[:, -4:] += np.array([[1e8], [-1e8]])
    info = join(H, oracle, np.ascontiguousarray(np.concatenate(parts + [far])), eps, "bf16")
    assert info["band_rechecks"] >= m


@pytest.mark.parametrize("dim", [16, 24, 40, 62, 126])
def test_split_bf16_pair_list_overflow(H, oracle, dim):
    """A first pair list far too small: from the tiles, and (one outlier draws
    the mean away from the rest: every pair is in the band) from the recheck."""
    rng = np.random.default_rng(dim)
    for both in (True, False):
        pts, eps = cloud(rng, 1500, dim, 1e8 if both else 1e10, both)
        pts[100:700] = pts[100] + 0.1 * eps / np.sqrt(dim) * rng.random((600, dim))  # 360k near pairs
        info = join(H, oracle, pts, eps, "bf16", result_capacity=1)
        if not both:
            assert info["band_rechecks"] >= info["total_neighbors"] > 300000


def test_split_bf16_band_list_overflow(H, oracle):
    """More band pairs than the first band list holds (2^22)."""
    rng = np.random.default_rng(1)
    pts = 0.5 + 0.01 * rng.random((2300, 16))
    pts[3, -4:] = 1e10
    info = join(H, oracle, pts, 0.02, "bf16")
    assert info["band_rechecks"] > 1 << 22


@pytest.mark.parametrize("dim", [16, 18, 32, 64, 90, 124])
@pytest.mark.parametrize("far, operands", [(100, "f16"), (800, "f16"), (6400, "bf16"), (100000, "bf16")])
def test_outliers_choose_the_operands(H, oracle, dim, far, operands):
    """Outliers `far` eps out set the FP16 scale.  At 6400 the norms' low parts
    are below FP16's normal range by more than eps^2 can bear: FP16 tiles would
    send most near pairs to the FP64 recheck."""
    pts, eps = cloud(np.random.default_rng(dim), 900, dim, 0)
    pts[7, -2:], pts[8, -2:] = far * eps, -far * eps
    info = join(H, oracle, pts, eps, operands)
    assert info["band_rechecks"] < info["total_neighbors"] / 2


def test_clusters_keep_fp16(H, oracle):
    """Centres 60 eps from the mean: wide guards in both, FP16 the faster."""
    rng = np.random.default_rng(2)
    pts, eps = cloud(rng, 1500, 18, 0)
    centre = rng.standard_normal((12, 18))
    centre[:, :6] = 0
    centre *= 60 * eps / np.linalg.norm(centre, axis=1, keepdims=True)
    pts += centre[rng.integers(0, 12, len(pts))]
    join(H, oracle, pts, eps, "f16")
