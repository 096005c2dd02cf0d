"""Ascending neighbour rows, sorted on the device: every row length at which
the sorting changes (16, 32 and 64 lanes, registers per lane, LDS, beyond
LDS), checked against the unsorted rows sorted by numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024,
           1025, 2047, 2048, 2049, 5000, 16383, 16384, 16385, 32768, 32769, 40000]


@pytest.fixture(scope="module")
def H():
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    return H


def rows_match(t):
    off, nb = t.csr(sort_rows=True)
    off0, nb0 = t.csr(sort_rows=False)
    assert np.array_equal(off, off0)
    row = np.repeat(np.arange(len(off) - 1), np.diff(off).astype(np.int64))
    want = nb0[np.lexsort((nb0, row))]
    assert np.array_equal(nb, want)
    return np.diff(off)


@pytest.mark.parametrize("shuffle", [False, True])
def test_every_row_length(H, shuffle):
    """Hubs with L - 1 points on a sphere of radius eps (1 - 1e-9) around
    each: in 18-D those see few of each other, so the hub's row is the long
    one.  Unshuffled ids also put short and long rows side by side."""
    rng = np.random.default_rng(9)
    eps, parts, hubs, at = 0.01, [], [], 0
    for i, length in enumerate(LENGTHS):
        hub = np.full((1, 18), 0.5)
        hub[0, :2] = 0.05 + 0.1 * (i % 9), 0.05 + 0.1 * (i // 9)
        d = rng.standard_normal((length - 1, 18))
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        parts += [hub, hub + d * eps * (1 - 1e-9)]
        hubs.append(at)
        at += length
    pts = np.concatenate(parts)
    order = rng.permutation(len(pts)) if shuffle else np.arange(len(pts))
    where = np.empty(len(pts), np.int64)
    where[order] = np.arange(len(pts))
    print("case", pts.shape, "shuffle", shuffle, flush=True)
    with H.GridIndex(np.ascontiguousarray(pts[order]), eps) as ix:
        t = ix.selfjoin()
        counts = rows_match(t)
        t.close()
    assert counts[where[hubs]].tolist() == LENGTHS


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1001])
def test_last_rows_of_a_wave(H, n):
    """Four rows per wave: every remainder, and rows spread over result batches."""
    pts = np.random.default_rng(n).random((n, 2)) * 0.05
    with H.GridIndex(pts, 0.01) as ix:
        for cap in (0, 20000):
            t = ix.selfjoin(result_capacity=cap)
            rows_match(t)
            t.close()
