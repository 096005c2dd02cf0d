"""The unit queues of the entry points beside hegj_selfjoin, at the sizes where
they change: runs of units in hegj_selfjoin_noalloc (fewer units than waves,
one run each, and more), one or two units per grab in the hybrid pieces."""
import numpy as np
import pytest

from hiprt import Buf, runtime

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    return H


@pytest.mark.parametrize("n, dim, eps", [(1, 2, 0.01), (9, 6, 0.05), (30000, 2, 0.0002), (400000, 2, 0.00005)])
def test_noalloc_runs(H, oracle, n, dim, eps):
    rt = runtime()
    pts = oracle.generate_expo(n, dim, seed=51)
    total, want = oracle.join_stats(pts, dim, eps)
    print("case noalloc", n, dim, total, flush=True)
    nb, off, cnt = bufs = [Buf(rt, t, m) for m, t in ((total + 1, np.uint32), (n, np.uint64), (n, np.uint32))]
    with H.GridIndex(pts, eps) as ix:
        ix.selfjoin().close()  # its lazily built arrays are inputs
        for _ in range(2):
            info = ix.selfjoin_noalloc(nb.p, total + 1, off.p, cnt.p)
            assert (info["total_neighbors"], info["pair_hash"]) == (total, want)
            assert int(cnt.get().sum()) == total
    for b in bufs:
        b.free()


@pytest.mark.parametrize("piece", [100, 8191, 8192, 16383, 16384, 60000])
def test_hybrid_pieces(H, oracle, piece):
    pts = oracle.generate_expo(50000, 6, seed=52)
    total, want = oracle.join_stats(pts, 6, 0.012)
    with H.GridIndex(pts, 0.012) as ix:
        print("case piece", piece, flush=True)
        t = ix.selfjoin_hybrid("static", gpu_fraction=0.99, gpu_chunk=piece, cpu_threads=2)
        info = t.info
        t.close()
    assert info["n_units"] > 16384
    assert (info["total_neighbors"], info["pair_hash"]) == (total, want)


def test_noalloc_beyond_its_scratch(H):
    """3M cells of a point each: units and their weights need more than the
    fixed scratch, which is a matter of capacity."""
    rt = runtime()
    n = 3_000_000
    pts = np.random.default_rng(5).permutation(n).astype(np.float64)[:, None] / n
    nb, off, cnt = bufs = [Buf(rt, t, n) for t in (np.uint32, np.uint64, np.uint32)]
    with H.GridIndex(pts, 0.4 / n) as ix:
        ix.selfjoin().close()
        with pytest.raises(H.HegjError) as e:
            ix.selfjoin_noalloc(nb.p, n, off.p, cnt.p)
        assert e.value.status == 6 and "scratch" in str(e.value)
    for b in bufs:
        b.free()


@pytest.mark.parametrize("grab", [20000, 20001, 1 << 30, (1 << 32) - 1])
def test_grabs_larger_than_the_join(H, oracle, grab):
    """More units per grab than there are, up to the largest 32-bit number, in
    every entry point: one grab, all of the result."""
    rt = runtime()
    pts = oracle.generate_expo(20000, 6, seed=53)
    total, want = oracle.join_stats(pts, 6, 0.012)
    nb, off, cnt = bufs = [Buf(rt, t, m) for m, t in ((total, np.uint32), (20000, np.uint64), (20000, np.uint32))]
    with H.GridIndex(pts, 0.012) as ix:
        print("case grab", grab, flush=True)
        for t in (ix.selfjoin(units_per_grab=grab), ix.selfjoin(units_per_grab=grab, use_graph=True),
                  ix.selfjoin(units_per_grab=grab, result_capacity=total // 3),
                  ix.selfjoin_hybrid("static", gpu_fraction=0.99, cpu_threads=2, units_per_grab=grab)):
            info = t.info
            t.close()
            assert (info["total_neighbors"], info["pair_hash"]) == (total, want)
        info = ix.selfjoin_noalloc(nb.p, total, off.p, cnt.p, units_per_grab=grab)
        assert (info["total_neighbors"], info["pair_hash"]) == (total, want)
    for b in bufs:
        b.free()
