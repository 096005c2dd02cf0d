"""What a call does around its kernels: results copied out in chunks by
several threads (sizes around every switch), buffers that pass from call to
call, and several threads with an index each."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    return H


@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 2048, 524287, 1048575, 1048576, 1048577, 1310720, 4194303,
                               4194304, 4194305, 5000011])
def test_copies_of_every_size(H, n):
    """Points farther apart than eps: each row is its own id, so the ids
    (4 n bytes), the offsets (8 n + 8) and the counts are known."""
    pts = np.random.default_rng(n).permutation(n).astype(np.float64)[:, None] / n
    with H.GridIndex(pts, 0.4 / n) as ix:
        t = ix.selfjoin()
        for sort_rows in (True, False):
            off, nb = t.csr(sort_rows=sort_rows)
            assert np.array_equal(off, np.arange(n + 1, dtype=np.uint64))
            assert np.array_equal(nb, np.arange(n, dtype=np.uint32))
        assert np.array_equal(t.counts(), np.ones(n, np.uint32))
        t.close()


def test_threads_and_reused_buffers(H):
    """Four threads, each building, joining (grid and MFMA refines) and
    closing indexes of its own sizes over and over, so buffers freed by one
    are taken by another; every result equals the one of a lone run."""
    cases = []
    for i in range(4):
        rng = np.random.default_rng(i)
        cases.append([(rng.exponential(1 / 40, (n, d)), eps) for n, d, eps in
                      ((30000 + 7 * i, 6, 0.012), (20000 + i, 2, 0.001), (9000 + i, 18, 0.06))])

    def one(pts, eps):
        with H.GridIndex(pts, eps) as ix:
            t = ix.selfjoin()
            off, nb = t.csr()
            h = t.info["pair_hash"]
            t.close()
            return off, nb, h

    want = [[one(*c) for c in cs] for cs in cases]
    bad = []

    def work(i):
        try:
            for _ in range(6):
                for c, w in zip(cases[i], want[i]):
                    g = one(*c)
                    if not (np.array_equal(g[0], w[0]) and np.array_equal(g[1], w[1]) and g[2] == w[2]):
                        bad.append((i, c[0].shape))
        except Exception as e:  # reported by the main thread
            bad.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    H.release_cached_memory()
    g, w = one(*cases[0][0]), want[0][0]
    assert np.array_equal(g[0], w[0]) and np.array_equal(g[1], w[1])
