"""Results copied into memory that is not pageable: pinned by the caller, or on
the device (a program that goes on there).  Sizes on both sides of the switches
of the pageable path, which stages and copies with the CPU."""
import numpy as np
import pytest

from hiprt import Buf, runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["pinned", "device"])
@pytest.mark.parametrize("n", [100, 4097, 700001, 3000001])
def test_destination(where, n):
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    lib = H.library()
    pts = np.random.default_rng(n).permutation(n).astype(np.float64)[:, None] / n
    rt = runtime()
    off, nb, cnt = bufs = [Buf(rt, t, m, where == "pinned")
                           for m, t in ((n + 1, np.uint64), (n, np.uint32), (n, np.uint32))]
    with H.GridIndex(pts, 0.4 / n) as ix:  # every point is its own neighbour only
        t = ix.selfjoin()
        print("case", where, n, flush=True)
        assert lib.hegj_result_copy_csr(t._h, off.p, nb.p, 1) == 0
        assert lib.hegj_result_copy_counts(t._h, cnt.p) == 0
        t.close()
    assert np.array_equal(off.get(), np.arange(n + 1))
    assert np.array_equal(nb.get(), np.arange(n))
    assert np.array_equal(cnt.get(), np.ones(n))
    for b in bufs:
        b.free()
