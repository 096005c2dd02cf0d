"""A result holds about the memory of its rows, also where its join sized the
output by the candidates (they are many times the pairs at 6-D)."""
import numpy as np
import pytest

from hiprt import free_bytes, runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [False, True])
def test_held_memory(oracle, use_graph):
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    rt = runtime()
    pts = oracle.generate_expo(60013, 6, seed=41)
    with H.GridIndex(pts, 0.0131) as ix:
        off, nb = (lambda t: (t.csr(), t.close())[0])(ix.selfjoin(use_graph=use_graph))  # everything lazily built
        H.release_cached_memory()
        before = free_bytes(rt)
        tables = [ix.selfjoin(use_graph=use_graph) for _ in range(3)]
        H.release_cached_memory()
        held = before - free_bytes(rt)
        rows = 4 * len(nb) + 12 * len(pts)
        print("held", held, "rows", rows, "candidates", tables[0].info["total_candidates"], flush=True)
        # twice the rows and 16 MiB in 2 MiB pieces; the candidates would be over 400 MB a table
        assert tables[0].info["total_candidates"] > 20 * len(nb) and held <= 3 * (2 * rows + (20 << 20))
        for t in tables:
            o, b = t.csr()
            assert np.array_equal(o, off) and np.array_equal(b, nb)
            t.close()
