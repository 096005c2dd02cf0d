"""What is left behind when device memory runs out: a call that fails with
"out of memory" leaves its index usable, wherever in the call it failed, and
the same call afterwards gives the whole result.  No reference counterpart."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

OUT_OF_MEMORY = 4  # HEGJ_ERR_OUT_OF_MEMORY


@pytest.fixture(scope="module")
def H():
    import hegjoin_amd as H
    if H.device_count() == 0:
        pytest.fail("no HIP device visible for a GPU test")
    yield H
    H.library().hegj_fail_device_allocations(0, 0)


def data(oracle, kind):
    """Points, eps, options: each lazily built part of an index."""
    rng = np.random.default_rng(11)
    if kind == "f32 copy, Morton order":
        return oracle.generate_expo(4000, 6, seed=31), 0.03, dict(refine="f32", unit_order="morton")
    if kind == "FP16 operands":
        return oracle.generate_expo(1500, 18, seed=32), 0.12, dict(refine="mfma", unit_order="morton")
    pts = rng.random((900, 24)) * 0.1
    pts[7, 20:] = 1e7  # one point too far for FP16: split-BF16 operands
    return pts, 0.15, dict(refine="mfma", unit_order="workload")


@pytest.mark.parametrize("kind", ["f32 copy, Morton order", "FP16 operands", "BF16 operands"])
def test_a_failed_first_join_can_be_repeated(H, oracle, kind):
    """Every allocation of the first join on an index fails once, each on an
    index of its own (no kept buffers, so each request reaches the driver)."""
    pts, eps, kw = data(oracle, kind)
    eoff, enb = oracle.join(pts, 6, eps)
    lib = H.library()
    failures = 0
    for skip in range(200):
        with H.GridIndex(pts, eps, indexed_dims=6) as ix:
            H.release_cached_memory()
            print("case", kind, "allocation", skip, flush=True)
            lib.hegj_fail_device_allocations(skip, 1 << 30)
            try:
                ix.selfjoin(**kw).close()
                done = True
            except H.HegjError as e:
                assert e.status == OUT_OF_MEMORY, str(e)
                done = False
            finally:
                lib.hegj_fail_device_allocations(0, 0)
            t = ix.selfjoin(**kw)
            off, nb = t.csr(sort_rows=True)
            t.close()
            assert np.array_equal(off, eoff) and np.array_equal(nb, enb)
        if done:
            break
        failures += 1
    assert done and failures >= 8


def test_kept_buffers_make_room(H, oracle):
    """A device full with the library's own kept buffers: every allocation of
    a server that opens, and of an index, is served after they went back."""
    base = oracle.generate_expo(5000, 6, seed=33)
    q = oracle.generate_expo(50, 6, seed=34)
    eoff, enb = oracle.range_join(base, q, 0.05)
    lib = H.library()
    for skip in range(30):
        with H.GridIndex(base, 0.03) as ix:
            ix.selfjoin().close()
        print("case allocation", skip, flush=True)
        lib.hegj_fail_device_allocations(skip, 1)
        try:
            S = H.Server(base, [0.051], slots=1, result_bytes=1 << 20, max_queries=64)
        finally:
            lib.hegj_fail_device_allocations(0, 0)
        with S:
            off, nb = S.result(S.submit(q, 0.05))
        rows = np.concatenate([np.sort(nb[off[i]:off[i + 1]]) for i in range(50)])
        assert np.array_equal(off, eoff) and np.array_equal(rows, enb)


def test_the_rounding_of_kept_sizes_is_no_reason_to_fail(H, oracle):
    """Sizes are rounded up so that later calls find each other's buffers.
    Where the rounded size does not fit the device, the exact one is taken:
    100003 points of 6 coordinates are 4800144 bytes, rounded up to 5242880."""
    pts = oracle.generate_expo(100003, 6, seed=35)
    H.release_cached_memory()
    H.library().hegj_fail_device_allocations(0, 2)  # the rounded size, before and after giving buffers back
    try:
        ix = H.GridIndex(pts, 0.01)
    finally:
        H.library().hegj_fail_device_allocations(0, 0)
    assert ix.info["n"] == len(pts)
    ix.close()


def test_graph_without_room_for_its_batch(H, oracle):
    """A replay whose output batch does not fit the device runs eagerly, with
    batches cut to the free memory, and the next one replays again."""
    pts = oracle.generate_expo(20000, 6, seed=36)
    eoff, enb = oracle.join(pts, 6, 0.02)
    with H.GridIndex(pts, 0.02, indexed_dims=6) as ix:
        for fail in (0, 3, 0):  # of a batch: the rounded size twice, the exact one
            if fail:
                H.release_cached_memory()
                H.library().hegj_fail_device_allocations(1, fail)  # after the row table
            try:
                t = ix.selfjoin(use_graph=True)
            finally:
                H.library().hegj_fail_device_allocations(0, 0)
            assert t.info["graph_replay"] == (0 if fail else 1)
            off, nb = t.csr(sort_rows=True)
            t.close()
            assert np.array_equal(off, eoff) and np.array_equal(nb, enb)


@pytest.mark.parametrize("kind", ["FP16 operands", "BF16 operands"])
def test_mfma_lists_shrink_to_the_memory(H, oracle, kind):
    """The first size of the pair and survivor lists is a guess: where one of
    them does not fit the device, the join runs with smaller ones."""
    pts, eps, kw = data(oracle, kind)
    eoff, enb = oracle.join(pts, 6, eps)
    lib = H.library()
    with H.GridIndex(pts, eps, indexed_dims=6) as ix:
        ix.selfjoin(**kw).close()  # everything lazily built

        def attempt(skip, count):
            H.release_cached_memory()
            print("case", kind, "allocation", skip, count, flush=True)
            lib.hegj_fail_device_allocations(skip, count)
            try:
                t = ix.selfjoin(**kw)
            except H.HegjError as e:
                assert e.status == OUT_OF_MEMORY
                return False
            finally:
                lib.hegj_fail_device_allocations(0, 0)
            off, nb = t.csr(sort_rows=True)
            t.close()
            assert np.array_equal(off, eoff) and np.array_equal(nb, enb)
            return True

        total = next(k for k in range(200) if attempt(k, 1 << 30))
        # one request in vain: at its rounded size, again, and at the exact one
        served = sum(attempt(k, 3) for k in range(total))
        assert served >= (3 if kind == "FP16 operands" else 2)
