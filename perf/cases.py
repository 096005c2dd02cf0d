"""Workloads whose speed this framework is judged by, through its public entry points.

Three kinds of work, over sizes from launch-bound to the largest workloads that
bench.py names:

  join     a self-join over a resident grid index (hegj_selfjoin), whose result
           is taken either as the neighbour counts (density estimates, DBSCAN
           core points) or as the whole neighbour table in host memory
           (hegj_result_copy_csr, rows ascending);
  oneshot  host points in, neighbour table out: index build, join and table
           (what hegjoin_amd.selfjoin() does);
  serve    one range-join request against a resident server: host queries in,
           CSR rows out.

Points follow the reference generator's law (exponential, rate 40) or are
uniform in the unit cube.  Every output is a whole number: neighbour ids,
offsets, counts, and the multiset hash of the pairs.  The pair set is defined
bit for bit (sqrt of the FP64 fma chain <= eps), so there is no value that
would be nearer to the truth than another and no exact() here.
"""
import ctypes as C
import math

import numpy as np
import torch

import hegjoin_amd as H

_lib = H.library()
_INDEX_OPTS_P = _lib.hegj_index_opts_default.argtypes[0]
_RESULT_INFO_P = _lib.hegj_result_get_info.argtypes[1]
_SERVE_OPTS_P = _lib.hegj_serve_open.argtypes[2]
_REQUEST_INFO_P = _lib.hegj_serve_wait.argtypes[2]

RATE = 40.0
# eps of the workloads in bench.py at (points, mean neighbours): other sizes
# of the same dimensionality scale it by the volume of the ball
ANCHOR = {2: (1_000_000, 1060.0, 0.001), 6: (5_000_000, 64.0, 0.0063131373103199606),
          18: (2_000_000, 32.0, 0.041121185939337571), 90: (1_000_000, 16.0, 0.19773135137186568)}
SERVE_SIDES = [0.02 * (1 + 1e-6) / 2 ** (i / 4) for i in range(8, -1, -1)]  # 0.005 .. 0.02


def ball(dim):
    return math.pi ** (dim / 2) / math.gamma(dim / 2 + 1)


def eps_for(dim, n, mean, dist):
    """An eps with about `mean` neighbours a point (within a factor of a few
    above 18 dimensions, where the number turns on a small change of eps)."""
    if dist == "uniform":
        return (mean / (n * ball(dim))) ** (1.0 / dim)
    if dim >= 18:
        # between the calibrated 18 and 90 dimensions eps grows about linearly
        # (a little faster at first); the exponential's tail makes the number
        # of neighbours grow slower than the ball's volume
        t = (dim - 18) / 72.0
        e = ANCHOR[18][2] + (ANCHOR[90][2] - ANCHOR[18][2]) * t
        m0, n0 = 32.0 * 0.5 ** t, 2e6 * 0.5 ** t
        return e * (1 + 0.3 * max(0.0, t * (1 - t))) * (mean / m0 * n0 / n) ** (1.3 / dim)
    if dim in ANCHOR:
        n0, m0, e0 = ANCHOR[dim]
        return e0 * (mean / m0 * n0 / n) ** (1.0 / dim)
    # integral of the squared density is (RATE / 2)^dim; the 8% is what the
    # 6-D calibration needs on top (points near the axes lack neighbours)
    return 1.08 * (mean / (n * ball(dim))) ** (1.0 / dim) / (RATE / 2)


def join(name, dim, n, mean, take, dist="expo", dtype="f64", kind="join"):
    c = {"kind": kind, "dim": dim, "n": n, "mean": mean, "eps": eps_for(dim, n, mean, dist), "dist": dist,
         "dtype": dtype, "take": take}
    return dict(c, name=name) if name else c


def serve(name, n, nq, eps):
    c = {"kind": "serve", "dim": 6, "n": n, "nq": nq, "eps": eps}
    return dict(c, name=name) if name else c


def listed():
    return [
        # an interactive query on a small 2-D set (map data): launch and call latency
        join("join 2d 20k table", 2, 20_011, 32.0, "csr"),
        # the 2-D workload of bench.py: the densest output (a billion pairs), counts for density clustering
        join("join 2d 1M counts", 2, 1_000_000, 1060.0, "counts"),
        # point clouds: 3-D, uniform, neighbour table on the host
        join("join 3d 500k table", 3, 500_009, 24.0, "csr", dist="uniform"),
        # 6-D feature vectors, a size met while exploring data
        join("join 6d 60k table", 6, 60_013, 64.0, "csr"),
        # the whole call on host data: upload, index, join, sorted neighbour table
        join("oneshot 6d 1M", 6, 1_000_000, 32.0, "csr", kind="oneshot"),
        # single precision (DTYPE=float)
        join("join 6d 1.5M float counts", 6, 1_500_007, 32.0, "counts", dtype="f32"),
        # the 6-D workload of bench.py (its default)
        join("join 6d 5M counts", 6, 5_000_000, 64.0, "counts"),
        # 18-D descriptors: a medium set with its table, and the workload of bench.py
        join("join 18d 250k table", 18, 250_007, 32.0, "csr"),
        join("join 18d 2M counts", 18, 2_000_000, 32.0, "counts"),
        # 90-D (the MillionSong width): the workload of bench.py
        join("join 90d 1M table", 90, 1_000_000, 16.0, "csr"),
        # serving: a small request, where latency counts, and a heavy one
        serve("serve 6d 2M small", 2_000_003, 1_000, 0.0081),
        serve("serve 6d 10M large", 10_000_000, 150_000, 0.0075),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["2d", "low", "6d", "6d", "18d", "high", "oneshot", "serve"])
    if what == "serve":
        return serve(None, _log(rng, 500_000, 10_000_000), _log(rng, 100, 150_000),
                     math.exp(rng.uniform(math.log(0.005), math.log(0.009))))
    dist = "expo"
    if what == "2d":
        dim, n, mean = 2, _log(rng, 10_000, 1_000_000), math.exp(rng.uniform(math.log(8), math.log(400)))
        dist = rng.choice(["expo", "uniform"])
    elif what == "low":
        dim, n, mean = rng.choice([3, 4, 5]), _log(rng, 10_000, 500_000), rng.uniform(8, 64)
        dist = rng.choice(["expo", "uniform"])
    elif what == "6d":
        dim, n, mean = 6, _log(rng, 20_000, 5_000_000), rng.uniform(8, 64)
    elif what == "18d":
        dim, n, mean = 18, _log(rng, 20_000, 1_500_000), rng.uniform(8, 32)
    elif what == "high":
        dim, n, mean = rng.choice([24, 32, 50, 64, 90, 100]), _log(rng, 20_000, 600_000), rng.uniform(4, 16)
    else:
        dim, n, mean = rng.choice([2, 6, 6, 18]), _log(rng, 10_000, 800_000), rng.uniform(8, 48)
        return join(None, dim, n, mean, "csr", kind="oneshot")
    dtype = "f32" if dim in (2, 6) and rng.random() < 0.25 else "f64"
    take = "csr" if n * mean < 2.5e7 and rng.random() < 0.5 else "counts"
    return join(None, dim, n, mean, take, dist, dtype)


def _points(n, dim, dist, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.empty((n, dim), dtype=torch.float64, device="cuda")
    if dist == "uniform":
        return x.uniform_(generator=g)
    return x.exponential_(RATE, generator=g).clamp_(max=1.0)


class _Opts(C.Structure):  # hegj_index_opts
    _fields_ = [("dim", C.c_uint32), ("indexed_dims", C.c_uint32), ("dtype", C.c_uint32),
                ("emulate_cell0", C.c_uint32), ("device", C.c_int32)]


class _ResultInfo(C.Structure):  # the head of hegj_result_info
    _fields_ = [("total_neighbors", C.c_uint64), ("pair_hash", C.c_uint64), ("rest", C.c_uint64 * 32)]


class _ServeOpts(C.Structure):  # hegj_serve_opts
    _fields_ = [("dim", C.c_uint32), ("indexed_dims", C.c_uint32), ("n_levels", C.c_uint32), ("slots", C.c_uint32),
                ("cell_sides", C.c_double * 32), ("result_bytes", C.c_uint64), ("max_queries", C.c_uint32),
                ("device", C.c_int32)]


class _RequestInfo(C.Structure):  # the head of hegj_request_info
    _fields_ = [("ticket", C.c_uint64), ("status", C.c_int32), ("level", C.c_uint32), ("n_queries", C.c_uint32),
                ("refine_used", C.c_uint32), ("pairs", C.c_uint64), ("rest", C.c_uint64 * 16)]


def _check(status):
    if status:
        raise RuntimeError("hegj status %d: %s" % (status, _lib.hegj_last_error().decode()))


class _Owner:
    """A library handle, freed with the state that holds it."""

    def __init__(self, free):
        self.h, self._free = C.c_void_p(), free

    def __del__(self):
        if self.h:
            self._free(self.h)


def _build(points, case, device):
    """hegj_index_build[_device] with the default options (the reference's)."""
    o = _Opts()
    _lib.hegj_index_opts_default(C.cast(C.byref(o), _INDEX_OPTS_P), case["dim"])
    o.dtype = 1 if case["dtype"] == "f32" else 0
    ix = _Owner(_lib.hegj_index_free)
    f = _lib.hegj_index_build_device if device else _lib.hegj_index_build
    _check(f(points, case["n"], case["eps"], C.cast(C.byref(o), _INDEX_OPTS_P), C.byref(ix.h)))
    return ix


def _pairs(case):
    """About how many pairs come out."""
    if case["kind"] == "serve":  # from the 6-D calibration: 64 neighbours in 5M at the anchor's eps
        return case["nq"] * 64.0 * case["n"] / 5e6 * (case["eps"] / ANCHOR[6][2]) ** 6 * 0.9
    return case["n"] * (case["mean"] + 1)


def prepare(case, seed):
    n, dim = case["n"], case["dim"]
    state = {"case": case}
    rows = case["nq"] if case["kind"] == "serve" else n
    if case.get("take") != "counts":
        # the program's own arrays for the neighbour table, with room to spare
        state["offsets"] = np.zeros(rows + 1, np.uint64)
        state["neighbors"] = np.zeros(int(2 * _pairs(case)) + 65536, np.uint32)
    else:
        state["counts"] = np.zeros(rows, np.uint32)
    if case["kind"] == "serve":
        pts = _points(n, dim, "expo", seed).cpu().numpy()
        state["queries"] = _points(case["nq"], dim, "expo", seed + 1_000_003).cpu().numpy()
        o = _ServeOpts(dim, 6, len(SERVE_SIDES), 2, result_bytes=8 << 30, max_queries=case["nq"], device=0)
        o.cell_sides[:len(SERVE_SIDES)] = SERVE_SIDES
        state["server"] = _Owner(_lib.hegj_serve_close)
        _check(_lib.hegj_serve_open(pts.ctypes.data, n, C.cast(C.byref(o), _SERVE_OPTS_P),
                                    C.byref(state["server"].h)))
        return state
    pts = _points(n, dim, case["dist"], seed)
    if case["kind"] == "oneshot":
        state["host"] = pts.cpu().numpy()
    else:
        torch.cuda.synchronize()  # the index reads the points on a stream of its own
        state["index"] = _build(pts.data_ptr(), case, True)
    return state


def _room(state, pairs):
    if pairs > len(state["neighbors"]):
        raise RuntimeError("%d pairs, room for %d" % (pairs, len(state["neighbors"])))
    return state["neighbors"].ctypes.data


def _join(state, ix):
    table = _Owner(_lib.hegj_result_free)
    _check(_lib.hegj_selfjoin(ix.h, None, C.byref(table.h)))  # the tuned options of the dimensionality
    info = _ResultInfo()
    _check(_lib.hegj_result_get_info(table.h, C.cast(C.byref(info), _RESULT_INFO_P)))
    if state["case"]["take"] == "counts":
        _check(_lib.hegj_result_copy_counts(table.h, state["counts"].ctypes.data))
        # the hash is 64 bits unsigned: as two halves it fits signed integers
        return {"counts": state["counts"], "pairs": info.total_neighbors,
                "hash": [info.pair_hash >> 32, info.pair_hash & 0xFFFFFFFF]}
    _check(_lib.hegj_result_copy_csr(table.h, state["offsets"].ctypes.data, _room(state, info.total_neighbors), 1))
    return {"offsets": state["offsets"], "neighbors": state["neighbors"]}


def run(state):
    case = state["case"]
    if case["kind"] == "join":
        return _join(state, state["index"])
    if case["kind"] == "oneshot":
        return _join(state, _build(state["host"].ctypes.data, case, False))
    srv, ticket, info = state["server"].h, C.c_uint64(), _RequestInfo()
    _check(_lib.hegj_serve_submit(srv, state["queries"].ctypes.data, case["nq"], case["eps"], C.byref(ticket)))
    _check(_lib.hegj_serve_wait(srv, ticket, C.cast(C.byref(info), _REQUEST_INFO_P)))
    _check(_lib.hegj_serve_copy(srv, ticket, state["offsets"].ctypes.data, _room(state, info.pairs)))
    _check(_lib.hegj_serve_release(srv, ticket))
    return {"offsets": state["offsets"], "neighbors": state["neighbors"]}


def _stencil_share(case):
    """Share of all points in the 3^k cells around a point: what the grid
    (min(dim, 6) indexed dimensions, cell side eps) leaves as candidates."""
    eps, k = case["eps"], min(case["dim"], 6)
    if case.get("dist", "expo") == "uniform":
        return min(1.0, 3 * eps) ** k
    r = math.exp(-RATE * eps)  # cell coordinates are geometric
    return ((1 - r) * (1 + 2 * r) / (1 + r)) ** k


def work(case):
    """Bytes: points (and queries) read once, neighbour ids with their row
    bounds (or the counts) written once.  Operations: a subtraction and a
    fused multiply-add a dimension for every candidate of the grid."""
    n, dim = case["n"], case["dim"]
    pairs = _pairs(case)
    if case["kind"] == "serve":
        candidates = case["nq"] * n * _stencil_share(case)
        return {"bytes": 8.0 * dim * (min(n, candidates) + case["nq"]) + 4 * pairs + 8.0 * case["nq"],
                "flops": 3.0 * dim * candidates}
    size = 4 if case["dtype"] == "f32" else 8
    out = 4.0 * n if case["take"] == "counts" else 8.0 * (n + 1) + 4.0 * pairs
    return {"bytes": size * n * dim + out, "flops": 3.0 * dim * n * n * _stencil_share(case)}
