// hegj_query.hip -- range join of external query points against a resident
// grid index: the device side of the serving loop.
//
// The reference has no query path (its only join is the self-join of
// kernel.cu:727-802); this follows the same grid semantics with the intended
// stencil (no cell-0 wrap) and the same distance chain and predicate:
//   a query q and an index point p pair when sqrt(acc) <= eps, with
//   acc = fma(p_l - q_l, p_l - q_l, acc) over l = 0..dim-1 (kernel.cu:350-355),
//   evaluated as acc <= T, T the largest double with sqrt(T) <= eps.
// The index level's cell side c satisfies eps <= c (1 - 2^-30), so every
// point within eps lies in the 3^k cells around the query's cell even after
// the rounding of (x - min) / c.
//
// Pipeline for one request (one stream):
//   k_qcell_keys    query -> key of its cell in the grid widened by one cell
//                   on each side (coordinates -1 .. nCells), or `dead` when
//                   the query lies further out (no point can be in range);
//   radix sort      (key, query id), dead keys last;
//   items           units of up to 4 queries of one cell, heavy ones split into
//                   segments of their candidates; each builds its stencil
//                   rows, pruned to the cells within eps of one of its queries
//                   (requests of at most 4096 queries: these three steps in
//                   three launches, without a readback);
//   k_qjoin<count>  per-query neighbour counts, and per group a bitmap of the
//                   candidate chunks in which one of its queries has a hit;
//   scan            CSR offsets, exact result size (admission happens here);
//   k_qjoin<fill>   each query's neighbours written at its own offset in
//                   candidate (cell) order, visiting only the hit chunks --
//                   no atomics, deterministic.
#include <type_traits>

#include "hegj_stencil.h"

namespace hegj {

namespace {

constexpr int kQWaves = 4;
// Queries evaluated together against one candidate chunk, on the FP64 path
// (their coordinates fill 48 scalar registers at 6-D) and on the FP32 filter.
// 8 on the FP32 filter measured slower at 6-D (10M points, 93k queries,
// eps 0.0172): the group's pruned stencil grows (+12% distance evaluations)
// and its registers spill.
constexpr int kQB = 4;
constexpr int kQBF32 = 4;
constexpr uint32_t kHitWords = kQueryHitWords;

__global__ __launch_bounds__(256) void k_qcell_keys(const double *__restrict__ q, uint32_t nq,
                                                    QueryGeom qg, uint64_t *__restrict__ keys,
                                                    uint32_t *__restrict__ ids) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nq) return;
    uint64_t key = 0, mult = 1;
    bool dead = false;
    for (uint32_t j = 0; j < qg.g.k; j++) {
        const double x = q[(uint64_t)i * qg.g.dim + j];
        const double f = floor((x - qg.g.minArr[j]) / qg.g.eps);
        // widened coordinate: -1 .. nCells map to 0 .. nCells + 1
        if (!(f >= -1.0) || f > (double)qg.g.nCells[j]) {
            dead = true;
        } else {
            key += (uint64_t)(int64_t)(f + 1.0) * mult;
        }
        mult *= (uint64_t)qg.g.nCells[j] + 2;
    }
    keys[i] = dead ? qg.dead_key : key;
    ids[i] = i;
}

// Unit r starts at the r-th run of equal live keys; n_live = first dead slot.
__global__ __launch_bounds__(256) void k_qrun_flags(const uint64_t *__restrict__ keys, uint32_t nq,
                                                    uint64_t dead, uint32_t *__restrict__ flag,
                                                    uint32_t *__restrict__ n_live) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nq) return;
    const uint64_t k = keys[i];
    flag[i] = (k != dead && (i == 0 || keys[i - 1] != k)) ? 1u : 0u;
    const bool last_live = k != dead && (i + 1 == nq || keys[i + 1] == dead);
    if (last_live) *n_live = i + 1;
}

__global__ __launch_bounds__(256) void k_qrun_fill(const uint32_t *__restrict__ flag,
                                                   const uint32_t *__restrict__ rank, uint32_t nq,
                                                   uint32_t *__restrict__ starts) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < nq && flag[i]) starts[rank[i]] = i;
}

// A unit is one group: at most kQB queries of one cell, so the groups of a
// dense cell go to different waves (with units of four groups the heaviest
// unit was the request's critical path: 6-D, 10M points, 150k queries, with
// the sweeps by group size below, count pass 13.5 -> 6.4 ms, fill 5.8 -> 3.1).
constexpr uint32_t kUnitQueries = kQB;
static_assert(kQB == kQBF32, "a unit is one group on either path");

// An item is a unit, or one of up to 16 equal segments of a unit's candidates
// where the unit looks heavy: a request of fewer units than the chip's 3072
// resident waves takes as long as its densest group.  Each wave builds the
// group's rows for itself (about 20 us at 6-D), so a segment is meant to have
// kSegCandidates.  A unit's candidates are estimated from the points of its
// home row's three cells, times the 3^(k-1) rows of the stencil, of which the
// box pruning leaves a share that falls with k (0.25 at 6-D).  6-D, 2M points,
// 3000 queries: request 0.78 -> 0.43 ms, 12000 queries 1.33 -> 0.84; segments
// of 2048 measured 0.47 and 0.89.
// .x = first sorted query, .y = segment | segments << 8 | queries << 16.
constexpr uint32_t kMaxSegments = 16;
constexpr float kSegCandidates = 4096.0f;

__device__ uint32_t unit_segments(const QueryGeom &qg, const DevIndex &ix, uint64_t key, uint32_t min_seg, uint32_t max_seg) {
    if (max_seg <= min_seg) return max_seg;
    const GridGeom &g = qg.g;
    uint64_t rkey = 0, mult = 1;
    int64_t c0 = 0;
    float rows = 1.0f;
    for (uint32_t j = 0; j < g.k; j++) {
        const uint64_t w = (uint64_t)g.nCells[j] + 2, rest = key / w;
        const int64_t c = (int64_t)(key - rest * w) - 1;
        key = rest;
        if (j == 0) {
            c0 = c;
            continue;
        }
        if (c < 0 || c >= (int64_t)g.nCells[j]) return min_seg;
        rkey += (uint64_t)c * mult;
        mult *= g.nCells[j];
        rows *= 3.0f;
    }
    uint32_t a, e;
    if (!row_lookup(ix.hrows, ix.hmask, rkey, &a, &e)) return min_seg;
    // the row's cells by coordinate 0: [c0 - 1, c0 + 1]
    auto lower = [&](int64_t v) {
        uint32_t lo = a, hi = e;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if ((int64_t)ix.cell_xyz[mid] < v)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo;
    };
    const uint32_t first = lower(c0 - 1), last = lower(c0 + 2);
    const float est = (float)(ix.cell_start[last] - ix.cell_start[first]) * rows * (1.15f - 0.15f * (float)g.k);
    return min(max((uint32_t)fminf(est / kSegCandidates, 1024.0f), min_seg), max_seg);
}

__device__ __forceinline__ uint2 make_item(uint32_t g0, uint32_t nqg, uint32_t seg, uint32_t nseg) {
    return make_uint2(g0, seg | nseg << 8 | nqg << 16);
}

// ---- requests of at most kSmallPlan queries: the plan in three launches ----
// The general plan (a radix sort of up to 8 passes, two scans, two readbacks)
// is about 40 launches, 0.25 ms of a 1 ms request; here each key's place is
// its rank among all of them, and nothing is read back: the join reads the
// number of units on the device.
constexpr uint32_t kSmallPlan = 4096;
constexpr uint32_t kSmallScan = 16384;  // counts scanned by one workgroup
// Largest number of items that splitting may make of a request (131072
// measured the same within 5% either way).
constexpr uint32_t kSplitItems = 49152;
// A request of fewer items leaves waves idle whatever it does: its units are
// split, up to 8 times, without asking for their weight (20 queries: 0.18 ms
// without, 0.13 with; at 2048 items 500 queries took 0.27 ms instead of 0.245).
constexpr uint32_t kSpareItems = 1024;

// place[i] = keys below keys[i] + equal keys before i (the stable sort's
// order); the second term also says which queries begin a unit.  64 queries
// a workgroup, its four waves a quarter of the keys each: bound by the LDS
// broadcasts (a key and its compare for every lane), 4096 keys 12 us.
__global__ __launch_bounds__(256) void k_qsmall_rank(const uint64_t *__restrict__ keys, uint32_t nq, QueryGeom qg,
                                                     DevIndex ix, uint32_t min_seg, uint32_t max_seg,
                                                     uint64_t *__restrict__ skeys,
                                                     uint32_t *__restrict__ sids, uint32_t *__restrict__ flags,
                                                     uint32_t *__restrict__ counts) {
    __shared__ uint64_t sh[kSmallPlan];
    __shared__ uint32_t part[2][4][64];
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (uint32_t j = threadIdx.x; j < nq; j += 256) sh[j] = keys[j];
    __syncthreads();
    const uint32_t i = blockIdx.x * 64 + lane;
    const uint64_t k = sh[min(i, nq - 1)];
    const uint32_t per = (nq + 3) / 4, b = min(w * per, nq), e = min(b + per, nq);
    uint32_t below = 0, before = 0;
#pragma unroll 8
    for (uint32_t j = b; j < e; j++) {
        const uint64_t o = sh[j];
        below += o < k;
        before += o == k && j < i;
    }
    part[0][w][lane] = below;
    part[1][w][lane] = before;
    __syncthreads();
    if (w != 0 || i >= nq) return;
    below = part[0][0][lane] + part[0][1][lane] + part[0][2][lane] + part[0][3][lane];
    before = part[1][0][lane] + part[1][1][lane] + part[1][2][lane] + part[1][3][lane];
    const uint32_t at = below + before;
    skeys[at] = k;
    sids[at] = i;
    // 2: live, 1: first of a unit, with the unit's segments above
    uint32_t f = k == qg.dead_key ? 0 : 2u;
    if (f && before % kUnitQueries == 0) f |= 1u | unit_segments(qg, ix, k, min_seg, max_seg) << 8;
    flags[at] = f;
    counts[i] = 0;
}

// Exclusive prefix of one value per thread over a workgroup of 1024.
__device__ uint64_t block_prefix(uint64_t v, uint64_t *sh, uint64_t *total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint64_t x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint64_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) sh[w] = x;
    __syncthreads();
    uint64_t base = 0, all = 0;
    for (int i = 0; i < 16; i++) {
        base += i < w ? sh[i] : 0;
        all += sh[i];
    }
    *total = all;
    return base + x - v;
}

// The items and their number from the flags in sorted order.
__global__ __launch_bounds__(1024) void k_qsmall_items(const uint32_t *__restrict__ flags, uint32_t nq,
                                                       uint2 *__restrict__ items, uint32_t *__restrict__ n_items) {
    constexpr uint32_t kPer = kSmallPlan / 1024;
    __shared__ uint64_t sh[16];
    const uint32_t i0 = threadIdx.x * kPer;
    uint32_t f[kPer + kUnitQueries - 1], mine = 0;
#pragma unroll
    for (uint32_t t = 0; t < kPer + kUnitQueries - 1; t++) {
        f[t] = i0 + t < nq ? flags[i0 + t] : 0;
        if (t < kPer) mine += f[t] >> 8;
    }
    uint64_t total;
    uint32_t o = (uint32_t)block_prefix(mine, sh, &total);
#pragma unroll
    for (uint32_t t = 0; t < kPer; t++) {
        uint32_t nqg = 1;
        bool more = true;
#pragma unroll
        for (uint32_t x = 1; x < kUnitQueries; x++) {
            more = more && (f[t + x] & 3) == 2;
            nqg += more;
        }
        for (uint32_t seg = 0; seg < f[t] >> 8; seg++) items[o++] = make_item(i0 + t, nqg, seg, f[t] >> 8);
    }
    if (threadIdx.x == 0) *n_items = (uint32_t)total;
}

// CSR offsets of at most kSmallScan counts in one workgroup.
__global__ __launch_bounds__(1024) void k_qsmall_offsets(const uint32_t *__restrict__ counts, uint32_t nq,
                                                         uint64_t *__restrict__ offsets) {
    constexpr uint32_t kPer = kSmallScan / 1024;
    __shared__ uint64_t sh[16];
    const uint32_t i0 = threadIdx.x * kPer;
    uint32_t c[kPer];
    uint64_t mine = 0, total;
#pragma unroll
    for (uint32_t t = 0; t < kPer; t++) {
        c[t] = i0 + t < nq ? counts[i0 + t] : 0;
        mine += c[t];
    }
    uint64_t o = block_prefix(mine, sh, &total);
#pragma unroll
    for (uint32_t t = 0; t < kPer; t++) {
        if (i0 + t < nq) offsets[i0 + t] = o;
        o += c[t];
    }
    if (threadIdx.x == 0) offsets[nq] = total;
}

// Items of each run of queries sharing a cell: its units times their segments.
__global__ __launch_bounds__(256) void k_item_counts(const uint32_t *__restrict__ starts, uint32_t nr,
                                                     const uint64_t *__restrict__ keys, QueryGeom qg, DevIndex ix,
                                                     uint32_t max_seg, uint32_t *__restrict__ nseg,
                                                     uint32_t *__restrict__ cnt) {
    const uint32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= nr) return;
    nseg[r] = unit_segments(qg, ix, keys[starts[r]], 1, max_seg);
    cnt[r] = (starts[r + 1] - starts[r] + kUnitQueries - 1) / kUnitQueries * nseg[r];
}

__global__ __launch_bounds__(256) void k_item_fill(const uint32_t *__restrict__ starts, uint32_t nr,
                                                   const uint32_t *__restrict__ nseg,
                                                   const uint32_t *__restrict__ first,
                                                   uint2 *__restrict__ items) {
    const uint32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= nr) return;
    const uint32_t b = starts[r], e = starts[r + 1], ns = nseg[r];
    uint32_t o = first[r];
    for (uint32_t i = b; i < e; i += kUnitQueries)
        for (uint32_t seg = 0; seg < ns; seg++) items[o++] = make_item(i, min(kUnitQueries, e - i), seg, ns);
}

// Stencil rows of a group of queries (all in the cell whose widened key is
// `key`) into the wave's LDS list; returns the candidate count.
//
// Cell-box pruning, as in the self-join: a stencil cell whose box lies
// farther than eps from every query of the group holds no neighbour and is
// left out.  With f_j the query's position inside its cell along indexed dim
// j (in cell sides), the gap to the -1 cell is f_j, to the +1 cell 1 - f_j;
// a cell is kept when the smallest sum of squared gaps over the group is at
// most T / side^2.  Gaps are shrunk by 1e-6 + 2e-15 (|c_j| + 2) (the FP64
// rounding of the cell assignments) and the bound raised by 1e-5 relative
// (FP32 sums), so the kept set can only be larger than the exact one.
template <int QB>
__device__ uint32_t qbuild_rows(const QJoinArgs &a, uint64_t key, const uint32_t *qid, uint32_t nqg,
                                StencilList &rl, StencilTabs<QB> &tb, uint32_t *nslots) {
    const GridGeom &g = a.qg.g;
    const int lane = threadIdx.x & 63;
    // lane j takes coordinate j of the widened cell (-1 .. nCells): two
    // divisions for all of them
    int64_t cl = 0;
    {
        uint64_t stride = 1, w = 1;
#pragma unroll
        for (int j = 0; j < kMaxK; j++) {
            if ((uint32_t)j >= g.k) break;
            const uint64_t wj = (uint64_t)g.nCells[j] + 2;
            if (lane > j) stride *= wj;
            if (lane == j) w = wj;
        }
        if ((uint32_t)lane < g.k) cl = (int64_t)((key / stride) % w) - 1;
    }
    CellBox box;
    int64_t c0 = 0;
    bool ok = true;
#pragma unroll
    for (int j = 0; j < kMaxK; j++) {
        // a coordinate of -1 wraps; the offset is added modulo 2^32
        box.c[j] = lane_u32((uint32_t)cl, j);
        box.lo[j] = box.hi[j] = 0;
        if ((uint32_t)j >= g.k) continue;
        const int64_t cj = (int64_t)(((uint64_t)lane_u32((uint32_t)((uint64_t)cl >> 32), j) << 32) | box.c[j]);
        if (j == 0) c0 = cj;
        const int64_t l = cj - 1 < 0 ? 0 : cj - 1;
        const int64_t h = cj + 1 > (int64_t)g.nCells[j] - 1 ? (int64_t)g.nCells[j] - 1 : cj + 1;
        ok &= l <= h;
        box.lo[j] = (uint32_t)l;
        box.hi[j] = (uint32_t)(h < 0 ? 0 : h);
    }
    if (!ok) {
        *nslots = 0;
        return 0;
    }
    const uint32_t k = g.k, dim = g.dim;
    const double inv_side = 1.0 / g.eps;
    wave_lds_sync();  // the previous group's reads of the list are done
    for (uint32_t e = (uint32_t)lane; e < nqg * k; e += 64) {
        const uint32_t qi = e / k, j = e - qi * k;
        uint32_t id = 0;
#pragma unroll
        for (int t = 0; t < QB; t++) id = (uint32_t)t == qi ? qid[t] : id;
        uint32_t cu = 0;
        double mn = 0.0;
#pragma unroll
        for (int jj = 0; jj < kMaxK; jj++) {
            cu = (uint32_t)jj == j ? box.c[jj] : cu;
            mn = (uint32_t)jj == j ? g.minArr[jj] : mn;
        }
        const double cj = cu == ~0u ? -1.0 : (double)cu;  // (a grid has under 2^32 - 1 cells a dim with two more)
        const double x = a.queries[(uint64_t)id * dim + j];
        double f = (x - mn) * inv_side - cj;
        f = f < 0.0 ? 0.0 : (f > 1.0 ? 1.0 : f);
        const double mg = 1e-6 + 2e-15 * (fabs(cj) + 2.0);
        const double gm = f - mg > 0.0 ? f - mg : 0.0, gp = 1.0 - f - mg > 0.0 ? 1.0 - f - mg : 0.0;
        tb.gap[qi * kMaxK + j] = make_float2((float)(gm * gm), (float)(gp * gp));
    }
    wave_lds_sync();
    const float thr = (float)(a.thresh * inv_side * inv_side) * (1.0f + 1e-5f);
    const uint32_t total = stencil_rows<QB>(g, a.ix, rl, tb, box, c0, nqg, thr, nslots);
    wave_lds_sync();
    return total;
}

// The kernel arguments, to be read again from here on: kept live through a
// unit's loops they would be spilled to vector lanes.
typedef __attribute__((address_space(4))) const QJoinArgs *QArgsPtr;
__device__ __forceinline__ const QJoinArgs &reload(QArgsPtr p) {
    __asm__ volatile("" : "+s"(p));
    return *(const QJoinArgs *)p;
}

// D > 0: coordinates in registers; D == 0: any dimensionality, one
// dimension at a time.
// F32: candidates from the level's centred FP32 copy, queries from the
// request's (centred the same way); acc32 <= tacc32 accepts, acc32 > trej32
// rejects, the band between is decided by the exact FP64 chain.
// Held to 3 waves per SIMD (130 registers): at 2 waves the candidate loads of
// too few waves are in flight (6-D, 10M points, 93k queries: 290 -> 270 ms per
// request); 4 waves measured the same.
template <int D, bool FILL, bool F32 = false, int QB = kQB>
__global__ __launch_bounds__(64 * kQWaves) __attribute__((amdgpu_waves_per_eu(3))) void k_qjoin(QJoinArgs) {
    static_assert(!F32 || D > 0, "FP32 filter needs a fixed dimensionality");
    __shared__ StencilList rls[kQWaves];
    __shared__ StencilTabs<QB> tabs[kQWaves];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    StencilList &rl = rls[wid];
    const QArgsPtr args = (QArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    __shared__ unsigned long long sh_stats[2];
    if (threadIdx.x < 2) sh_stats[threadIdx.x] = 0;
    __syncthreads();
    uint64_t my_evals = 0, my_band = 0;
    uint32_t n_items;
    {
        const QJoinArgs &a = reload(args);
        n_items = a.items_dev ? *a.items_dev : a.n_items;
    }
    // the first item of a wave is its number, the others come from the queue
    for (uint32_t w = blockIdx.x * kQWaves + wid; w < n_items;) {
        const QJoinArgs &a = reload(args);
        const uint32_t dim = D > 0 ? (uint32_t)D : a.qg.g.dim;
        const uint2 item = a.items[w];
        const uint32_t g0 = wave_bcast_u32(item.x), iy = wave_bcast_u32(item.y);
        const uint32_t seg = iy & 0xFF, nseg = (iy >> 8) & 0xFF, nqg = iy >> 16;
        {
            uint32_t qid[QB];
            uint64_t base[QB];
            uint32_t cnt[QB];
#pragma unroll
            for (int qi = 0; qi < QB; qi++) {
                qid[qi] = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.ids[g0 + min((uint32_t)qi, nqg - 1)]);
                base[qi] = FILL ? a.offsets[qid[qi]] : 0;
                cnt[qi] = 0;
            }
            if (FILL && seg > 0) {  // behind the unit's segments before this one
                uint32_t v = (uint32_t)lane / QB < seg ? a.seg_counts[(uint64_t)(w - seg) * QB + lane] : 0;
#pragma unroll
                for (int o = QB; o < 64; o *= 2) v += __shfl_xor(v, o, 64);
#pragma unroll
                for (int qi = 0; qi < QB; qi++) base[qi] += lane_u32(v, qi);
            }
            uint32_t nslots;
            const uint32_t M = qbuild_rows<QB>(a, a.keys[g0], qid, nqg, rl, tabs[wid], &nslots);
            // the group's query coordinates, once (lane i loads element i;
            // scalar registers), so no load in the candidate loop waits on
            // anything but the candidates
            constexpr int DQ = D > 0 ? D : 1;
            double qreg[F32 ? 1 : QB][DQ];
            float qregf[F32 ? QB : 1][DQ];
            if constexpr (F32) {
#pragma unroll
                for (int h = 0; h < (QB * DQ + 63) / 64; h++) {
                    const int e = h * 64 + lane, qi = e / DQ, l = e % DQ;
                    float v = 0.0f;
                    if (e < QB * DQ) {
                        uint32_t id = 0;
#pragma unroll
                        for (int k = 0; k < QB; k++) id = k == qi ? qid[k] : id;
                        v = a.q32[(uint64_t)id * dim + l];
                    }
#pragma unroll
                    for (int j = h * 64; j < QB * DQ && j < h * 64 + 64; j++)
                        qregf[j / DQ][j % DQ] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), j - h * 64));
                }
            } else if constexpr (D > 0) {
                static_assert(QB * D <= 64, "one load per lane");
                const int qi = lane / DQ, l = lane % DQ;
                double v = 0.0;
                if (lane < QB * DQ) {
                    uint32_t id = 0;
#pragma unroll
                    for (int k = 0; k < QB; k++) id = k == qi ? qid[k] : id;
                    v = a.queries[(uint64_t)id * dim + l];
                }
#pragma unroll
                for (int j = 0; j < QB * DQ; j++) {
                    const uint64_t u = (uint64_t)__double_as_longlong(v);
                    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, j);
                    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), j);
                    qreg[j / DQ][j % DQ] = __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
                }
            }
            // this wave's segment of the candidates, in whole chunks
            const uint32_t nch_all = (M + 63) / 64;
            const uint32_t per = nseg > 1 ? (nch_all + nseg - 1) / nseg : nch_all;
            const uint32_t clo = min(seg * per, nch_all), nch = min(clo + per, nch_all);
            const uint32_t mend = min(M, nch * 64);
            SlotCursor cur;
            cur.reset(rl);
            // NQ >= nqg queries evaluated: most cells of a sparse request hold
            // a single query (72% of the groups of 150k queries over 10M 6-D
            // points), and a group's unused places would cost as much as its
            // queries.
            auto sweep = [&](auto nqc) __attribute__((always_inline)) {
            constexpr int NQ = decltype(nqc)::value;
            const QJoinArgs &a = reload(args);
            const uint64_t n = a.qg.g.n;
            const double T = a.thresh;
            const double *__restrict__ soa = a.ix.soa;
            if constexpr (D > 0) {
                // Candidate chunks kDepth ahead in a register ring (coordinates,
                // positions and, when filling, point ids), so a wave keeps
                // several chunks of loads in flight instead of waiting on each.
                // A slot's position and id are copied out before the slot is
                // refilled; its coordinates are read by the distances first.
                constexpr int kDepth = 4;
                typedef typename std::conditional<F32, float, double>::type CT;
                CT ring[kDepth][DQ];
                uint32_t posr[kDepth], pidr[kDepth];
                auto load = [&](uint32_t t0, int p) __attribute__((always_inline)) {
                    const uint32_t t = t0 + lane;
                    const uint32_t pos = t < mend ? cur.pos(rl, t) : 0u;
                    posr[p] = pos;
                    if constexpr (F32) {
                        if constexpr (DQ % 2 == 0) {
                            typedef float f2 __attribute__((ext_vector_type(2)));
                            const f2 *src = reinterpret_cast<const f2 *>(a.aos32 + (uint64_t)pos * DQ);
#pragma unroll
                            for (int l = 0; l < DQ / 2; l++) {
                                const f2 v = src[l];
                                ring[p][2 * l] = v.x;
                                ring[p][2 * l + 1] = v.y;
                            }
                        } else {
#pragma unroll
                            for (int l = 0; l < DQ; l++) ring[p][l] = a.soa32[(uint64_t)l * n + pos];
                        }
                    } else if constexpr (D <= (int)kAosMaxDim) {
                        const double *src = a.ix.aos + (uint64_t)pos * DQ;
#pragma unroll
                        for (int l = 0; l < DQ; l++) ring[p][l] = src[l];
                    } else {
#pragma unroll
                        for (int l = 0; l < DQ; l++) ring[p][l] = soa[(uint64_t)l * n + pos];
                    }
                    if (FILL) pidr[p] = a.ix.ila[pos];
                };
                // Hit-chunk bitmap of the group (a.hitbits: kHitWords words
                // per query, the group's at its first query), one bit per
                // `span` chunks.  The count pass sets the bits of chunks in
                // which some query of the group has a neighbour; the fill
                // pass, which does the same arithmetic, visits only those.
                const uint32_t words = nqg * kHitWords / nseg, nown = nch - clo;
                uint64_t *hb = a.hitbits ? a.hitbits + (uint64_t)g0 * kHitWords + seg * words : nullptr;
                const uint32_t capb = words * 64;
                const uint32_t span = nown > capb ? (nown + capb - 1) / capb : 1u;
                const uint32_t nw = ((nown + span - 1) / span + 63) / 64;
                uint32_t cur = clo, cend = 0, wi = 0, bitpos = 0, subc = 0;
                uint64_t w = (FILL && hb && nw > 0) ? hb[0] : 0ull, hitw = 0;
                // next chunk to visit (nch when none is left)
                auto next = [&]() __attribute__((always_inline)) -> uint32_t {
                    if (!FILL || !hb) return cur < nch ? cur++ : nch;
                    if (cur + 1 < cend) return ++cur;
                    while (w == 0) {
                        if (++wi >= nw) return cur = cend = nch;
                        w = hb[wi];
                    }
                    const uint32_t b = wi * 64 + (uint32_t)__builtin_ctzll(w);
                    w &= w - 1;
                    cur = clo + b * span;
                    cend = min(cur + span, nch);
                    return cur;
                };
                uint32_t chr[kDepth];
#pragma unroll
                for (int p = 0; p < kDepth; p++) {
                    chr[p] = next();
                    load(chr[p] * 64, p);
                }
                while (chr[0] < nch) {
#pragma unroll
                    for (int p = 0; p < kDepth; p++) {
                        const uint32_t ch = chr[p];
                        const uint32_t t0 = ch * 64;
                        const bool valid = t0 + lane < mend;
                        const uint64_t vmask = __builtin_amdgcn_ballot_w64(valid);
                        const uint32_t pos = posr[p];
                        const uint32_t pid = FILL ? pidr[p] : 0u;
                        CT accv[NQ];
#pragma unroll
                        for (int qi = 0; qi < NQ; qi++) {
                            accv[qi] = (CT)0;
#pragma unroll
                            for (int l = 0; l < DQ; l++) {
                                if constexpr (F32) {
                                    const float d = ring[p][l] - qregf[qi][l];
                                    accv[qi] = __builtin_fmaf(d, d, accv[qi]);
                                } else {
                                    const double d = ring[p][l] - qreg[qi][l];
                                    accv[qi] = __builtin_fma(d, d, accv[qi]);
                                }
                            }
                        }
#pragma unroll
                        for (int qi = 0; qi < NQ; qi++) __asm__ volatile("" ::"v"(accv[qi]) : "memory");
                        chr[p] = next();
                        load(chr[p] * 64, p);
                        uint64_t anyhit = 0;
#pragma unroll
                        for (int qi = 0; qi < NQ; qi++) {
                            const uint64_t vq = (uint32_t)qi < nqg ? vmask : 0ull;
                            uint64_t m;
                            if constexpr (F32) {
                                m = __builtin_amdgcn_ballot_w64(accv[qi] <= a.tacc32) & vq;
                                const uint64_t mb = vq & ~m & ~__builtin_amdgcn_ballot_w64(accv[qi] > a.trej32);
                                if (mb) {
                                    // the band: the exact FP64 chain decides
                                    bool hit = false;
                                    if (__builtin_amdgcn_inverse_ballot_w64(mb)) {
                                        double e = 0.0;
#pragma unroll
                                        for (int l = 0; l < DQ; l++) {
                                            const double d = soa[(uint64_t)l * n + pos] - a.queries[(uint64_t)qid[qi] * dim + l];
                                            e = __builtin_fma(d, d, e);
                                        }
                                        hit = e <= T;
                                    }
                                    m |= __builtin_amdgcn_ballot_w64(hit);
                                    my_band += (uint64_t)__popcll(mb);
                                }
                            } else {
                                m = __builtin_amdgcn_ballot_w64(accv[qi] <= T) & vq;
                            }
                            if (FILL && m && __builtin_amdgcn_inverse_ballot_w64(m))
                                a.out[base[qi] + cnt[qi] + lanes_below(m)] = pid;
                            cnt[qi] += (uint32_t)__popcll(m);
                            anyhit |= m;
                        }
                        if (!FILL && hb && ch < nch) {
                            hitw |= (uint64_t)(anyhit != 0) << (bitpos & 63);
                            if (++subc == span) {
                                subc = 0;
                                if ((++bitpos & 63) == 0) {
                                    if (lane == 0) hb[(bitpos >> 6) - 1] = hitw;
                                    hitw = 0;
                                }
                            }
                        }
                    }
                }
                if (!FILL && hb && ((bitpos & 63) != 0 || subc != 0) && lane == 0) hb[bitpos >> 6] = hitw;
            } else {
                for (uint32_t t0 = clo * 64; t0 < mend; t0 += 64) {
                    const uint32_t t = t0 + lane;
                    const bool valid = t < mend;
                    const uint32_t pos = valid ? cur.pos(rl, t) : 0u;
                    // one compare per ballot, validity applied to the scalar
                    // masks; the hit lanes of a fill store under the mask itself
                    const uint64_t vmask = __builtin_amdgcn_ballot_w64(valid);
                    uint32_t pid = 0;
                    if (FILL) pid = a.ix.ila[pos];
                    double acc[NQ] = {};
                    for (uint32_t l = 0; l < dim; l++) {
                        const double xl = valid ? soa[(uint64_t)l * n + pos] : 0.0;
#pragma unroll
                        for (int qi = 0; qi < NQ; qi++) {
                            const double d = xl - a.queries[(uint64_t)qid[qi] * dim + l];
                            acc[qi] = __builtin_fma(d, d, acc[qi]);
                        }
                    }
#pragma unroll
                    for (int qi = 0; qi < NQ; qi++) {
                        const uint64_t m = __builtin_amdgcn_ballot_w64(acc[qi] <= T) & ((uint32_t)qi < nqg ? vmask : 0ull);
                        if (FILL && m && __builtin_amdgcn_inverse_ballot_w64(m))
                            a.out[base[qi] + cnt[qi] + lanes_below(m)] = pid;
                        cnt[qi] += (uint32_t)__popcll(m);
                    }
                }
            }
            };
            if (nqg == 1)
                sweep(std::integral_constant<int, 1>());
            else if (nqg == 2)
                sweep(std::integral_constant<int, 2>());
            else
                sweep(std::integral_constant<int, QB>());
            if (!FILL && lane < (int)nqg) {
                uint32_t mine = 0, id = 0;
#pragma unroll
                for (int qi = 0; qi < QB; qi++) {
                    mine = qi == lane ? cnt[qi] : mine;
                    id = qi == lane ? qid[qi] : id;
                }
                if (nseg == 1) {
                    a.counts[id] = mine;
                } else {
                    a.seg_counts[(uint64_t)w * QB + lane] = mine;
                    if (mine) atomicAdd(&a.counts[id], mine);
                }
            }
            if (lane == 0) my_evals += (uint64_t)(mend - min(mend, clo * 64)) * nqg;
        }
        if (lane == 0) w = gridDim.x * kQWaves + atomicAdd(reload(args).queue_head, 1u);
        w = (uint32_t)__builtin_amdgcn_readfirstlane((int)w);
    }
    if (!FILL) {
        if (lane == 0) {
            atomicAdd(&sh_stats[0], (unsigned long long)my_evals);
            atomicAdd(&sh_stats[1], (unsigned long long)my_band);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            const QJoinArgs &a = reload(args);
            if (sh_stats[0]) atomicAdd(a.evals, sh_stats[0]);
            if (sh_stats[1] && a.band) atomicAdd(a.band, sh_stats[1]);
        }
    }
}

// Pair hash of a request's CSR result: sum of mix64(query << 32 | neighbour)
// over its rows, G lanes per row; one atomic per workgroup (atomics on one
// address take 12 ns each, one after the other).
template <int G>
__global__ __launch_bounds__(256) void k_csr_hash(const uint64_t *__restrict__ off, const uint32_t *__restrict__ nb,
                                                  uint32_t n, unsigned long long *hash) {
    const uint32_t sub = threadIdx.x & (G - 1);
    const uint32_t grp = (blockIdx.x * 256 + threadIdx.x) / G, ngrp = (gridDim.x * 256) / G;
    uint64_t h = 0;
    for (uint32_t q = grp; q < n; q += ngrp) {
        const uint64_t b = off[q], e = off[q + 1];
        for (uint64_t j = b + sub; j < e; j += G) h += mix64(((uint64_t)q << 32) | nb[j]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) h += __shfl_xor(h, o, 64);
    __shared__ uint64_t sh[4];
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = h;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(hash, (unsigned long long)(sh[0] + sh[1] + sh[2] + sh[3]));
}

// q32 = fl32(fl64(q - centre)) and the largest |q - centre| (as ordered bits).
__global__ __launch_bounds__(256) void k_q32(const double *__restrict__ q, uint64_t total, uint32_t dim,
                                             const double *__restrict__ centre, float *__restrict__ q32,
                                             unsigned long long *rmax_bits) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    double r = 0.0;
    if (i < total) {
        const double d = q[i] - centre[i % dim];
        q32[i] = (float)d;
        r = fabs(d);
    }
    for (int o = 32; o > 0; o >>= 1) r = fmax(r, __shfl_xor(r, o, 64));
    if ((threadIdx.x & 63) == 0 && r > 0.0)
        atomicMax(rmax_bits, (unsigned long long)__double_as_longlong(r));
}

__global__ __launch_bounds__(256) void k_q_u32_u64(const uint32_t *__restrict__ in, uint32_t n,
                                                   uint64_t *__restrict__ out) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = in[i];
}

template <int D, bool FILL>
hegj_status launch_q(const QJoinArgs &a, uint32_t blocks, hipStream_t s) {
    if constexpr (D > 0) {
        if (a.f32)
            k_qjoin<D, FILL, true, kQBF32><<<blocks, 64 * kQWaves, 0, s>>>(a);
        else
            k_qjoin<D, FILL><<<blocks, 64 * kQWaves, 0, s>>>(a);
    } else {
        if (a.f32) return fail(HEGJ_ERR_UNSUPPORTED, "FP32 filter needs dim 2 or 6");
        k_qjoin<D, FILL><<<blocks, 64 * kQWaves, 0, s>>>(a);
    }
    HIP_TRY(hipGetLastError());
    return HEGJ_OK;
}

template <bool FILL>
hegj_status launch_qd(const QJoinArgs &a, uint32_t blocks, hipStream_t s) {
    switch (a.qg.g.dim) {
        case 2: return launch_q<2, FILL>(a, blocks, s);
        case 6: return launch_q<6, FILL>(a, blocks, s);
        default: return launch_q<0, FILL>(a, blocks, s);
    }
}

}  // namespace

hegj_status query_geom(const GridGeom &g, QueryGeom *qg) {
    qg->g = g;
    uint64_t prod = 1;
    for (uint32_t j = 0; j < g.k; j++) {
        const uint64_t w = (uint64_t)g.nCells[j] + 2;
        if (prod > (~0ull >> 1) / w) return fail(HEGJ_ERR_UNSUPPORTED, "query grid needs more than 63 bits");
        prod *= w;
    }
    qg->dead_key = prod;  // one past the largest live key
    int bits = 0;
    while (bits < 64 && (prod >> bits) != 0) bits++;
    qg->key_bits = bits;
    return HEGJ_OK;
}

hegj_status query_plan(QueryPlan *p, Scratch &keep, const QueryGeom &qg, const DevIndex &ix, const double *queries,
                       uint32_t nq, hipStream_t s) {
    *p = QueryPlan{};
    if (nq == 0) return HEGJ_OK;
    const uint32_t max_seg = std::min(std::max(kSplitItems / nq, 1u), kMaxSegments);
    HIP_TRY(keep.get(&p->keys, nq));
    HIP_TRY(keep.get(&p->ids, nq));
    HIP_TRY(keep.get(&p->items, (size_t)nq * max_seg));
    HIP_TRY(keep.get(&p->counts, nq));
    if (max_seg > 1) HIP_TRY(keep.get(&p->seg_counts, (size_t)nq * max_seg * kUnitQueries));
    Scratch sc;
    uint64_t *keys_alt;
    uint32_t *ids_alt, *flag;
    HIP_TRY(sc.get(&keys_alt, nq));
    HIP_TRY(sc.get(&ids_alt, nq));
    HIP_TRY(sc.get(&flag, nq));
    if (nq <= kSmallPlan) {
        HIP_TRY(keep.get(&p->items_dev, 1));
        k_qcell_keys<<<ceil_div(nq, 256), 256, 0, s>>>(queries, nq, qg, keys_alt, ids_alt);
        HIP_TRY(hipGetLastError());
        const uint32_t min_seg = std::min(std::max(kSpareItems / nq, 1u), kMaxSegments / 2);
        k_qsmall_rank<<<ceil_div(nq, 64), 256, 0, s>>>(keys_alt, nq, qg, ix, min_seg, max_seg, p->keys, p->ids,
                                                       flag, p->counts);
        HIP_TRY(hipGetLastError());
        k_qsmall_items<<<1, 1024, 0, s>>>(flag, nq, p->items, p->items_dev);
        HIP_TRY(hipGetLastError());
        p->n_items = nq * max_seg;  // at most: the device holds their number
        return scratch_done(s);
    }
    uint32_t *rank, *starts, *d_small;
    HIP_TRY(sc.get(&rank, nq));
    HIP_TRY(sc.get(&starts, (size_t)nq + 1));
    HIP_TRY(sc.get(&d_small, 2));
    HIP_TRY(hipMemsetAsync(p->counts, 0, sizeof(uint32_t) * nq, s));
    k_qcell_keys<<<ceil_div(nq, 256), 256, 0, s>>>(queries, nq, qg, p->keys, p->ids);
    HIP_TRY(hipGetLastError());
    HEGJ_TRY(radix_sort_u64(p->keys, p->ids, keys_alt, ids_alt, nq, qg.key_bits, s));
    HIP_TRY(hipMemsetAsync(d_small, 0, 2 * sizeof(uint32_t), s));
    k_qrun_flags<<<ceil_div(nq, 256), 256, 0, s>>>(p->keys, nq, qg.dead_key, flag, d_small + 1);
    HIP_TRY(hipGetLastError());
    HEGJ_TRY(scan_u32(flag, rank, nq, d_small, s));
    k_qrun_fill<<<ceil_div(nq, 256), 256, 0, s>>>(flag, rank, nq, starts);
    HIP_TRY(hipGetLastError());
    uint32_t h[2];
    HEGJ_TRY(read_back(h, d_small, s, 2));
    const uint32_t runs = h[0];
    // starts[runs] = end of the live queries
    HIP_TRY(hipMemcpyAsync(starts + runs, &h[1], sizeof(uint32_t), hipMemcpyHostToDevice, s));
    if (runs > 0) {
        uint32_t *cnt, *nseg, *first, *d_total;
        HIP_TRY(sc.get(&cnt, runs));
        HIP_TRY(sc.get(&nseg, runs));
        HIP_TRY(sc.get(&first, runs));
        HIP_TRY(sc.get(&d_total, 1));
        k_item_counts<<<ceil_div(runs, 256), 256, 0, s>>>(starts, runs, p->keys, qg, ix, max_seg, nseg, cnt);
        HIP_TRY(hipGetLastError());
        HEGJ_TRY(scan_u32(cnt, first, runs, d_total, s));
        k_item_fill<<<ceil_div(runs, 256), 256, 0, s>>>(starts, runs, nseg, first, p->items);
        HIP_TRY(hipGetLastError());
        HEGJ_TRY(read_back(&p->n_items, d_total, s));
    }
    return scratch_done(s);
}

hegj_status query_run(const QJoinArgs &base, bool fill, int device, hipStream_t s) {
    if (base.n_items == 0) return HEGJ_OK;
    // resident workgroups of the join on this device (thread-safe, once)
    static const uint32_t resident = [device]() {
        hipDeviceProp_t prop;
        int per_cu = 0;
        if (hipGetDeviceProperties(&prop, device) != hipSuccess) return 1024u;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, reinterpret_cast<const void *>(&k_qjoin<6, true>), 64 * kQWaves, 0) != hipSuccess)
            per_cu = 1;
        return (uint32_t)std::max(per_cu, 1) * (uint32_t)prop.multiProcessorCount;
    }();
    const uint32_t blocks =
        std::max<uint32_t>(1, std::min<uint32_t>(resident, ceil_div(base.n_items, kQWaves)));
    return fill ? launch_qd<true>(base, blocks, s) : launch_qd<false>(base, blocks, s);
}

hegj_status query_hash(const uint64_t *offsets, const uint32_t *nbrs, uint32_t nq, uint64_t total,
                       unsigned long long *hash, hipStream_t s) {
    if (nq == 0 || total == 0) return HEGJ_OK;
    const bool longrows = total / nq >= 256;
    const uint32_t G = longrows ? 64 : 16;
    const uint32_t blocks = std::min<uint32_t>(std::max<uint32_t>(ceil_div((uint64_t)nq * G, 256), 1), 4096);
    if (longrows)
        k_csr_hash<64><<<blocks, 256, 0, s>>>(offsets, nbrs, nq, hash);
    else
        k_csr_hash<16><<<blocks, 256, 0, s>>>(offsets, nbrs, nq, hash);
    HIP_TRY(hipGetLastError());
    return HEGJ_OK;
}

hegj_status query_to_f32(const double *q, uint32_t nq, uint32_t dim, const double *centre, float *q32,
                         unsigned long long *rmax_bits, hipStream_t s) {
    const uint64_t total = (uint64_t)nq * dim;
    if (total == 0) return HEGJ_OK;
    k_q32<<<ceil_div(total, 256), 256, 0, s>>>(q, total, dim, centre, q32, rmax_bits);
    HIP_TRY(hipGetLastError());
    return HEGJ_OK;
}

hegj_status query_offsets(const uint32_t *counts, uint32_t nq, uint64_t *offsets, hipStream_t s) {
    if (nq <= kSmallScan) {
        k_qsmall_offsets<<<1, 1024, 0, s>>>(counts, nq, offsets);
        HIP_TRY(hipGetLastError());
        return HEGJ_OK;
    }
    Scratch sc;
    uint64_t *c64;
    HIP_TRY(sc.get(&c64, nq));
    k_q_u32_u64<<<ceil_div(nq, 256), 256, 0, s>>>(counts, nq, c64);
    HIP_TRY(hipGetLastError());
    return scan_u64(c64, offsets, nq, offsets + nq, s);
}

}  // namespace hegj
