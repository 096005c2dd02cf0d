// hegj_stencil.h -- the stencil rows of one cell, found by one wave.
//
// A row is a position in indexed dims 1..k-1 (3^(k-1) of them around a cell);
// the cells of a row that lie in the dim-0 window are one run of candidate
// positions.  A work unit needs the non-empty runs, less the cells that
// cell-box pruning leaves out, as a compacted list in LDS.
//
// This was a third of the 6-D join (12 of 37 ms at 5M points, 2.4M units), as
// much issue as waiting: five 64-bit divisions to take the cell's id apart,
// per row a digit loop with 64-bit products and, per query, five gap lookups,
// a 64-bit mixing hash, and for rows of more than 4 cells two binary searches
// per row, one row after the other.  Here
//   - the cell's coordinates come from the index (cell_xyz);
//   - a row number splits as a + 9 b: a covers dims 1 and 2, b dims 3 to 5, so
//     its key and its gap to a query are sums of two table entries (9 and 27,
//     made once per unit by as many lanes);
//   - a lane's rows (l, l + 64, ..) take each dependent step together, the
//     binary search included; its upper end comes from the three keys at the
//     lower one (the window is three cells wide at most).
#pragma once

#include "hegj_internal.h"

namespace hegj {

// One wave's list of runs, in LDS.
struct StencilList {
    uint32_t start[kMaxRows + 1];  // first candidate position of slot s (+1: a padding slot)
    uint32_t off[kMaxRows + 1];    // prefix of slot lengths
};
// LDS tables needed only while the list is made.  QB: queries.
template <int QB>
struct StencilTabs {
    float2 gap[QB * kMaxK];        // per (query, indexed dim): squared gaps to the -1 / +1 cell
    uint64_t key9[9], key27[27];   // row key parts of dims 1, 2 and of dims 3..5
    float g9[QB * 9], g27[QB * 27];  // squared gap parts, per query
};

// Coordinates and dim bounds of a cell, wave-uniform.
struct CellBox {
    uint32_t c[kMaxK], lo[kMaxK], hi[kMaxK];
};

__device__ __forceinline__ uint32_t lane_u32(uint32_t v, int l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}

// The box of a non-empty cell; false when the cell-0 wrap silences it.
__device__ __forceinline__ bool cell_box(const GridGeom &g, const DevIndex &ix, uint32_t cell, CellBox &b) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t x = lane < g.k ? ix.cell_xyz[(uint64_t)lane * ix.C + cell] : 0u;
    bool ok = true;
#pragma unroll
    for (int j = 0; j < kMaxK; j++) {
        b.c[j] = lane_u32(x, j);
        b.lo[j] = b.hi[j] = 0;
        if ((uint32_t)j < g.k) ok &= stencil_dim(b.c[j], g.nCells[j], g.emulate_cell0, &b.lo[j], &b.hi[j]);
    }
    return ok;
}

// A lane's rows (l, l + 64, ..): the row's cells [ca, re), none where the row
// is empty or left out, and the dim-0 window [lo, hi].
constexpr int kLaneRows = (kMaxRows + 63) / 64;
struct LaneRows {
    uint32_t ca[kLaneRows], re[kLaneRows], lo[kLaneRows], hi[kLaneRows];
};

// The rows of the box `b`.  tb.gap holds the gaps of nq queries (written and
// ordered by the caller); a cell is kept when the sum of its squared gaps is
// at most thr for one of them (nq = 0 with thr = +inf: every cell).  c0: the
// dim-0 coordinate, signed (a query's cell may lie one outside the grid).
template <int QB>
__device__ __forceinline__ void stencil_probe(const GridGeom &g, const DevIndex &ix, StencilTabs<QB> &tb,
                                              const CellBox &b, int64_t c0, uint32_t nq, float thr, LaneRows &w) {
    const uint32_t lane = threadIdx.x & 63, k = g.k;
    // tables: lanes 0..8 take part a (dims 1, 2), lanes 16..42 part b (dims 3..5)
    const bool isb = lane >= 16;
    const uint32_t t = isb ? lane - 16 : lane;
    const uint32_t o0 = t % 3, o1 = (t / 3) % 3, o2 = t / 9;
    const bool has = isb ? t < 27 : t < 9;
    bool inside = has;
    uint64_t key = 0;
    float2 *const gap = tb.gap;
    const int ja = isb ? 3 : 1;
    {
        uint64_t mult = 1;
#pragma unroll
        for (int j = 1; j < kMaxK; j++) {
            if ((uint32_t)j >= k) break;
            const bool mine = isb ? j >= 3 : j < 3;
            const uint32_t o = j == 1 || j == 3 ? o0 : j == 2 || j == 4 ? o1 : o2;
            const uint32_t cj = b.c[j] + o - 1;  // wraps below 0, rejected here
            if (mine) {
                inside &= cj >= b.lo[j] && cj <= b.hi[j];
                key += (uint64_t)cj * mult;
            }
            mult *= g.nCells[j];
        }
    }
    const uint64_t in = __builtin_amdgcn_ballot_w64(inside);
    const uint32_t in9 = (uint32_t)in & 0x1FFu, in27 = (uint32_t)(in >> 16);
    if (has) (isb ? tb.key27 : tb.key9)[t] = key;
    for (uint32_t qi = 0; qi < nq; qi++) {
        if (!has) continue;
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            if (i == 2 && !isb) break;
            if ((uint32_t)(ja + i) >= k) break;
            const float2 v = gap[qi * kMaxK + ja + i];
            const uint32_t o = i == 0 ? o0 : i == 1 ? o1 : o2;
            s += o == 0 ? v.x : (o == 2 ? v.y : 0.0f);
        }
        if (isb)
            tb.g27[qi * 27 + t] = s;
        else
            tb.g9[qi * 9 + t] = s;
    }
    wave_lds_sync();
    const uint32_t nrows = pow3(k - 1);
    constexpr int R = kLaneRows;
    uint32_t slot[R];
    uint64_t rkey[R];
    bool want[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
        const uint32_t r = min(lane + 64u * i, (uint32_t)kMaxRows - 1), rb = r / 9, ra = r - rb * 9;
        want[i] = lane + 64u * i < nrows && ((in9 >> ra) & (in27 >> rb) & 1u);
        rkey[i] = tb.key9[ra] + tb.key27[rb];
        int64_t l = b.lo[0], h = b.hi[0];
        float mmid = 3.4e38f, mleft = 3.4e38f, mright = 3.4e38f;
        for (uint32_t qi = 0; qi < nq; qi++) {
            const float rd = tb.g9[qi * 9 + ra] + tb.g27[qi * 27 + rb];
            const float2 v0 = gap[qi * kMaxK];
            mmid = fminf(mmid, rd);
            mleft = fminf(mleft, rd + v0.x);
            mright = fminf(mright, rd + v0.y);
        }
        if (!(mleft <= thr) && c0 > l) l = c0;
        if (!(mright <= thr) && c0 < h) h = c0;
        want[i] = want[i] && mmid <= thr && l <= h;
        w.lo[i] = (uint32_t)l;
        w.hi[i] = (uint32_t)h;
        slot[i] = hash_slot(rkey[i]) & ix.hmask;
    }
    // hash probes: first slots together, collisions one by one
    {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        const u32x4 *const tab = reinterpret_cast<const u32x4 *>(ix.hrows);
        u32x4 e[R];
#pragma unroll
        for (int i = 0; i < R; i++) {
            e[i] = u32x4{~0u, ~0u, 0u, 0u};
            if (want[i]) e[i] = tab[slot[i]];
        }
#pragma unroll
        for (int i = 0; i < R; i++) {
            const uint32_t k0 = (uint32_t)rkey[i], k1 = (uint32_t)(rkey[i] >> 32);
            bool hit = e[i].x == k0 && e[i].y == k1;
            while (want[i] && !hit && (e[i].x & e[i].y) != ~0u) {
                slot[i] = (slot[i] + 1) & ix.hmask;
                e[i] = tab[slot[i]];
                hit = e[i].x == k0 && e[i].y == k1;
            }
            w.ca[i] = want[i] && hit ? e[i].z : 0u;
            w.re[i] = want[i] && hit ? e[i].w : 0u;
        }
    }
}

// Candidate positions [pstart, pstart + plen) of a lane's rows.
__device__ __forceinline__ void stencil_ranges(const DevIndex &ix, const LaneRows &w, uint32_t (&pstart)[kLaneRows],
                                               uint32_t (&plen)[kLaneRows]) {
    constexpr int R = kLaneRows;
    uint32_t ca[R], longest = 0;
#pragma unroll
    for (int i = 0; i < R; i++) {
        ca[i] = w.ca[i];
        longest = max(longest, w.re[i] - ca[i]);
    }
    // first cell at or after the window's start, all rows in step, by the
    // cells' dim-0 coordinates (ascending within a row)
    const uint32_t *const x0 = ix.cell_xyz;
    uint32_t end[R];
#pragma unroll
    for (int i = 0; i < R; i++) end[i] = w.re[i];
    while (__builtin_amdgcn_ballot_w64(longest > 3)) {
        uint32_t v[R];
#pragma unroll
        for (int i = 0; i < R; i++) v[i] = end[i] > ca[i] ? x0[(ca[i] + end[i]) >> 1] : 0u;
        longest = 0;
#pragma unroll
        for (int i = 0; i < R; i++) {
            if (end[i] > ca[i]) {
                const uint32_t mid = (ca[i] + end[i]) >> 1;
                if (v[i] < w.lo[i])
                    ca[i] = mid + 1;
                else
                    end[i] = mid;
            }
            longest = max(longest, end[i] - ca[i]);
        }
    }
    // at most 3 cells are left before the lower bound and 3 from it on are in
    // the window: six coordinates decide both ends
    uint32_t ck[R][6], cb[R];
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
        for (int j = 0; j < 6; j++) ck[i][j] = ca[i] + j < w.re[i] ? x0[ca[i] + j] : ~0u;
#pragma unroll
    for (int i = 0; i < R; i++) {
        uint32_t na = 0, nb = 0;
#pragma unroll
        for (int j = 0; j < 6; j++) {
            const bool in_row = ca[i] + j < w.re[i];
            na += in_row && ck[i][j] < w.lo[i] ? 1u : 0u;
            nb += in_row && ck[i][j] <= w.hi[i] ? 1u : 0u;
        }
        cb[i] = ca[i] + nb;
        ca[i] += na;
    }
#pragma unroll
    for (int i = 0; i < R; i++) {
        const bool any = cb[i] > ca[i];
        pstart[i] = any ? ix.cell_start[ca[i]] : 0u;
        plen[i] = any ? ix.cell_start[cb[i]] - pstart[i] : 0u;
    }
}

// Rows of the box `b` into rl; returns the number of candidates, *nslots the
// number of rows kept.  The other arguments as for stencil_probe.
template <int QB, typename L>
__device__ __forceinline__ uint32_t stencil_rows(const GridGeom &g, const DevIndex &ix, L &rl,
                                                 StencilTabs<QB> &tb, const CellBox &b, int64_t c0, uint32_t nq,
                                                 float thr, uint32_t *nslots) {
    LaneRows w;
    stencil_probe<QB>(g, ix, tb, b, c0, nq, thr, w);
    uint32_t pstart[kLaneRows], plen[kLaneRows];
    stencil_ranges(ix, w, pstart, plen);
    // compact the non-empty rows, in row order, into the LDS list
    const uint32_t lane = threadIdx.x & 63, nrows = pow3(g.k - 1);
    uint32_t slots = 0, total = 0;
#pragma unroll
    for (int i = 0; i < kLaneRows; i++) {
        if (64u * i >= nrows) break;
        const uint64_t nz = __ballot(plen[i] > 0);
        uint32_t x = plen[i];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (plen[i] > 0) {
            const uint32_t s = slots + lanes_below(nz);
            rl.start[s] = pstart[i];
            rl.off[s] = total + x - plen[i];
        }
        slots += (uint32_t)__popcll(nz);
        total += lane_u32(x, 63);
    }
    if (lane == 0) rl.off[slots] = total;
    *nslots = slots;
    return total;
}

}  // namespace hegj
