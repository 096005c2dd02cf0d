// hegj_gb.h -- device code shared by the two MFMA guard-band joins
// (hegj_mfma.hip: split BF16, hegj_gram16.hip: FP16): the key lists they
// append to and the stencil-row list of a workgroup's work unit.
#pragma once

#include "hegj_internal.h"

namespace hegj {

constexpr int kGbBlk = 256;          // pair-list slots reserved per wave at a time
constexpr uint64_t kSentinel = ~0ull;
// A band key with this bit stands for both ordered pairs (query positions are
// below 2^29, so the bit is free).
constexpr uint64_t kGbMirror = 1ull << 63;

// Bit moves between float and uint32 that compile for host and device.
__host__ __device__ __forceinline__ uint32_t f2u(float f) {
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    return u;
}
__host__ __device__ __forceinline__ float u2f(uint32_t u) {
    float f;
    __builtin_memcpy(&f, &u, 4);
    return f;
}

// Neighbouring FP32 values (finite inputs), by bit arithmetic.
__host__ __device__ __forceinline__ float f32_next_up(float f) {
    uint32_t u = f2u(f);
    if (f == 0.0f) return u2f(1u);
    return u2f((u >> 31) ? u - 1 : u + 1);
}
__host__ __device__ __forceinline__ float f32_next_down(float f) {
    uint32_t u = f2u(f);
    if (f == 0.0f) return u2f(0x80000001u);
    return u2f((u >> 31) ? u + 1 : u - 1);
}

// Stencil-row list shared by the workgroup.
struct GbRows {
    uint32_t start[kMaxRows];
    uint32_t off[kMaxRows + 1];
};

// One wave builds the stencil rows of `cell` (ascending positions; nothing
// when the cell is silenced).  *below: candidates at positions under `pos0`.
__device__ __forceinline__ void gb_build_rows(const GridGeom &g, const DevIndex &ix, uint32_t cell,
                                              uint32_t pos0, GbRows &rl, uint32_t *n_slots,
                                              uint32_t *n_cand, uint32_t *below) {
    const int lane = threadIdx.x & 63;
    uint32_t c[kMaxK], lo[kMaxK], hi[kMaxK];
    decode_cell(ix.cell_key[cell], g, c);
    bool ok = true;
    for (uint32_t j = 0; j < g.k; j++)
        ok &= stencil_dim(c[j], g.nCells[j], g.emulate_cell0, &lo[j], &hi[j]);
    uint32_t slots = 0, total = 0, under = 0;
    if (ok) {
        const uint32_t nrows = pow3(g.k - 1);
        for (uint32_t r0 = 0; r0 < nrows; r0 += 64) {
            const uint32_t r = r0 + lane;
            uint32_t pstart = 0, plen = 0;
            if (r < nrows) {
                uint32_t cf, cl;
                stencil_row(c, lo, hi, r, g, ix, &cf, &cl);
                if (cl > cf) {
                    pstart = ix.cell_start[cf];
                    plen = ix.cell_start[cl] - pstart;
                }
            }
            const uint64_t nz = __ballot(plen > 0);
            uint32_t x = plen;
            for (int o = 1; o < 64; o <<= 1) {
                uint32_t y = __shfl_up(x, o, 64);
                if (lane >= o) x += y;
            }
            if (plen > 0) {
                const uint32_t s = slots + lanes_below(nz);
                rl.start[s] = pstart;
                rl.off[s] = total + x - plen;
            }
            slots += (uint32_t)__popcll(nz);
            total += __shfl(x, 63, 64);
            under += pstart < pos0 ? min(plen, pos0 - pstart) : 0u;
        }
    }
    if (lane == 0) rl.off[slots] = total;
    for (int o = 32; o > 0; o >>= 1) under += __shfl_xor(under, o, 64);
    *n_slots = slots;
    *n_cand = total;
    *below = under;
}

// Next work unit for a workgroup (thread 0): its XCD's range first
// (neighbouring cells share candidates in that XCD's L2), then the others.
// `tried`: ranges found empty so far.  ~0u when all are drained.
__device__ __forceinline__ uint32_t gb_next_unit(uint32_t *queue_heads, uint32_t n_parts,
                                                 const uint32_t *part_end, uint32_t part0,
                                                 uint32_t &tried) {
    while (tried < n_parts) {
        const uint32_t p = (part0 + tried) % n_parts;
        const uint32_t k = (p ? part_end[p - 1] : 0u) + atomicAdd(&queue_heads[p], 1u);
        if (k < part_end[p]) return k;
        tried++;
    }
    return ~0u;
}

// Per-wave append buffer into a global key list (blocks of kGbBlk slots;
// unused tails are filled with the sentinel, which sorts last).
struct Appender {
    uint64_t cur, end;
};

__device__ __forceinline__ void append_keys(uint64_t key, bool pred, Appender &ap,
                                            uint64_t *list, uint64_t cap,
                                            unsigned long long *cursor, uint32_t *overflow) {
    const int lane = threadIdx.x & 63;
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    const uint32_t k = (uint32_t)__popcll(m);
    if (ap.cur + k > ap.end) {
        // pad the rest of the block, then take a new one
        for (uint64_t i = ap.cur + lane; i < ap.end; i += 64) list[i] = kSentinel;
        uint64_t b = 0;
        if (lane == 0) b = atomicAdd(cursor, (unsigned long long)kGbBlk);
        b = wave_bcast_u64(b);
        if (b + kGbBlk > cap) {
            if (lane == 0) atomicOr(overflow, 1u);
            ap.cur = ap.end = 0;
            return;
        }
        ap.cur = b;
        ap.end = b + kGbBlk;
    }
    if (pred) list[ap.cur + lanes_below(m)] = key;
    ap.cur += k;
}

__device__ __forceinline__ void close_appender(Appender &ap, uint64_t *list) {
    const int lane = threadIdx.x & 63;
    for (uint64_t i = ap.cur + lane; i < ap.end; i += 64) list[i] = kSentinel;
}

// Arguments of both joins (launch_gb / g16_launch pick the kernel).
struct GbArgs {
    GridGeom g;
    DevIndex ix;
    const uint2 *units;           // (cell, first query offset in cell)
    const uint4 *units16;         // FP16 join: (cell, query offset, first candidate, end)
    uint32_t n_units;
    uint32_t *queue_heads;        // [kMaxParts] units taken per range
    uint32_t n_parts;             // unit ranges: range p is [part_end[p - 1], part_end[p])
    uint32_t part_end[kMaxParts];
    const uint16_t *Av;
    const uint16_t *Bv;
    const float *w;
    uint32_t kp;
    uint32_t mirror;              // FP16 join: each unordered pair evaluated once
    float trej;                   // FP16 join: s' > trej is out
    double tacc;                  // FP16 join: s' + w_q + w_c <= tacc is in
    uint64_t *raw;                // FP16 join: survivors of the reject test, keys
    float *raw_s;                 // and their s'
    uint64_t raw_cap;             // a multiple of kGbBlk below 2^32
    unsigned long long *raw_cursor;
    unsigned long long *raw_lost; // survivors that did not fit
    uint64_t *pairs;              // accepted keys (qpos << 32 | cpos)
    uint64_t pair_cap;
    unsigned long long *pair_cursor;
    uint64_t *band;               // band keys
    uint64_t band_cap;
    unsigned long long *band_cursor;
    unsigned long long *n_accept;
    unsigned long long *n_band;
    unsigned long long *evals;
    uint32_t *overflow;
};

}  // namespace hegj
