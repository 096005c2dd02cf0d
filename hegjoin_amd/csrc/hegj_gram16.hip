// hegj_gram16.hip -- the MFMA refine at one FP16 product per dimension: Gram
// tiles with a proven guard band, each unordered pair evaluated once.
//
// The split-BF16 join (hegj_mfma.hip) spends three products per dimension to
// make its distances good to ~2^-15.  A filter needs less: the pairs it
// cannot decide go to the exact FP64 chain anyway, and near the threshold
// there are few of them.  Here a point is one FP16 vector
//     z = fp16((x - mean) * sigma),  sigma a power of two
// and its own rounding error E >= ||z - sigma (x - mean)|| is measured in FP64
// when the operands are made, so the guard is what the data need and not a
// worst case over the format.  With tau = sigma sqrt(T), G = ||z_q - z_c||^2:
//     acc <= T  =>  sqrt(G) <= tau + E_q + E_c
//               =>  G <= tau^2 + (2 tau E_q + 2 E_q^2) + (2 tau E_c + 2 E_c^2)
//     sqrt(G) <= tau - E_q - E_c  <=  G <= tau^2 - 2 tau E_q - 2 tau E_c
//                                  =>  acc <= T
// The per-point terms fold into the operands.  A' = [-2z, n, 1, 1] and
// B' = [z, 1, 1, n], n = hi + lo <= ||z||^2 - (2 tau E + 2 E^2) - a, so one
// v_mfma_f32_16x16x32_f16 chain of K = dim + 4 (18-D: one instruction for 256
// pairs, the split BF16 took two; 90-D: three against nine) gives
//     s' = -2 z_q.z_c + n_q + n_c,   s' > tau^2            => acc > T (reject)
//     w >= ||z||^2 - n + 2 tau E + a,  s' + w_q + w_c <= tau^2 => acc <= T
// and the pairs in between are the band.  a covers the FP32 accumulation
// inside the MFMAs (any order and rounding mode, twice its bound); tau^2 is
// moved outwards (inwards to accept) by the rounding of the FP64 chain
// itself.  The pair set is the FP64 one.  Elements below 2^-14 become zero
// (their value goes to E), so no FP16 denormal enters an MFMA.
//
// Both (q, c) and (c, q) have the same FP64 chain value (the differences are
// negated exactly), so a unit visits only candidates at or after its first
// query in cell order and emits both keys for those beyond its last query.
// With the cell-0 wrap some points are candidates but never queries: then
// (args.mirror = 0) every unit visits its whole stencil.
//
// What bounds it: 2 K flops per evaluated pair on the matrix cores.  The
// running minimum that rejects a tile costs two v_min3 per MFMA (8 of its 16
// cycles, in the shadow of the other waves' MFMAs).  18-D, 2M points, 32
// neighbours: 488 ms split BF16 -> 67.7 ms, 1.35e12 pairs, 1.28 PFLOP/s;
// 90-D, 1M points, 16 neighbours: 701 -> 67.6 ms, 5e11 pairs, 1.42 PFLOP/s.
// A large library FP16 matrix product runs at 1.37 PFLOP/s on the same card.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "hegj_gb.h"

namespace hegj {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kRt = 8;                             // 16-query row tiles per wave
constexpr uint32_t kUnitQ = kWaves * kRt * 16;     // queries per unit
// Candidates per LDS chunk: 8 KB to 16 KB of operands, so a chunk keeps every
// wave busy for ~1000 cycles per barrier and three to four workgroups fit.
constexpr int chunk_of(int kb) { return kb == 1 ? 128 : 64; }
constexpr uint32_t kMaxChunk = 128;
constexpr float kPadNorm = 65504.0f;

// ---- operands ------------------------------------------------------------
// max_p ||x_p - mean||^2 as the bits of a positive double, over the points
// whose coordinates are all finite (the others have no neighbour: their chain
// is inf or NaN against every point, and they get the padding row).
__global__ __launch_bounds__(256) void k_g16_maxnorm(const double *__restrict__ soa, uint32_t n,
                                                     uint32_t dim, const double *__restrict__ mean,
                                                     unsigned long long *max_bits) {
    __shared__ double sh[4];
    double m = 0.0;
    for (uint64_t p = (uint64_t)blockIdx.x * 256 + threadIdx.x; p < n; p += (uint64_t)gridDim.x * 256) {
        double s = 0.0;
        bool fin = true;
        for (uint32_t l = 0; l < dim; l++) {
            const double x = soa[(uint64_t)l * n + p], y = x - mean[l];
            fin &= __builtin_isfinite(x);
            s = __builtin_fma(y, y, s);
        }
        if (fin) m = fmax(m, s);  // +inf when finite coordinates overflow it
    }
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
        atomicMax(max_bits, (unsigned long long)__double_as_longlong(m));
    }
}

__host__ __device__ __forceinline__ uint16_t h_bits(_Float16 h) {
    uint16_t b;
    __builtin_memcpy(&b, &h, 2);
    return b;
}

// fp16 of v (FP64), elements below the normal range to zero.
__host__ __device__ __forceinline__ _Float16 to_h16(double v) {
    const _Float16 h = (_Float16)(float)v;
    return __builtin_fabs((double)(float)h) < 6.103515625e-05 ? (_Float16)0.0f : h;
}

// fp16 not above v (|v| in the normal range or moved down into it).
__host__ __device__ __forceinline__ _Float16 h16_down(double v) {
    if (v >= 0.0 && v < 6.103515625e-05) return (_Float16)0.0f;
    if (v < 0.0 && v > -6.103515625e-05) return (_Float16)-6.103515625e-05f;
    _Float16 h = (_Float16)(float)v;
    if ((double)(float)h > v) {
        uint16_t b = h_bits(h);
        b = h > (_Float16)0.0f ? b - 1 : b + 1;  // one step toward -inf
        __builtin_memcpy(&h, &b, 2);
        if (__builtin_fabs((double)(float)h) < 6.103515625e-05) h = (_Float16)0.0f;  // stepped out of the normals
    }
    return h;
}

// One point's rows A' and B' (kp values, a multiple of 32) and its accept
// guard w, from its coordinates x (stride `stride` between dims); its rounding
// error E and squared norm N are returned.  real = false, or a coordinate that is not finite: the
// padding row (s' >= 65504 against anything, above any tau^2), E = N = 0.
// Built for the host too, where the guards are tested: guard_scale (1 in the
// join) shrinks them.
struct G16Point {
    double err, norm;
};
__host__ __device__ __forceinline__ G16Point g16_point(const double *x, uint64_t stride, uint32_t dim, int kp,
                                                     const double *mean, double sigma, double tau, double gamma,
                                                     double guard_scale, bool real, uint16_t *A, uint16_t *B,
                                                     float *w) {
    const bool point = real;
    f16x8 az, bz;
    double N = 0.0, e2 = 0.0, y2 = 0.0;
    G16Point r{0.0, 0.0};
    f16x8 *arow = reinterpret_cast<f16x8 *>(A);
    f16x8 *brow = reinterpret_cast<f16x8 *>(B);
    for (int k0 = 0; k0 < kp; k0 += 8) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t l = (uint32_t)(k0 + i);
            _Float16 z = (_Float16)0.0f;
            if (l < dim && point) {
                const double xl = x[(uint64_t)l * stride], y = (xl - mean[l]) * sigma;
                real &= __builtin_isfinite(xl);
                z = real ? to_h16(y) : (_Float16)0.0f;
                const double zd = (double)(float)z, e = y - zd;
                N = __builtin_fma(zd, zd, N);
                e2 = __builtin_fma(e, e, e2);
                y2 = __builtin_fma(y, y, y2);
            }
            bz[i] = z;
            az[i] = z * (_Float16)-2.0f;  // exact
        }
        if (k0 < kp - 8) {
            arow[k0 / 8] = az;
            brow[k0 / 8] = bz;
        }
    }
    // the last group of 8 ends with the norm slots (dim <= kp - 4); a
    // point with a coordinate that is not finite becomes a padding row
    _Float16 nhi = (_Float16)kPadNorm, nlo = (_Float16)kPadNorm;
    if (point && !real) {
        *w = 0.0f;
        az = bz = (f16x8)(_Float16)0.0f;
        for (int j = 0; j < kp / 8 - 1; j++) arow[j] = brow[j] = az;
    }
    if (real) {
        const double u64 = 1.1102230246251565e-16;
        const double rel = 4.0 * (dim + 4) * u64;
        // measured error, its own rounding, and that of x - mean
        const double err = (__builtin_sqrt(e2) * (1.0 + rel) + 4.0 * u64 * __builtin_sqrt(y2)) * guard_scale;
        const double s0 = (2.0 * tau * err + 2.0 * err * err) * (1.0 + 1e-12);
        const double acc = 2.0 * gamma * guard_scale * (2.1 * N + 1.1 * s0);
        const double v = N * (1.0 - rel) - s0 - acc;
        nhi = to_h16(v);
        nlo = h16_down(v - (double)(float)nhi);
        const double nt = (double)(float)nhi + (double)(float)nlo;
        const double wd = (N * (1.0 + rel) - nt) + 2.0 * tau * err * (1.0 + 1e-12) + acc;
        float wf = (float)wd;
        if ((double)wf < wd) wf = f32_next_up(wf);
        *w = wf;
        r = G16Point{err, N};
    }
    az[4] = nhi;
    az[5] = nlo;
    az[6] = az[7] = (_Float16)1.0f;
    bz[4] = bz[5] = (_Float16)1.0f;
    bz[6] = nhi;
    bz[7] = nlo;
    arow[kp / 8 - 1] = az;
    brow[kp / 8 - 1] = bz;
    return r;
}

// Sums over the points, each on a line of its own: E, and the shares of tau^2
// that the guards of a pair of such points take, here and in the split-BF16
// join (at most 1: then every near pair is in the band).
enum G16Sum { kSumErr, kSumShare, kSumShareBf, kSums };
constexpr int kLineDoubles = kLineWords / 2;

// One thread per point (cell order); row n of A and B is the padding row.
// bf: the split-BF16 join's guard of two points per unit of N.
template <int KB>
__global__ __launch_bounds__(256) void k_g16_prepare(const double *__restrict__ soa, uint32_t n,
                                                     uint32_t dim, const double *__restrict__ mean,
                                                     double sigma, double tau, double gamma, double bf,
                                                     uint16_t *__restrict__ A, uint16_t *__restrict__ B,
                                                     float *__restrict__ w, double *sums) {
    constexpr int KP = KB * 32;
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    double v[kSums] = {};
    if (p <= n) {
        const G16Point r = g16_point(soa + (p < n ? p : 0), n, dim, KP, mean, sigma, tau, gamma, 1.0, p < n,
                                     A + (uint64_t)p * KP, B + (uint64_t)p * KP, w + p);
        if (p < n) {
            v[kSumErr] = r.err;
            v[kSumShare] = fmin(1.0, 2.0 * (double)w[p] / (tau * tau));
            v[kSumShareBf] = fmin(1.0, bf * r.norm / (tau * tau));
        }
    }
    __shared__ double sh[kSums][4];
#pragma unroll
    for (int k = 0; k < kSums; k++) {
        for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
        if ((threadIdx.x & 63) == 0) sh[k][threadIdx.x >> 6] = v[k];
    }
    __syncthreads();
    if (threadIdx.x < kSums) {
        const double *s = sh[threadIdx.x];
        atomicAdd(sums + threadIdx.x * kLineDoubles, s[0] + s[1] + s[2] + s[3]);
    }
}

// ---- work units ------------------------------------------------------------
// Cell i of the order contributes (query blocks of kUnitQ) x (segments of
// `seg` candidates of its stencil); none when the cell is silenced (work 0).
__global__ __launch_bounds__(256) void k_g16_unit_counts(DevIndex ix, const uint32_t *__restrict__ order,
                                                         const uint32_t *__restrict__ work, uint32_t seg,
                                                         uint32_t *__restrict__ cnt) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= ix.C) return;
    const uint32_t cell = order ? order[i] : i;
    const uint32_t sz = ix.cell_start[cell + 1] - ix.cell_start[cell];
    cnt[i] = ((sz + kUnitQ - 1) / kUnitQ) * ((work[cell] + seg - 1) / seg);
}

// One thread per unit: within a cell segment-major, so the query blocks that
// run at the same time stream the same candidates.
__global__ __launch_bounds__(256) void k_g16_unit_fill(DevIndex ix, const uint32_t *__restrict__ order,
                                                       const uint32_t *__restrict__ work, uint32_t seg,
                                                       const uint32_t *__restrict__ off, uint32_t U,
                                                       uint4 *__restrict__ units) {
    const uint32_t u = blockIdx.x * 256 + threadIdx.x;
    if (u >= U) return;
    uint32_t lo = 0, hi = ix.C;  // last i with off[i] <= u
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (off[mid] <= u)
            lo = mid;
        else
            hi = mid;
    }
    const uint32_t cell = order ? order[lo] : lo;
    const uint32_t sz = ix.cell_start[cell + 1] - ix.cell_start[cell];
    const uint32_t nb = (sz + kUnitQ - 1) / kUnitQ, k = u - off[lo];
    const uint32_t s = k / nb, b = k - s * nb;
    units[u] = make_uint4(cell, b * kUnitQ, s * seg, min(work[cell], (s + 1) * seg));
}

// ---- the join --------------------------------------------------------------
// Survivors of the reject test go to one global list as they are found: the
// query position (bit 31: stands for both ordered pairs), the candidate
// position and s'.  They are a few in a million, and what decides them (two
// dependent loads of guards each, the FP64 chain for the band) is done for 64
// at a time by k_g16_decide instead of stalling this kernel's waves.
// One wave's share of a candidate chunk on its way to LDS: column tiles wid,
// wid + 4, ..; lane l carries 16 bytes of candidate l % 16 per K block.  The
// walk over the unit's stencil rows keeps the lane's slot in registers.
template <int KB>
struct G16Stage {
    static constexpr int KP = KB * 32;
    static constexpr int TPW = chunk_of(KB) / 16 / kWaves;
    static_assert(TPW <= 2, "one or two column tiles per wave");
    struct Tile {
        u32x4 v[KB];
        uint32_t pos;
    };
    Tile x, y;
    uint32_t slot, base, next;
    __device__ __forceinline__ void init(const GbRows &rl) {
        slot = 0;
        base = rl.start[0] - rl.off[0];
        next = rl.off[1];
    }
    __device__ __forceinline__ void fetch_tile(Tile &d, const uint16_t *Bv, const GbRows &rl, uint32_t nslots,
                                               uint32_t t, uint32_t t1, uint32_t npad) {
        while (t < t1 && next <= t && slot + 1 < nslots) {
            slot++;
            base = rl.start[slot] - rl.off[slot];
            next = rl.off[slot + 1];
        }
        d.pos = t < t1 ? base + t : npad;
        const u32x4 *src = reinterpret_cast<const u32x4 *>(Bv) + (uint64_t)d.pos * (KP / 8) + ((threadIdx.x & 63) >> 4);
#pragma unroll
        for (int kb = 0; kb < KB; kb++) d.v[kb] = src[kb * 4];
    }
    // candidates tc .. (absent ones, t >= t1, read the padding row)
    __device__ __forceinline__ void fetch(const uint16_t *Bv, const GbRows &rl, uint32_t nslots, uint32_t tc,
                                          uint32_t t1, uint32_t npad) {
        const uint32_t t = tc + (threadIdx.x >> 6) * 16 + (threadIdx.x & 15);
        fetch_tile(x, Bv, rl, nslots, t, t1, npad);
        if constexpr (TPW > 1) fetch_tile(y, Bv, rl, nslots, t + kWaves * 16, t1, npad);
    }
    __device__ __forceinline__ void store_tile(const Tile &d, u32x4 *cb, uint32_t *cpos, uint32_t tile) const {
        const uint32_t lane = threadIdx.x & 63;
#pragma unroll
        for (int kb = 0; kb < KB; kb++) cb[(tile * KB + kb) * 64 + lane] = d.v[kb];
        if (lane < 16) cpos[tile * 16 + lane] = d.pos;
    }
    __device__ __forceinline__ void store(u32x4 *cb, uint32_t *cpos) const {
        store_tile(x, cb, cpos, threadIdx.x >> 6);
        if constexpr (TPW > 1) store_tile(y, cb, cpos, kWaves + (threadIdx.x >> 6));
    }
};

template <int KB>
__global__ __launch_bounds__(64 * kWaves, KB == 1 ? 4 : KB == 2 ? 3 : 2) void k_g16_join(GbArgs a) {
    constexpr int KP = KB * 32;
    constexpr int CH = chunk_of(KB);
    constexpr int CT = CH / 16;       // column tiles per chunk
    __shared__ GbRows rl;
    // operand tiles in fragment order: [tile][kb][lane], 16 bytes per lane, so
    // staging and fragment reads are linear (no bank conflicts)
    __shared__ u32x4 cb[2][CT * KB * 64];
    __shared__ uint32_t cpos[2][CH];
    __shared__ uint32_t sh_unit[4];

    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const float Trej = a.trej;
    const uint32_t npad = a.g.n;
    uint2 blk = make_uint2(0, 0);  // the wave's block of the survivor list (wave-uniform)
    uint64_t my_evals = 0;

    const uint32_t part0 = xcc_id() % a.n_parts;
    uint32_t tried = 0;
    while (true) {
        if (tid == 0) sh_unit[0] = gb_next_unit(a.queue_heads, a.n_parts, a.part_end, part0, tried);
        __syncthreads();
        const uint32_t ui = wave_bcast_u32(sh_unit[0]);
        if (ui >= a.n_units) break;
        const uint4 unit = a.units16[ui];
        const uint32_t cstart = a.ix.cell_start[unit.x];
        const uint32_t csize = a.ix.cell_start[unit.x + 1] - cstart;
        const uint32_t nq = wave_bcast_u32(min(kUnitQ, csize - unit.y));
        const uint32_t qpos0 = wave_bcast_u32(cstart + unit.y);
        if (wid == 0) {
            uint32_t slots, total, below;
            gb_build_rows(a.g, a.ix, unit.x, qpos0, rl, &slots, &total, &below);
            if (lane == 0) {
                sh_unit[1] = total;
                sh_unit[2] = slots;
                sh_unit[3] = below;
            }
        }
        __syncthreads();
        const uint32_t t1 = wave_bcast_u32(min(sh_unit[1], unit.w)), nslots = wave_bcast_u32(sh_unit[2]);
        const uint32_t t0 = wave_bcast_u32(max(unit.z, a.mirror ? sh_unit[3] : 0u));
        if (t0 >= t1) {  // its candidates all precede its queries
            __syncthreads();
            continue;
        }
        if (tid == 0) my_evals += (uint64_t)(t1 - t0) * nq;
        const uint32_t nchunks = (t1 - t0 + CH - 1) / CH;
        // candidates from here on are beyond the unit's queries: both directions
        const uint32_t mir0 = a.mirror ? qpos0 + nq : ~0u;
        // the unit's row tiles, spread evenly over the waves
        const uint32_t tiles = (nq + 15) / 16, per = (tiles + kWaves - 1) / kWaves;
        const uint32_t q0 = (uint32_t)wid * per * 16;  // the wave's first query

        // NR row tiles of this wave against every candidate chunk
        auto run = [&](auto nrc, uint32_t cur, uint32_t end) __attribute__((always_inline)) {
            constexpr int NR = decltype(nrc)::value;
            G16Stage<KB> st;
            st.init(rl);
            st.fetch(a.Bv, rl, nslots, t0, t1, npad);
            st.store(cb[0], cpos[0]);
            __syncthreads();
            f16x8 afr[NR > 0 ? NR : 1][KB];
#pragma unroll
            for (int rt = 0; rt < NR; rt++) {
                const uint32_t q = q0 + rt * 16 + (lane & 15);
                const bool in = (uint32_t)rt < per && q < nq;
                const f16x8 *src = reinterpret_cast<const f16x8 *>(a.Av) + (uint64_t)(in ? qpos0 + q : npad) * (KP / 8) + (lane >> 4);
#pragma unroll
                for (int kb = 0; kb < KB; kb++) {
                    afr[rt][kb] = src[kb * 4];
                    // arrived before the loop, whose waits are for the chunk in flight
                    __asm__ volatile("" : "+v"(afr[rt][kb]));
                }
            }
            for (uint32_t ch = 0; ch < nchunks; ch++) {
                const uint32_t buf = ch & 1;
                if (ch + 1 < nchunks) st.fetch(a.Bv, rl, nslots, t0 + (ch + 1) * CH, t1, npad);
#pragma unroll 1
                for (int ct = 0; NR > 0 && ct < CT; ct++) {
                    f32x4 acc[NR > 0 ? NR : 1];
#pragma unroll
                    for (int kb = 0; kb < KB; kb++) {
                        const f16x8 b = *reinterpret_cast<const f16x8 *>(&cb[buf][(ct * KB + kb) * 64 + lane]);
#pragma unroll
                        for (int rt = 0; rt < NR; rt++)
                            acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                afr[rt][kb], b, kb == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[rt], 0, 0, 0);
                    }
                    // the lane's smallest s' (all finite), one vote per tile column
                    float mn = acc[0][0];
#pragma unroll
                    for (int rt = 0; rt < NR; rt++) {
                        mn = fminf(fminf(mn, acc[rt][0]), acc[rt][1]);
                        mn = fminf(fminf(mn, acc[rt][2]), acc[rt][3]);
                    }
                    if (__builtin_amdgcn_ballot_w64(mn <= Trej)) {
                        // rare: keep its addresses out of the loop's registers
                        uint32_t ln = (uint32_t)lane;
                        __asm__ volatile("" : "+v"(ln));
                        const uint32_t cp = cpos[buf][ct * 16 + (ln & 15)];
                        const uint32_t qrow = q0 + (ln >> 4) * 4;
#pragma unroll
                        for (int rt = 0; rt < NR; rt++) {
                            const float m4 = fminf(fminf(acc[rt][0], acc[rt][1]), fminf(acc[rt][2], acc[rt][3]));
                            if (!__builtin_amdgcn_ballot_w64(m4 <= Trej)) continue;
#pragma unroll 1
                            for (int j = 0; j < 4; j++) {
                                const float v = j == 0 ? acc[rt][0] : j == 1 ? acc[rt][1] : j == 2 ? acc[rt][2] : acc[rt][3];
                                const uint32_t q = qrow + rt * 16 + j;
                                // padding never passes (s' >= 65504); checked all the same
                                const bool hit = v <= Trej && q < nq && cp < npad;
                                const uint64_t m = __builtin_amdgcn_ballot_w64(hit);
                                if (m == 0) continue;
                                const uint32_t k = (uint32_t)__popcll(m);
                                if (cur + k > end) {
                                    // pad the rest of the block, then take a new one
                                    if (cur + ln < end) a.raw[cur + ln] = kSentinel;
                                    unsigned long long b = 0;
                                    if (ln == 0) b = atomicAdd(a.raw_cursor, (unsigned long long)kGbBlk);
                                    b = wave_bcast_u64(b);
                                    if (b + kGbBlk > a.raw_cap) {  // full: counted, the join runs again
                                        if (ln == 0) atomicAdd(a.raw_lost, (unsigned long long)k);
                                        cur = end = 0;
                                        continue;
                                    }
                                    cur = (uint32_t)b;
                                    end = cur + kGbBlk;
                                }
                                if (hit) {
                                    const uint32_t at = cur + lanes_below(m);
                                    const uint32_t qp = (qpos0 + q) | (cp >= mir0 ? 0x80000000u : 0u);
                                    a.raw[at] = ((uint64_t)qp << 32) | cp;
                                    a.raw_s[at] = v;
                                }
                                cur += k;
                            }
                        }
                    }
                }
                if (ch + 1 < nchunks) st.store(cb[buf ^ 1], cpos[buf ^ 1]);
                __syncthreads();
            }
            return make_uint2(cur, end);
        };
        if (q0 >= nq) {  // no queries for this wave: it only stages candidates
            blk = run(std::integral_constant<int, 0>{}, blk.x, blk.y);
        } else if (per > 4) {
            blk = run(std::integral_constant<int, 8>{}, blk.x, blk.y);
        } else if (per > 2) {
            blk = run(std::integral_constant<int, 4>{}, blk.x, blk.y);
        } else {
            blk = run(std::integral_constant<int, 2>{}, blk.x, blk.y);
        }
    }
    for (uint32_t i = blk.x + lane; i < blk.y; i += 64) a.raw[i] = kSentinel;
    if (lane == 0) {
        if (my_evals) atomicAdd(a.evals, (unsigned long long)my_evals);
    }
}

// Decides the survivors: accepted by their guards, or by the reference's
// exact FP64 chain (kernel.cu:350-355) over the points' own rows (pts, by
// point id: 8 dim contiguous bytes, where the cell-ordered planes cost a
// cache line per coordinate).  The band is queued per wave, so the chain runs
// on full waves.  Keys (query, candidate position) go to the pair list, both
// directions for a mirrored survivor.
__global__ __launch_bounds__(256) void k_g16_decide(GbArgs a) {
    __shared__ uint64_t queue[4][128];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint64_t total = *a.raw_cursor < a.raw_cap ? *a.raw_cursor : a.raw_cap;
    const uint32_t dim = a.g.dim;
    uint64_t *const q = queue[wid];
    Appender ap{0, 0};
    uint32_t nq = 0;
    uint64_t my_acc = 0, my_band = 0;
    auto emit = [&](uint64_t key, bool ok) __attribute__((always_inline)) {
        const bool mir = ok && (key >> 63);
        const uint64_t kd = key & ~kGbMirror, km = (kd << 32) | (kd >> 32);
        append_keys(kd, ok, ap, a.pairs, a.pair_cap, a.pair_cursor, a.overflow);
        append_keys(km, mir, ap, a.pairs, a.pair_cap, a.pair_cursor, a.overflow);
        my_acc += (ok ? 1u : 0u) + (mir ? 1u : 0u);
    };
    auto recheck = [&](uint32_t m) __attribute__((always_inline)) {  // the queue's first m <= 64
        bool ok = false;
        uint64_t key = 0;
        wave_lds_sync();
        if ((uint32_t)lane < m) {
            key = q[lane];
            const uint32_t qp = (uint32_t)(key >> 32) & 0x7FFFFFFFu, cp = (uint32_t)key;
            const double *xq = a.ix.pts + (uint64_t)a.ix.ila[qp] * dim, *xc = a.ix.pts + (uint64_t)a.ix.ila[cp] * dim;
            double acc = 0.0;
            for (uint32_t l = 0; l < dim; l++) {
                const double d = xc[l] - xq[l];
                acc = __builtin_fma(d, d, acc);
            }
            ok = acc <= a.g.thresh;
        }
        emit(key, ok);
        my_band += (uint32_t)lane < m ? 1u : 0u;
    };
    const uint64_t step = (uint64_t)gridDim.x * 256;
    for (uint64_t i0 = (uint64_t)blockIdx.x * 256 + wid * 64; i0 < total; i0 += step) {
        const uint64_t i = i0 + lane;
        uint64_t key = i < total ? a.raw[i] : kSentinel;
        bool acc_ok = false, band = false;
        if (key != kSentinel) {
            const uint32_t qp = (uint32_t)(key >> 32) & 0x7FFFFFFFu, cp = (uint32_t)key;
            const double hi = (double)a.raw_s[i] + (double)a.w[qp] + (double)a.w[cp];
            acc_ok = hi <= a.tacc;
            band = !acc_ok;
        }
        emit(key, acc_ok);
        const uint64_t m = __ballot(band);
        if (m) {
            if (band) q[nq + lanes_below(m)] = key;
            nq += (uint32_t)__popcll(m);
            if (nq >= 64) {
                recheck(64);
                wave_lds_sync();
                const uint64_t rest = (uint32_t)lane + 64 < nq ? q[lane + 64] : 0;
                wave_lds_sync();
                if ((uint32_t)lane + 64 < nq) q[lane] = rest;
                nq -= 64;
            }
        }
    }
    if (nq) recheck(nq);
    close_appender(ap, a.pairs);
    for (int o = 32; o > 0; o >>= 1) {
        my_acc += __shfl_xor(my_acc, o, 64);
        my_band += __shfl_xor(my_band, o, 64);
    }
    if (lane == 0) {
        if (my_acc) atomicAdd(a.n_accept, (unsigned long long)my_acc);
        if (my_band) atomicAdd(a.n_band, (unsigned long long)my_band);
    }
}

template <int KB>
hegj_status occ16(int device, uint32_t *blocks) {
    int per_cu = 0, cus = 0;
    HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, reinterpret_cast<const void *>(&k_g16_join<KB>), 64 * kWaves, 0));
    HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    *blocks = (uint32_t)std::max(per_cu, 1) * (uint32_t)cus;
    return HEGJ_OK;
}

}  // namespace

// K blocks of 32 for dim coordinates and 4 norm slots; 0: not built.
uint32_t g16_kblocks(uint32_t dim) {
    const uint32_t kb = (dim + 4 + 31) / 32;
    return kb <= 4 ? kb : 0;
}

// FP32 accumulation inside the MFMAs, relative to the sum of the magnitudes
// of its terms, for any order and rounding mode.
static double g16_gamma(uint32_t kb) {
    const double up = std::ldexp(1.0, -23), nadd = 32.0 * kb + kb + 8.0;
    return nadd * up / (1.0 - nadd * up);
}

// Scale and thresholds of the operands, from the largest squared norm of the
// centred points.
struct G16Scale {
    double sigma, tau;
    float trej;
    double tacc;
};
static G16Scale g16_scale(double max2, double thresh, double eps, uint32_t dim) {
    // sigma: norms and eps below 112, so every s' of a real pair stays far
    // below the padding's and all norms fit FP16
    const double top = std::max(std::sqrt(max2) * 1.0001, eps);
    const int e = std::min(1000, (int)std::floor(std::log2(112.0 / top)));
    G16Scale r;
    r.sigma = std::ldexp(1.0, e);
    // the FP64 chain against the exact sum, relative to T: its roundings, and
    // where squares underflow half of the smallest FP64 number for each of them
    const double u64 = std::ldexp(1.0, -53);
    const double slop = 4.0 * (dim + 8) * u64 + (dim + 8) * std::ldexp(1.0, -1074) / thresh;
    const double tau2 = thresh * r.sigma * r.sigma;
    r.tau = std::sqrt(tau2) * (1.0 + slop);
    const double rej = r.tau * r.tau * (1.0 + 4.0 * u64);
    float rf = (float)rej;
    if ((double)rf < rej) rf = f32_next_up(rf);
    r.trej = rf;
    r.tacc = tau2 * (1.0 - slop);
    return r;
}

// Operands for one index and its threshold; ops->A stays null when FP16
// cannot serve the data: a norm overflows FP64, or the band would hold a large
// share of the near pairs and the split BF16, whose exponent range is FP32's,
// is the better filter.  A far outlier does that: it sets the scale, and what is
// below 2^-14 of it (coordinates, and the norms' low parts) is lost.
// `share`, the part of tau^2 that a pair's guards take, decides; total join
// time FP16 / split BF16 with two opposite outliers, by share:
//     18-D 250k  .029 3.7 / 19.2 ms   .106 4.1 / 19.0   .41 576 / 19
//     18-D 1M    .037 25.6 / 160      .134 61 / 160     .50 5309 / 160
//     32-D 200k  .029 145 / 318       .107 416 / 317    .42 2673 / 320
//     64-D 100k  .040 2.2 / 11.9      .154 35 / 11.7    .52 1555 / 11.9
//     90-D 100k  .027 1.6 / 10.3      .103 2.4 / 10.5   .40 852 / 10.4
//     124-D 60k  .020 0.8 / 4.5       .073 0.9 / 4.5    .28 16.6 / 4.5
// Clusters far from their mean widen the split BF16's guards no less, and FP16
// stays ahead (18-D 200k, 50 centres 100 eps out: shares .64 and 1, 1.6 / 793
// ms), until its mean error exceeds 1/16 of eps.
hegj_status g16_prepare(const GridGeom &g, const DevIndex &ix, const double *mean, GbOperands *ops,
                        hipStream_t s) {
    const uint32_t n = g.n, dim = g.dim, kb = g16_kblocks(dim);
    if (kb == 0) return HEGJ_OK;
    Scratch sc;
    unsigned long long *d_bits;
    double *d_sums;
    HIP_TRY(sc.get(&d_bits, 1));
    HIP_TRY(sc.get(&d_sums, kSums * kLineDoubles));
    HIP_TRY(hipMemsetAsync(d_bits, 0, sizeof(*d_bits), s));
    HIP_TRY(hipMemsetAsync(d_sums, 0, sizeof(double) * kSums * kLineDoubles, s));
    k_g16_maxnorm<<<std::min<uint32_t>(ceil_div(n, 256), 2048), 256, 0, s>>>(ix.soa, n, dim, mean, d_bits);
    HIP_TRY(hipGetLastError());
    unsigned long long bits = 0;
    HEGJ_TRY(read_back(&bits, d_bits, s));
    double max2;
    std::memcpy(&max2, &bits, sizeof(max2));
    if (!std::isfinite(max2)) return HEGJ_OK;
    const G16Scale sc16 = g16_scale(max2, g.thresh, g.eps, dim);
    const double sigma = sc16.sigma, tau = sc16.tau;
    const size_t rows = (size_t)n + 1;
    uint16_t *A = nullptr, *B = nullptr;
    float *w = nullptr;
    DevHold hold(s);
    HIP_TRY(hold.get(&A, rows * kb * 32));
    HIP_TRY(hold.get(&B, rows * kb * 32));
    HIP_TRY(hold.get(&w, rows));
    const uint32_t blocks = ceil_div(rows, 256);
    const double gamma = g16_gamma(kb);
    // twice 4 delta (hegj_mfma.hip); without such a kernel its share is 1
    const uint32_t kbf = gb_kblocks(dim);
    const double bf = kbf ? 8.0 * gb_coefficient(dim, kbf * 32) : INFINITY;
    switch (kb) {
        case 1: k_g16_prepare<1><<<blocks, 256, 0, s>>>(ix.soa, n, dim, mean, sigma, tau, gamma, bf, A, B, w, d_sums); break;
        case 2: k_g16_prepare<2><<<blocks, 256, 0, s>>>(ix.soa, n, dim, mean, sigma, tau, gamma, bf, A, B, w, d_sums); break;
        case 3: k_g16_prepare<3><<<blocks, 256, 0, s>>>(ix.soa, n, dim, mean, sigma, tau, gamma, bf, A, B, w, d_sums); break;
        default: k_g16_prepare<4><<<blocks, 256, 0, s>>>(ix.soa, n, dim, mean, sigma, tau, gamma, bf, A, B, w, d_sums); break;
    }
    HIP_TRY(hipGetLastError());
    double sums[kSums * kLineDoubles];
    HEGJ_TRY(read_back(sums, d_sums, s, kSums * kLineDoubles));
    const double err = sums[kSumErr * kLineDoubles] / n, share = sums[kSumShare * kLineDoubles] / n,
                 share_bf = sums[kSumShareBf * kLineDoubles] / n;
    if (!(err <= tau / 16.0) || !(share <= 1.0 / 16 || share <= share_bf)) return HEGJ_OK;
    ops->A = A;
    ops->B = B;
    ops->w = w;
    hold.keep();
    ops->kp = kb * 32;
    ops->f16 = true;
    ops->trej = sc16.trej;
    ops->tacc = sc16.tacc;
    return HEGJ_OK;
}

// Units of the FP16 join.  The segment length aims at ~8192 units (eight per
// resident workgroup, so the last round of a launch is short), within
// 1024 .. 65536 candidates: shorter ones would spend their time on the
// stencil build, longer ones overflow an XCD's L2 (64 bytes per candidate at
// K = 32) without saving anything.
hegj_status g16_units(const DevIndex &ix, const uint32_t *order, const uint32_t *work, uint64_t candidates,
                      uint4 **units, uint32_t *n_units, hipStream_t s) {
    const uint32_t C = ix.C;
    uint64_t seg = candidates / kUnitQ / 8192;
    seg = std::max<uint64_t>(1024, std::min<uint64_t>(seg, 65536));
    seg = (seg + kMaxChunk - 1) / kMaxChunk * kMaxChunk;
    Scratch sc;
    uint32_t *cnt, *off, *d_total;
    HIP_TRY(sc.get(&cnt, C));
    HIP_TRY(sc.get(&off, C));
    HIP_TRY(sc.get(&d_total, 1));
    k_g16_unit_counts<<<ceil_div(C, 256), 256, 0, s>>>(ix, order, work, (uint32_t)seg, cnt);
    HIP_TRY(hipGetLastError());
    HEGJ_TRY(scan_u32(cnt, off, C, d_total, s));
    uint32_t U = 0;
    HEGJ_TRY(read_back(&U, d_total, s));
    HIP_TRY(dev_malloc_n(units, (size_t)U + 1));
    if (U) k_g16_unit_fill<<<ceil_div(U, 256), 256, 0, s>>>(ix, order, work, (uint32_t)seg, off, U, *units);
    HIP_TRY(hipGetLastError());
    *n_units = U;
    return scratch_done(s);
}

hegj_status g16_occupancy(uint32_t kp, int device, uint32_t *blocks) {
    switch (kp / 32) {
        case 1: return occ16<1>(device, blocks);
        case 2: return occ16<2>(device, blocks);
        case 3: return occ16<3>(device, blocks);
        case 4: return occ16<4>(device, blocks);
    }
    return fail(HEGJ_ERR_UNSUPPORTED, "no FP16 MFMA kernel for this dimensionality");
}

hegj_status g16_decide(const GbArgs &a, uint32_t blocks, hipStream_t s) {
    k_g16_decide<<<blocks, 256, 0, s>>>(a);
    HIP_TRY(hipGetLastError());
    return HEGJ_OK;
}

hegj_status g16_launch(const GbArgs &a, uint32_t blocks, hipStream_t s) {
    switch (a.kp / 32) {
        case 1: k_g16_join<1><<<blocks, 64 * kWaves, 0, s>>>(a); break;
        case 2: k_g16_join<2><<<blocks, 64 * kWaves, 0, s>>>(a); break;
        case 3: k_g16_join<3><<<blocks, 64 * kWaves, 0, s>>>(a); break;
        case 4: k_g16_join<4><<<blocks, 64 * kWaves, 0, s>>>(a); break;
        default: return fail(HEGJ_ERR_UNSUPPORTED, "no FP16 MFMA kernel for this dimensionality");
    }
    HIP_TRY(hipGetLastError());
    return HEGJ_OK;
}

}  // namespace hegj

extern "C" hegj_status hegj_g16_operands(const double *pts, uint32_t n, uint32_t dim, const double *centre, double epsilon,
                                         double guard_scale, uint16_t *A, uint16_t *B, float *w, uint32_t *kp,
                                         float *trej, double *tacc) {
    using namespace hegj;
    const uint32_t kb = g16_kblocks(dim);
    if (dim == 0 || kb == 0) return fail(HEGJ_ERR_UNSUPPORTED, "no FP16 MFMA refine for this dimensionality");
    if (kp) *kp = kb * 32;
    if (!A && !B && !w) return HEGJ_OK;
    if (!pts || !centre || !A || !B || !w || !trej || !tacc || !(epsilon > 0.0))
        return fail(HEGJ_ERR_INVALID_ARG, "NULL argument or bad epsilon");
    double max2 = 0.0;
    for (uint32_t p = 0; p < n; p++) {
        double s = 0.0;
        bool fin = true;
        for (uint32_t l = 0; l < dim; l++) {
            const double x = pts[(uint64_t)p * dim + l], y = x - centre[l];
            fin &= std::isfinite(x);
            s = std::fma(y, y, s);
        }
        if (fin) max2 = std::max(max2, s);
    }
    const G16Scale r = g16_scale(max2, sqrt_threshold(epsilon), epsilon, dim);
    std::vector<f16x8> a(kb * 4), b(kb * 4);  // (the caller's rows may not be aligned)
    for (uint32_t p = 0; p < n; p++) {
        g16_point(pts + (uint64_t)p * dim, 1, dim, (int)kb * 32, centre, r.sigma, r.tau, g16_gamma(kb), guard_scale, true,
                  reinterpret_cast<uint16_t *>(a.data()), reinterpret_cast<uint16_t *>(b.data()), w + p);
        std::memcpy(A + (uint64_t)p * kb * 32, a.data(), kb * 64);
        std::memcpy(B + (uint64_t)p * kb * 32, b.data(), kb * 64);
    }
    *trej = r.trej;
    *tacc = r.tacc;
    return HEGJ_OK;
}
