// E8 shell codebook encoder: nearest table row by argmin_k( |c_k|^2 - 2 <x, c_k> ), strict "<"
// so that the lowest index wins ties (glq/codebook.py:253-278; glq/codebook_kernel.py:12-83).
//
// One lane owns VPT vectors (8 fp32 each, in registers) and every wave walks the whole table:
// the table row is uniform over the wave, so it arrives through the scalar data path (one
// 32-byte scalar load per row) and feeds the multiply-adds as a scalar operand -- no LDS, no
// expansion, 8 FMAs + 1 FMA + compare + 2 selects per (vector, row).  The dot product is
// summed in coordinate order in fp32 with fused multiply-adds and the distance is
// fma(-2, dot, norm): for fp32 inputs this is the arithmetic of the reference's CPU branch.
#include "common.h"

namespace {

typedef float f32x4v __attribute__((ext_vector_type(4)));

constexpr int EQ_THREADS = 256;
constexpr int EQ_VPT = 4;

__global__ void __launch_bounds__(EQ_THREADS)
e8_quantize_kernel(const float *__restrict__ x, const float *__restrict__ table,
                   const float *__restrict__ norms, int64_t N, int K, int64_t *__restrict__ idx_out,
                   float *__restrict__ dec_out) {
    const int64_t v0 = ((int64_t)blockIdx.x * EQ_THREADS + threadIdx.x) * EQ_VPT;
    float xv[EQ_VPT][8], best[EQ_VPT];
    int bi[EQ_VPT];
#pragma unroll
    for (int u = 0; u < EQ_VPT; ++u) {
        const int64_t v = v0 + u < N ? v0 + u : N - 1;
        const f32x4v a = *(const f32x4v *)(x + v * 8), b = *(const f32x4v *)(x + v * 8 + 4);
        xv[u][0] = a.x; xv[u][1] = a.y; xv[u][2] = a.z; xv[u][3] = a.w;
        xv[u][4] = b.x; xv[u][5] = b.y; xv[u][6] = b.z; xv[u][7] = b.w;
        best[u] = __builtin_inff();
        bi[u] = 0;
    }
#pragma unroll 4
    for (int k = 0; k < K; ++k) {
        const float *c = table + (int64_t)k * 8;               // uniform: scalar loads
        const float nk = norms[k];
#pragma unroll
        for (int u = 0; u < EQ_VPT; ++u) {
            float dot = 0.0f;
#pragma unroll
            for (int d = 0; d < 8; ++d) dot = __builtin_fmaf(xv[u][d], c[d], dot);
            const float dist = __builtin_fmaf(-2.0f, dot, nk);
            const bool better = dist < best[u];
            best[u] = better ? dist : best[u];
            bi[u] = better ? k : bi[u];
        }
    }
#pragma unroll
    for (int u = 0; u < EQ_VPT; ++u) {
        if (v0 + u < N) {
            idx_out[v0 + u] = bi[u];
            if (dec_out) {
                const float *c = table + (int64_t)bi[u] * 8;
#pragma unroll
                for (int d = 0; d < 8; ++d) dec_out[(v0 + u) * 8 + d] = c[d];
            }
        }
    }
}

// ---- the whole shell table, by its symmetry --------------------------------------------
// The 65536-row table is every E8 point of norm up to 10 and a part of the shell of norm 12.  A
// full shell is a union of orbits of the even signed permutations (Weyl group of D8), and on one
// orbit the largest <x, c> is <y, p>: y = |x| in descending order, its last entry carrying the
// sign of the product of x's entries, p the orbit's representative ordered the same way.  20 orbits
// of prefix sums of y replace 56881 distances; the second largest value on an orbit is one of the
// eight simple reflections of p away, so the gap to every other row is known too.  The index of
// the row found comes from a hash of the codewords.
//
// Which row the table walk above would return depends on fp32 rounding only where two distances are
// closer than what rounding can move them; `es_margin` bounds that: 128 roundings of
// 12 + 2 sqrt(12) |x|, where the walk's own sums take 9, the ones here 12 and the place bits in y 16,
// all twice for a difference.  Vectors inside it (a few in 10^4 of N(0, 1)), and any that are not
// finite or large, take the table walk, spread over the whole chip (e8_slow_kernel): same indices always.
//
// The part of shell 12 that the table holds has no symmetry: vectors for which some point of the
// full shell would be nearer (a quarter of N(0, 1)) meet its rows on the matrix cores, f16 codewords against x as
// two f16 parts (22 bits), and the winning 32 rows are then compared exactly.
//
// 524288 vectors of N(0, 1): 12.06 ms (walk) -> 0.098 ms (70 us, of which the rows of norm 12 are most,
// + 28 us for the walk of the 200 left over); 960 vectors: 12.7 ms -> 21 us, latency.
typedef f16 f16x8v __attribute__((ext_vector_type(8)));
typedef float f32x16v __attribute__((ext_vector_type(16)));

constexpr int ES_THREADS = 256;
constexpr int ES_SLOTS = 1 << 17;                              // hash slots for at most 65536 keys
constexpr uint32_t ES_EMPTY = 0xFFFFFFFFu;
constexpr int ES_CHUNK = 128;                                  // vectors of one pass over shell 12
constexpr int ES_SPLIT = 128;                                  // parts of the table in the exact walk

__device__ __forceinline__ uint32_t es_hash(uint32_t code) { return (code * 2654435761u) >> 15; }

__global__ void __launch_bounds__(256)
es_clear_kernel(uint32_t *__restrict__ keys, int *__restrict__ counts) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < ES_SLOTS) keys[i] = ES_EMPTY;
    if (i < 8) counts[i] = 0;
}

// counts[s]: distinct rows of norm 2s (s = 0..6) that are E8 points with that norm in `norms`;
// rows of norm 12 also go to rem_rows.  counts[7]: everything else.
__global__ void __launch_bounds__(256)
es_index_kernel(const float *__restrict__ table, const float *__restrict__ norms, int n, uint32_t *__restrict__ keys,
                int *__restrict__ vals, int *__restrict__ counts, int *__restrict__ rem_rows) {
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    uint32_t code = 0, odd = 0;
    int sum = 0, n4 = 0;
    bool ok = true;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        const float t = 2.0f * table[(int64_t)r * 8 + d] + 6.0f;
        ok = ok && t >= 0.0f && t <= 12.0f && t == (float)(int)t;
        const int v = ok ? (int)t : 0;
        code |= (uint32_t)v << (4 * d);
        odd += v & 1;
        sum += v - 6;
        n4 += (v - 6) * (v - 6);
    }
    ok = ok && (odd == 0 || odd == 8) && (sum & 3) == 0 && n4 <= 48 && norms[r] == 0.25f * (float)n4;
    int s = 7;
    if (ok) {
        uint32_t h = es_hash(code);
        for (int probe = 0; probe < ES_SLOTS; ++probe) {       // ends: fewer keys than slots
            const uint32_t was = atomicCAS(keys + h, ES_EMPTY, code);
            if (was == ES_EMPTY) { vals[h] = r; s = n4 >> 3; break; }
            if (was == code) break;                            // a second row with these values
            h = (h + 1) & (ES_SLOTS - 1);
        }
    }
    // one add per wave and class: the rows are sorted by norm, so a wave has one or two
#pragma unroll 1
    for (int q = 0; q < 8; ++q) {
        const unsigned long long who = __ballot(s == q);
        if (s != q) continue;
        const int first = __builtin_ctzll(who), lane = threadIdx.x & 63;
        int at = 0;
        if (lane == first) at = atomicAdd(counts + q, __builtin_popcountll(who));
        at = __builtin_amdgcn_readlane(at, first) + __builtin_popcountll(who & ((1ull << lane) - 1));
        if (q == 6) rem_rows[at] = r;
    }
}

// MFMA operands of the rows of shell 12, 32 to a tile: lanes 0..31 hold a row's eight values, lanes
// 32..63 the same times 2^-11, for the low parts of x.  Rows past n_rem are zeros (index -1).
__global__ void __launch_bounds__(256)
es_operands_kernel(const float *__restrict__ table, int *__restrict__ rem_rows, int n_rem, int n_tiles, f16 *__restrict__ ops) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n_tiles * 64) return;
    const int at = (i >> 6) * 32 + (i & 31);
    const float scale = (i & 32) ? 1.0f / 2048.0f : 1.0f;
    f16x8v v;
#pragma unroll
    for (int d = 0; d < 8; ++d) v[d] = at < n_rem ? (f16)(table[(int64_t)rem_rows[at] * 8 + d] * scale) : (f16)0.0f;
    *(f16x8v *)(ops + (int64_t)i * 8) = v;
    if (at >= n_rem && !(i & 32)) rem_rows[at] = -1;
}

// the walk's distance of one row
__device__ __forceinline__ float es_dist(const float x[8], const float *__restrict__ c, float norm) {
    float dot = 0.0f;
#pragma unroll
    for (int d = 0; d < 8; ++d) dot = __builtin_fmaf(x[d], c[d], dot);
    return __builtin_fmaf(-2.0f, dot, norm) + 0.0f;            // + 0: one zero
}

__device__ __forceinline__ void es_load(const float *__restrict__ x, int64_t v, float xv[8]) {
    const f32x4v a = *(const f32x4v *)(x + v * 8), b = *(const f32x4v *)(x + v * 8 + 4);
    xv[0] = a.x; xv[1] = a.y; xv[2] = a.z; xv[3] = a.w;
    xv[4] = b.x; xv[5] = b.y; xv[6] = b.z; xv[7] = b.w;
}

__device__ __forceinline__ float es_margin(const float xv[8]) {
    float q = 0.0f;
#pragma unroll
    for (int d = 0; d < 8; ++d) q += xv[d] * xv[d];
    return (12.0f + 6.93f * __builtin_sqrtf(q)) * 0x1p-17f;
}

struct es_args {
    const float *x, *table, *norms;
    int64_t N;
    const uint32_t *keys;
    const int *vals;
    const f16 *ops;
    const int *rem_rows;
    int n_groups, n_entries;                                   // groups: pairs of 32-row tiles
    int64_t *idx_out;
    float *dec_out;                                            // may be null
    int *slow_count;                                           // per workgroup of the first kernel
    int *slow_list, *slow_arrive;                              // N each
    unsigned long long *slow_key;                              // N
};

__device__ __forceinline__ void es_store(const es_args &a, int64_t v, int row) {
    a.idx_out[v] = row;
    if (a.dec_out) {
        const f32x4v *c = (const f32x4v *)(a.table + (int64_t)row * 8);
        const f32x4v lo = c[0], hi = c[1];
        *(f32x4v *)(a.dec_out + v * 8) = lo;
        *(f32x4v *)(a.dec_out + v * 8 + 4) = hi;
    }
}

// p of an orbit: 2 p_r + 1 in nibble r - 1
constexpr uint32_t es_p(int a, int b, int c, int d, int e, int f, int g, int h) {
    return (uint32_t)(a + 1) | (uint32_t)(b + 1) << 4 | (uint32_t)(c + 1) << 8 | (uint32_t)(d + 1) << 12 |
           (uint32_t)(e + 1) << 16 | (uint32_t)(f + 1) << 20 | (uint32_t)(g + 1) << 24 | (uint32_t)(h + 1) << 28;
}

template <int V>                                               // vectors of a workgroup
__global__ void __launch_bounds__(ES_THREADS, 3)
e8_shell_kernel(const es_args a) {
    __shared__ int n_flag, n_slow, n_exact;
    __shared__ unsigned short flag_v[V], exact_j[ES_CHUNK];
    __shared__ float flag_a[V], flag_m[V];                     // distance and margin
    __shared__ int flag_row[V], exact_group[ES_CHUNK];
    __shared__ float m1s[8][ES_CHUNK], m2s[8][ES_CHUNK];
    __shared__ int ids[8][ES_CHUNK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t v0 = (int64_t)blockIdx.x * V;
    if (tid == 0) n_flag = n_slow = 0;
    __syncthreads();
    auto slow = [&](int local) {
        const int64_t at = v0 + atomicAdd(&n_slow, 1);
        a.slow_list[at] = local;
        a.slow_arrive[at] = 0;
        a.slow_key[at] = 0xFF800000ull << 32;                  // +inf, row 0: the walk's start
    };
#pragma unroll 1
    for (int local = tid; local < V && v0 + local < a.N; local += ES_THREADS) {
        const int64_t v = v0 + local;
        float xv[8];
        es_load(a.x, v, xv);
        uint32_t k[8], signs = 0;
        float total = 0.0f;
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const uint32_t b = __builtin_bit_cast(uint32_t, xv[d]);
            signs |= (b >> 31) << d;
            k[d] = (b & 0x7ffffff8u) | (uint32_t)d;            // |x| and its place: 2^-20 of the value at most
            total += __builtin_fabsf(xv[d]);
        }
        if (!(total < 4096.0f)) { slow(local); continue; }     // f16 parts below; infinities and NaN
        const float margin = es_margin(xv);
        // descending, 19 exchanges
#define ES_X(i, j) { const uint32_t hi = k[i] > k[j] ? k[i] : k[j], lo = k[i] > k[j] ? k[j] : k[i]; k[i] = hi; k[j] = lo; }
        ES_X(0, 1) ES_X(2, 3) ES_X(4, 5) ES_X(6, 7)
        ES_X(0, 2) ES_X(1, 3) ES_X(4, 6) ES_X(5, 7)
        ES_X(1, 2) ES_X(5, 6) ES_X(0, 4) ES_X(3, 7)
        ES_X(1, 5) ES_X(2, 6)
        ES_X(1, 4) ES_X(3, 6)
        ES_X(2, 4) ES_X(3, 5)
        ES_X(3, 4)
#undef ES_X
        float y[8];
#pragma unroll
        for (int d = 0; d < 8; ++d) y[d] = __builtin_bit_cast(float, k[d] & ~7u);
        const bool flip = __builtin_popcount(signs) & 1;
        if (flip) y[7] = -y[7];
        const float s2 = y[0] + y[1], s3 = s2 + y[2], s4 = s3 + y[3], s5 = s4 + y[4], s6 = s5 + y[5], s7 = s6 + y[6];
        const float s8 = s7 + y[7], t8 = s7 - y[7];
        float b1 = 0.0f, b2 = __builtin_inff();                // the origin
        uint32_t p = es_p(0, 0, 0, 0, 0, 0, 0, 0);
        auto orbit = [&](float score, uint32_t code) {
            b2 = __builtin_amdgcn_fmed3f(b1, b2, score);
            if (score < b1) p = code;
            b1 = __builtin_fminf(b1, score);
        };
        orbit(2.0f - 2.0f * s2, es_p(2, 2, 0, 0, 0, 0, 0, 0));
        orbit(2.0f - s8, es_p(1, 1, 1, 1, 1, 1, 1, 1));
        orbit(4.0f - 4.0f * y[0], es_p(4, 0, 0, 0, 0, 0, 0, 0));
        orbit(4.0f - 2.0f * s4, es_p(2, 2, 2, 2, 0, 0, 0, 0));
        orbit(4.0f - t8 - 2.0f * y[0], es_p(3, 1, 1, 1, 1, 1, 1, -1));
        orbit(6.0f - 2.0f * (s3 + y[0]), es_p(4, 2, 2, 0, 0, 0, 0, 0));
        orbit(6.0f - 2.0f * s6, es_p(2, 2, 2, 2, 2, 2, 0, 0));
        orbit(6.0f - s8 - 2.0f * s2, es_p(3, 3, 1, 1, 1, 1, 1, 1));
        orbit(8.0f - 4.0f * s2, es_p(4, 4, 0, 0, 0, 0, 0, 0));
        orbit(8.0f - 2.0f * (s5 + y[0]), es_p(4, 2, 2, 2, 2, 0, 0, 0));
        orbit(8.0f - 2.0f * s8, es_p(2, 2, 2, 2, 2, 2, 2, 2));
        orbit(8.0f - 2.0f * t8, es_p(2, 2, 2, 2, 2, 2, 2, -2 + 0));
        orbit(8.0f - t8 - 2.0f * s3, es_p(3, 3, 3, 1, 1, 1, 1, -1));
        orbit(8.0f - s8 - 4.0f * y[0], es_p(5, 1, 1, 1, 1, 1, 1, 1));
        orbit(10.0f - 2.0f * (s2 + 2.0f * y[0]), es_p(6, 2, 0, 0, 0, 0, 0, 0));
        orbit(10.0f - 2.0f * (s4 + s2), es_p(4, 4, 2, 2, 0, 0, 0, 0));
        orbit(10.0f - 2.0f * (s7 + y[0]), es_p(4, 2, 2, 2, 2, 2, 2, 0));
        orbit(10.0f - s8 - 2.0f * s4, es_p(3, 3, 3, 3, 1, 1, 1, 1));
        orbit(10.0f - t8 - 2.0f * (s2 + y[0]), es_p(5, 3, 1, 1, 1, 1, 1, -1));
        // the full shell of norm 12, of which the table holds a part
        float b12 = 12.0f - 4.0f * s3;
        b12 = __builtin_fminf(b12, 12.0f - 2.0f * (s6 + s2));
        b12 = __builtin_fminf(b12, 12.0f - 2.0f * (s4 + 2.0f * y[0]));
        b12 = __builtin_fminf(b12, 12.0f - t8 - 2.0f * s5);
        b12 = __builtin_fminf(b12, 12.0f - s8 - 2.0f * (s3 + y[0]));
        // gap to the other rows: other orbits, and the simple reflections of p on its own
        float gap = b2 - b1;
        int q[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) q[r] = (int)((p >> (4 * r)) & 15u) - 1;
        if (q[7] == 14) q[7] = -2;                             // the one entry below -1
#pragma unroll
        for (int r = 0; r < 7; ++r)
            if (q[r] != q[r + 1]) gap = __builtin_fminf(gap, (float)(q[r] - q[r + 1]) * (y[r] - y[r + 1]));
        if (q[6] + q[7] != 0) gap = __builtin_fminf(gap, (float)(q[6] + q[7]) * (y[6] + y[7]));
        if (!(gap > margin)) { slow(local); continue; }
        uint32_t code = 0;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const uint32_t i = k[r] & 7u;
            bool neg = (signs >> i) & 1u;
            if (r == 7) neg = neg != flip;
            code |= (uint32_t)(6 + (neg ? -q[r] : q[r])) << (4 * i);
        }
        uint32_t h = es_hash(code);
        for (int probe = 0; a.keys[h] != code && probe < ES_SLOTS; ++probe) h = (h + 1) & (ES_SLOTS - 1);
        const int row = a.vals[h];
        a.idx_out[v] = row;
        if (a.dec_out) {
            f32x4v lo, hi;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                lo[d] = (float)((code >> (4 * d)) & 15u) * 0.5f - 3.0f;
                hi[d] = (float)((code >> (4 * d + 16)) & 15u) * 0.5f - 3.0f;
            }
            *(f32x4v *)(a.dec_out + v * 8) = lo;
            *(f32x4v *)(a.dec_out + v * 8 + 4) = hi;
        }
        if (b12 < b1 + 2.0f * margin) {
            const int j = atomicAdd(&n_flag, 1);
            flag_v[j] = (unsigned short)local;
            flag_a[j] = b1;
            flag_m[j] = 2.0f * margin;
            flag_row[j] = row;
        }
    }
    __syncthreads();
    const int nf = n_flag;
    for (int c0 = 0; c0 < nf; c0 += ES_CHUNK) {
        if (tid == 0) n_exact = 0;
        f16x8v bop[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int j = c0 + 32 * t + (lane & 31);
            float xv[8];
            if (j < nf) es_load(a.x, v0 + flag_v[j], xv);
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const float f = j < nf ? xv[d] : 0.0f;
                f16 hi = (f16)f;
                if (__builtin_fabsf(f) < 0x1p-13f) hi = (f16)0.0f;      // no subnormal operands
                bop[t][d] = lane < 32 ? hi : (f16)((f - (float)hi) * 2048.0f);
            }
        }
        float m1[4], m2[4];
        int id[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) { m1[t] = m2[t] = -__builtin_inff(); id[t] = 0; }
        const f16x8v *ops = (const f16x8v *)a.ops + lane;
        // row tiles requested two steps ahead (a step's products take less than a round trip to the L2)
        f16x8v nx[2][2];
        auto request = [&](int slot, int g) {
            const int64_t at = (int64_t)(g < a.n_groups ? g : 0) * 128;
            nx[slot][0] = ops[at];
            nx[slot][1] = ops[at + 64];
        };
        if (wave < a.n_groups) { request(0, wave); request(1, wave + 4); }
        auto step = [&](int slot, int g) {
            const f16x8v a0 = nx[slot][0], a1 = nx[slot][1];
            request(slot, g + 8);
            __builtin_amdgcn_sched_barrier(0);                 // the requests stay up here
            const f32x16v zero = {};
            const int tiles = (nf - c0 + 31) >> 5;             // of vectors; 4 and more: all of them
            f32x16v d0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, bop[0], zero, 0, 0, 0);
            f32x16v d1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, bop[0], zero, 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 4; ++t) {                      // the next products run under this maximum
                if (t >= tiles) break;
                f32x16v e0, e1;
                if (t < 3) {
                    e0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, bop[t + 1], zero, 0, 0, 0);
                    e1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, bop[t + 1], zero, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                float m = __builtin_fmaxf(d0[0], d1[0]);
#pragma unroll
                for (int i = 1; i < 16; ++i) m = __builtin_fmaxf(__builtin_fmaxf(m, d0[i]), d1[i]);
                m2[t] = __builtin_amdgcn_fmed3f(m1[t], m2[t], m);
                if (m > m1[t]) id[t] = g;
                m1[t] = __builtin_fmaxf(m1[t], m);
                d0 = e0;
                d1 = e1;
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll 1
        for (int g = wave; g < a.n_groups; g += 8) {
            step(0, g);
            if (g + 4 < a.n_groups) step(1, g + 4);
        }
        const int part = wave * 2 + (lane >> 5);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            m1s[part][32 * t + (lane & 31)] = m1[t];
            m2s[part][32 * t + (lane & 31)] = m2[t];
            ids[part][32 * t + (lane & 31)] = id[t] * 2 + (lane >> 5);
        }
        __syncthreads();
        if (tid < ES_CHUNK && c0 + tid < nf) {
            float w1 = m1s[0][tid], w2 = m2s[0][tid];
            int wid = ids[0][tid];
#pragma unroll
            for (int q = 1; q < 8; ++q) {
                const float o1 = m1s[q][tid];
                w2 = __builtin_fmaxf(__builtin_fmaxf(w2, m2s[q][tid]), __builtin_fminf(w1, o1));
                if (o1 > w1) { w1 = o1; wid = ids[q][tid]; }
            }
            const int local = flag_v[c0 + tid];
            const float margin = flag_m[c0 + tid], best = flag_a[c0 + tid];
            const float d1 = 12.0f - 2.0f * w1, d2 = 12.0f - 2.0f * w2;
            if (d1 <= best + margin) {
                if (d2 <= __builtin_fminf(d1, best) + margin) slow(local);
                else {
                    const int e = atomicAdd(&n_exact, 1);
                    exact_j[e] = (unsigned short)(c0 + tid);
                    exact_group[e] = wid;
                }
            }
        }
        __syncthreads();
        // the 32 rows of the winning half pair of tiles, a lane each, and the row of the full shells
        const int ne = n_exact;
        for (int e = tid >> 5; e < ne; e += ES_THREADS / 32) {
            const int j = exact_j[e], grp = exact_group[e], i = lane & 31;
            const int64_t v = v0 + flag_v[j];
            float xv[8];
            es_load(a.x, v, xv);
            const int at = (grp >> 1) * 64 + (i >> 4) * 32 + 8 * ((i >> 2) & 3) + 4 * (grp & 1) + (i & 3);
            int row = a.rem_rows[at];
            const f16x8v c16 = ((const f16x8v *)a.ops)[(at >> 5) * 64 + (at & 31)];   // the row's values, exactly
            float c[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) c[q] = (float)c16[q];
            float d = es_dist(xv, c, 12.0f);
            if (row < 0) { d = __builtin_inff(); row = 0x7fffffff; }
            const int fr = flag_row[j];
            const float fd = es_dist(xv, a.table + (int64_t)fr * 8, a.norms[fr]);
            if (fd < d || (fd == d && fr < row)) { d = fd; row = fr; }
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) {
                const float od = __shfl_xor(d, o, 64);
                const int orow = __shfl_xor(row, o, 64);
                if (od < d || (od == d && orow < row)) { d = od; row = orow; }
            }
            if (i == 0 && row != fr) es_store(a, v, row);
        }
        __syncthreads();
    }
    if (tid == 0) a.slow_count[blockIdx.x] = n_slow;
}

// The table walk for the vectors left over, 64 at a time, a lane each: workgroup (64 vectors, part of
// the table), its waves walking a quarter of the part.  The lowest (distance, row) of a part goes to the
// vector's 64-bit minimum; the last part to arrive writes the row.
__global__ void __launch_bounds__(ES_THREADS)
e8_slow_kernel(const es_args a, int n_src, int per_src) {
    constexpr int ROWS = 65536 / ES_SPLIT;                     // of one part, at most
    __shared__ int sums[4];
    __shared__ int64_t item[64];                               // the vector's list position
    __shared__ unsigned long long keys[4][64];
    __shared__ f32x4v rows[ROWS][2];
    __shared__ float row_norm[ROWS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the vectors' ranks over all source workgroups: a run of sources per thread
    const int per = (n_src + ES_THREADS - 1) / ES_THREADS;
    const int s0 = min(tid * per, n_src), s1 = min(s0 + per, n_src);
    int mine = 0;
    for (int s = s0; s < s1; ++s) mine += a.slow_count[s];
    int first = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(first, o, 64);
        if (lane >= o) first += v;
    }
    if (lane == 63) sums[wave] = first;
    __syncthreads();
    int total = 0;
    first -= mine;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (q < wave) first += sums[q];
        total += sums[q];
    }
    const int64_t work = (int64_t)((total + 63) / 64) * ES_SPLIT;
    for (int64_t w = blockIdx.x; w < work; w += gridDim.x) {
        const int base = (int)(w / ES_SPLIT) * 64, part = (int)(w % ES_SPLIT);
        if (first < base + 64 && first + mine > base) {
            int rank = first;
            for (int s = s0; s < s1; ++s)
                for (int j = 0, c = a.slow_count[s]; j < c; ++j, ++rank)
                    if (rank >= base && rank < base + 64) item[rank - base] = (int64_t)s * per_src + j;
        }
        const int r0 = (int)((int64_t)a.n_entries * part / ES_SPLIT), n = (int)((int64_t)a.n_entries * (part + 1) / ES_SPLIT) - r0;
        for (int i = tid; i < n; i += ES_THREADS) {
            const f32x4v *c = (const f32x4v *)(a.table + (int64_t)(r0 + i) * 8);
            rows[i][0] = c[0];
            rows[i][1] = c[1];
            row_norm[i] = a.norms[r0 + i];
        }
        __syncthreads();
        const bool on = base + lane < total;
        const int64_t at = item[on ? lane : 0];
        const int64_t v = at / per_src * per_src + a.slow_list[at];
        float xv[8], best = __builtin_inff();
        es_load(a.x, v, xv);
        int row = 0;
        const int i1 = n * (wave + 1) / 4;
#pragma unroll 4
        for (int i = n * wave / 4; i < i1; ++i) {
            const float d = es_dist(xv, (const float *)rows[i], row_norm[i]);
            if (d < best) { best = d; row = r0 + i; }
        }
        uint32_t b = __builtin_bit_cast(uint32_t, best);
        b = (b >> 31) ? ~b : b | 0x80000000u;                  // ordered like the floats
        keys[wave][lane] = (unsigned long long)b << 32 | (uint32_t)row;
        __syncthreads();
        if (wave == 0 && on) {
            unsigned long long key = keys[0][lane];
            for (int o = 1; o < 4; ++o) key = keys[o][lane] < key ? keys[o][lane] : key;
            // the minimum has been taken before the arrival is counted: its old value is waited for
            const unsigned long long old = atomicMin(a.slow_key + at, key);
            asm volatile("" ::"v"(old));
            __builtin_amdgcn_s_waitcnt(0);
            if (atomicAdd(a.slow_arrive + at, 1) == ES_SPLIT - 1)
                es_store(a, v, (int)(uint32_t)__hip_atomic_load(a.slow_key + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        }
        __syncthreads();
    }
}

// Vectors per workgroup: few while the chip is not filled, so that shell 12 is passed once with one tile of
// them; more when it is, for fewer reads of the shell.
int es_per_wg(int64_t N) {
    const int64_t cus = glqh_device_cus();
    return N <= 2 * 64 * cus ? 64 : N < 4 * 256 * cus ? 256 : 512;
}

}  // namespace

int glqh_launch_e8_quantize(const float *x, const float *table, const float *norms, int64_t N, int K,
                            int64_t *idx_out, float *dec_out, hipStream_t stream) {
    const int64_t per_wg = (int64_t)EQ_THREADS * EQ_VPT;
    const int64_t wgs = (N + per_wg - 1) / per_wg;
    GLQH_REQUIRE(wgs <= 2147483647ll, "e8 quantize: too many vectors");
    hipLaunchKernelGGL(e8_quantize_kernel, dim3((unsigned)wgs), dim3(EQ_THREADS), 0, stream, x, table, norms, N,
                       K, idx_out, dec_out);
    GLQH_LAUNCH_CHECK("e8 quantize launch");
    return 0;
}

int glqh_launch_e8_shell_index(const float *table, const float *norms, int n, uint32_t *keys, int *vals, int *counts,
                               int *rem_rows, hipStream_t stream) {
    hipLaunchKernelGGL(es_clear_kernel, dim3(ES_SLOTS / 256), dim3(256), 0, stream, keys, counts);
    hipLaunchKernelGGL(es_index_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, table, norms, n, keys, vals,
                       counts, rem_rows);
    GLQH_LAUNCH_CHECK("e8 shell index launch");
    return 0;
}

int glqh_launch_e8_shell_operands(const float *table, int *rem_rows, int n_rem, void *ops, hipStream_t stream) {
    const int tiles = ((n_rem + 63) / 64) * 2;
    if (tiles == 0) return 0;
    hipLaunchKernelGGL(es_operands_kernel, dim3((unsigned)((tiles * 64 + 255) / 256)), dim3(256), 0, stream, table, rem_rows,
                       n_rem, tiles, (f16 *)ops);
    GLQH_LAUNCH_CHECK("e8 shell operands launch");
    return 0;
}

size_t glqh_e8_shell_ws_bytes(int64_t N) { return (size_t)N * 16 + (size_t)((N + 63) / 64) * 4; }

int glqh_launch_e8_shell_quantize(const float *x, int64_t N, const float *table, const float *norms, int n_entries,
                                  const uint32_t *keys, const int *vals, const void *ops, const int *rem_rows, int n_rem,
                                  int64_t *idx_out, float *dec_out, void *ws, hipStream_t stream) {
    const int per = es_per_wg(N);
    const int64_t wgs = (N + per - 1) / per;
    GLQH_REQUIRE(wgs <= 2147483647ll && N <= 2147483647ll, "e8 quantize: too many vectors");
    es_args a;
    a.x = x; a.table = table; a.norms = norms; a.N = N; a.keys = keys; a.vals = vals; a.ops = (const f16 *)ops;
    a.rem_rows = rem_rows; a.n_groups = (n_rem + 63) / 64; a.n_entries = n_entries; a.idx_out = idx_out; a.dec_out = dec_out;
    a.slow_key = (unsigned long long *)ws;
    a.slow_list = (int *)(a.slow_key + N);
    a.slow_arrive = a.slow_list + N;
    a.slow_count = a.slow_arrive + N;
    if (per == 512) hipLaunchKernelGGL(e8_shell_kernel<512>, dim3((unsigned)wgs), dim3(ES_THREADS), 0, stream, a);
    else if (per == 256) hipLaunchKernelGGL(e8_shell_kernel<256>, dim3((unsigned)wgs), dim3(ES_THREADS), 0, stream, a);
    else hipLaunchKernelGGL(e8_shell_kernel<64>, dim3((unsigned)wgs), dim3(ES_THREADS), 0, stream, a);
    const int grid = 2 * glqh_device_cus();
    hipLaunchKernelGGL(e8_slow_kernel, dim3((unsigned)grid), dim3(ES_THREADS), 0, stream, a, (int)wgs, per);
    GLQH_LAUNCH_CHECK("e8 shell quantize launch");
    return 0;
}
