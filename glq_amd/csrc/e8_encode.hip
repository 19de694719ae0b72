// E8 shell codebook encoder: nearest table row by argmin_k( |c_k|^2 - 2 <x, c_k> ), strict "<"
// so that the lowest index wins ties (glq/codebook.py:253-278; glq/codebook_kernel.py:12-83).
//
// One lane owns VPT vectors (8 fp32 each, in registers) and every wave walks the whole table:
// the table row is uniform over the wave, so it arrives through the scalar data path (one
// 32-byte scalar load per row) and feeds the multiply-adds as a scalar operand -- no LDS, no
// expansion, 8 FMAs + 1 FMA + compare + 2 selects per (vector, row).  The dot product is
// summed in coordinate order in fp32 with fused multiply-adds and the distance is
// fma(-2, dot, norm): for fp32 inputs this is the arithmetic of the reference's CPU branch.
#include <type_traits>
#include "common.h"

namespace {

typedef float f32x4v __attribute__((ext_vector_type(4)));

constexpr int EQ_THREADS = 256;
constexpr int EQ_VPT = 4;

// the vectors of workgroup `block`
__device__ __forceinline__ void
e8_quantize_block(const float *__restrict__ x, const float *__restrict__ table, const float *__restrict__ norms, int64_t N,
                  int K, int64_t *__restrict__ idx_out, float *__restrict__ dec_out, int64_t block) {
    const int64_t v0 = (block * EQ_THREADS + threadIdx.x) * EQ_VPT;
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

__global__ void __launch_bounds__(EQ_THREADS)
e8_quantize_kernel(const float *__restrict__ x, const float *__restrict__ table,
                   const float *__restrict__ norms, int64_t N, int K, int64_t *__restrict__ idx_out,
                   float *__restrict__ dec_out) {
    e8_quantize_block(x, table, norms, N, K, idx_out, dec_out, blockIdx.x);
}

// ---- the whole shell table, by its symmetry --------------------------------------------
// The 65536-row table is every E8 point of norm up to 10 and a part of the shell of norm 12.  A
// full shell is a union of orbits of the even signed permutations (Weyl group of D8), and on one
// orbit the largest <x, c> is <y, p>: y = |x| in descending order, its last entry carrying the
// sign of the product of x's entries, p the orbit's representative ordered the same way.  20 orbits
// of prefix sums of y replace 56881 distances; the second largest value on an orbit is one of the
// eight simple reflections of p away, so the gap to every other row is known too.
//
// Nothing about a table is taken on trust or kept from one call for the next.  Every E8 point of norm up to 12 has a
// place of its own (es_map), a matter of the lattice alone; the first launch of a call writes each row's number to its
// place, and what the search assumes of the table is checked on the way: rows that are such points, with their norms
// in `norms`, the number of those of norm up to 10, and (in the second launch) that no two rows share a place.  For
// any other table the third launch walks it, every vector against every row.
//
// Which row the table walk above would return depends on fp32 rounding only where two distances are
// closer than what rounding can move them; `es_margin` bounds that: 128 roundings of
// 12 + 2 sqrt(12) |x|, where the walk's own sums take 9, the ones here 12 and the place bits in y 16,
// all twice for a difference.  A vector with a second point inside the margin, or with a point of
// norm 12 that may be nearer (a fifth of N(0, 1)), has all of them listed: orbit by orbit, every
// point follows from a nearer one by a simple reflection, so the points within reach form a tree
// that a workgroup walks in its LDS, 2.5 of them on average.  Those that the table holds are compared
// by the walk's own arithmetic, lowest row on ties: the walk's answer, always.  Vectors that are not
// finite, or have too many points in reach for the list, take the walk itself (e8_walk_kernel).
//
// 524288 vectors of N(0, 1): 12.06 ms (walk) -> 98 us (points of norm 12 on the matrix cores, all 8655 rows for
// every vector they may win) -> 34 us (points in reach only; 38 MB in and out, 8 us) -> 33.2 us with the table read
// by every call (es_index_kernel 4 us; 250 -> 52 us where the table is new); 960 vectors 12.7 ms -> 13.4 ->
// 17.3 us: three dependent launches.  Then the lists, which a workgroup had filled an addition at a time and walked level
// by level, a barrier each: with the first points and their children from the 25 known orbits, counted before they are placed,
// and the rest to each wave alone, 33.5 -> 32 us, 131072 vectors 21.4 -> 18.5, 960 17.7 -> 15.8; of scale 2, where nearly all
// vectors have them, 131072 vectors 109 -> 49 us, and of scale 20, 201 -> 175.  Of 32 us the kernel takes 28: half of that
// the first pass (bound by VALU instructions), a quarter the first points, the rest trips through the lists and the table.
constexpr int ES_THREADS = 256;
constexpr int ES_PLACES = 117361;                              // E8 points of norm up to 12
constexpr int ES_FULL = GLQH_E8_SHELL_MIN_ROWS;                // of norm up to 10: all of them are rows of the table
enum { ES_SHARED, ES_IN_FULL, ES_WALKS, ES_FOUND };            // two rows of one place; rows of the full shells; vectors to walk
constexpr int ES_CHECKS = 128;                                 // workgroups, at least, that look for rows of one place
constexpr int ES_CHUNK = 128;                                  // vectors whose points are listed together, fewer far out,
constexpr int ES_LIST = 3584;                                  // and the points: 3.6 each at unit scale, up to 106 far out
constexpr int ES_GROWN = ES_LIST - 1200;                       // (four workgroups' lists fill a CU's LDS); the nearest points
constexpr int ES_WAVE = ES_GROWN / 4;                          // of the orbits behind this, the others in a part for each wave
// Points in wait from which a wave takes a lane for each rather than eight: times of 16, 24, 40, 64 are 149, 149, 152, 169 us
// at 131072 vectors of scale 4 and level at unit scale.
constexpr int ES_MANY = 24;
// Vectors to list up to which a workgroup's first points go to the waves as they are found.  (Those of the known orbits and their
// children, counted and then placed, are some 1500 instructions, whoever has them: with them for every workgroup 960 vectors of scale 0.5 took
// 13.6 us, not 12.5, 8000 of scale 0.25 13.8, not 12.7, 524288 21.6, not 21.0.  At 8 and 16 vectors for the line level or slower.)
constexpr int ES_FEW = 32;
static_assert(ES_THREADS == 2 * ES_CHUNK && 16 * 25 <= ES_LIST - ES_GROWN && 16 * 25 * 8 <= 2 * ES_GROWN,
              "two threads a vector; the orbits of the fewest vectors fit, and most of their points' children");
constexpr int ES_SPLIT = 128;                                  // parts of the table in the exact walk

// Places.  A point is two halves of four coordinates (2 c + 6 in a nibble each).  Halves are integers or half-integers
// and have an even or an odd sum of coordinates (of 2 c: 0 or 2 mod 4), and two of them make a point when they agree in
// both.  With the halves of a class in the order of their norms, those that a first half h can take are a prefix, as
// long as there are halves of norm up to 12 - |h|^2: the place of (h, l) is base(h) + rank(l).
struct es_map_t {
    uint32_t at[65536];                                        // by half: base << 11 | rank; 0 where it is none
    int places, ranks;
};

constexpr es_map_t es_make_map() {
    es_map_t m = {};
    int count[4][50] = {};                                     // halves of a class by 4 * norm, then those before them
    int base = 0, most = 0;
    for (int pass = 0; pass < 2; ++pass) {
        int upto[4][50] = {};                                  // halves of 4 * norm up to n
        int next[4][50] = {};
        if (pass == 1)
            for (int c = 0; c < 4; ++c) {
                int sum = 0;
                for (int n = 0; n <= 48; ++n) {
                    next[c][n] = sum;
                    sum += count[c][n];
                    upto[c][n] = sum;
                }
                most = sum > most ? sum : most;
            }
        for (int odd = 0; odd < 2; ++odd)
            for (int a = odd; a <= 12; a += 2)
                for (int b = odd; b <= 12; b += 2)
                    for (int c = odd; c <= 12; c += 2)
                        for (int d = odd; d <= 12; d += 2) {
                            const int n = (a - 6) * (a - 6) + (b - 6) * (b - 6) + (c - 6) * (c - 6) + (d - 6) * (d - 6);
                            const int k = 2 * odd + (((a + b + c + d) >> 1) & 1);
                            if (n > 48) continue;
                            if (pass == 0) ++count[k][n];
                            else {
                                m.at[a | b << 4 | c << 8 | d << 12] = (uint32_t)base << 11 | (uint32_t)next[k][n]++;
                                base += upto[k][48 - n];
                            }
                        }
    }
    m.places = base;
    m.ranks = most;
    return m;
}

__device__ constexpr es_map_t es_map = es_make_map();
static_assert(es_map.places == ES_PLACES && es_map.ranks <= 2048, "places of the points");

// the place of a point of norm up to 12
__device__ __forceinline__ int es_place(uint32_t code) {
    const uint32_t h = es_map.at[code & 0xffffu], l = es_map.at[code >> 16];
    return (int)((h >> 11) + (l & 2047u));
}

// the walk's distance of one row
__device__ __forceinline__ float es_dist(const float x[8], const float *__restrict__ c, float norm) {
    float dot = 0.0f;
#pragma unroll
    for (int d = 0; d < 8; ++d) dot = __builtin_fmaf(x[d], c[d], dot);
    return __builtin_fmaf(-2.0f, dot, norm) + 0.0f;            // + 0: one zero
}

// (distance, row) in the walk's order
__device__ __forceinline__ unsigned long long es_key(float dist, int row) {
    uint32_t b = __builtin_bit_cast(uint32_t, dist);
    b = (b >> 31) ? ~b : b | 0x80000000u;                      // ordered like the floats
    return (unsigned long long)b << 32 | (uint32_t)row;
}

__device__ __forceinline__ void es_load(const float *__restrict__ x, int64_t v, float xv[8]) {
    const f32x4v a = *(const f32x4v *)(x + v * 8), b = *(const f32x4v *)(x + v * 8 + 4);
    xv[0] = a.x; xv[1] = a.y; xv[2] = a.z; xv[3] = a.w;
    xv[4] = b.x; xv[5] = b.y; xv[6] = b.z; xv[7] = b.w;
}

// row_at[place] = row; place_of[row], -1 where the row is not such a point with its norm in `norms`.
// counts[r / 64]: rows of norm up to 10, negative if one of the 64 rows is no point.
__global__ void __launch_bounds__(ES_THREADS)
es_index_kernel(const float *__restrict__ table, const float *__restrict__ norms, int n, int *__restrict__ row_at,
                int *__restrict__ place_of, int *__restrict__ counts, int *__restrict__ found) {
    const int r = blockIdx.x * ES_THREADS + threadIdx.x;
    if (r == 0) found[ES_SHARED] = found[ES_IN_FULL] = found[ES_WALKS] = 0;
    if (r >= n) return;
    float c[8];
    es_load(table, r, c);
    const float norm = norms[r];
    uint32_t code = 0, odd = 0;
    int sum = 0, n4 = 0;
    bool ok = true;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        const float t = 2.0f * c[d] + 6.0f;
        ok = ok && t >= 0.0f && t <= 12.0f && t == (float)(int)t;
        const int v = ok ? (int)t : 0;
        code |= (uint32_t)v << (4 * d);
        odd += v & 1;
        sum += v - 6;
        n4 += (v - 6) * (v - 6);
    }
    ok = ok && (odd == 0 || odd == 8) && (sum & 3) == 0 && n4 <= 48 && norm == 0.25f * (float)n4;
    const int place = ok ? es_place(code) : -1;
    place_of[r] = place;
    if (ok) row_at[place] = r;
    const unsigned long long full = __ballot(ok && n4 <= 40), bad = __ballot(!ok);
    if ((threadIdx.x & 63) == 0) counts[r >> 6] = bad ? -ES_FULL - 1 : __builtin_popcountll(full);
}

struct es_args {
    const float *x, *table, *norms;
    int64_t N;
    int n_entries;
    int *row_at, *place_of, *counts;                           // written by es_index_kernel
    int *found;                                                // what the search finds out, cleared by es_index_kernel
    int64_t *idx_out;
    float *dec_out;                                            // may be null
    int *walk_count;                                           // per workgroup of the first kernel
    int *walk_list, *walk_arrive;                              // N each
    unsigned long long *walk_key;                              // N
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

// x in its dominant chamber: k_r = |x| and, in the low three bits, its place (2^-20 of the value at most),
// descending; signs of x by place; the last of the order carries the product of the signs
struct es_vec {
    uint32_t k[8], signs;
    bool flip;
    float y[8], margin;
};

// false: not finite, or large enough for a sum to leave fp32
__device__ __forceinline__ bool es_sort(const float xv[8], es_vec &s) {
    float total = 0.0f, q = 0.0f;
    s.signs = 0;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        const uint32_t b = __builtin_bit_cast(uint32_t, xv[d]);
        s.signs |= (b >> 31) << d;
        s.k[d] = (b & 0x7ffffff8u) | (uint32_t)d;
        total += __builtin_fabsf(xv[d]);
        q += xv[d] * xv[d];
    }
    s.margin = (12.0f + 6.93f * __builtin_sqrtf(q)) * 0x1p-17f;
#define ES_X(i, j) { const uint32_t hi = s.k[i] > s.k[j] ? s.k[i] : s.k[j], lo = s.k[i] > s.k[j] ? s.k[j] : s.k[i]; s.k[i] = hi; s.k[j] = lo; }
    ES_X(0, 1) ES_X(2, 3) ES_X(4, 5) ES_X(6, 7)
    ES_X(0, 2) ES_X(1, 3) ES_X(4, 6) ES_X(5, 7)
    ES_X(1, 2) ES_X(5, 6) ES_X(0, 4) ES_X(3, 7)
    ES_X(1, 5) ES_X(2, 6)
    ES_X(1, 4) ES_X(3, 6)
    ES_X(2, 4) ES_X(3, 5)
    ES_X(3, 4)
#undef ES_X
#pragma unroll
    for (int d = 0; d < 8; ++d) s.y[d] = __builtin_bit_cast(float, s.k[d] & ~7u);
    s.flip = __builtin_popcount(s.signs) & 1;
    if (s.flip) s.y[7] = -s.y[7];
    return total < 1e15f;
}

// a point in that order: 2 c_r + 6 in nibble r
constexpr uint32_t es_p(int a, int b, int c, int d, int e, int f, int g, int h) {
    return (uint32_t)(a + 6) | (uint32_t)(b + 6) << 4 | (uint32_t)(c + 6) << 8 | (uint32_t)(d + 6) << 12 |
           (uint32_t)(e + 6) << 16 | (uint32_t)(f + 6) << 20 | (uint32_t)(g + 6) << 24 | (uint32_t)(h + 6) << 28;
}

__device__ __forceinline__ int es_q(uint32_t p, int r) { return (int)((p >> (4 * r)) & 15u) - 6; }

// the codeword in x's own order
__device__ __forceinline__ uint32_t es_code(uint32_t p, const uint32_t k[8], uint32_t signs, bool flip) {
    uint32_t code = 0;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const uint32_t i = k[r] & 7u;
        bool neg = (signs >> i) & 1u;
        if (r == 7) neg = neg != flip;
        const int q = es_q(p, r);
        code |= (uint32_t)(6 + (neg ? -q : q)) << (4 * i);
    }
    return code;
}

// f(distance - |x|^2 of the orbit's nearest point, that point) for the orbits of the full shells ...
template <typename F>
__device__ __forceinline__ void es_orbits(const float y[8], F f) {
    const float s2 = y[0] + y[1], s3 = s2 + y[2], s4 = s3 + y[3], s5 = s4 + y[4], s6 = s5 + y[5], s7 = s6 + y[6];
    const float s8 = s7 + y[7], t8 = s7 - y[7];
    f(0.0f, es_p(0, 0, 0, 0, 0, 0, 0, 0));
    f(2.0f - 2.0f * s2, es_p(2, 2, 0, 0, 0, 0, 0, 0));
    f(2.0f - s8, es_p(1, 1, 1, 1, 1, 1, 1, 1));
    f(4.0f - 4.0f * y[0], es_p(4, 0, 0, 0, 0, 0, 0, 0));
    f(4.0f - 2.0f * s4, es_p(2, 2, 2, 2, 0, 0, 0, 0));
    f(4.0f - t8 - 2.0f * y[0], es_p(3, 1, 1, 1, 1, 1, 1, -1));
    f(6.0f - 2.0f * (s3 + y[0]), es_p(4, 2, 2, 0, 0, 0, 0, 0));
    f(6.0f - 2.0f * s6, es_p(2, 2, 2, 2, 2, 2, 0, 0));
    f(6.0f - s8 - 2.0f * s2, es_p(3, 3, 1, 1, 1, 1, 1, 1));
    f(8.0f - 4.0f * s2, es_p(4, 4, 0, 0, 0, 0, 0, 0));
    f(8.0f - 2.0f * (s5 + y[0]), es_p(4, 2, 2, 2, 2, 0, 0, 0));
    f(8.0f - 2.0f * s8, es_p(2, 2, 2, 2, 2, 2, 2, 2));
    f(8.0f - 2.0f * t8, es_p(2, 2, 2, 2, 2, 2, 2, -2));
    f(8.0f - t8 - 2.0f * s3, es_p(3, 3, 3, 1, 1, 1, 1, -1));
    f(8.0f - s8 - 4.0f * y[0], es_p(5, 1, 1, 1, 1, 1, 1, 1));
    f(10.0f - 2.0f * (s2 + 2.0f * y[0]), es_p(6, 2, 0, 0, 0, 0, 0, 0));
    f(10.0f - 2.0f * (s4 + s2), es_p(4, 4, 2, 2, 0, 0, 0, 0));
    f(10.0f - 2.0f * (s7 + y[0]), es_p(4, 2, 2, 2, 2, 2, 2, 0));
    f(10.0f - s8 - 2.0f * s4, es_p(3, 3, 3, 3, 1, 1, 1, 1));
    f(10.0f - t8 - 2.0f * (s2 + y[0]), es_p(5, 3, 1, 1, 1, 1, 1, -1));
}

// ... and of the shell of norm 12, of which the table holds a part
template <typename F>
__device__ __forceinline__ void es_orbits_12(const float y[8], F f) {
    const float s2 = y[0] + y[1], s3 = s2 + y[2], s4 = s3 + y[3], s5 = s4 + y[4], s6 = s5 + y[5], s7 = s6 + y[6];
    const float s8 = s7 + y[7], t8 = s7 - y[7];
    f(12.0f - 4.0f * s3, es_p(4, 4, 4, 0, 0, 0, 0, 0));
    f(12.0f - 2.0f * (s6 + s2), es_p(4, 4, 2, 2, 2, 2, 0, 0));
    f(12.0f - 2.0f * (s4 + 2.0f * y[0]), es_p(6, 2, 2, 2, 0, 0, 0, 0));
    f(12.0f - t8 - 2.0f * s5, es_p(3, 3, 3, 3, 3, 1, 1, -1));
    f(12.0f - s8 - 2.0f * (s3 + y[0]), es_p(5, 3, 3, 1, 1, 1, 1, 1));
}

// f(gap, child) for the children of point p in its orbit's tree whose distance is at most `room` more than p's: a
// simple reflection that takes p further away, and is the first to bring the child back.  (Of points known at compile time little
// but the comparisons with `room` is left.)
template <typename F>
__device__ __forceinline__ void es_children(uint32_t p, const float y[8], float room, F f) {
    int q[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) q[r] = es_q(p, r);
    bool before = true;                                        // the pairs ahead of (i - 1, i) descend
#pragma unroll
    for (int i = 0; i < 7; ++i) {
        if (i >= 2) before = before && q[i - 2] >= q[i - 1];
        const float gap = (float)(q[i] - q[i + 1]) * (y[i] - y[i + 1]);
        if (before && q[i] > q[i + 1] && (i == 0 || q[i - 1] >= q[i + 1]) && gap <= room) {
            const uint32_t d = ((p >> (4 * i)) ^ (p >> (4 * i + 4))) & 15u;
            f(gap, p ^ (d << (4 * i)) ^ (d << (4 * i + 4)));
        }
    }
    const float gap = (float)(q[6] + q[7]) * (y[6] + y[7]);
    if (before && q[4] >= q[5] && q[5] >= -q[7] && q[6] >= q[7] && q[6] + q[7] > 0 && gap <= room)
        f(gap, (p & 0x00FFFFFFu) | (uint32_t)(6 - q[7]) << 24 | (uint32_t)(6 - q[6]) << 28);
}

// The same with eight lanes to a point, lane i: whether reflection i (7: of the last two places, with their signs) makes a child, and how
// much further away it is.  ya, yb: y of the two places.
__device__ __forceinline__ bool es_child(uint32_t p, int i, float ya, float yb, float room, float &gap) {
    const int k = i < 7 ? i : 6, qa = es_q(p, k), qb = es_q(p, k + 1), qp = es_q(p, i < 7 ? max(i - 1, 0) : 5);
    // the pairs ahead of (i - 1, i) descend
    const uint32_t descends = (uint32_t)(__ballot(qa >= qb) >> (threadIdx.x & 56)) & 255u;
    const uint32_t ahead = i == 7 ? 31u : (1u << max(i - 1, 0)) - 1u;
    bool child = (descends & ahead) == ahead;
    if (i < 7) {
        gap = (float)(qa - qb) * (ya - yb);
        child = child && qa > qb && (i == 0 || qp >= qb);
    } else {
        gap = (float)(qa + qb) * (ya + yb);
        child = child && qp >= -qb && qa >= qb && qa + qb > 0;
    }
    return child && gap <= room;
}
__device__ __forceinline__ uint32_t es_reflect(uint32_t p, int i) {
    if (i == 7) return (p & 0x00FFFFFFu) | (uint32_t)(6 - es_q(p, 7)) << 24 | (uint32_t)(6 - es_q(p, 6)) << 28;
    const uint32_t d = ((p >> (4 * i)) ^ (p >> (4 * i + 4))) & 15u;
    return p ^ (d << (4 * i)) ^ (d << (4 * i + 4));
}

// The lanes' counts up to this one's, and of all of them.  The whole wave calls.
__device__ __forceinline__ int es_before(int count, int &total) {
    int sum = count;
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x111, 0xf, 0xf, true);   // row_shr:1, 2, 4, 8
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x112, 0xf, 0xf, true);
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x114, 0xf, 0xf, true);
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x118, 0xf, 0xf, true);
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x142, 0xa, 0xf, false);  // row_bcast:15, 31
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x143, 0xc, 0xf, false);
    total = __builtin_amdgcn_readlane(sum, 63);
    return sum - count;
}
// Places for `count` entries of each lane in a list of the workgroup, in one addition to its length: this lane's first one.  The
// whole wave calls.  (An addition for each
// orbit would be 25 trips to LDS, one after the other.)
__device__ __forceinline__ int es_places(int count, int *length) {
    int total;
    const int before = es_before(count, total);
    if (total == 0) return 0;
    int at = 0;
    if ((threadIdx.x & 63) == 0) at = atomicAdd(length, total);
    return __builtin_amdgcn_readfirstlane(at) + before;
}

template <int V>                                               // vectors of a workgroup
__global__ void __launch_bounds__(ES_THREADS, 4)
e8_shell_kernel(const es_args a) {
    __shared__ int n_flag, n_walk, n_seed, n_child, n_grown[4], n_left[4];
    __shared__ unsigned short flags[V];
    __shared__ uint32_t list_p[ES_LIST], sk[8][ES_CHUNK];
    __shared__ unsigned char list_j[ES_LIST];
    __shared__ float list_room[ES_LIST];
    __shared__ uint32_t s_signs[ES_CHUNK];                     // bit 8: flip
    __shared__ unsigned char s_walk[ES_CHUNK];                 // left to the walk
    __shared__ float s_margin[ES_CHUNK];
    __shared__ unsigned long long best[ES_CHUNK];
    const int tid = threadIdx.x;
    const int64_t v0 = (int64_t)blockIdx.x * V;
    if (tid == 0) n_flag = n_walk = 0;
    // two rows of one place: one of them is not the row found there.  (What the last launch asks of the table is summed up
    // here, so that with nothing to walk it reads three words: 524288 vectors 35.9 -> 33.2 us, 960 20 -> 17.3.)
    for (int64_t r = (int64_t)blockIdx.x * ES_THREADS + tid; r < a.n_entries; r += (int64_t)gridDim.x * ES_THREADS) {
        const int place = a.place_of[r];
        if (place >= 0 && a.row_at[place] != (int)r) a.found[ES_SHARED] = 1;
    }
    if (blockIdx.x == gridDim.x - 1) {                         // rows of the full shells; other rows make the sum differ
        int full = 0;
        for (int i = tid; i < (a.n_entries + 63) / 64; i += ES_THREADS) full += a.counts[i];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) full += __shfl_xor(full, o, 64);
        if ((tid & 63) == 0) atomicAdd(a.found + ES_IN_FULL, full);
    }
    if (v0 >= a.N) return;                                     // here for that only
    __syncthreads();
    auto walk = [&](int local) {
        const int64_t at = v0 + atomicAdd(&n_walk, 1);
        a.walk_list[at] = local;
        a.walk_arrive[at] = 0;
        a.walk_key[at] = es_key(__builtin_inff(), 0);          // the walk's start
    };
#pragma unroll 1
    for (int local = tid; local < V && v0 + local < a.N; local += ES_THREADS) {
        const int64_t v = v0 + local;
        float xv[8];
        es_load(a.x, v, xv);
        es_vec s;
        if (!es_sort(xv, s)) { walk(local); continue; }
        float b1 = __builtin_inff(), b2 = b1, b12 = b1;
        uint32_t p = 0;
        es_orbits(s.y, [&](float d, uint32_t code) {
            b2 = __builtin_amdgcn_fmed3f(b1, b2, d);
            if (d < b1) p = code;
            b1 = __builtin_fminf(b1, d);
        });
        es_orbits_12(s.y, [&](float d, uint32_t) { b12 = __builtin_fminf(b12, d); });
        float gap = __builtin_fminf(b2, b12) - b1;             // to other orbits, and to p's own by a reflection
        int q[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) q[r] = es_q(p, r);
#pragma unroll
        for (int r = 0; r < 7; ++r)
            if (q[r] != q[r + 1]) gap = __builtin_fminf(gap, (float)(q[r] - q[r + 1]) * (s.y[r] - s.y[r + 1]));
        if (q[6] + q[7] != 0) gap = __builtin_fminf(gap, (float)(q[6] + q[7]) * (s.y[6] + s.y[7]));
        if (!(gap > s.margin)) {
            const int at = atomicAdd(&n_flag, 1);
            flags[at] = (unsigned short)local;
            if (at < ES_CHUNK) {                               // the first chunk's are at hand
#pragma unroll
                for (int r = 0; r < 8; ++r) sk[r][at] = s.k[r];
                s_signs[at] = s.signs | (s.flip ? 256u : 0u);
                s_margin[at] = s.margin;
            }
            continue;
        }
        const uint32_t code = es_code(p, s.k, s.signs, s.flip);
        a.idx_out[v] = a.row_at[es_place(code)];               // a row of the table, of norm up to 10
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
    }
    __syncthreads();
    const int nf = n_flag;
    // As many vectors at a time as the lists hold the first points of, with room for as many again.  (32 where more than half are
    // here and 128 otherwise, without the second try below: 1.5 and 2 times as long at scale 4 and 2.)
    int step = ES_CHUNK;
    for (int c0 = 0; c0 < nf;) {
        const int nc = nf - c0 < step ? nf - c0 : step;
        if (tid == 0) n_seed = n_child = 0;
        if (tid < ES_CHUNK) s_walk[tid] = 0;
        __syncthreads();
        auto put = [&](int at, int end, uint32_t p, int j, float room) {
            if (at < end) {
                list_p[at] = p;
                list_j[at] = (unsigned char)j;
                list_room[at] = room;
            } else s_walk[j] = 1;
        };
        // the nearest points of the orbits in reach, and their children: half of the orbits each to two threads of a vector
        const int mine = tid & (ES_CHUNK - 1), half = __builtin_amdgcn_readfirstlane(tid / ES_CHUNK);
        if ((mine & ~63) < nc) {
            const bool on = mine < nc;
            const int slot = on ? mine : 0;
            float y[8], margin;
            if (c0 == 0) {
#pragma unroll
                for (int r = 0; r < 8; ++r) y[r] = __builtin_bit_cast(float, sk[r][slot] & ~7u);
                if (s_signs[slot] & 256u) y[7] = -y[7];
                margin = s_margin[slot];
            } else {
                float xv[8];
                es_load(a.x, v0 + flags[c0 + slot], xv);
                es_vec s;
                es_sort(xv, s);
                if (on && half == 0) {
#pragma unroll
                    for (int r = 0; r < 8; ++r) sk[r][mine] = s.k[r];
                    s_signs[mine] = s.signs | (s.flip ? 256u : 0u);
                }
#pragma unroll
                for (int r = 0; r < 8; ++r) y[r] = s.y[r];
                margin = s.margin;
            }
            if (on && half == 0) best[mine] = ~0ull;
            float b1 = __builtin_inff(), room[25];
            int o = 0;
            es_orbits(y, [&](float v, uint32_t) {
                b1 = __builtin_fminf(b1, v);
                room[o++] = v;
            });
            es_orbits_12(y, [&](float v, uint32_t) { room[o++] = v; });
            const float reach = b1 + margin;
#pragma unroll
            for (o = 0; o < 25; ++o) room[o] = on ? reach - room[o] : -1.0f;
            if (nf <= ES_FEW) {                                // points like the others, whose children the waves find
                o = 0;
                auto list = [&](float, uint32_t code) {
                    if (o / 13 == half && room[o] >= 0.0f) {
                        const int to = atomicAdd(&n_child, 1);
                        put((to & 3) * ES_WAVE + (to >> 2), ((to & 3) + 1) * ES_WAVE, code, mine, room[o]);
                    }
                    ++o;
                };
                es_orbits(y, list);
                es_orbits_12(y, list);
            } else {
                int seeds = 0, children = 0;
                o = 0;
                auto count = [&](float, uint32_t code) {
                    if (o / 13 == half) {
                        seeds += room[o] >= 0.0f;
                        es_children(code, y, room[o], [&](float, uint32_t) { ++children; });
                    }
                    ++o;
                };
                es_orbits(y, count);
                es_orbits_12(y, count);
                int at = ES_GROWN + es_places(seeds, &n_seed), to = es_places(children, &n_child);
                if (step == 16 || __ballot(at + seeds > ES_LIST || to + children > ES_GROWN / 2) == 0) {
                    o = 0;
                    auto list = [&](float, uint32_t code) {
                        if (o / 13 == half) {
                            if (room[o] >= 0.0f) put(at++, ES_LIST, code, mine, 0.0f);
                            es_children(code, y, room[o], [&](float gap, uint32_t child) {   // dealt out to the waves
                                put((to & 3) * ES_WAVE + (to >> 2), ((to & 3) + 1) * ES_WAVE, child, mine, room[o] - gap);
                                ++to;
                            });
                        }
                        ++o;
                    };
                    es_orbits(y, list);
                    es_orbits_12(y, list);
                }
            }
        }
        __syncthreads();
        if (step > 16 && (n_seed > ES_LIST - ES_GROWN || n_child > ES_GROWN / 2)) {
            int of = 1;                                        // too many for the lists: again with fewer vectors
            do of *= 2;
            while (step > 16 * of && (n_seed > of * (ES_LIST - ES_GROWN) || n_child > of * (ES_GROWN / 2)));
            step /= of;
            __syncthreads();
            continue;
        }
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), first = wave * ES_WAVE;
        int n = min((n_child + 3 - wave) >> 2, ES_WAVE), done = 0, seeds = min(n_seed, ES_LIST - ES_GROWN);
        for (;;) {
            // a wave's own points, with no wait for the others, until none is added or its part of the list is full: a lane
            // each while there are many, eight lanes each when there are few
            while (done < n) {
                if (n - done >= ES_MANY) {
                    // the last added ones first where the list fills up, so that fewer wait
                    const bool last = n > ES_WAVE / 2 && n - done >= 128;
                    const int at = (last ? n - 64 : done) + (tid & 63), e = first + min(at, n - 1), j = list_j[e];
                    const float room = at < n ? list_room[e] : -1.0f;
                    const uint32_t p = list_p[e];
                    if (last) {                                // they change places with the longest waiting
                        const int with = first + done + (tid & 63);
                        const uint32_t wp = list_p[with];
                        const unsigned char wj = list_j[with];
                        const float wr = list_room[with];
                        list_p[with] = p;
                        list_j[with] = (unsigned char)j;
                        list_room[with] = room;
                        list_p[e] = wp;
                        list_j[e] = wj;
                        list_room[e] = wr;
                    }
                    float y[8];
#pragma unroll
                    for (int r = 0; r < 8; ++r) y[r] = __builtin_bit_cast(float, sk[r][j] & ~7u);
                    if (s_signs[j] & 256u) y[7] = -y[7];
                    int children = 0, total;
                    es_children(p, y, room, [&](float, uint32_t) { ++children; });
                    int to = first + n + es_before(children, total);
                    if (n + total > ES_WAVE && done > 0) break;
                    es_children(p, y, room, [&](float gap, uint32_t child) { put(to++, first + ES_WAVE, child, j, room - gap); });
                    done = min(done + 64, n);
                    n = min(n + total, ES_WAVE);
                    __builtin_amdgcn_wave_barrier();
                    continue;
                }
                const int i = tid & 7, k = i < 7 ? i : 6, at = done + (tid >> 3 & 7), e = first + min(at, n - 1), j = list_j[e];
                const float room = list_room[e];
                const uint32_t p = list_p[e], kb = sk[k + 1][j] & ~7u;
                const float ya = __builtin_bit_cast(float, sk[k][j] & ~7u);
                const float yb = __builtin_bit_cast(float, k == 6 && (s_signs[j] & 256u) ? kb ^ 0x80000000u : kb);
                float gap;
                const bool child = es_child(p, i, ya, yb, room, gap) && at < n;
                const unsigned long long all = __ballot(child);
                if (n + __builtin_popcountll(all) > ES_WAVE && done > 0) break;
                const int to = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(all >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)all, 0));
                if (child) put(first + to, first + ES_WAVE, es_reflect(p, i), j, room - gap);
                done = min(done + 8, n);
                n = min(n + __builtin_popcountll(all), ES_WAVE);
                __builtin_amdgcn_wave_barrier();
            }
            if ((tid & 63) == 0) {
                n_grown[wave] = done;
                n_left[wave] = n - done;
            }
            __syncthreads();
            // the points that the table holds, by the walk's arithmetic: three trips to memory each, two points at a time where there
            // are more than threads (where there are not, the second one's trips cost 0.1-0.3 us)
            const int g0 = n_grown[0], g1 = g0 + n_grown[1], g2 = g1 + n_grown[2], g3 = g2 + n_grown[3];
            const int some = g3 + seeds;
            auto compare = [&](int q0, auto points) {
                constexpr int U = decltype(points)::value;
                int j[U], row[U];
                uint32_t code[U];
                float xv[U][8];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int q = min(q0 + u * ES_THREADS, some - 1);
                    const int e = q < g0 ? q : q < g1 ? ES_WAVE + q - g0 : q < g2 ? 2 * ES_WAVE + q - g1 : q < g3 ? 3 * ES_WAVE + q - g2 : ES_GROWN + q - g3;
                    j[u] = list_j[e];
                    es_load(a.x, v0 + flags[c0 + j[u]], xv[u]);
                    uint32_t k[8];
#pragma unroll
                    for (int r = 0; r < 8; ++r) k[r] = sk[r][j[u]];
                    code[u] = es_code(list_p[e], k, s_signs[j[u]], (s_signs[j[u]] >> 8) & 1u);
                }
                int place[U];
#pragma unroll
                for (int u = 0; u < U; ++u) place[u] = es_place(code[u]);
#pragma unroll
                for (int u = 0; u < U; ++u) row[u] = a.row_at[place[u]];
#pragma unroll
                for (int u = 0; u < U; ++u)                        // not held: the place is not set
                    if ((uint32_t)row[u] >= (uint32_t)a.n_entries || a.place_of[row[u]] != place[u]) row[u] = -1;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (row[u] < 0 || q0 + u * ES_THREADS >= some) continue;
                    float c[8];
                    int n4 = 0;
#pragma unroll
                    for (int d = 0; d < 8; ++d) {
                        const int q = es_q(code[u], d);
                        c[d] = 0.5f * (float)q;
                        n4 += q * q;
                    }
                    atomicMin(&best[j[u]], es_key(es_dist(xv[u], c, 0.25f * (float)n4), row[u]));
                }
            };
            if (some <= ES_THREADS) {
                if (tid < some) compare(tid, std::integral_constant<int, 1>());
            } else {
                for (int q0 = tid; q0 < some; q0 += 2 * ES_THREADS) compare(q0, std::integral_constant<int, 2>());
            }
            if ((n_left[0] | n_left[1] | n_left[2] | n_left[3]) == 0) break;
            __syncthreads();
            // those that are not tried for children yet go to the front
            for (int e = tid & 63; e < n - done; e += 64) {
                list_p[first + e] = list_p[first + done + e];
                list_j[first + e] = list_j[first + done + e];
                list_room[first + e] = list_room[first + done + e];
            }
            __builtin_amdgcn_wave_barrier();
            n -= done;
            done = seeds = 0;
        }
        __syncthreads();
        if (tid < nc) {
            const int local = flags[c0 + tid];
            if (s_walk[tid]) walk(local);
            else if (best[tid] != ~0ull) es_store(a, v0 + local, (int)(uint32_t)best[tid]);   // none: not the shell table
        }
        __syncthreads();
        c0 += step;
    }
    if (tid == 0) {
        a.walk_count[blockIdx.x] = n_walk;
        if (n_walk) atomicAdd(a.found + ES_WALKS, n_walk);
    }
}

// The table walk for the vectors left over, 64 at a time, a lane each: workgroup (64 vectors, part of
// the table), its waves walking a quarter of the part.  The lowest (distance, row) of a part goes to the
// vector's 64-bit minimum; the last part to arrive writes the row.
__global__ void __launch_bounds__(ES_THREADS)
e8_walk_kernel(const es_args a, int n_src, int per_src) {
    constexpr int ROWS = 65536 / ES_SPLIT;                     // of one part, at most
    __shared__ int sums[4];
    __shared__ int64_t item[64];                               // the vector's list position
    __shared__ unsigned long long keys[4][64];
    __shared__ f32x4v rows[ROWS][2];
    __shared__ float row_norm[ROWS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (a.found[ES_SHARED] != 0 || a.found[ES_IN_FULL] != ES_FULL) {   // not what the search assumed: every vector, every row
        const int64_t blocks = (a.N + EQ_THREADS * EQ_VPT - 1) / (EQ_THREADS * EQ_VPT);
        for (int64_t b = blockIdx.x; b < blocks; b += gridDim.x)
            e8_quantize_block(a.x, a.table, a.norms, a.N, a.n_entries, a.idx_out, a.dec_out, b);
        return;
    }
    const int total = a.found[ES_WALKS];
    if (total == 0) return;
    // the vectors' ranks over all source workgroups: a run of sources per thread
    const int per = (n_src + ES_THREADS - 1) / ES_THREADS;
    const int s0 = min(tid * per, n_src), s1 = min(s0 + per, n_src);
    int mine = 0;
    for (int s = s0; s < s1; ++s) mine += a.walk_count[s];
    int first = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(first, o, 64);
        if (lane >= o) first += v;
    }
    if (lane == 63) sums[wave] = first;
    __syncthreads();
    first -= mine;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (q < wave) first += sums[q];
    const int64_t work = (int64_t)((total + 63) / 64) * ES_SPLIT;
    for (int64_t w = blockIdx.x; w < work; w += gridDim.x) {
        const int base = (int)(w / ES_SPLIT) * 64, part = (int)(w % ES_SPLIT);
        if (first < base + 64 && first + mine > base) {
            int rank = first;
            for (int s = s0; s < s1; ++s)
                for (int j = 0, c = a.walk_count[s]; j < c; ++j, ++rank)
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
        const int64_t v = at / per_src * per_src + a.walk_list[at];
        float xv[8], best = __builtin_inff();
        es_load(a.x, v, xv);
        int row = 0;
        const int i1 = n * (wave + 1) / 4;
#pragma unroll 4
        for (int i = n * wave / 4; i < i1; ++i) {
            const float d = es_dist(xv, (const float *)rows[i], row_norm[i]);
            if (d < best) { best = d; row = r0 + i; }
        }
        keys[wave][lane] = es_key(best, row);
        __syncthreads();
        if (wave == 0 && on) {
            unsigned long long key = keys[0][lane];
            for (int o = 1; o < 4; ++o) key = keys[o][lane] < key ? keys[o][lane] : key;
            // the minimum has been taken before the arrival is counted: its old value is waited for
            const unsigned long long old = atomicMin(a.walk_key + at, key);
            asm volatile("" ::"v"(old));
            __builtin_amdgcn_s_waitcnt(0);
            if (atomicAdd(a.walk_arrive + at, 1) == ES_SPLIT - 1)
                es_store(a, v, (int)(uint32_t)__hip_atomic_load(a.walk_key + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        }
        __syncthreads();
    }
}

// Vectors per workgroup: few while the chip is not filled, for latency; more when it is, so that the vectors with
// more than one point in reach fill the threads that list the points.
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

static size_t es_align(size_t v) { return (v + 15) & ~(size_t)15; }

size_t glqh_e8_shell_ws_bytes(int64_t N) {
    return es_align((size_t)N * 16 + (size_t)((N + 63) / 64) * 4) + (size_t)(ES_PLACES + 65536 + 65536 / 64 + ES_FOUND) * 4;
}

int glqh_launch_e8_shell_quantize(const float *x, int64_t N, const float *table, const float *norms, int n_entries,
                                  int64_t *idx_out, float *dec_out, void *ws, hipStream_t stream) {
    const int per = es_per_wg(N);
    const int64_t wgs = (N + per - 1) / per;
    GLQH_REQUIRE(N <= 2147483647ll, "e8 quantize: too many vectors");
    es_args a;
    a.x = x; a.table = table; a.norms = norms; a.N = N; a.n_entries = n_entries;
    a.idx_out = idx_out; a.dec_out = dec_out;
    a.walk_key = (unsigned long long *)ws;
    a.walk_list = (int *)(a.walk_key + N);
    a.walk_arrive = a.walk_list + N;
    a.walk_count = a.walk_arrive + N;
    a.row_at = (int *)((char *)ws + es_align((size_t)N * 16 + (size_t)((N + 63) / 64) * 4));
    a.place_of = a.row_at + ES_PLACES;
    a.counts = a.place_of + 65536;
    a.found = a.counts + 65536 / 64;
    const dim3 grid((unsigned)(wgs > ES_CHECKS ? wgs : ES_CHECKS));
    hipLaunchKernelGGL(es_index_kernel, dim3((unsigned)((n_entries + ES_THREADS - 1) / ES_THREADS)), dim3(ES_THREADS), 0, stream, table,
                       norms, n_entries, a.row_at, a.place_of, a.counts, a.found);
    if (per == 512) hipLaunchKernelGGL(e8_shell_kernel<512>, grid, dim3(ES_THREADS), 0, stream, a);
    else if (per == 256) hipLaunchKernelGGL(e8_shell_kernel<256>, grid, dim3(ES_THREADS), 0, stream, a);
    else hipLaunchKernelGGL(e8_shell_kernel<64>, grid, dim3(ES_THREADS), 0, stream, a);
    hipLaunchKernelGGL(e8_walk_kernel, dim3(2 * glqh_device_cus()), dim3(ES_THREADS), 0, stream, a, (int)wgs, per);
    GLQH_LAUNCH_CHECK("e8 shell quantize launch");
    return 0;
}
