// Tail-biting Viterbi search of the trellis-3INST quantizer on the GPU
// (bitshift_codebook.viterbi / quantize, glq/trellis.py:253-296, 467-484;
// _viterbi_acs_step, glq/trellis_step_kernel.py:30-109).
//
// A tile is a sequence of T = 256 values; the trellis has 2^16 states, a step shifts K new
// bits in (state' = (state << K | b) & 0xFFFF) and costs (lut[state'] - x)^2.  With
// G = 2^(16-K), the predecessors of state' are the 2^K states k*G + (state' >> K), so only
//     best_i[g] = min_k ( err_{i-1}[k*G + g] + best_{i-1}[(k*G + g) >> K] ),  lowest k on ties,
// has to be carried from step to step (G floats in LDS).  The search runs twice
// (glq/trellis.py:479-482): on the sequence rolled by T/2 without constraints, then on the
// sequence itself with first and last state tied to the overlap the first pass found.
// All arithmetic is fp32 with separate subtract, multiply and add (no contraction), the
// input is rounded to fp16 first (glq/trellis.py:468).
//
// viterbi_kernel does that for every tile of 1-bit calls and, at 2 and 3 bits, of small ones; elsewhere for those that the
// search on lower bounds, further down, does not try or leaves to it.
//
// What bounds it is vector-ALU issue: 65536 states per step, 510 steps per tile.  A workgroup
// therefore keeps the whole table in registers, two fp16 values to a register (v_fma_mix_f32
// subtracts the input from either half with fp32 rounding), and a state costs 3.5 instructions:
// subtract, multiply, add, half a three-way minimum.  The arg-min is not tracked: every
// `VT_DEPTH`-th cost row goes to scratch and the backtrack, one wave, recomputes the 2^(K*depth)
// costs below its state for `depth` steps at a time.  2048 x 2048 weights at K = 4: 165 ms (hash per
// state and step, compare and two selects per state, a byte of arg-min per step and group) -> 69.6 ms,
// vector ALUs issuing in 74 % of the cycles at 2.4 GHz (30.8 M instructions per SIMD, of which 29.9 M
// are the 3.5 per state).
#include <algorithm>
#include <type_traits>
#include "common.h"
#include "trellis_device.h"

#pragma clang fp contract(off)

size_t glqh_viterbi_scratch_bytes(int K, int64_t n_tiles, int less);

namespace {

constexpr int VT_T = 256;

struct vt_best {
    float cost;
    int state;
};

// A thread owns UNITS units of LOWS neighbouring groups that share their predecessors' groups
// (g >> K): unit u holds groups u*LOWS .. u*LOWS + LOWS-1 under predecessor group hi(u), and
// neighbouring threads own neighbouring units, so that cost reads are conflict-free and cost
// writes are whole 8..32-byte runs.  512 threads and at most 128 registers for K >= 2: two
// workgroups per CU, one of which computes while the other's single wave walks back.  At K = 1 the
// cost row alone is 128 KB of LDS: one workgroup of 1024.
template <int K>
struct vt_cfg {
    static constexpr int G = 1 << (16 - K), NK = 1 << K;
    static constexpr int THREADS = K == 1 ? 1024 : 512;
    static constexpr int PER = G / THREADS;                    // groups per thread
    static constexpr int LOWS = K == 4 ? 8 : NK;               // K = 4: two threads per predecessor group
    static constexpr int UNITS = PER / LOWS;
    static constexpr int HI = G >> K;                          // predecessor groups
    // two cost rows where they fit the LDS twice per CU, else one (every thread reads, then all write)
    static constexpr bool TWO_ROWS = K >= 3;
    static constexpr int ROWS = TWO_ROWS ? 2 : 1;
    // steps per stored cost row: 16 KB of cost rows per step at most (8 KB at K = 4), 64 or 256 leaves
    static constexpr int DEPTH = K == 1 ? 8 : K == 2 ? 4 : 2;
};

// LDS only: a __syncthreads() would also wait for the cost rows on their way to scratch
__device__ __forceinline__ void vt_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// (float)half - x, rounded once; exact halves of a packed register, x the same for the whole wave
__device__ __forceinline__ float vt_sub_lo(f16x2 w, float x) {
    float d;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(w), "s"(x));
    return d;
}
__device__ __forceinline__ float vt_sub_hi(f16x2 w, float x) {
    float d;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(w), "s"(x));
    return d;
}

__device__ __forceinline__ float vt_err(int s, float x) {
    const float d = (float)tr_weight((uint32_t)s) - x;
    return d * d;
}

// States i-1 .. i-D from state s of step i (one wave): the costs of the NK^D paths into s from the
// cost row of step i-D, minimised level by level, lowest k on ties.  cost, pick: 256 words each of LDS.
template <int K, int D>
__device__ __forceinline__ int vt_back(int i, int s, const float *__restrict__ row, const float *x, float *cost,
                                       int *pick, int *states) {
    constexpr int G = vt_cfg<K>::G, NK = vt_cfg<K>::NK;
    constexpr int LEAVES = 1 << (K * D);
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));                             // keeps what follows from it out of the callers' registers
    // state reached from s by the digits of p (e digits, most significant first)
    auto walk = [&](int p, int e) {
        int st = s;
        for (int q = e - 1; q >= 0; --q) st = (st >> K) + ((p >> (K * q)) & (NK - 1)) * G;
        return st;
    };
#pragma unroll
    for (int r = 0; r < (LEAVES + 63) / 64; ++r) {
        const int p = lane + 64 * r;
        if (p < LEAVES) {
            const int st = walk(p, D);
            // rows were written by other waves of this workgroup: past the L1
            const float b = __hip_atomic_load(row + (st >> K), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            cost[p] = vt_err(st, x[i - D]) + b;
        }
    }
    __builtin_amdgcn_wave_barrier();
    int base = 0;                                              // pick: level D first, then D-1, ...
#pragma unroll
    for (int e = D; e >= 1; --e) {
        const int groups = 1 << (K * (e - 1));
        float nc[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int p = lane + 64 * r;
            if (p < groups) {
                float bc = cost[p * NK];
                int bk = 0;
#pragma unroll
                for (int k = 1; k < NK; ++k) {
                    const float c = cost[p * NK + k];
                    if (c < bc) { bc = c; bk = k; }
                }
                pick[base + p] = bk;
                nc[r] = e > 1 ? vt_err(walk(p, e - 1), x[i - e + 1]) + bc : bc;
            }
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < 2; ++r)
            if (lane + 64 * r < groups) cost[lane + 64 * r] = nc[r];
        __builtin_amdgcn_wave_barrier();
        base += groups;
    }
    // the picks from the top: level 1 is the last one stored
    int p = 0;
#pragma unroll
    for (int e = 1; e <= D; ++e) {
        base -= 1 << (K * (e - 1));
        p = p * NK + pick[base + p];
        const int st = walk(p, e);
        if (lane == 0) states[i - e] = st;
        if (e == D) s = st;
    }
    __builtin_amdgcn_wave_barrier();
    return __builtin_amdgcn_readfirstlane(s);
}

// One pass.  x: T inputs in LDS; best: ROWS * G floats in LDS; hist: cost rows of steps 0, DEPTH,
// 2*DEPTH, ... in scratch; overlap < 0: unconstrained.  Leaves the best state sequence in `states`
// (LDS), from step `first` on.
template <int K>
__device__ __forceinline__ void viterbi_pass(const f16x2 (&w)[32768 / vt_cfg<K>::THREADS], const float *x, float *best,
                                             float *__restrict__ hist, int overlap, int first, int *states, vt_best *red,
                                             float *cost, int *pick) {
    using C = vt_cfg<K>;
    constexpr int G = C::G, NK = C::NK, LOWS = C::LOWS, UNITS = C::UNITS, D = C::DEPTH;
    const int tid = threadIdx.x;
    const float inf = __builtin_inff();
    float *cur = best, *nxt = C::TWO_ROWS ? best + G : best;
    for (int g = tid; g < G; g += C::THREADS) {
        const float v = (overlap < 0 || g == overlap) ? 0.0f : inf;
        cur[g] = v;
        if (first == 0) hist[g] = v;
    }
    vt_barrier();
    auto hi_of = [&](int q) { return K == 4 ? tid >> 1 : tid + q * C::THREADS; };
    float xn = x[0];                                           // a step's input, read a step ahead
#pragma unroll 1
    for (int i = 1; i < VT_T; ++i) {
        const float xi = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, xn)));
        xn = x[i];
        float *row = (i % D == 0 && i >= first - D) ? hist + (int64_t)(i / D) * G : nullptr;   // uniform
        float c[UNITS][NK];
        auto load = [&](int q) {
#pragma unroll
            for (int k = 0; k < NK; ++k) c[q][k] = cur[k * C::HI + hi_of(q)];
        };
        if constexpr (!C::TWO_ROWS) {
#pragma unroll
            for (int q = 0; q < UNITS; ++q) load(q);
            vt_barrier();
        }
#pragma unroll
        for (int q = 0; q < UNITS; ++q) {
            if constexpr (C::TWO_ROWS) load(q);
            float m[LOWS];
#pragma unroll
            for (int j = 0; j < LOWS; j += 2) {
                float a[NK], b[NK];
#pragma unroll
                for (int k = 0; k < NK; ++k) {
                    const f16x2 wk = w[(k * UNITS + q) * (LOWS / 2) + j / 2];
                    const float d0 = vt_sub_lo(wk, xi), d1 = vt_sub_hi(wk, xi);
                    a[k] = d0 * d0 + c[q][k];
                    b[k] = d1 * d1 + c[q][k];
                }
                float ma = a[0], mb = b[0];
                if constexpr (NK == 2) {
                    ma = __builtin_fminf(ma, a[1]);
                    mb = __builtin_fminf(mb, b[1]);
                } else {
#pragma unroll
                    for (int k = 1; k + 1 < NK; k += 2) {
                        ma = __builtin_fminf(__builtin_fminf(ma, a[k]), a[k + 1]);
                        mb = __builtin_fminf(__builtin_fminf(mb, b[k]), b[k + 1]);
                    }
                    ma = __builtin_fminf(ma, a[NK - 1]);
                    mb = __builtin_fminf(mb, b[NK - 1]);
                }
                m[j] = ma;
                m[j + 1] = mb;
                __builtin_amdgcn_sched_barrier(0);             // one pair of groups at a time: no spills in this loop
            }
            const int g = (tid + q * C::THREADS) * LOWS;
            if constexpr (LOWS == 2) {
                *(f32x2 *)(nxt + g) = f32x2{m[0], m[1]};
                if (row) *(f32x2 *)(row + g) = f32x2{m[0], m[1]};
            } else {
#pragma unroll
                for (int j = 0; j < LOWS; j += 4) {
                    const f32x4 v = {m[j], m[j + 1], m[j + 2], m[j + 3]};
                    *(f32x4 *)(nxt + g + j) = v;
                    if (row) *(f32x4 *)(row + g + j) = v;
                }
            }
        }
        vt_barrier();
        if constexpr (C::TWO_ROWS) { float *t = cur; cur = nxt; nxt = t; }
    }
    // final costs, with the tail-biting mask on the low 16-K bits; lowest state on ties
    const float xl = x[VT_T - 1];
    float bc = inf;
    int bs = 0x7fffffff;
#pragma unroll 1
    for (int s = tid; s < 65536; s += C::THREADS) {
        float c = vt_err(s, xl) + cur[s >> K];
        if (overlap >= 0 && (s & (G - 1)) != overlap) c = inf;
        if (c < bc || (c == bc && s < bs)) { bc = c; bs = s; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float oc = __shfl_xor(bc, o, GLQH_WAVE);
        const int os = __shfl_xor(bs, o, GLQH_WAVE);
        if (oc < bc || (oc == bc && os < bs)) { bc = oc; bs = os; }
    }
    if ((tid & 63) == 0) red[tid >> 6] = vt_best{bc, bs};
    __syncthreads();                                           // and every stored cost row has arrived
    if (tid < GLQH_WAVE) {
        vt_best b = red[0];
        for (int v = 1; v < C::THREADS / 64; ++v)
            if (red[v].cost < b.cost || (red[v].cost == b.cost && red[v].state < b.state)) b = red[v];
        // every state is infinite only if the constraint is unsatisfiable, which the
        // first pass rules out; argmin of an all-inf row is state 0 in the reference
        int s = __builtin_amdgcn_readfirstlane(b.state == 0x7fffffff ? 0 : b.state);
        if (tid == 0) states[VT_T - 1] = s;
        constexpr int REST = (VT_T - 1) % D;                   // steps above the last stored row
        int i = VT_T - 1;
        s = vt_back<K, REST>(i, s, hist + (int64_t)((i - REST) / D) * G, x, cost, pick, states);
        i -= REST;
#pragma unroll 1
        for (; i > first; i -= D) s = vt_back<K, D>(i, s, hist + (int64_t)(i / D - 1) * G, x, cost, pick, states);
    }
    __syncthreads();
}

// Position (row * 16 + col) of trellis step t = 8l + j inside its 16x16 tile (glq/trellis.py:99-101).
__device__ __forceinline__ int64_t vt_step_pos(int t, int64_t ld) {
    const int l = t >> 3, j = t & 7;
    return (int64_t)((l >> 2) + 8 * ((j >> 1) & 1)) * ld + 2 * (l & 3) + 8 * (j >> 2) + (j & 1);
}

// Element `t` of a tile.  ld > 0: of (m, n) matrices of row length ld, the tiles their 16x16 blocks in row-major order;
// ld == 0: of (tiles, 256) rows in step order.
__device__ __forceinline__ int64_t vt_pos(int64_t tile, int t, int64_t ld) {
    const int64_t per_row = ld >> 4;
    return ld ? (tile / per_row) * 16 * ld + (tile % per_row) * 16 + vt_step_pos(t, ld) : tile * VT_T + t;
}

// Which tiles of a call are searched how: those for the search on bounds, from order[0] on, those that it does not try, from
// order[n_tiles - 1] back, and those that it tried and left.
struct vb_lists {
    int *counts;                           // how many it tries, how many it left, and before this batch, and how many of the first go
                                           // through vm_kernel; null: no such search
    int *order, *left;
};

// Persistent workgroups walk the tiles (lists: those that are not found on bounds) with a fixed stride, each owning one
// slab of cost rows.
template <int K>
__global__ void __launch_bounds__(vt_cfg<K>::THREADS, 4)
viterbi_kernel(const float *__restrict__ tiles_in, int64_t n_tiles, int64_t ld, float *__restrict__ scratch,
               int32_t *__restrict__ states_out, float *__restrict__ hat_out, vb_lists lists) {
    using C = vt_cfg<K>;
    constexpr int G = C::G;
    extern __shared__ float best[];                            // ROWS * G floats
    __shared__ float x[VT_T], xr[VT_T], cost[VT_T];
    __shared__ int states[VT_T], pick[VT_T];
    __shared__ vt_best red[C::THREADS / 64];
    const int tid = threadIdx.x;
    float *hist = scratch + (int64_t)blockIdx.x * (VT_T / C::DEPTH) * G;
    const int64_t untried = lists.counts ? n_tiles - lists.counts[0] : 0, todo = lists.counts ? untried + lists.counts[1] : n_tiles;
    if ((int64_t)blockIdx.x >= todo) return;
    f16x2 w[32768 / C::THREADS];
#pragma unroll
    for (int k = 0; k < C::NK; ++k)
#pragma unroll
        for (int q = 0; q < C::UNITS; ++q)
#pragma unroll
            for (int j = 0; j < C::LOWS; j += 2) {
                const uint32_t s = (uint32_t)(k * G + (tid + q * C::THREADS) * C::LOWS + j);
                f16x2 v = {tr_weight(s), tr_weight(s + 1)};
                asm volatile("" : "+v"(v));                    // finished here: neither spilled half-done nor recomputed
                w[(k * C::UNITS + q) * (C::LOWS / 2) + j / 2] = v;
            }
    for (int64_t item = blockIdx.x; item < todo; item += gridDim.x) {
        int64_t tile = item;
        if (lists.counts) tile = item < untried ? lists.order[n_tiles - 1 - item] : lists.left[item - untried];
        const int64_t pos = vt_pos(tile, tid & 255, ld);
        if (tid < VT_T) {
            const float v = (float)(f16)tiles_in[pos];
            x[tid] = v;
            xr[(tid + VT_T / 2) & (VT_T - 1)] = v;             // np.roll(x, T/2)
        }
        __syncthreads();
        viterbi_pass<K>(w, xr, best, hist, -1, VT_T / 2, states, red, cost, pick);
        const int overlap = states[VT_T / 2] >> K;
        __syncthreads();
        viterbi_pass<K>(w, x, best, hist, overlap, 0, states, red, cost, pick);
        if (tid < VT_T) {
            const int s = states[tid];
            states_out[tile * VT_T + tid] = s;
            hat_out[pos] = (float)tr_weight((uint32_t)s);
        }
        __syncthreads();
    }
}

// ---- the search on lower bounds ----------------------------------------------------------
// The costs that decide are fp32, but most of what viterbi_kernel spends on them goes to states that no good path comes
// near.  Here the forward pass carries LOWER BOUNDS of the costs in packed fp16, two states to an instruction and rounded
// towards zero, and the few paths that their bounds do not exclude are compared in the exact arithmetic of
// viterbi_kernel: the same states, the same ties.
//
// Bounds (vb_forward).  l_i[g] <= best_i[g] - B_i for every group: the subtraction and the multiply-add of a state
// round towards zero, a minimum does not round, and every VB_NORM steps the row's minimum moves from the row into B
// (values stay small, where fp16 is fine; a difference of two fp16 numbers that is >= 0 rounds down too).  The pass runs
// one step past the last input, so that L = min l_T + B_T bounds the whole search.
// Backtrack (vb_backtrack, a wave a tile).  From the end, keep every way whose bound (its cost to the end + l + B)
// is at most L (1 + SLACK) + VB_LOST: what the fp16 roundings lose is 0.3-0.5 % of the cost, so a level keeps 1.4 ways on
// average.  (Below 2^-14 they lose up to 2^-24 a step whatever the cost: on values that are decoded ones again, or a rounding
// off them, L is 0 where the best path costs 10^-9.)
// At the start the cheapest kept path costs U.  If U (1 + VB_NEAR) is within the limit, no path that was dropped can be the
// search's answer, and the kept ones contain that and all its ties; else the backtrack runs again with that limit.  (Four
// fp32 sums stand between the two, each off by at most e = (256 + 8) 2^-24 of itself: U, the bound of what was dropped,
// and viterbi_kernel's costs of both paths, from which it takes the cheaper; 4 e < VB_NEAR.)  Where another kept path is
// within VB_NEAR of the cheapest (3 % of the tiles), fp32 costs are evaluated forward over the kept ways, minima and lowest
// states as in viterbi_kernel.
// Tiles with inputs above VB_X, not finite or all equal are not tried, and those with more kept ways than fit, behind vm_kernel also at half the
// slack, are left: lists of both go to viterbi_kernel (with marks instead of lists, every workgroup walking its share of all tiles, it took the
// time of all of them where half were marked).  Far beyond the weights' range the cost is mostly what no path can avoid,
// and SLACK of that lets everything through: tiles with more than WIDE of it are not tried either (K = 4: 5 % of those with
// 2-3 are left, 23 % with 4-5, 64 % with 10-14; K = 3 and 2: 20 and 18 % of the first beyond), nor is a minority of up to two
// chips full, nor the rest of a call after batches of which more than half were left.  4096 tiles, exact / so, ms:
//   normal values of sigma      1e-4         0.9          1.6          1.8          2.2          3 and more
//     K = 4                     17.5 / 17.2  17.5 / 7.9   17.5 / 10.9  17.5 / 15.6  17.5 / 17.5  17.5 / 17.6
//     K = 4, through vm_kernel         9.8          6.3          9.0         15.0         17.5         17.5
//     K = 3                     14.7 / 9.9   14.7 / 9.5   14.6 / 10.8  14.6 / 11.0  14.6 / 14.5  14.6 / 14.6
//     K = 2                     16.7 / 8.0   16.7 / 8.9   16.7 / 9.0   16.7 / 10.4  16.7 / 11.0  16.7 / 16.6
// Slower is what fills the lists and shows nothing beforehand, as slow ramps do (-3 to 3 over the tile's steps): 17.5 / 19.1 (20.4
// through vm_kernel, whose batches are larger; 70 % of a chip behind normal tiles 18.2 / 19.5), 14.6 / 16.3, 16.7 / 18.6, up to 1.3 times
// in calls of one or two batches.  2048 x 2048 weights: 69.6 -> 32.7 at K = 4 (24.0 through vm_kernel), 58.6 -> 38.0 at 3, 66.6 -> 35.4 at 2.
constexpr int VB_THREADS = 512;
constexpr int VB_NORM = 2;                 // steps between two moves of the row's minimum into B
constexpr float VB_X = 16.0f;              // largest input: (16 + 4)^2 for 16 / K steps stays far below 65504
constexpr float VB_W = 4.0f;               // the weights' range: 3.97
constexpr int VB_MOST = 64;                // kept groups of a step: a lane each
constexpr float VB_NEAR = 1100 * 0x1p-24f; // paths this close, relative to the limit, are compared in viterbi_kernel's sums
static_assert(4 * (VT_T + 8) * 0x1p-24f < VB_NEAR, "four sums of 256 rounded squares");
constexpr float VB_LOST = VT_T * 0x1p-24f; // what fp16 roundings of the smallest numbers take off a bound, at most

template <int K>
struct vb_cfg {
    static constexpr int G = 1 << (16 - K), NK = 1 << K, HI = G >> K;
    static constexpr int CW = NK / 2;                          // words of a group's predecessor costs
    static constexpr int DEPTH = K == 2 ? 4 : 2;               // steps per stored row
    static constexpr int STORED = VT_T / DEPTH;
    static constexpr float SLACK = K == 4 ? 0.0042f : K == 3 ? 0.0049f : 0.0058f;
    static constexpr int ROW = K == 4 ? 32 * 72 : K == 3 ? 128 * 36 : 4096 * 2 + 256 * 2;   // words of a row, with its padding
    static constexpr int ROWS = K == 2 ? 1 : 2;                // cost rows in LDS per tile; one: read by all, then written
    static constexpr float WIDE = 4.0f * (1 << (2 * (4 - K)));   // of a tile that is tried: cost beyond the weights' range
    static constexpr int FEW = K == 2 ? 2 : 1;                 // tiles a workgroup in calls that do not fill the chip
};

__device__ __forceinline__ f16x2 vb_pair(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t vb_bits(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ float vb_half(uint32_t bits) { return (float)__builtin_bit_cast(f16, (uint16_t)bits); }

// Where cost rows lie in LDS: the NK predecessor costs of a group (a = g >> K) are one run, read in one or two
// accesses, and what a wave writes of one low digit falls on different banks: runs are padded, and the words of a run
// (predecessors 2j, 2j+1) exchanged by an exclusive-or that is constant for a reader and for a writer.
template <int K>
__device__ __forceinline__ int vb_run(int a) {                 // in words
    if constexpr (K == 4) return (a >> 3) * 72 + (a & 7) * 8;
    if constexpr (K == 3) return (a >> 3) * 36 + (a & 7) * 4;
    return a * 2 + (a >> 4) * 2;
}
template <int K>
__device__ __forceinline__ int vb_word(int a) {
    if constexpr (K == 4) return (a >> 5) & 7;
    if constexpr (K == 3) return (a >> 7) & 3;
    return (a >> 6) & 1;
}
// group g's cost, in halves; the groups of a thread's slots are NK halves apart
template <int K>
__device__ __forceinline__ int vb_at(int g) {
    using C = vb_cfg<K>;
    const int k = g / C::HI, a = g % C::HI;
    return vb_run<K>(a) * 2 + (((k >> 1) ^ vb_word<K>(a)) << 1) + (k & 1);
}
// Stored rows are the runs without the padding: what a thread has read of the row goes out as it is, and the ways into
// one group, whose digits are the high ones, lie in 64-byte pieces.  Position of group g's cost, and back:
template <int K>
__device__ __forceinline__ int vb_stored(int g) {
    using C = vb_cfg<K>;
    const int k = g / C::HI, a = g % C::HI;
    return a * C::NK + (((k >> 1) ^ vb_word<K>(a)) << 1) + (k & 1);
}
template <int K>
__device__ __forceinline__ int vb_group(int at) {
    using C = vb_cfg<K>;
    const int a = at >> K, k = at & (C::NK - 1);
    return ((((k >> 1) ^ vb_word<K>(a)) << 1) + (k & 1)) * C::HI + a;
}

// vm_kernel's rows have all ways into a group in one piece, its NK^DEPTH runs one after the other (512 bytes at K = 4, where
// sixteen pieces of 32 touch sixteen cache lines: the walk back over 4096 tiles 694 -> 612 us).  vb_forward's threads write a run
// each of neighbouring groups, which would scatter.  Where a place of theirs lies then, and back:
template <int K>
__device__ __forceinline__ int vb_together(int at) {
    constexpr int E = 16 - K - K * vb_cfg<K>::DEPTH, HIGH = 16 - 2 * K - E;   // bits of a that the ways share, and the others
    const int a = at >> K;
    return ((a & ((1 << E) - 1)) << HIGH | a >> E) << K | (at & (vb_cfg<K>::NK - 1));
}
template <int K>
__device__ __forceinline__ int vb_apart(int at) {
    constexpr int E = 16 - K - K * vb_cfg<K>::DEPTH, HIGH = 16 - 2 * K - E;
    const int a = at >> K;
    return ((a & ((1 << HIGH) - 1)) << E | a >> HIGH) << K | (at & (vb_cfg<K>::NK - 1));
}

// the least of a wave's values, in every lane
__device__ __forceinline__ uint32_t vb_wave_min(uint32_t v) {
    auto step = [&](uint32_t u) { v = u < v ? u : v; };
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x111, 0xf, 0xf, false));   // row_shr:1, 2, 4, 8
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x112, 0xf, 0xf, false));
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x114, 0xf, 0xf, false));
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x118, 0xf, 0xf, false));
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xa, 0xf, false));   // row_bcast:15, 31
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xc, 0xf, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ int vb_lane(int v, int from) { return __builtin_amdgcn_readlane(v, from); }
__device__ __forceinline__ float vb_lane(float v, int from) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), from));
}
__device__ __forceinline__ int vb_below(uint64_t mask) {       // lanes of the mask below this one
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}

// What the two kernels of a pass hand each other, per tile
struct vb_tile {
    float pre[VT_T / VB_NORM + 1];         // B at step j * VB_NORM
    int over;                              // the tail-biting overlap, -1: left to viterbi_kernel
};

// Tiles order[vb_first .. vb_first + count - 1], as far as that many are tried, and one of their two passes: 0 on the inputs rolled by T/2, unconstrained; 1 from and
// to the overlap that the first backtrack found.  rows: of every tile a row of G halves, STORED times.
struct vb_part {
    int64_t first;
    int count, pass;
    uint16_t *rows;
    vb_tile *info;
    bool product;                          // bounds of vm_kernel
};
__device__ __forceinline__ int64_t vb_first(const vb_part &part, const vb_lists &lists) {
    return part.first + (part.product ? 0 : __builtin_amdgcn_readfirstlane(lists.counts[3]));   // behind vm_kernel's
}
__device__ __forceinline__ int vb_count(const vb_part &part, const vb_lists &lists) {
    const int tried = __builtin_amdgcn_readfirstlane(lists.counts[0]), products = __builtin_amdgcn_readfirstlane(lists.counts[3]);
    const int64_t left = (part.product && products < tried ? products : tried) - vb_first(part, lists);
    return left < part.count ? (left < 0 ? 0 : (int)left) : part.count;
}

// How many of `tiles` go through vm_kernel: whole chips of them, and the rest where it is `fewest` or more
__host__ __device__ __forceinline__ int64_t vm_share(int64_t tiles, int64_t chip, int64_t fewest) {
    const int64_t rest = tiles % chip;
    return rest < fewest ? tiles - rest : tiles;
}

// The lists, in two launches (10 us together, where the smallest call takes 730): a wave a tile notes in `left` whether it is tried, and one workgroup deals the tiles out.
__global__ void __launch_bounds__(256)
vb_try_kernel(const float *__restrict__ tiles_in, int64_t n_tiles, int64_t ld, float most, vb_lists lists) {
    const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (tile >= n_tiles) return;
    float v[VT_T / 64];
#pragma unroll
    for (int j = 0; j < VT_T / 64; ++j) v[j] = (float)(f16)tiles_in[vt_pos(tile, 64 * j + lane, ld)];
    bool within = true, varied = false;                        // equal inputs leave every other path a tie
    float wide = 0.0f;
    const float first = __shfl(v[0], 0, GLQH_WAVE);
#pragma unroll
    for (int j = 0; j < VT_T / 64; ++j) {
        within = within && __builtin_fabsf(v[j]) <= VB_X;
        varied = varied || v[j] != first;
        const float past = __builtin_fmaxf(__builtin_fabsf(v[j]) - VB_W, 0.0f);
        wide += past * past;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) wide += __shfl_xor(wide, d, GLQH_WAVE);
    within = __ballot(!within) == 0 && __ballot(varied) != 0 && wide <= most;
    if (lane == 0) lists.left[tile] = within;
}

__global__ void __launch_bounds__(1024)
vb_order_kernel(int n_tiles, int few, int chip, int fewest, vb_lists lists) {
    __shared__ int of_wave[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int tried = 0;
    int next = tid < n_tiles ? lists.left[tid] : 0;
    for (int base = 0; base < n_tiles; base += 1024) {
        const int i = base + tid, mine = next;
        next = i + 1024 < n_tiles ? lists.left[i + 1024] : 0;
        const uint64_t mask = __ballot(mine);
        if (lane == 0) of_wave[wave] = __builtin_popcountll(mask);
        __syncthreads();
        int at = tried + vb_below(mask);
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            at += w < wave ? of_wave[w] : 0;
            tried += of_wave[w];
        }
        if (i < n_tiles) lists.order[mine ? at : n_tiles - 1 - (i - at)] = i;   // i - at: tiles before it that are not tried
        __syncthreads();
    }
    if (tid == 0) {
        tried = tried <= few && tried < n_tiles - tried ? 0 : tried;
        lists.counts[0] = tried;
        lists.counts[1] = 0;
        lists.counts[3] = chip ? vm_share(tried, chip, fewest) : 0;
    }
}

// Before a batch: where more than half of those before it were left, it and the rest are not tried.
__global__ void vb_stop_kernel(vb_part part, vb_lists lists) {
    if (threadIdx.x != 0) return;
    const int64_t first = vb_first(part, lists);
    if (2 * (int64_t)lists.counts[1] > first && lists.counts[0] > first) lists.counts[0] = (int)first;
    lists.counts[2] = lists.counts[1];
}

// Between the passes of a large batch: where the first one left fewer than `worth` of those tried, none of it is tried.  (The exact
// search takes as long over three tiles a CU as the second pass over any number.  Given up at half of a chip, 8192 tiles that are half
// slow ramps took 36.1 ms, not 33, and 4096 that are 70 % ramps 20.7, not 19.)
__global__ void vm_stop_kernel(vb_part part, int worth, vb_lists lists) {
    const int count = vb_count(part, lists);
    if (threadIdx.x != 0 || count == 0 || count - (lists.counts[1] - lists.counts[2]) >= worth) return;
    lists.counts[0] = (int)part.first;
    lists.counts[1] = lists.counts[2];
}

// One forward pass, the rows of every DEPTH-th step to part.rows.  TPW tiles a workgroup: their steps share the table and
// the barriers; workgroups walk the tiles with a fixed stride.
//
// What bounds it is vector issue: 2.5 instructions for two states, 4.4-4.7 clocks each.  A loop of nothing else takes 6.0
// clocks a state, where subtract, multiply, add and half a minimum in fp32 take 14.4 (fma_mix 4.3, the others 2.5); the
// pass over 1024 tiles at K = 4 takes 0.93 ms, of which such loops would be 0.65.
template <int K, int TPW>
__device__ __forceinline__ void vb_forward(const float *__restrict__ tiles_in, int64_t ld, const vb_lists &lists,
                                           const vb_part &part, int worker, int workers, uint32_t *lds) {
    using C = vb_cfg<K>;
    constexpr int THREADS = VB_THREADS;
    const int64_t first = vb_first(part, lists);
    const int count = vb_count(part, lists), pass = part.pass;
    if (count <= 0) return;
    uint16_t *const __restrict__ rows = part.rows;
    vb_tile *const __restrict__ info = part.info;
    constexpr int G = C::G, NK = C::NK, CW = C::CW, D = C::DEPTH, ROWS = C::ROWS;
    // SHARE threads to a predecessor group, UNITS such groups to a thread, LP pairs of their groups
    constexpr int SHARE = K == 4 ? 2 : 1, LOWS = NK / SHARE, LP = LOWS / 2;
    constexpr int UNITS = G / THREADS / LOWS;
    constexpr int ROUND = D > VB_NORM ? D : VB_NORM;
    __shared__ uint32_t xh[TPW][VT_T];                         // inputs, twice each
    __shared__ uint32_t low[TPW][2];                           // the least cost of the last row, of alternate moves
    __shared__ int over[TPW];
    const int tid = threadIdx.x, lane = tid & 63;
    auto row_of = [&](int t, int which) { return lds + (t * ROWS + which) * C::ROW; };
    // This thread's predecessor group and first slot of unit q.  Below K = 4, units 2i and 2i + 1 are predecessors 2j and
    // 2j + 1 of the same groups: their costs go out as one word.
    auto a_of = [&](int q) {
        const int t = tid / SHARE;
        if constexpr (K == 4) return t;
        if constexpr (K == 3) return (t & 127) + 128 * (2 * (t >> 7) + q);
        return t + THREADS * ((q & 4) | (q & 1) << 1 | (q >> 1 & 1));
    };
    const int slot0 = tid % SHARE * LOWS;
    f16x2 w[UNITS * LP * NK];
#pragma unroll
    for (int q = 0; q < UNITS; ++q)
#pragma unroll
        for (int p = 0; p < LP; ++p)
#pragma unroll
            for (int j = 0; j < NK; ++j) {
                const int a = a_of(q);
                const int k = (((j >> 1) ^ vb_word<K>(a)) << 1) + (j & 1);
                const int s = k * G + a * NK;
                f16x2 v = {tr_weight((uint32_t)(s + slot0 + 2 * p)), tr_weight((uint32_t)(s + slot0 + 2 * p + 1))};
                asm volatile("" : "+v"(v));                    // finished here, in the usual rounding
                w[(q * LP + p) * NK + j] = v;
            }
    const int turn = pass ? 0 : VT_T / 2, pairs = (count + TPW - 1) / TPW;
#pragma unroll 1
    for (int pair = worker; pair < pairs; pair += workers) {
        if (tid < TPW) over[tid] = pair * TPW + tid >= count ? -1 : pass ? info[pair * TPW + tid].over : 0;
        {
            const int t = tid >> 8, i = tid & 255;
            if (t < TPW) {
                const bool there = pair * TPW + t < count;
                const f16 v = there ? (f16)tiles_in[vt_pos(lists.order[first + pair * TPW + t], i, ld)] : (f16)0.0f;
                xh[t][i] = vb_bits(f16x2{v, v});
            }
        }
        __syncthreads();
        bool any = false;
#pragma unroll
        for (int t = 0; t < TPW; ++t) any = any || over[t] >= 0;
        if (!any) {
            __syncthreads();
            continue;
        }
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            uint16_t *r = (uint16_t *)row_of(t, 0);
            for (int g = tid; g < G; g += THREADS) r[vb_at<K>(g)] = pass == 0 || g == over[t] ? 0 : 0x7C00;
            if (tid < 2) low[t][tid] = 0xFFFFFFFFu;
        }
        __syncthreads();
        asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 3" ::: "memory");   // fp16 rounds towards zero
        uint32_t xn[TPW];
        float moved[TPW];
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            xn[t] = xh[t][turn];
            moved[t] = 0.0f;
            if (tid == 0 && pair * TPW + t < count) info[pair * TPW + t].pre[0] = 0.0f;
        }
        auto load = [&](int t, int which, uint32_t (&c)[UNITS][CW]) {
#pragma unroll
            for (int q = 0; q < UNITS; ++q) {
                const uint32_t *r = row_of(t, which) + vb_run<K>(a_of(q));
                if constexpr (CW == 2) {
                    const u32x2 v = *(const u32x2 *)r;
                    c[q][0] = v.x; c[q][1] = v.y;
                } else {
#pragma unroll
                    for (int j = 0; j < CW; j += 4) {
                        const u32x4 v = *(const u32x4 *)(r + j);
                        c[q][j] = v.x; c[q][j + 1] = v.y; c[q][j + 2] = v.z; c[q][j + 3] = v.w;
                    }
                }
            }
        };
        auto keep = [&](int t, int level, uint32_t (&c)[UNITS][CW]) {   // the row of a level, as read
            uint16_t *h = rows + ((int64_t)(level - 1) * part.count + pair * TPW + t) * G;
#pragma unroll
            for (int q = 0; q < UNITS; ++q) {
                if constexpr (K == 4) {                        // two threads have read the same: a half each
                    const uint32_t odd = 0u - (tid & 1);
                    u32x4 v;
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = c[q][j] ^ ((c[q][j] ^ c[q][j + 4]) & odd);
                    *(u32x4 *)(h + (uint32_t)(tid * 8)) = v;
                } else if constexpr (K == 3) {
                    *(u32x4 *)(h + (uint32_t)(a_of(q) * NK)) = u32x4{c[q][0], c[q][1], c[q][2], c[q][3]};
                } else {
                    *(u32x2 *)(h + (uint32_t)(a_of(q) * NK)) = u32x2{c[q][0], c[q][1]};
                }
            }
        };
#pragma unroll 1
        for (int i0 = 0; i0 < VT_T; i0 += ROUND)
#pragma unroll
        for (int u = 1; u <= ROUND; ++u) {
            const int i = i0 + u, cur = ROWS == 2 ? (u + 1) & 1 : 0, nxt = ROWS == 2 ? u & 1 : 0;
            const bool move = u % VB_NORM == 0, least = u % VB_NORM == VB_NORM - 1;
            f16x2 x[TPW];
            uint32_t c[TPW][UNITS][CW];
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                if (ROWS == 2) load(t, cur, c[t]);
                x[t] = vb_pair(__builtin_amdgcn_readfirstlane(xn[t]));
                xn[t] = xh[t][(i + turn) & (VT_T - 1)];        // read a step ahead
            }
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                if constexpr (ROWS == 1) {
                    load(t, 0, c[t]);
                    vt_barrier();                              // read by all: the row may change
                }
                f16x2 shift = vb_pair(0);
                if (move) shift = vb_pair(__builtin_amdgcn_readfirstlane(low[t][i / VB_NORM & 1]));
                const bool there = pair * TPW + t < count;
                if ((u - 1) % D == 0 && i > 1 && there) keep(t, (i - 1) / D, c[t]);
                f16x2 least_of = vb_pair(0x7C007C00u), m[2][LP];
#pragma unroll
                for (int q = 0; q < UNITS; ++q) {
                    f16x2(&mq)[LP] = m[q & 1];
#pragma unroll
                    for (int p = 0; p < LP; ++p) {
                        f16x2 e[NK];
#pragma unroll
                        for (int j = 0; j < NK; ++j) {
                            const f16x2 d = w[(q * LP + p) * NK + j] - x[t], cj = vb_pair(c[t][q][j >> 1]);
                            e[j] = __builtin_elementwise_fma(d, d, j & 1 ? f16x2{cj.y, cj.y} : f16x2{cj.x, cj.x});
                        }
                        f16x2 v = e[0];
#pragma unroll
                        for (int j = 1; j + 1 < NK; j += 2)
                            v = __builtin_elementwise_minimum(__builtin_elementwise_minimum(v, e[j]), e[j + 1]);
                        mq[p] = __builtin_elementwise_minimum(v, e[NK - 1]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (move) {
#pragma unroll
                        for (int p = 0; p < LP; ++p) mq[p] -= shift;
                    }
                    if (least) {
#pragma unroll
                        for (int p = 0; p < LP; ++p) least_of = __builtin_elementwise_minimum(least_of, mq[p]);
                    }
                    if constexpr (K == 4) {
                        uint16_t *o = (uint16_t *)row_of(t, nxt) + vb_at<K>((a_of(0) << K) + slot0);
#pragma unroll
                        for (int p = 0; p < LP; ++p) {
                            o[2 * p * NK] = (uint16_t)vb_bits(mq[p]);
                            o[(2 * p + 1) * NK] = (uint16_t)(vb_bits(mq[p]) >> 16);
                        }
                    } else if (q & 1) {
                        uint32_t *o = row_of(t, nxt) + (vb_at<K>((a_of(q - 1) << K) + slot0) >> 1);
#pragma unroll
                        for (int p = 0; p < LP; ++p) {
                            o[2 * p * CW] = vb_bits(f16x2{m[0][p].x, m[1][p].x});
                            o[(2 * p + 1) * CW] = vb_bits(f16x2{m[0][p].y, m[1][p].y});
                        }
                    }
                }
                if (least) {                                   // numbers >= 0 order as their bits
                    least_of = __builtin_elementwise_minimum(least_of, f16x2{least_of.y, least_of.x});
                    const uint32_t v = vb_wave_min(vb_bits(least_of));
                    if (lane == 0) atomicMin(&low[t][(i + 1) / VB_NORM & 1], v);
                    if (tid == 0 && i > VB_NORM) low[t][i / VB_NORM & 1] = 0xFFFFFFFFu;   // the word of the move before
                }
                if (move && tid == 0 && there) {
                    moved[t] += (float)shift.x;
                    info[pair * TPW + t].pre[i / VB_NORM] = moved[t];
                }
            }
            if (ROWS == 2) vt_barrier();
        }
        vt_barrier();
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            uint32_t c[UNITS][CW];
            load(t, 0, c);
            if (pair * TPW + t < count) keep(t, C::STORED, c);
        }
        asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 0" ::: "memory");
        __syncthreads();
    }
}

// ---- the forward pass on the matrix cores (K = 4, chips full of tiles) ---------------------
// w^2 - 2xw + c is a product of matrices: rows are states, with w, w^2 and a one, columns are tiles, with -2x, a one and c.
// w and x are fp16 numbers, w^2 two of them (rounded, and what that left), c the bound of the predecessor's group as it is
// stored: the products are exact, and the sums are fp32.  A v_mfma_f32_32x32x16_f16 costs 1024 states in 32 clocks, where
// vb_forward's two packed instructions take 75, and leaves the vector units the minima, three numbers to an instruction, and
// x^2 and what moves into B once to a minimum.
//
// Operands.  Of the sixteen numbers of a row a product needs three and the one: a lane's eight hold two states each (its
// halves of tw, of their squares and of what those lack), and lanes 32-63 two more; columns are sixteen tiles, twice, and
// pick by their zeros: the first product of a pair takes the states of lanes 0-31 (their first halves in columns 0-15, their
// second ones in 16-31), the second product those of lanes 32-63.  The ones meet the bounds in lanes 0-31 only, whose rows
// 0-15 and 16-31 are two neighbouring predecessor groups a, in the order of their low digits, at one high digit k; bounds of
// two such groups lie in one word.  So a pair of products costs the states of 4 predecessor groups at 2 high digits, eight
// pairs are all 16 digits (a unit), and the minimum over them stays in its lane.
//
// A workgroup has sixteen tiles, a CU to itself: one row of bounds, 128 KB, is read by all and written by all in turn, and
// eight waves have eight units each, with their table in 64 registers and the new bounds, until all have read, in 64 more.
//
// Rounding.  A sum is off by at most VM_OFF times its terms' magnitudes (measured, not derived: 2.6 * 2^-24 is the most that 3 * 10^7 sums
// of such terms showed, and a rounding follows; the rows that come of it are held to costs in 64 bits, group by group); with e the state's cost those are at most (2 |x| + sqrt e)^2 <= 5 x^2 + 5 e, and c, and
// what moves, which is no more than c.  So 5 VM_OFF x^2 comes off every step's bounds, with what w^2 may lack below fp16's
// smallest numbers, and VM_LESS of c + e.  Bounds are rounded once a step, towards zero; a row's least one stays at VM_FLOOR,
// above what comes off until the next move, so that none is negative.
//
// 4096 tiles, a pass: 2.6 ms, where vb_forward takes 3.7, and 0.6 for the walk back, which nothing overlaps.  Vector ALUs issue
// in 62 % of the cycles (three quarters of that the minima) and the matrix cores work in 38 %, at 2.1 GHz; the rows on their
// way to memory take 0.4 ms of it.  Measured and not kept: products a pair ahead of the minima (2.6, with the rows in one
// piece; no registers for more), four waves a SIMD (eight tiles a workgroup, 128 registers: 3.4), eight tiles and two rows
// (2.8), priorities of waves (level).
constexpr int VM_TILES = 16, VM_THREADS = 512;
constexpr float VM_OFF = 6 * 0x1p-24f, VM_LESS = 0x1p-19f, VM_FLOOR = 0x1p-9f;
static_assert(5 * VM_OFF < VM_LESS && VB_NORM * 2 * 5 * VM_OFF * VB_X * VB_X < 0.99f * VM_FLOOR, "all of a sum; no bound is negative");
constexpr int VM_ROW = 2048 * VM_TILES, VM_LDS = (VM_ROW + VT_T * VM_TILES) * 4;   // words of the row; bytes

template <int N, int END, typename F>
__device__ __forceinline__ void vm_unroll(const F &f) {        // f(0), f(1), ... for more than a pragma unrolls
    if constexpr (N < END) {
        f(std::integral_constant<int, N>());
        vm_unroll<N + 1, END>(f);
    }
}
__device__ __forceinline__ float vm_loss(float x) { return 5 * VM_OFF * x * x + 0x1p-24f; }

// Word of the bounds of groups k * 256 + 2p and + 1 (p < 128), tile t.  A product's lanes read 16 tiles at one or two p, what goes
// to memory is 32 p at two k of one tile: the exclusive-or keeps both on different banks.
__device__ __forceinline__ int vm_word(int k, int p, int t) { return (k * 128 + p) * VM_TILES + (t ^ ((p >> 2 & 7) | (k >> 3) << 3)); }

__global__ void __launch_bounds__(VM_THREADS, 2)
vm_kernel(const float *__restrict__ tiles_in, int64_t ld, vb_lists lists, vb_part part) {
    using C = vb_cfg<4>;
    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
    typedef float f32x16 __attribute__((ext_vector_type(16)));
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    uint32_t *const xs = lds + VM_ROW;                         // inputs [step][tile], twice each
    __shared__ uint32_t low[2][VM_TILES];                      // the least bound of the last row, of alternate moves
    __shared__ int over[VM_TILES];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, t = lane & 15, second = lane >> 4 & 1;
    const int first = blockIdx.x * VM_TILES, count = vb_count(part, lists) - first;
    if (count <= 0) return;
    if (tid < VM_TILES) over[tid] = tid < count && part.pass ? part.info[first + tid].over : -1;
    if (tid < 2 * VM_TILES) low[tid >> 4][tid & 15] = 0xFFFFFFFFu;
    for (int i = tid; i < VT_T * VM_TILES; i += VM_THREADS) {
        const int to = i >> 8, step = i & 255;
        const f16 v = to < count ? (f16)tiles_in[vt_pos(lists.order[part.first + first + to], step, ld)] : (f16)0.0f;
        xs[step * VM_TILES + to] = vb_bits(f16x2{v, v});
    }
    __syncthreads();
    for (int i = tid; i < VM_ROW; i += VM_THREADS) {           // step 0: the group that the overlap names, or all
        const int to = i & 15, p = i >> 4 & 127, k = i >> 11, g = over[to] - k * 256 - 2 * p;
        const f16 in = (f16)VM_FLOOR, out = (f16)30000.0f;     // (far above any that matters, and finite: zeros meet it)
        lds[vm_word(k, p, to)] = part.pass ? vb_bits(f16x2{g == 0 ? in : out, g == 1 ? in : out}) : vb_bits(f16x2{in, in});
    }
    uint32_t tw[8][8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t s = (uint32_t)((2 * j + half) * C::G + (4 * (8 * wave + u) + second) * C::NK + t);
            tw[u][j] = vb_bits(f16x2{tr_weight(s), tr_weight(s + 2 * C::NK)});
            asm volatile("" : "+v"(tw[u][j]));                 // finished here
        }
    // the operands' fixed parts, kept apart from what changes
    const uint32_t pick = second ? 0xFFFF0000u : 0x0000FFFFu, one = 0x3C003C00u & pick;
    const uint32_t pick1 = half ? 0 : pick, pick2 = half ? pick : 0;
    u32x4 a = {0, 0, 0, half ? 0u : second ? 0x3C000000u : 0x00003C00u}, b1[2], b2[2];
    asm volatile("" : "+v"(a));
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        b1[n] = half ? u32x4{0, 0, 0, 0} : u32x4{0, one, one, 0};
        b2[n] = half ? u32x4{0, one, one, 0} : u32x4{0, 0, 0, 0};
        asm volatile("" : "+v"(b1[n]), "+v"(b2[n]));
    }
    const int read0 = (16 * wave + second) * VM_TILES * 4 + ((t ^ (wave & 1) << 2) << 2);
    const int write0 = (2 * wave * 128 + 16 * second + 2 * half) * VM_TILES * 4 + ((t ^ second << 2 ^ (wave >> 2) << 3) << 2);
    char *const row = (char *)lds;
    const int turn = part.pass ? 0 : VT_T / 2;
    float moved = -VM_FLOOR;
    if (tid < VM_TILES && tid < count) part.info[first + tid].pre[0] = 0.0f;
    __syncthreads();

    // An eighth of what a wave writes of a level's row: 32 words p at eight of the digits, of one of its two tiles
    const int high = lane & 1;
    auto fetch = [&](int q, u32x4 (&v)[2]) __attribute__((always_inline)) {
        const int to = 2 * wave + (q >> 2), p = 32 * (q & 3) + (lane >> 1), w = p >> 4 & 7;
        const int from = vm_word(8 * high, p, to) * 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            typedef __attribute__((address_space(3))) const uint32_t lds_word;
            __attribute__((address_space(3))) const char *at = (__attribute__((address_space(3))) const char *)row + (from + ((j ^ (w & 3)) << 14));
            v[0][j] = *(lds_word *)at;
            v[1][j] = *(lds_word *)(at + 8192);
        }
    };
    auto keep = [&](int level, int q, const u32x4 (&v)[2]) __attribute__((always_inline)) {
        const int to = 2 * wave + (q >> 2), p = 32 * (q & 3) + (lane >> 1), w = p >> 4 & 7;
        uint16_t *o = part.rows + ((int64_t)(level - 1) * part.count + first + to) * C::G + vb_together<4>(2 * p * C::NK) + 8 * (high ^ w >> 2);
        u32x4 even, odd;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            even[j] = __builtin_amdgcn_perm(v[1][j], v[0][j], 0x05040100u);
            odd[j] = __builtin_amdgcn_perm(v[1][j], v[0][j], 0x07060302u);
        }
        if (to < count) {
            *(u32x4 *)o = even;
            *(u32x4 *)(o + vb_together<4>(C::NK)) = odd;
        }
    };
    uint32_t next = xs[turn * VM_TILES + t];
#pragma unroll 1
    for (int i = 1; i <= VT_T; ++i) {
        const bool move = i % VB_NORM == 0;
        const uint32_t xh = next;
        next = xs[((i + turn) & (VT_T - 1)) * VM_TILES + t];   // read a step ahead
        const float x = vb_half(xh & 0xFFFFu);
        float shift = 0.0f;
        if (move) {
            shift = vb_half(low[i / VB_NORM & 1][t] & 0xFFFFu) - VM_FLOOR;
            moved += shift;
            if (tid < VM_TILES && tid < count) part.info[first + tid].pre[i / VB_NORM] = moved;
        }
        const bool store = !move && i > 1;                     // the row that this step reads
        const float add = x * x * (1 - VM_LESS) - shift - vm_loss(x);
        const uint32_t twice = vb_bits(vb_pair(xh) * f16x2{(f16)-2.0f, (f16)-2.0f});
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            b1[n].x = twice & pick1;
            b2[n].x = twice & pick2;
        }
        f32x16 least;
        u32x4 kept[2];
        int at[2];
        uint32_t out[8][8];
        auto ask = [&](int n) {                                // the bounds of pair n
            const int u = n >> 3, k = 2 * (n & 7);
            if ((n & 15) == 0) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    at[q] = (read0 ^ ((u >> 1 | q << 3) << 2)) + q * 65536;
                    asm volatile("" : "+v"(at[q]));            // addresses of their own would all be kept
                }
            }
            typedef __attribute__((address_space(3))) const volatile char lds_byte;   // volatile: into the operand, not two at once and moved
            typedef __attribute__((address_space(3))) const volatile uint32_t lds_word;
            lds_byte *from = (lds_byte *)row + at[k >> 3] + ((k & 7) * 8192 + u * 128);
            b1[n & 1].w = *(lds_word *)from;
            b2[n & 1].w = *(lds_word *)(from + 8192);
        };
        ask(0);
        ask(1);
        vm_unroll<0, 64>([&](auto at_n) __attribute__((always_inline)) {
            constexpr int n = decltype(at_n)::value;
            u32x4 &p1 = b1[n & 1], &p2 = b2[n & 1];
            if (n % 8 == 0 && store) fetch(n >> 3, kept);
            if (n % 8 == 4 && store) keep((i - 1) / C::DEPTH, n >> 3, kept);
            a.x = tw[n >> 3][n & 7];
            asm volatile("" : "+v"(a.x));                      // or the squares of all would be kept, for which there is no room
            const f16x2 w = vb_pair(a.x), sq = w * w;
            a.y = vb_bits(sq);
            a.z = vb_bits(__builtin_elementwise_fma(w, w, -sq));
            const f32x16 d1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, p1), f32x16{}, 0, 0, 0);
            const f32x16 d2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, p2), f32x16{}, 0, 0, 0);
            asm("" : "+v"(a), "+v"(p1), "+v"(p2));             // changed in place
            if (n + 2 < 64) ask(n + 2);
#pragma unroll
            for (int r = 0; r < 16; ++r)
                least[r] = n % 8 == 0 ? __builtin_elementwise_minimum(d1[r], d2[r])
                                      : __builtin_elementwise_minimum(__builtin_elementwise_minimum(least[r], d1[r]), d2[r]);
            if (n % 8 == 3) asm volatile("" : "+v"(least));    // here, and not behind the branch
            if (n % 8 == 7) {
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    out[n >> 3][r] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(__builtin_fmaf(least[2 * r], 1 - VM_LESS, add),
                                                                                                      __builtin_fmaf(least[2 * r + 1], 1 - VM_LESS, add)));
                    asm volatile("" : "+v"(out[n >> 3][r]));   // now, and not where it is written: there is no room for the products
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        vt_barrier();                                          // read by all
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int r = 0; r < 8; ++r)
                *(uint32_t *)(row + (write0 ^ (r >> 1) << 2) + (u >> 2) * 8192 + (u & 3) * 2048 + (r >> 1) * 256 + (r & 1) * 64) = out[u][r];
        if (!move) {                                           // numbers >= 0 order as their bits
            f16x2 v = vb_pair(0x7C007C00u);
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int r = 0; r < 8; r += 2)
                    v = __builtin_elementwise_minimum(__builtin_elementwise_minimum(v, vb_pair(out[u][r])), vb_pair(out[u][r + 1]));
            v = __builtin_elementwise_minimum(v, f16x2{v.y, v.x});
            atomicMin(&low[(i + 1) / VB_NORM & 1][t], vb_bits(v) & 0xFFFFu);
            if (tid < VM_TILES && i > VB_NORM) low[i / VB_NORM & 1][tid] = 0xFFFFFFFFu;   // the word of the move before
        }
        vt_barrier();
    }
#pragma unroll 1
    for (int q = 0; q < 8; ++q) {
        u32x4 v[2];
        fetch(q, v);
        keep(C::STORED, q, v);
    }
}

// A tile's working memory in LDS during the backtrack.  Level l is step l * DEPTH; its entries are the
// kept ways from the groups of level l (parents: where the states lead) to those of level l - 1 (children).
template <bool PRODUCT>
struct vb_pool {
    // 550 at most in 3 * 10^4 tiles of Gaussian values, 170 on average; behind vm_kernel what lets sixteen walk on a CU.  (672 behind
    // vb_kernel too: of 2048 tiles of sigma 0.0001 891 left, not 657, 9.8 ms, not 8.9; of 0.001 368, not 133.)
    static constexpr int ENTRIES = PRODUCT ? 672 : 768;
    float cost[ENTRIES];                   // of the entries: to the end
    uint16_t entry[ENTRIES];               // the digits of its states, nearest step first | parent << 8
    uint16_t via[ENTRIES];                 // of child j at j: best entry | its parent << 8 | close second << 14
    uint16_t group[ENTRIES];               // the groups of level l at groups[l]
    uint8_t child[ENTRIES];
    uint16_t at[VT_T / 2 + 2], groups[VT_T / 2 + 2];   // entries of level l: at[l] .. at[l-1]
    float best[VB_MOST];
    int kept[VB_MOST];
};
static_assert(vb_pool<true>::ENTRIES >= VB_MOST, "a level fits");
// states from group g by the digits p, nearest step first
template <int K>
__device__ __forceinline__ void vb_walk(int g, int p, int (&st)[vb_cfg<K>::DEPTH]) {
    using C = vb_cfg<K>;
    int at = g;
#pragma unroll
    for (int e = 0; e < C::DEPTH; ++e) {
        st[e] = ((p >> (K * (C::DEPTH - 1 - e))) & (C::NK - 1)) * C::G + at;
        at = st[e] >> K;
    }
}

// The backtrack of one tile by one wave: true, and the states in `states`; or false, and `limit` the one to try next,
// infinity where the tile has to be searched exactly.
// n, gv: the groups of step T (a lane each) whose bounds are within `limit`; x[i]: input of step i; the bounds' row of
// level l at hist + (l - 1) * step; pre[j]: B at step j * VB_NORM; tie: the only group of step 0, or -1; the states up to
// step `upto` are wanted.
template <int K, bool PRODUCT>
__device__ __forceinline__ bool vb_trace(int n, int gv, float &limit, const f16 *x, const uint16_t *__restrict__ hist,
                                         int64_t step, const float *pre, int tie, int upto, vb_pool<PRODUCT> *P, uint16_t *states) {
    using C = vb_cfg<K>;
    constexpr int D = C::DEPTH, LEVELS = C::STORED, R = (1 << (K * D)) / 64;
    const int lane = threadIdx.x & 63;
    const float close = limit * VB_NEAR, inf = __builtin_inff();
    float cv = 0.0f;                                           // lane j: cost from group gv of this level to the end
    int ne = 0, ns = 0;
    bool full = false, empty = false;
    typedef f16 inputs __attribute__((ext_vector_type(D)));
    inputs xn = *(const inputs *)(x + VT_T - D);               // read a level ahead
    float pn = pre[(LEVELS - 1) * D / VB_NORM];
    // The ways from a group, R to a lane, by where their bounds lie: digits of a lane's ways, and the first one's place.
    constexpr int E = 16 - K - K * D;                          // what of the group is left above the digits
    int ways[R], place;
    {
        const int run = K == 4 ? lane >> 2 : K == 3 ? lane >> 3 : lane;   // the digits but the farthest, the nearest lowest
        const int in = K == 4 ? (lane & 3) * 4 : K == 3 ? lane & 7 : 0;
        place = (run << (PRODUCT ? K : E + K)) + in;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int k = in + r;
            k ^= vb_word<K>(run << E) << 1;
            ways[r] = K == 2 ? (run & 3) << 6 | (run >> 2 & 3) << 4 | run >> 4 << 2 | k : run << K | k;
        }
    }
    // their bounds, in the row below level l (of level 1, whose row is not stored, any row); requested as soon as a level's
    // first group is known: they take longer than everything else here
    u32x2 ahead = {0, 0};
    auto ask = [&](int l, int g, u32x2 &into) {
        const uint16_t *row = hist + (l > 1 ? l - 2 : 0) * step + place + (uint32_t)((g >> (K * D)) << (PRODUCT ? K * D : K));
        if constexpr (R == 4) into = *(const u32x2 *)row;
        else into.x = *row;
    };
    auto bound_of = [&](u32x2 v, int r) { return vb_half((r & 2 ? v.y : v.x) >> (16 * (r & 1)) & 0xFFFFu); };
    // of the ways from group g, c0 from the end: the groups they come from, their costs, the lanes of those within the limit
    float xs[D], room;
    auto look = [&](int l, int g, float c0, u32x2 bounds, int (&front)[R], float (&c)[R], uint64_t (&mask)[R]) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int st[D];
            vb_walk<K>(g, ways[r], st);
            front[r] = st[D - 1] >> K;
            c[r] = c0;
#pragma unroll
            for (int e = 0; e < D; ++e) c[r] += vt_err(st[e], xs[e]);
        }
        if (l == 1) {                                          // from the start, or from its only group
            auto start = [&](int r) { return tie < 0 || front[r] == tie ? 0u : 0x7C00u; };
            bounds.x = start(0) | (R > 1 ? start(R > 1 ? 1 : 0) << 16 : 0u);
            if constexpr (R == 4) bounds.y = start(2) | start(3) << 16;
        }
        int count = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            mask[r] = __ballot(c[r] + bound_of(bounds, r) <= room);
            count += __builtin_popcountll(mask[r]);
        }
        return count;
    };
    ask(LEVELS, vb_lane(gv, 0), ahead);
#pragma unroll 1
    for (int l = LEVELS; l > 0; --l) {
        full = ns + n > P->ENTRIES;
        if (full) break;
        room = limit - pn;
#pragma unroll
        for (int e = 0; e < D; ++e) xs[e] = (float)xn[D - 1 - e];
        xn = *(const inputs *)(x + ((l - 2) * D & (VT_T - 1)));
        pn = pre[(l > 1 ? l - 2 : 0) * D / VB_NORM];
        int front[R];
        float c[R];
        uint64_t mask[R];
        if (n == 1) {                                          // one group: its ways lead to different ones
            const int g = vb_lane(gv, 0), m = look(l, g, vb_lane(cv, 0), ahead, front, c, mask);
            full = ne + m > P->ENTRIES || m > VB_MOST;
            empty = m == 0;
            if (full || empty) break;
            int cs = __builtin_bit_cast(int, c[R - 1]), ws = ways[R - 1];   // a lane's first way in reach
            uint64_t first = mask[R - 1];
#pragma unroll
            for (int r = R - 2; r >= 0; --r) {
                const bool in = mask[r] >> lane & 1;
                cs = in ? __builtin_bit_cast(int, c[r]) : cs;
                ws = in ? ways[r] : ws;
                first = mask[r] ? mask[r] : first;
            }
            const int from = __builtin_ctzll(first), way = vb_lane(ws, from);
            int st[D];
            vb_walk<K>(g, way, st);
            ask(l - 1, st[D - 1] >> K, ahead);
            if (lane == 0) {
                P->at[l] = (uint16_t)ne;
                P->groups[l] = (uint16_t)ns;
                P->group[ns] = (uint16_t)g;
            }
            if (m == 1) {                                      // three levels in four
                gv = st[D - 1] >> K;
                cv = __builtin_bit_cast(float, vb_lane(cs, from));
                if (lane == 0) {
                    P->entry[ne] = (uint16_t)way;
                    P->cost[ne] = cv;
                    P->child[ne] = 0;
                    P->via[ne] = 0;
                }
            } else {
                int k = 0;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int to = k + vb_below(mask[r]);
                    if (mask[r] >> lane & 1) {
                        P->entry[ne + to] = (uint16_t)ways[r];
                        P->kept[to] = front[r];
                        P->cost[ne + to] = c[r];
                    }
                    k += __builtin_popcountll(mask[r]);
                }
                __builtin_amdgcn_wave_barrier();
                gv = P->kept[lane];
                cv = P->cost[ne + (lane < m ? lane : 0)];
                if (lane < m) {
                    P->child[ne + lane] = (uint8_t)lane;
                    P->via[ne + lane] = (uint16_t)lane;
                }
                __builtin_amdgcn_wave_barrier();
            }
            ns += 1;
            ne += m;
            n = m;
            continue;
        }
        if (lane == 0) {
            P->at[l] = (uint16_t)ne;
            P->groups[l] = (uint16_t)ns;
        }
        if (lane < n) P->group[ns + lane] = (uint16_t)gv;
        ns += n;
        // lane j: child j, its cheapest entry, and the next one's cost
        int m = 0, nn = 0, ng = -1, nvia = lane;
        float nc = inf, second = inf;
#pragma unroll 1
        for (int j = 0; j < n; ++j) {
            const u32x2 bounds = ahead;
            if (j + 1 < n) ask(l, vb_lane(gv, j + 1), ahead);  // one group ahead, too
            const int count = look(l, vb_lane(gv, j), vb_lane(cv, j), bounds, front, c, mask);
            full = m + count > 256 || ne + m + count > P->ENTRIES;
            if (full) break;
            int k = m;                                         // one entry after the other, in registers: there are a few
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (mask[r] >> lane & 1) {
                    const int to = ne + k + vb_below(mask[r]);
                    P->entry[to] = (uint16_t)(ways[r] | j << 8);
                    P->cost[to] = c[r];
                }
#pragma unroll 1
                for (uint64_t rest = mask[r]; rest; rest &= rest - 1, ++k) {
                    const int from = __builtin_ctzll(rest), f = vb_lane(front[r], from);
                    const float cf = vb_lane(c[r], from);
                    const uint64_t same = __ballot(ng == f);
                    const int child = same ? __builtin_ctzll(same) : nn;
                    nn = __builtin_amdgcn_readfirstlane(nn + (same ? 0 : 1));
                    P->child[ne + k] = (uint8_t)child;
                    const bool mine = lane == child, better = mine && cf < nc;
                    const float other = __builtin_fmaxf(nc, cf);   // the new one's or, where that is better, the old one's
                    second = mine && other < second ? other : second;
                    nvia = better ? k | j << 8 : nvia;
                    nc = better ? cf : nc;
                    ng = mine ? f : ng;
                }
            }
            m += count;
        }
        full = full || nn > VB_MOST;
        empty = m == 0;
        if (full || empty) break;
        ask(l - 1, vb_lane(ng, 0) & (C::G - 1), ahead);
        if (lane < nn) P->via[ne + lane] = (uint16_t)(nvia | (second - nc <= close ? 1 << 14 : 0));
        ne += m;
        n = nn;
        gv = ng & (C::G - 1);
        cv = nc;
    }
    if (full || empty) {
        limit = full ? inf : limit * (1.0f + 0.5f * C::SLACK);
        return false;
    }
    if (lane == 0) P->at[0] = (uint16_t)ne;
    float u = inf, second = inf;
    int take = 0;
#pragma unroll 1
    for (int q = 0; q < n; ++q) {
        const float cq = vb_lane(cv, q);
        take = cq < u ? q : take;
        second = __builtin_fminf(second, __builtin_fmaxf(u, cq));
        u = __builtin_fminf(u, cq);
    }
    if (!(u * (1.0f + VB_NEAR) <= limit)) {
        limit = vb_lane(u * (1.0f + 2 * VB_NEAR), 0);
        return false;
    }
    // the cheapest path, from the start; where no other one is close to it, it is the answer
    bool near = second - u <= close;
    __builtin_amdgcn_wave_barrier();
#pragma unroll 1
    for (int l0 = 0; l0 * D <= upto; l0 += 64) {
        const int ats = P->at[l0 + 1 + lane], gs = P->groups[l0 + 1 + lane];
        int mine = 0;                                          // lane k: the path's way from level l0 + k to the next
#pragma unroll 1
        for (int k = 0; k < 64 && (l0 + k) * D <= upto; ++k) {
            const int v = __builtin_amdgcn_readfirstlane(P->via[vb_lane(ats, k) + take]);
            mine = lane == k ? v : mine;
            near = near || (v >> 14);
            take = v >> 8 & 63;
        }
        if ((l0 + lane) * D <= upto) {
            int st[D];
            vb_walk<K>(P->group[gs + (mine >> 8 & 63)], P->entry[ats + (mine & 255)] & 255, st);
#pragma unroll
            for (int e = 0; e < D; ++e) states[(l0 + lane + 1) * D - 1 - e] = (uint16_t)st[e];
        }
    }
    if (!near) return true;

    // exact costs, forward over the kept ways that a path close to the cheapest may take; lane e: entry e of the level,
    // best, cheap: exact cost from the start, cost to the end, of group `lane` of the level below
    // (what of a level is known beforehand is read a level ahead: trips to LDS, each behind the last, were half of its time)
    struct level_data {
        int m, nb, parent, child, way, group;
        float cost, cheap;                                     // of the entry; of group `lane` of the level above
    };
    auto read = [&](int l) {
        level_data L;
        const int eb = P->at[l];
        L.m = (int)P->at[l - 1] - eb, L.nb = P->at[l < LEVELS ? l + 1 : l];
        const int e = eb + (lane < L.m ? lane : 0), en = P->entry[e];
        L.parent = en >> 8, L.way = en & 255, L.child = P->child[e], L.cost = P->cost[e];
        L.group = P->group[P->groups[l] + L.parent];
        L.cheap = P->cost[L.nb + (P->via[L.nb + lane] & 255)];
        return L;
    };
    float cheap = P->cost[P->at[1] + (P->via[P->at[1] + lane] & 255)];
    float best = lane < n && cheap <= u + close ? 0.0f : inf;
    level_data next = read(1);
#pragma unroll 1
    for (int l = 1; l <= LEVELS; ++l) {
        const level_data L = next;
        next = read(l < LEVELS ? l + 1 : l);
        const int m = __builtin_amdgcn_readfirstlane(L.m), nb = L.nb, parent = L.parent;
        if (m > 64) {
            limit = inf;
            return false;
        }
        int st[D];
        vb_walk<K>(L.group, L.way, st);
        float v[D], c = __shfl(best, L.child, GLQH_WAVE);
        const float room = __shfl(cheap, L.child, GLQH_WAVE) + close;
        const uint64_t live = __ballot(lane < m && c < inf && L.cost <= room);
        const inputs xl = *(const inputs *)(x + (l - 1) * D);
#pragma unroll
        for (int d = D - 1; d >= 0; --d) {
            c = vt_err(st[d], (float)xl[D - 1 - d]) + c;
            v[d] = c;
        }
        bool least = live >> lane & 1;     // of its parent (at the end: of all): the lowest cost, then the lowest state, step by step
#pragma unroll 1
        for (uint64_t rest = live & (live - 1) ? live : 0; rest; rest &= rest - 1) {
            const int q = __builtin_ctzll(rest);
            bool under = false, level = l == LEVELS || vb_lane(parent, q) == parent;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const float vq = vb_lane(v[d], q);
                const int sq = vb_lane(st[d], q);
                under = under || (level && (vq < v[d] || (vq == v[d] && sq < st[d])));
                level = level && vq == v[d] && sq == st[d];
            }
            least = least && !under;
        }
        const uint64_t won = __ballot(least);
        if (l == LEVELS) {
            take = __builtin_ctzll(won);
            break;
        }
        cheap = L.cheap;
        if ((won & (won - 1)) == 0) {
            const int q = __builtin_ctzll(won);
            best = lane == vb_lane(parent, q) ? vb_lane(v[0], q) : inf;
        } else {
            P->best[lane] = inf;
            __builtin_amdgcn_wave_barrier();
            if (least) P->best[parent] = v[0];
            __builtin_amdgcn_wave_barrier();
            best = P->best[lane];
        }
        __builtin_amdgcn_wave_barrier();
        if (least) P->via[nb + parent] = (uint16_t)lane;       // now: the entry that the group's exact cost comes from
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll 1
    for (int l0 = LEVELS; l0 > 0; l0 -= 64) {
        const int ats = P->at[l0 - lane], gs = P->groups[l0 - lane];
        int mine = 0;                                          // lane k: the path's entry of level l0 - k
#pragma unroll 1
        for (int k = 0; k < 64; ++k) {
            mine = lane == k ? take : mine;
            const int at = vb_lane(ats, k);
            if (l0 - k > 1) take = __builtin_amdgcn_readfirstlane(P->via[at + P->child[at + take]]);
        }
        const int en = P->entry[ats + mine];
        int st[D];
        vb_walk<K>(P->group[gs + (en >> 8)], en & 255, st);
#pragma unroll
        for (int e = 0; e < D; ++e) states[(l0 - lane) * D - 1 - e] = (uint16_t)st[e];
    }
    return true;
}

// A wave's memory while it walks back
template <bool PRODUCT>
struct vb_work {
    vb_pool<PRODUCT> pool;
    float pre[VT_T / VB_NORM + 1];
    alignas(8) f16 x[VT_T];
    uint16_t states[VT_T];
    int start[VB_MOST];
};
static_assert(sizeof(vb_work<true>) <= 160 * 1024 / 16, "sixteen on a CU");

// The backtrack of tile vb_first + at (one wave): after pass 0 the overlap, after pass 1 the states and values.
// What bounds it is latency: a chain of STORED levels, each a look into a row of which only the last level's group tells
// where (a microsecond), some 150 instructions and trips to LDS.  150 us on average, 340 for the slowest of 256 tiles.
// Sixteen waves a CU over 4096 tiles of vm_kernel: 0.19 ms on average, 0.46 for the slowest tile, which is what the launch takes (four ways
// a level, and another near).  0.73 -> 0.58 by the kept groups' bounds in one piece, a short way where one way is in reach, and
// the exact comparison's levels read ahead and its path found by the lanes.  (Two groups at a time, or the next level's
// first two asked for: 0.69, in spilled scalar registers; a loop of its own for levels of one way: level.)
template <int K, bool PRODUCT>
__device__ __forceinline__ void vb_backtrack(const float *__restrict__ tiles_in, int64_t ld, const vb_lists &lists,
                                             const vb_part &part, int at, vb_work<PRODUCT> *W, int32_t *__restrict__ states_out, float *__restrict__ hat_out) {
    using C = vb_cfg<K>;
    float *const pre = W->pre;
    f16 *const x = W->x;
    uint16_t *const states = W->states;
    int *const start = W->start;
    const int lane = threadIdx.x & 63, pass = part.pass;
    const int64_t tile = __builtin_amdgcn_readfirstlane(lists.order[vb_first(part, lists) + at]);
    vb_tile *const mine = part.info + at;
    const int over = pass ? __builtin_amdgcn_readfirstlane(mine->over) : 0;
    if ((uint32_t)over >= (uint32_t)C::G) return;              // left after the first pass
    const int turn = pass ? 0 : VT_T / 2, tie = pass ? over : -1;
    float lost = 0.0f;                                         // off the bounds, beside their roundings
    for (int i = lane; i < VT_T; i += 64) {
        x[i] = (f16)tiles_in[vt_pos(tile, (i + turn) & (VT_T - 1), ld)];
        lost += vm_loss((float)x[i]);
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) lost += __shfl_xor(lost, d, GLQH_WAVE);
    lost = PRODUCT ? VT_T * VM_FLOOR * 0x1p-10f + lost : VB_LOST;   // (2^-10: a rounding of the least bounds)
    for (int i = lane; i <= VT_T / VB_NORM; i += 64) pre[i] = mine->pre[i];
    const int64_t step = (int64_t)part.count * C::G;
    const uint16_t *hist = part.rows + (int64_t)at * C::G, *last = hist + (C::STORED - 1) * step;
    __builtin_amdgcn_wave_barrier();
    const float bt = pre[VT_T / VB_NORM];
    uint32_t lo = 0xFFFFu;                                     // the least bound of the groups that may be last
    if (pass) {
        lo = last[PRODUCT ? vb_together<K>(vb_stored<K>(tie)) : vb_stored<K>(tie)];
    } else {
#pragma unroll 8
        for (int g = 0; g < C::G; g += 64) {
            const uint32_t v = last[g + lane];
            lo = v < lo ? v : lo;
        }
        lo = vb_wave_min(lo);
    }
    const float least = vb_lane(vb_half(lo) + bt, 0);
    float limit = vb_lane(least * (1.0f + C::SLACK) + lost, 0);
    // behind vb_kernel a second walk takes longer than the exact search over what it saves, a tile a CU at a time (K = 2, 1024 slow ramps 5.2 ->
    // 7.1 ms with it; K = 3, 4096 tiles of sigma 2.0 12.7 -> 13.0; K = 4, 1024 of 1.5 3.8 -> 4.4, though 3000 of 1.7 10.4 -> 9.6)
    float lower = PRODUCT ? limit - 0.5f * (limit - least) : __builtin_inff();
    bool good = false;
#pragma unroll 1
    for (int tries = 0; tries < 4; ++tries) {
        int n = pass;                                          // the groups of step T within the limit
        if (pass) {
            if (lane == 0) start[0] = tie;
        } else {
#pragma unroll 1
            for (int g0 = 0; g0 < C::G; g0 += 512) {
                float b[8], least = __builtin_inff();
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    b[k] = vb_half(last[g0 + 64 * k + lane]) + bt;
                    least = __builtin_fminf(least, b[k]);
                }
                if (!__ballot(least <= limit)) continue;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const uint64_t mask = __ballot(b[k] <= limit);
                    const int at = n + vb_below(mask);
                    if (b[k] <= limit && at < VB_MOST) start[at] = vb_group<K>(PRODUCT ? vb_apart<K>(g0 + 64 * k + lane) : g0 + 64 * k + lane);
                    n += __builtin_popcountll(mask);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
        n = __builtin_amdgcn_readfirstlane(n);
        if (n > VB_MOST) limit = __builtin_inff();
        else good = vb_trace<K, PRODUCT>(n, lane < n ? start[lane] : 0, limit, x, hist, step, pre, tie, pass ? VT_T - 1 : VT_T / 2, &W->pool, states);
        if (good) break;
        if (limit == __builtin_inff()) {                       // too many ways for the lists: half the slack may do
            limit = lower;
            lower = __builtin_inff();
        }
        if (limit == __builtin_inff()) break;
        __builtin_amdgcn_wave_barrier();
    }
    __builtin_amdgcn_wave_barrier();
    if (!good && lane == 0) lists.left[atomicAdd(lists.counts + 1, 1)] = (int)tile;
    if (pass == 0 && lane == 0) mine->over = good ? states[VT_T / 2] >> K : -1;
    if (pass == 0 || !good) return;
    for (int i = lane; i < VT_T; i += 64) {
        const int s = states[i];
        states_out[tile * VT_T + i] = s;
        hat_out[vt_pos(tile, i, ld)] = (float)tr_weight((uint32_t)s);
    }
}

// The first workgroups walk back, a tile to each of their first VB_WALK waves; the others run a forward pass.  Neither
// part reads what the other one writes: a launch walks back over one batch of tiles while the vector units, which that
// leaves idle, run another batch forward (1024 and 1024 tiles, K = 2: 1.11 ms, 0.91 + 0.40 in two launches).
constexpr int VB_WALK = 4;
template <int K, int TPW>
constexpr int vb_lds() {
    constexpr int rows = TPW * vb_cfg<K>::ROWS * vb_cfg<K>::ROW * 4, walk = VB_WALK * (int)sizeof(vb_work<false>);
    return rows > walk ? rows : walk;
}
template <int K, int TPW>
__global__ void __launch_bounds__(VB_THREADS, 4)
vb_kernel(const float *__restrict__ tiles_in, int64_t ld, vb_lists lists, vb_part forward, vb_part back, int walkers,
          int32_t *__restrict__ states_out, float *__restrict__ hat_out) {
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];   // (at 4, with the rows read 16 bytes at a time: a pass 228 -> 267 us)
    if ((int)blockIdx.x < walkers) {
        const int wave = threadIdx.x >> 6, at = blockIdx.x * VB_WALK + wave;
        if (wave >= VB_WALK || at >= vb_count(back, lists)) return;
        __builtin_amdgcn_s_setprio(3);
        vb_backtrack<K, false>(tiles_in, ld, lists, back, at, (vb_work<false> *)lds + wave, states_out, hat_out);
    } else {
        vb_forward<K, TPW>(tiles_in, ld, lists, forward, blockIdx.x - walkers, gridDim.x - walkers, lds);
    }
}

// The walk back over tiles that vm_kernel has run forward, a wave a workgroup: as many at a time as the LDS holds
__global__ void __launch_bounds__(GLQH_WAVE, 4)
vm_walk_kernel(const float *__restrict__ tiles_in, int64_t ld, vb_lists lists, vb_part back, int32_t *__restrict__ states_out,
               float *__restrict__ hat_out) {
    __shared__ vb_work<true> work;
    if ((int)blockIdx.x < vb_count(back, lists)) vb_backtrack<4, true>(tiles_in, ld, lists, back, blockIdx.x, &work, states_out, hat_out);
}

// states (tiles in row-major tile order, 256 steps each) -> packed kernel layout: the chunk of
// stream lane l is the top K bits of states 8l..8l+7, first state in the most significant
// position, stored little-endian (glq/trellis.py:486-523, 580-619).  One thread per chunk.
__global__ void __launch_bounds__(256)
pack_states_kernel(const int32_t *__restrict__ states, int m, int n, int K, uint8_t *__restrict__ packed) {
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t nblocks = (int64_t)(m >> 5) * (n >> 5);
    if (id >= nblocks * 128) return;
    const int c = (int)(id & 3), l = (int)((id >> 2) & 31);
    const int64_t blk = id >> 7;
    const int kpairs = n >> 5;
    const int mp = (int)(blk / kpairs), kp = (int)(blk % kpairs);
    const int tm = 2 * mp + (c & 1), tn = 2 * kp + (c >> 1);
    const int32_t *st = states + ((int64_t)tm * (n >> 4) + tn) * 256 + 8 * l;
    uint32_t chunk = 0;
    for (int j = 0; j < 8; ++j) chunk |= (((uint32_t)st[j] & 0xFFFFu) >> (16 - K)) << (K * (7 - j));
    uint8_t *dst = packed + (blk * 32 + l) * (4 * K) + c * K;
    for (int b = 0; b < K; ++b) dst[b] = (uint8_t)(chunk >> (8 * b));
}

// One add-compare-select step over cost rows that live in memory, for callers that drive the
// search step by step (bitshift_codebook.update, glq/trellis.py:230-251; its one-kernel form
// _viterbi_acs_step, glq/trellis_step_kernel.py:30-84).  V = 1, 2^16 states, NK = 2^K
// candidates: group j takes the minimum of cost[b, k*G + j] over ascending k (strict <, a NaN
// displaces a number and is never displaced), stores the predecessor j + (k << (16-K)) and
// the NK new costs (lut[s] - x[b])^2 + best of states s = j*NK .. j*NK + NK-1.  One thread per
// group: its loads are coalesced across the wave for every k, its stores are NK consecutive
// floats.  Streams 2 * B * 2^16 floats; bound by HBM.
template <int K>
__global__ void __launch_bounds__(256)
viterbi_acs_step_kernel(const float *__restrict__ cost, const f16 *__restrict__ x,
                        const float *__restrict__ lut, float *__restrict__ cost_out,
                        int32_t *__restrict__ prev) {
    constexpr int G = 1 << (16 - K);
    constexpr int NK = 1 << K;
    const int j = blockIdx.x * 256 + threadIdx.x;             // G is a multiple of 256
    const int b = blockIdx.y;
    const float *row = cost + (int64_t)b * 65536;
    float v[NK];
#pragma unroll
    for (int k = 0; k < NK; ++k) v[k] = row[k * G + j];
    float best = __builtin_inff();
    int bestk = 0;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        const bool take = (v[k] < best) || ((v[k] != v[k]) && (best == best));
        best = take ? v[k] : best;
        bestk = take ? k : bestk;
    }
    prev[(int64_t)b * G + j] = j + (bestk << (16 - K));
    const float xb = (float)x[b];
    float *o = cost_out + (int64_t)b * 65536 + (int64_t)j * NK;
    const float *l = lut + (int64_t)j * NK;
    if constexpr (NK >= 4) {
#pragma unroll
        for (int r = 0; r < NK; r += 4) {
            const f32x4 lv = *(const f32x4 *)(l + r);
            f32x4 e;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float d = lv[c] - xb;
                e[c] = d * d + best;                          // contraction is off in this file
            }
            *(f32x4 *)(o + r) = e;
        }
    } else {
        const f32x2 lv = *(const f32x2 *)l;
        f32x2 e;
        for (int c = 0; c < 2; ++c) {
            const float d = lv[c] - xb;
            e[c] = d * d + best;
        }
        *(f32x2 *)o = e;
    }
}

template <int K>
int acs_launch(const float *cost, const void *x, const float *lut, float *cost_out, int32_t *prev, int64_t B,
               hipStream_t stream) {
    hipLaunchKernelGGL(viterbi_acs_step_kernel<K>, dim3((1u << (16 - K)) / 256, (unsigned)B), dim3(256), 0, stream,
                       cost, (const f16 *)x, lut, cost_out, prev);
    GLQH_LAUNCH_CHECK("viterbi step launch");
    return 0;
}

// Two batches of tiles take turns: while one walks back, the other runs forward.  A batch is a chip full of pairs (two
// workgroups a CU); everything is one batch where that leaves none to overlap with.  less, what a caller short of memory has:
// 1, no vm_kernel; 2, batches of half as many besides, in the scratch that viterbi_kernel alone takes.  16384 tiles at K = 4
// 4 GB 24.8 ms, 2 GB 31.0, 1 GB 36.0 (4096: 6.5, 7.7, 9.1); at K = 3, where the first two are one, 4 GB 38.8, 2 GB 39.2, at 2 35.8, 38.9.
//
// At K = 4 chips full of sixteen tiles a CU come first, through vm_kernel, one after the other, and the rest too where that is
// VM_FEWEST tiles a CU or more: a part of a chip takes its whole time (3072 tiles 6.2 and 6.0 ms, 4096 8.2 and 6.5).  What counts is
// how many tiles are tried, which the device knows (vm_share): the launches of both ways are there, and those of one do nothing.
// (4096 tiles, all tried, 6.30 -> 6.33 ms for them.  By the tiles of the call alone 3072 of which 55 % were tried took 12.6 ms, not
// 10.1, 8192 28.1, not 23.9.)
struct vb_plan {
    int64_t batch;
    int batches;                           // in flight: 1 or 2
};
constexpr int VM_FEWEST = 12;
template <int K>
int64_t vm_tiles(int64_t n_tiles, int less) {
    const int64_t cus = glqh_device_cus();
    return K != 4 || less ? 0 : vm_share(n_tiles, VM_TILES * cus, VM_FEWEST * cus);
}
// tiles, at most, behind them
template <int K>
int64_t vb_rest(int64_t n_tiles, int less) {
    const int64_t most = VM_FEWEST * (int64_t)glqh_device_cus() - 1;
    return vm_tiles<K>(n_tiles, less) == 0 ? n_tiles : std::min(n_tiles, most);
}
vb_plan vb_plan_of(int64_t n_tiles, int less) {
    const int64_t full = (less > 1 ? 2 : 4) * (int64_t)glqh_device_cus();
    return n_tiles <= full ? vb_plan{n_tiles, 1} : vb_plan{full, 2};
}
template <int K>
size_t vb_bytes(int64_t n_tiles, int less) {
    const int64_t products = vm_tiles<K>(n_tiles, less), chip = std::min(products, VM_TILES * (int64_t)glqh_device_cus());
    const vb_plan p = vb_plan_of(vb_rest<K>(n_tiles, less), less);
    return (size_t)std::max(chip, p.batch * p.batches) * (vb_cfg<K>::STORED * vb_cfg<K>::G * 2 + sizeof(vb_tile));
}

// The lists, behind everything else (viterbi_kernel's rows take the place of the bounds'), the counts last
size_t vb_list_bytes(int64_t n_tiles) { return 2 * (((size_t)n_tiles * sizeof(int) + 255) & ~(size_t)255) + 256; }
vb_lists vb_lists_at(char *end, int64_t n_tiles) {
    char *at = end - vb_list_bytes(n_tiles);
    const size_t one = ((size_t)n_tiles * sizeof(int) + 255) & ~(size_t)255;
    return vb_lists{(int *)(at + 2 * one), (int *)at, (int *)(at + one)};
}

template <int K>
int vb_launch(const float *tiles, int64_t n_tiles, int64_t ld, void *scratch, int less, const vb_lists &lists, int32_t *states,
              float *hat, hipStream_t stream) {
    using C = vb_cfg<K>;
    hipLaunchKernelGGL(vb_try_kernel, dim3((unsigned)((n_tiles + 3) / 4)), dim3(256), 0, stream, tiles, n_tiles, ld, C::WIDE, lists);
    const int cus = glqh_device_cus();
    const int64_t products = vm_tiles<K>(n_tiles, less), rest = vb_rest<K>(n_tiles, less);
    hipLaunchKernelGGL(vb_order_kernel, dim3(1), dim3(1024), 0, stream, (int)n_tiles, 8 * cus, products ? VM_TILES * cus : 0,
                       VM_FEWEST * cus, lists);
    GLQH_LAUNCH_CHECK("viterbi lists launch");
    const vb_plan plan = vb_plan_of(rest, less);
    const size_t rows = (size_t)plan.batch * C::STORED * C::G;
    auto part = [&](int64_t batch, int pass) {
        const int64_t first = batch * plan.batch, left = rest - first;
        const int slab = (int)(batch & 1);
        return vb_part{first, (int)(left <= 0 ? 0 : left < plan.batch ? left : plan.batch), pass, (uint16_t *)scratch + slab * rows,
                       (vb_tile *)((uint16_t *)scratch + plan.batches * rows) + slab * plan.batch, false};
    };
    const vb_part none{0, 0, 0, nullptr, nullptr, false};
    auto launch = [&](const vb_part &forward, const vb_part &back) {
        const int walkers = (back.count + VB_WALK - 1) / VB_WALK;
        // one tile a workgroup while that gives no CU more than two workgroups (512 tiles: 1.58 ms at K = 4, 1.52 at 3); at
        // K = 2, with one cost row and a barrier to both its sides, a second tile is what fills the wait (2.9 -> 1.66)
        // (by the tiles that are there when all are tried)
        const int64_t all = n_tiles - products - forward.first;
        const bool few = (all > 0 ? std::min<int64_t>(all, forward.count) : forward.count) <= 2 * cus;
        const int per = few ? C::FEW : 2, work = (forward.count + per - 1) / per;
        const dim3 grid(walkers + (work < 2 * cus ? work : 2 * cus));
        if (grid.x == 0) return 0;
        if (few)
            hipLaunchKernelGGL((vb_kernel<K, C::FEW>), grid, dim3(VB_THREADS), (vb_lds<K, C::FEW>()), stream, tiles, ld, lists, forward,
                               back, walkers, states, hat);
        else
            hipLaunchKernelGGL((vb_kernel<K, 2>), grid, dim3(VB_THREADS), (vb_lds<K, 2>()), stream, tiles, ld, lists, forward, back,
                               walkers, states, hat);
        GLQH_LAUNCH_CHECK("viterbi launch");
        return 0;
    };
    if constexpr (K == 4) {
        const int64_t chip = std::min(products, VM_TILES * (int64_t)cus);
        for (int64_t first = 0; first < products; first += chip) {
            const int count = (int)std::min(products - first, chip);
            for (int pass = 0; pass < 2; ++pass) {
                const vb_part all{first, count, pass, (uint16_t *)scratch, (vb_tile *)((uint16_t *)scratch + chip * C::STORED * C::G), true};
                if (pass == 0) hipLaunchKernelGGL(vb_stop_kernel, dim3(1), dim3(64), 0, stream, all, lists);
                hipLaunchKernelGGL(vm_kernel, dim3((count + VM_TILES - 1) / VM_TILES), dim3(VM_THREADS), VM_LDS, stream, tiles, ld, lists, all);
                hipLaunchKernelGGL(vm_walk_kernel, dim3(count), dim3(GLQH_WAVE), 0, stream, tiles, ld, lists, all, states, hat);
                if (pass == 0) hipLaunchKernelGGL(vm_stop_kernel, dim3(1), dim3(64), 0, stream, all, 3 * cus, lists);
                GLQH_LAUNCH_CHECK("viterbi launch");
            }
        }
    }
    // batches 2i and 2i + 1: F0(a) | F0(b) B0(a) | F1(a) B0(b) | F1(b) B1(a) | F0(a') B1(b) | ...
    vb_part back = none;
    for (int64_t b = 0; b * plan.batch < rest; b += 2) {
        if (products + b) hipLaunchKernelGGL(vb_stop_kernel, dim3(1), dim3(64), 0, stream, part(b, 0), lists);
        for (int turn = 0; turn < 4; ++turn) {
            const vb_part forward = part(b + (turn & 1), turn >> 1);
            if (forward.count == 0 || plan.batches == 1) {     // nothing beside it
                if (launch(none, back)) return 1;
                back.count = 0;
            }
            if (forward.count == 0) continue;
            if (launch(forward, back)) return 1;
            back = forward;
        }
    }
    return launch(none, back);
}

// a tile a CU is as fast without the bounds' chain of launches (256 tiles, exact / on bounds: 1.38 / 1.62 ms at K = 2,
// 1.16 / 1.20 at 3, 1.40 / 1.16 at 4; 512: 2.15 / 1.68, 1.89 / 1.52, 2.18 / 1.58)
bool vb_takes(int K, int64_t n_tiles) { return K == 4 || (K >= 2 && n_tiles > glqh_device_cus()); }

template <int K>
int vt_launch(const float *tiles, int64_t n_tiles, int64_t ld, void *scratch, int less, int grid, int32_t *states, float *hat,
              hipStream_t stream) {
    vb_lists lists = {};
    if constexpr (K >= 2) {
        if (vb_takes(K, n_tiles)) {
            lists = vb_lists_at((char *)scratch + glqh_viterbi_scratch_bytes(K, n_tiles, less), n_tiles);
            if (int rc = vb_launch<K>(tiles, n_tiles, ld, scratch, less, lists, states, hat, stream)) return rc;
        }
    }
    constexpr size_t lds = vt_cfg<K>::ROWS * sizeof(float) * (size_t)vt_cfg<K>::G;
    hipLaunchKernelGGL(viterbi_kernel<K>, dim3((unsigned)grid), dim3(vt_cfg<K>::THREADS), lds, stream, tiles, n_tiles, ld,
                       (float *)scratch, states, hat, lists);
    GLQH_LAUNCH_CHECK("viterbi launch");
    return 0;
}

template <int K>
int vt_set_lds() {
    if constexpr (K >= 2) {
        auto set = [](const void *kernel, int lds) {
            return glqh_check_hip(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds), "viterbi attribute");
        };
        constexpr int FEW = vb_cfg<K>::FEW;
        if (int rc = set((const void *)vb_kernel<K, FEW>, vb_lds<K, FEW>()) || set((const void *)vb_kernel<K, 2>, vb_lds<K, 2>()))
            return rc;
        if constexpr (K == 4)
            if (int rc = set((const void *)vm_kernel, VM_LDS)) return rc;
    }
    return glqh_check_hip(hipFuncSetAttribute((const void *)viterbi_kernel<K>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                              (int)(vt_cfg<K>::ROWS * sizeof(float) * vt_cfg<K>::G)),
                          "viterbi attribute");
}

}  // namespace

int glqh_viterbi_init(void) { return vt_set_lds<1>() || vt_set_lds<2>() || vt_set_lds<3>() || vt_set_lds<4>(); }

// persistent workgroups: two per CU, one at K = 1 (its cost row fills the LDS)
int glqh_viterbi_grid(int K, int64_t n_tiles) {
    const int64_t g = (int64_t)glqh_device_cus() * (K >= 2 ? 2 : 1);
    return (int)(n_tiles < g ? n_tiles : g);
}

// less: 0, what the search is fastest with; 1 and 2, what it can do with too
size_t glqh_viterbi_scratch_bytes(int K, int64_t n_tiles, int less) {
    const size_t row = sizeof(float) << (16 - K);
    const int depth = K == 1 ? vt_cfg<1>::DEPTH : K == 2 ? vt_cfg<2>::DEPTH : K == 3 ? vt_cfg<3>::DEPTH : vt_cfg<4>::DEPTH;
    const size_t exact = (size_t)glqh_viterbi_grid(K, n_tiles) * (VT_T / depth) * row;
    if (!vb_takes(K, n_tiles)) return exact;
    const size_t bound = K == 2 ? vb_bytes<2>(n_tiles, less) : K == 3 ? vb_bytes<3>(n_tiles, less) : vb_bytes<4>(n_tiles, less);
    return (((exact > bound ? exact : bound) + 255) & ~(size_t)255) + vb_list_bytes(n_tiles);
}

// ld: 0 for tiles in step order, else the row length of the (m, n) matrices `tiles` and `hat`
int glqh_launch_viterbi(const float *tiles, int64_t n_tiles, int64_t ld, int K, void *scratch, int less, int32_t *states,
                        float *hat, hipStream_t stream) {
    const int grid = glqh_viterbi_grid(K, n_tiles);
    switch (K) {
    case 1: return vt_launch<1>(tiles, n_tiles, ld, scratch, less, grid, states, hat, stream);
    case 2: return vt_launch<2>(tiles, n_tiles, ld, scratch, less, grid, states, hat, stream);
    case 3: return vt_launch<3>(tiles, n_tiles, ld, scratch, less, grid, states, hat, stream);
    case 4: return vt_launch<4>(tiles, n_tiles, ld, scratch, less, grid, states, hat, stream);
    }
    return glqh_fail("trellis encoder supports K (bits/weight) 1-4, got %d", K);
}

int glqh_launch_pack_states(const int32_t *states, int64_t m, int64_t n, int K, void *packed, hipStream_t stream) {
    const int64_t threads = (m / 32) * (n / 32) * 128;
    hipLaunchKernelGGL(pack_states_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, states,
                       (int)m, (int)n, K, (uint8_t *)packed);
    GLQH_LAUNCH_CHECK("pack states launch");
    return 0;
}

int glqh_launch_viterbi_acs_step(const float *cost, const void *x_f16, const float *lut, float *cost_out,
                                 int32_t *prev, int64_t B, int K, hipStream_t stream) {
    switch (K) {
    case 1: return acs_launch<1>(cost, x_f16, lut, cost_out, prev, B, stream);
    case 2: return acs_launch<2>(cost, x_f16, lut, cost_out, prev, B, stream);
    case 3: return acs_launch<3>(cost, x_f16, lut, cost_out, prev, B, stream);
    case 4: return acs_launch<4>(cost, x_f16, lut, cost_out, prev, B, stream);
    }
    return glqh_fail("viterbi step supports K (bits/weight) 1-4, got %d", K);
}
