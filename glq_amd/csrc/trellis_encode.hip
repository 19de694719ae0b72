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
// What bounds it is vector-ALU issue: 65536 states per step, 510 steps per tile.  A workgroup
// therefore keeps the whole table in registers, two fp16 values to a register (v_fma_mix_f32
// subtracts the input from either half with fp32 rounding), and a state costs 3.5 instructions:
// subtract, multiply, add, half a three-way minimum.  The arg-min is not tracked: every
// `VT_DEPTH`-th cost row goes to scratch and the backtrack, one wave, recomputes the 2^(K*depth)
// costs below its state for `depth` steps at a time.  2048 x 2048 weights at K = 4: 165 ms (hash per
// state and step, compare and two selects per state, a byte of arg-min per step and group) -> 69.6 ms,
// vector ALUs issuing in 74 % of the cycles at 2.4 GHz (30.8 M instructions per SIMD, of which 29.9 M
// are the 3.5 per state).
#include "common.h"
#include "trellis_device.h"

#pragma clang fp contract(off)

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

// Persistent workgroups walk the tiles with a fixed stride, each owning one slab of cost rows.
// ld > 0: tiles_in and hat_out are (m, n) matrices of row length ld, the tiles their 16x16 blocks in
// row-major order; ld == 0: (tiles, 256) rows in step order.
template <int K>
__global__ void __launch_bounds__(vt_cfg<K>::THREADS, 4)
viterbi_kernel(const float *__restrict__ tiles_in, int64_t n_tiles, int64_t ld, float *__restrict__ scratch,
               int32_t *__restrict__ states_out, float *__restrict__ hat_out) {
    using C = vt_cfg<K>;
    constexpr int G = C::G;
    extern __shared__ float best[];                            // ROWS * G floats
    __shared__ float x[VT_T], xr[VT_T], cost[VT_T];
    __shared__ int states[VT_T], pick[VT_T];
    __shared__ vt_best red[C::THREADS / 64];
    const int tid = threadIdx.x;
    float *hist = scratch + (int64_t)blockIdx.x * (VT_T / C::DEPTH) * G;
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
    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int64_t per_row = ld >> 4;
        const int64_t at = ld ? (tile / per_row) * 16 * ld + (tile % per_row) * 16 : tile * VT_T;
        const int64_t pos = ld ? at + vt_step_pos(tid & 255, ld) : at + (tid & 255);
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

template <int K>
int vt_launch(const float *tiles, int64_t n_tiles, int64_t ld, void *scratch, int grid, int32_t *states, float *hat,
              hipStream_t stream) {
    constexpr size_t lds = vt_cfg<K>::ROWS * sizeof(float) * (size_t)vt_cfg<K>::G;
    hipLaunchKernelGGL(viterbi_kernel<K>, dim3((unsigned)grid), dim3(vt_cfg<K>::THREADS), lds, stream, tiles, n_tiles, ld,
                       (float *)scratch, states, hat);
    GLQH_LAUNCH_CHECK("viterbi launch");
    return 0;
}

template <int K>
int vt_set_lds() {
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

size_t glqh_viterbi_scratch_bytes(int K, int64_t n_tiles) {
    const size_t row = sizeof(float) << (16 - K);
    const int depth = K == 1 ? vt_cfg<1>::DEPTH : K == 2 ? vt_cfg<2>::DEPTH : K == 3 ? vt_cfg<3>::DEPTH : vt_cfg<4>::DEPTH;
    return (size_t)glqh_viterbi_grid(K, n_tiles) * (VT_T / depth) * row;
}

// ld: 0 for tiles in step order, else the row length of the (m, n) matrices `tiles` and `hat`
int glqh_launch_viterbi(const float *tiles, int64_t n_tiles, int64_t ld, int K, void *scratch, int32_t *states,
                        float *hat, hipStream_t stream) {
    const int grid = glqh_viterbi_grid(K, n_tiles);
    switch (K) {
    case 1: return vt_launch<1>(tiles, n_tiles, ld, scratch, grid, states, hat, stream);
    case 2: return vt_launch<2>(tiles, n_tiles, ld, scratch, grid, states, hat, stream);
    case 3: return vt_launch<3>(tiles, n_tiles, ld, scratch, grid, states, hat, stream);
    case 4: return vt_launch<4>(tiles, n_tiles, ld, scratch, grid, states, hat, stream);
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
