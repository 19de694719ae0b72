// E8 shell codebook GEMV / small-batch GEMM on the matrix cores with the table in LDS
// (gfx950, wave64).
//
// One 16-bit index stands for 8 consecutive weights of one row (glq/codebook.py:280-282):
// exactly the A operand a lane supplies to v_mfma_f32_16x16x32_f16 (row L & 15, k-group
// L >> 4, eight consecutive k).  A lane reads a 16-byte run of 8 indices of its row, looks
// each one up, expands the eight 4-bit codes to fp16 and issues one MFMA per index against
// the 8 activations of the same columns (B operand, 16 bytes per token, from LDS).  Up to
// 16 tokens share the decode.
//
// The lookup is what bounds this codebook: a random 4-byte gather from L2 sustains well
// under one lane per clock and CU, an LDS gather about twenty times that.  The nibble-packed
// table is 256 KiB and LDS 160 KiB, but the table is sorted by norm and both the first-stage
// indices and, more so, the residual-stage indices concentrate on the low-norm shells, so
// each workgroup keeps the first P entries (a launch parameter, ~120-144 KiB) in LDS and
// sends only the tail to L2.  Lanes that hit LDS all point their L2 load at entry 0, so the
// loads stay unconditional (exact wait counts) and coalesce.  Workgroups are persistent
// (one per CU, 16 waves) so the table prefix is loaded once per CU and launch.
//
// Layers whose folded streams exist (glqh_e8_fold_table) take e8_few.hip instead; this is the form on the indices.
//
// Work split: tile = (16*WR rows) x (one K slot); the 16 waves of a workgroup form WR row
// groups x WK k-parts (WK = 4 for up to 4 tokens, 1 above); k-parts are summed through LDS
// in a fixed order; every stage keeps its own accumulator and partial sum, combined by the
// consumer in stage order (glq/quantized_linear.py:1177-1194).
#include "e8_device.h"

namespace {


constexpr int EM_WAVES = 16;
constexpr int EM_THREADS = EM_WAVES * GLQH_WAVE;
constexpr int EM_STEP_BLKS = 32;               // 8-column blocks a wave covers per step

template <int NS>
struct em_idx {
    u32x4 v[NS];                               // 8 indices per stage, two per dword
};

template <int NS>
__device__ __forceinline__ em_idx<NS> em_load_idx(const uint16_t *const q[4], int64_t off) {
    em_idx<NS> r;
#pragma unroll
    for (int s = 0; s < NS; ++s) r.v[s] = __builtin_nontemporal_load((const u32x4 *)(q[s] + off));
    return r;
}

template <int NS, int TP, int WK>
__global__ void __launch_bounds__(EM_THREADS)
e8_mma_kernel(const uint16_t *__restrict__ q1, const uint16_t *__restrict__ q2,
              const uint16_t *__restrict__ q3, const uint16_t *__restrict__ q4,
              const uint32_t *__restrict__ t1, const uint32_t *__restrict__ t2, uint32_t n2,
              int t2_is_t1, const f16 *__restrict__ x, int B, int m_pad, int n_pad, int P, int slot_blks,
              int xs_slots, int ksplit, int ns_total, int s_off, float *__restrict__ part,
              glqh_e8_pscale ps) {                              // ps.v[s]: factor of stage s_off + s
    constexpr int WR = EM_WAVES / WK;
    constexpr int ROWS = 16 * WR;
    extern __shared__ u32x4 lds[];
    uint32_t *tab = (uint32_t *)lds;                           // P words
    u32x4 *xs = lds + P / 4;                                   // xs_slots slots, then 8*TP zero slots
    const int nblk = n_pad >> 3;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wr = wave / WK, wk = wave % WK;
    const int i = lane & 15, g = lane >> 4;
    const bool live = i < TP;                                  // token column of this lane
    u32x4 *zero_slots = xs + xs_slots;

    const uint16_t *const qs[4] = {q1, q2, q3, q4};
    const int RB = (m_pad + ROWS - 1) / ROWS;
    const int ntiles = RB * ksplit;
    const uint32_t P2 = t2_is_t1 ? (uint32_t)P : 0u;           // a separate stage-2 table stays in L2

    // The wave's steps over all of its workgroup's tiles form one sequence; the index runs
    // of the next steps are requested while step n is looked up, across tile boundaries,
    // and the first ones before the table is copied in.
    const int spt = slot_blks / (WK * EM_STEP_BLKS);           // steps per tile
    const int my_tiles = (ntiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
    const int nsteps = my_tiles * spt;
    auto idx_offset = [&](int sidx) -> int64_t {
        sidx = min(sidx, nsteps - 1);
        const int tile = blockIdx.x + (sidx / spt) * gridDim.x;
        const int slot = tile / RB, rb = tile % RB;
        const int row = rb * ROWS + wr * 16 + i;
        const int b0 = slot * slot_blks + ((sidx % spt) * WK + wk) * EM_STEP_BLKS;
        return (int64_t)min(row, m_pad - 1) * nblk + min(b0 + 8 * g, nblk - 8);
    };
    // a step whose 32 blocks all lie past the row (the last slot of a row that is not a multiple of the
    // step round) is skipped: no index run is requested for it, nothing is looked up (uniform over the wave)
    auto step_live = [&](int sidx) -> bool {
        if (sidx >= nsteps) return false;
        const int tile = blockIdx.x + (sidx / spt) * gridDim.x;
        return (tile / RB) * slot_blks + ((sidx % spt) * WK + wk) * EM_STEP_BLKS < nblk;
    };
    em_idx<NS> cur = em_load_idx<NS>(qs, idx_offset(0));
    em_idx<NS> nx1 = cur;                                      // the runs of steps n + 1 and n + 2 are in flight during step n
    if (step_live(1)) nx1 = em_load_idx<NS>(qs, idx_offset(1));

    // activations of a slot: one 16-byte LDS slot per (block, token), zero past B and n_pad
    auto x_load = [&](int sb0, int j) -> u32x4 {
        j = min(j, slot_blks * TP - 1);
        const int tl = j / slot_blks, blk = j % slot_blks;
        const u32x4 ld = *(const u32x4 *)(x + (int64_t)min(tl, B - 1) * n_pad + 8 * min(sb0 + blk, nblk - 1));
        return (tl < B && sb0 + blk < nblk) ? ld : u32x4{0u, 0u, 0u, 0u};
    };
    auto x_store = [&](int j, u32x4 v) {
        if (j < slot_blks * TP) xs[(j % slot_blks) * TP + j / slot_blks] = v;
    };
    // The first round of the first tile's activations is requested first, then the table prefix,
    // as loads that write LDS directly (1 KB per wave and instruction, no registers in between).
    // (P is a multiple of 1024 entries, so a wave's 64 x 16 bytes lie inside the prefix or outside.
    // Running the first step on L2 lookups alone while the table arrives was tried: that step then
    // asks L2 for six times the lines of a normal one, 36.4 us per call against 28.2.)
    {
        constexpr int U = 10;                                  // 10 * 1024 * 16 bytes = 160 KiB >= P * 4
        u32x4 xv[4];
        const int sb0 = ((int)blockIdx.x / RB) * slot_blks;
#pragma unroll
        for (int u = 0; u < 4; ++u) xv[u] = x_load(sb0, u * EM_THREADS + (int)threadIdx.x);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if ((u * EM_WAVES + wave) * GLQH_WAVE < P / 4)         // uniform over the wave
                __builtin_amdgcn_global_load_lds((const u32x4 *)t1 + u * EM_THREADS + threadIdx.x,
                                                 lds + (u * EM_WAVES + wave) * GLQH_WAVE, 16, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) x_store(u * EM_THREADS + (int)threadIdx.x, xv[u]);
    }
    for (int j = threadIdx.x; j < 8 * TP; j += EM_THREADS) zero_slots[j] = u32x4{0u, 0u, 0u, 0u};

    const int nblk_r = (nblk + EM_STEP_BLKS - 1) / EM_STEP_BLKS * EM_STEP_BLKS;
    int sidx = 0;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int slot = tile / RB, rb = tile % RB;
        const int sb0 = slot * slot_blks;
        const bool first = tile == (int)blockIdx.x;
        if (!first) __syncthreads();                           // previous tile is done with xs
        for (int j0 = first ? 4 * EM_THREADS : 0; j0 < slot_blks * TP; j0 += 4 * EM_THREADS) {
            u32x4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = x_load(sb0, j0 + u * EM_THREADS + (int)threadIdx.x);
#pragma unroll
            for (int u = 0; u < 4; ++u) x_store(j0 + u * EM_THREADS + (int)threadIdx.x, v[u]);
        }
        __syncthreads();                                       // (first tile: also drains the table loads)

        f32x4 acc[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};

        for (int st = 0; st < spt; ++st, ++sidx) {
            const int b0 = sb0 + (st * WK + wk) * EM_STEP_BLKS;  // blocks [b0, b0+32), lane's run b0 + 8g
            const u32x4 *xl = live ? xs + (b0 - sb0 + 8 * g) * TP + i : zero_slots;
            // all lookups of the step first: LDS for the prefix, L2 for the tail
            uint32_t wl[NS][8], wg[NS][8];
            bool hit[NS][8];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    uint32_t idx = (cur.v[s][t >> 1] >> (16 * (t & 1))) & 0xFFFFu;
                    const uint32_t *tg = s == 1 ? t2 : t1;
                    const uint32_t pre = s == 1 ? P2 : (uint32_t)P;
                    if (s == 1) idx = min(idx, n2 - 1);
                    // hits read LDS and aim their L2 load at one shared entry; misses the reverse
                    hit[s][t] = idx < pre;
                    wg[s][t] = tg[max(idx, pre)];
                    wl[s][t] = tab[min(idx, (uint32_t)P - 1)];
                }
            }
            // requested after the lookups, so that waiting for those does not wait for this
            em_idx<NS> nx2 = nx1;
            if (step_live(sidx + 2)) nx2 = em_load_idx<NS>(qs, idx_offset(sidx + 2));   // uniform
            if (b0 < nblk_r) {                                 // uniform; past the row the activations are zero
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const f16x8 bf = __builtin_bit_cast(f16x8, xl[t * TP]);
#pragma unroll
                    for (int s = 0; s < NS; ++s) {
                        const f16x8 af = em_expand(hit[s][t] ? wl[s][t] : wg[s][t]);
                        acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf, acc[s], 0, 0, 0);
                    }
                }
            }
            cur = nx1;
            nx1 = nx2;
        }

        // lane holds rows 4g .. 4g+3 of token i (D layout of the 16x16 MFMA)
        if constexpr (WK == 1) {
            if (live && i < B) {
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int orow = rb * ROWS + wr * 16 + 4 * g + r;
                        if (orow < m_pad) part[(((int64_t)slot * ns_total + s_off + s) * B + i) * m_pad + orow] = ps.v[s] * acc[s][r];
                    }
            }
        } else {
            __syncthreads();                                   // xs is free: reuse it for the k-part sums
            float *red = (float *)xs;                          // [WK][NS][TP][ROWS]
            if (live) {
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        red[((wk * NS + s) * TP + i) * ROWS + wr * 16 + 4 * g + r] = acc[s][r];
            }
            __syncthreads();
            for (int e = threadIdx.x; e < NS * TP * ROWS; e += EM_THREADS) {
                const int rl = e % ROWS, tl = (e / ROWS) % TP, s = e / (ROWS * TP);
                const int orow = rb * ROWS + rl;
                if (tl >= B || orow >= m_pad) continue;
                float v = red[e];
#pragma unroll
                for (int w = 1; w < WK; ++w) v += red[w * NS * TP * ROWS + e];
                part[(((int64_t)slot * ns_total + s_off + s) * B + tl) * m_pad + orow] = ps.v[s] * v;
            }
        }
    }
}

struct em_plan {
    int TP, WK, P, slot_blks, xs_slots, ksplit, grid;
    size_t lds;
};

constexpr size_t EM_LDS_TOTAL = 160 * 1024;

// 0 when the shape is better served by the plain gather kernel
int em_make_plan(int64_t m_pad, int64_t n_pad, int64_t B, int64_t n1, em_plan *p) {
    const int64_t nblk = n_pad / 8;
    if (B < 1 || B > 16 || nblk < 8 || (nblk & 7) || n1 < 4096) return 0;
    // the table load would dominate (2048 x 2048, two stages, whole linear: 15.7 us here against
    // 13.3 us with L2 gathers at one token, 16.5 against 16.6 at four; 3072 x 3072: 18.6 against 21.3)
    if (m_pad * n_pad < (B == 1 ? (int64_t)6 << 20 : (int64_t)1 << 22)) return 0;
    p->TP = B == 1 ? 1 : B <= 4 ? 4 : 16;
    p->WK = p->TP == 16 ? 1 : 4;
    const int rows = 16 * (EM_WAVES / p->WK);
    const int64_t RB = (m_pad + rows - 1) / rows;
    const int unit = p->WK * EM_STEP_BLKS;                      // blocks per workgroup step
    const int64_t nunits = (nblk + unit - 1) / unit;
    // activations: at most 32 KB of LDS; slots as long as that allows, so that a workgroup has one
    // tile (and one table fill per tile) where the shape permits
    const int slot_cap_blks = p->TP == 16 ? 128 : 512;
    const int cus = glqh_device_cus();
    int64_t ks = RB >= cus ? 1 : cus / RB;                      // one tile per workgroup where possible
    if (ks > nunits) ks = nunits;
    if (ks < 1) ks = 1;
    int64_t slot_units = (nunits + ks - 1) / ks;
    if (slot_units * unit > slot_cap_blks) slot_units = slot_cap_blks / unit;
    if (slot_units < 1) slot_units = 1;
    p->slot_blks = (int)(slot_units * unit);
    p->ksplit = (int)((nunits + slot_units - 1) / slot_units);
    // LDS: activations (or the k-part sums that reuse their space) + 8*TP zero slots + table
    size_t xbytes = (size_t)p->slot_blks * p->TP * 16;
    const size_t red = (size_t)p->WK * 4 * p->TP * rows * sizeof(float);
    if (p->WK > 1 && xbytes < red) xbytes = red;
    p->xs_slots = (int)(xbytes / 16);
    const size_t rest = xbytes + (size_t)8 * p->TP * 16;
    int64_t P = (int64_t)((EM_LDS_TOTAL - rest) / 4) & ~(int64_t)1023;
    if (P > n1) P = n1 & ~(int64_t)3;
    p->P = (int)P;
    p->lds = (size_t)P * 4 + rest;
    const int64_t ntiles = RB * p->ksplit;
    p->grid = (int)(ntiles < cus ? ntiles : cus);
    return 1;
}

template <int NS, int TP, int WK>
int em_launch(const em_plan &p, const void *x, int64_t B, const void *const q[4], const uint32_t *t1, const uint32_t *t2,
              int64_t n1, int64_t n2, int64_t m_pad, int64_t n_pad, int ns_total, int s_off, float *part, hipStream_t stream,
              glqh_e8_pscale ps) {
    hipLaunchKernelGGL((e8_mma_kernel<NS, TP, WK>), dim3((unsigned)p.grid), dim3(EM_THREADS), p.lds, stream,
                       (const uint16_t *)q[0], (const uint16_t *)q[1], (const uint16_t *)q[2],
                       (const uint16_t *)q[3], t1, t2, (uint32_t)n2, (int)(t1 == t2 && n1 == n2),
                       (const f16 *)x, (int)B, (int)m_pad, (int)n_pad, p.P, p.slot_blks, p.xs_slots, p.ksplit,
                       ns_total, s_off, part, ps);
    GLQH_LAUNCH_CHECK("e8 mma launch");
    return 0;
}

template <int NS>
int em_launch_NS(const em_plan &p, const void *x, int64_t B, const void *const q[4], const uint32_t *t1, const uint32_t *t2,
                 int64_t n1, int64_t n2, int64_t m_pad, int64_t n_pad, int ns_total, int s_off, float *part,
                 hipStream_t stream, const float *pscale) {
    glqh_e8_pscale ps = {{1.0f, 1.0f, 1.0f, 1.0f}};
    if (pscale)
        for (int i = 0; i + s_off < 4; ++i) ps.v[i] = pscale[s_off + i];
#define GLQH_EM(TP, WK) em_launch<NS, TP, WK>(p, x, B, q, t1, t2, n1, n2, m_pad, n_pad, ns_total, s_off, part, stream, ps)
    if (p.TP == 1) return GLQH_EM(1, 4);
    if (p.TP == 4) return GLQH_EM(4, 4);
    return GLQH_EM(16, 1);
#undef GLQH_EM
}

template <typename K>
int em_set_lds(K kernel) {
    return glqh_check_hip(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                              (int)EM_LDS_TOTAL),
                          "e8 mma attribute");
}

template <int NS>
int em_init_NS() {
    return em_set_lds(e8_mma_kernel<NS, 1, 4>) || em_set_lds(e8_mma_kernel<NS, 4, 4>) || em_set_lds(e8_mma_kernel<NS, 16, 1>);
}

}  // namespace

int glqh_e8_mma_init(void) { return em_init_NS<1>() || em_init_NS<2>(); }

// ksplit of the LDS-table kernel for this call, or 0 when the shape is not eligible
int glqh_e8_mma_ksplit(int64_t m_pad, int64_t n_pad, int64_t B, int64_t n1) {
    em_plan p;
    return em_make_plan(m_pad, n_pad, B, n1, &p) ? p.ksplit : 0;
}

// One launch covers two stages (the register budget of the three-deep pipeline); layers of
// three and four stages take a second launch for stages 3-4, which index the primary table.
int glqh_launch_e8_mma(const void *x, int64_t B, const void *const q[4], int nstages, const uint32_t *t1,
                       int64_t n1, const uint32_t *t2, int64_t n2, int64_t m_pad, int64_t n_pad, float *part,
                       hipStream_t stream, const float *pscale) {
    em_plan p;
    if (!em_make_plan(m_pad, n_pad, B, n1, &p)) return glqh_fail("e8 mma: shape not eligible");
    if (nstages < 1 || nstages > 4) return glqh_fail("e8 matmul: %d stages unsupported (1-4)", nstages);
    if (nstages == 1) return em_launch_NS<1>(p, x, B, q, t1, t2, n1, n2, m_pad, n_pad, 1, 0, part, stream, pscale);
    if (em_launch_NS<2>(p, x, B, q, t1, t2, n1, n2, m_pad, n_pad, nstages, 0, part, stream, pscale)) return 1;
    if (nstages == 2) return 0;
    const void *const q34[4] = {q[2], q[3], q[2], q[3]};
    if (nstages == 3) return em_launch_NS<1>(p, x, B, q34, t1, t1, n1, n1, m_pad, n_pad, 3, 2, part, stream, pscale);
    return em_launch_NS<2>(p, x, B, q34, t1, t1, n1, n1, m_pad, n_pad, 4, 2, part, stream, pscale);
}
