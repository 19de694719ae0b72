// E8 shell linear at a few tokens on folded streams: the input transform, the table lookups and the products of all
// stages in one launch (gfx950, wave64).
//
// Folded streams (glqh_e8_fold_table / glqh_e8_fold_indices): the 65536 codewords of the shell table are built from
// only 1286 distinct half codewords (columns 0..3 or 4..7 with their signs).  A table of those as finished fp16 values
// (8 bytes each, 10 KB) fits LDS whole: a lookup is two 8-byte LDS reads that are the A operand of one
// v_mfma_f32_16x16x32_f16 as they arrive, no lookup leaves the CU and nothing is expanded.  An index becomes two 11-bit
// half numbers, stored as a 16-bit word (first half | low 5 bits of the second << 11) and a byte (its high 6 bits): 3
// bytes instead of 2.
//
// What bounds the call at few tokens is the number of launches (each about 2.8 us before its first wave and after
// its last, 4 us for a transform of one row), not the 3 bytes per index and stage: so every workgroup transforms
// the rows itself, from the activations, while its first indices and the table are on their way.  A wave takes
// 1024 columns of one token: sixteen consecutive elements per lane, four butterfly levels in the lane and six across
// lanes, no LDS, no barrier.  In blocks of 2048, 4096 and 8192 columns a lane starts with the same columns of two,
// four or eight such segments, combines them, and one exchange through LDS puts every segment into a wave.  The result
// goes straight into the product's operand slots.
//
// Work split: tile = 16 * WR rows x one K slot; the sixteen waves of a workgroup form WR row groups x WK K parts
// (WK as large as the tiles still fill the chip at most once: no K slot leaves the workgroup where the shape
// permits).  K parts are summed in LDS in a fixed order; the finishing launch reads one scaled sum per K slot and
// stage.
//
// Kernel times of the whole linear, two stages, one / four tokens, microseconds; before: a launch for the transform, one
// for the product (two for three and four stages), one to finish: 960 x 960 12.8 -> 10.5 / 16.3 -> 11.2; 2048 x 2048 14.4
// -> 11.5 / 15.2 -> 12.8; 14336 x 4096 21.4 -> 18.9 / 22.7 -> 22.7; 4096 x 14336 21.0 -> 20.5 / 24.3 (not fused); four
// stages, one token: 4096 x 4096 22.6 -> 15.3, 14336 x 4096 35.7 -> 27.1; 2432 x 1152 at sixteen tokens 47.9 -> 19.5.
#include "e8_device.h"
#include "fht_device.h"

namespace {

constexpr int EF_WAVES = 16;
constexpr int EF_THREADS = EF_WAVES * GLQH_WAVE;
constexpr int EF_STEP_BLKS = 32;               // 8-column blocks a wave covers per step
constexpr int EF_SEG = 1024;                   // columns of one wave's part of the input transform
constexpr int EF_STG = EF_SEG + EF_SEG / 8;    // floats of a staging row: four of padding behind every 32
__device__ __forceinline__ int ef_pad(int p) { return p + ((p >> 5) << 2); }   // 16-byte groups stay whole
constexpr size_t EF_LDS_TOTAL = 160 * 1024;

struct ef_args {
    const uint16_t *q[4];                      // 16-bit words of the folded streams, per stage
    const uint8_t *hi[4];                      // their bytes
    const uint32_t *t1, *t2;                   // half codewords, two words each
    uint32_t n1, n2;
    int own2;                                  // stage 2 has a table of its own
    const void *x;
    int64_t x_stride;
    const f16 *sv;                             // NULL: x is transformed fp16 rows of n_pad
    int x_bf16, B, in_features, m_pad, n_pad;  // n_pad: also the canonical blocks (its bits)
    int lwk, slot_blks, ksplit;
    int direct;                                // one K slot: part is the (B, m_pad) sum of the scaled stages
    int xs_off, stg_off, red_off;              // LDS regions, in 16-byte units
    float *part;
    glqh_e8_pscale ps;
};

template <int NS>
struct ef_idx {
    u32x4 v[NS];                               // 8 indices per stage, two per dword
    u32x2 sg[NS];                              // their 8 high bytes
};

template <int NS>
__device__ __forceinline__ ef_idx<NS> ef_load_idx(const uint16_t *const (&q)[NS], const uint8_t *const (&hi)[NS], int64_t off,
                                                  uint32_t lane) {
    ef_idx<NS> r;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        r.v[s] = __builtin_nontemporal_load((const u32x4 *)(q[s] + off) + lane);
        r.sg[s] = __builtin_nontemporal_load((const u32x2 *)(hi[s] + off) + lane);
    }
    return r;
}

// sixteen consecutive activations and signs, as they arrive
struct ef_raw {
    u32x4 x[2], sv[2];
};

__device__ __forceinline__ void ef_unpack8(u32x4 w, bool bf16, float *f) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t we = w[e];
        if (bf16) {
            f[2 * e] = __builtin_bit_cast(float, we << 16);
            f[2 * e + 1] = __builtin_bit_cast(float, we & 0xffff0000u);
        } else {
            const f16x2 h = __builtin_bit_cast(f16x2, we);
            f[2 * e] = (float)h[0];
            f[2 * e + 1] = (float)h[1];
        }
    }
}

__device__ __forceinline__ u32x4 ef_pack8(const float *f, float norm) {
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const f16x2 h = {(f16)(f[2 * e] * norm), (f16)(f[2 * e + 1] * norm)};
        w[e] = __builtin_bit_cast(uint32_t, h);
    }
    return w;
}

// W consecutive 16-bit values (2, 4 or 8; p on 2 * W bytes) into W / 2 words
template <int W>
__device__ __forceinline__ void ef_load_run(const uint16_t *p, uint32_t *o) {
    if constexpr (W == 2) o[0] = *(const uint32_t *)p;
    else if constexpr (W == 4) *(u32x2 *)o = *(const u32x2 *)p;
    else *(u32x4 *)o = *(const u32x4 *)p;
}

// A wave's part `seg` of a token's row.  Inside a block of NB = 2, 4, 8 segments of 1024 columns: 16 / NB consecutive
// columns of every segment, so that the levels across segments are the lane's own; otherwise (NB 1) sixteen
// consecutive columns of the segment.  first: the lane's first column.  Columns from in_features (even) on read as
// zero, two at a time.
template <int NB>
__device__ __forceinline__ void ef_load_part(ef_raw &r, const ef_args &a, const uint16_t *xr, int first) {
    constexpr int W = NB == 1 ? 8 : 16 / NB;
#pragma unroll
    for (int k = 0; k < 16 / W; ++k) {
        const int c = first + k * (NB == 1 ? 8 : EF_SEG);
        if (a.in_features == a.n_pad) {                        // uniform
            ef_load_run<W>(xr + c, (uint32_t *)r.x + k * (W / 2));
        } else {
#pragma unroll
            for (int e = 0; e < W; e += 2) {
                const uint32_t w = *(const uint32_t *)(xr + min(c + e, a.in_features - 2));
                ((uint32_t *)r.x)[(k * W + e) / 2] = c + e < a.in_features ? w : 0u;
            }
        }
        ef_load_run<W>((const uint16_t *)a.sv + c, (uint32_t *)r.sv + k * (W / 2));
    }
}

// the block of a large-block segment: its first segment and log2 of its segments
struct ef_block {
    int seg0, log_nb;
};
__device__ __forceinline__ ef_block ef_block_of(int big, int seg) {
    ef_block b;
    uint32_t left = (uint32_t)big;
    b.seg0 = 0;
    for (;;) {                                                 // uniform; seg lies in one of the blocks
        b.log_nb = 31 - __builtin_clz(left) - 10;
        if (seg < b.seg0 + (1 << b.log_nb)) return b;
        b.seg0 += 1 << b.log_nb;
        left &= ~(1u << (b.log_nb + 10));
    }
}

__device__ __forceinline__ ef_raw ef_load_raw(const ef_args &a, int tok, int seg, int big, int lane) {
    const uint16_t *xr = (const uint16_t *)a.x + (int64_t)tok * a.x_stride;
    ef_raw r;
    r.x[0] = r.x[1] = r.sv[0] = r.sv[1] = u32x4{0u, 0u, 0u, 0u};
    if (seg * EF_SEG < big) {                                  // uniform
        const ef_block b = ef_block_of(big, seg);
        const int part = seg - b.seg0, base = b.seg0 * EF_SEG;
        if (b.log_nb == 1) ef_load_part<2>(r, a, xr, base + part * 512 + 8 * lane);
        else if (b.log_nb == 2) ef_load_part<4>(r, a, xr, base + part * 256 + 4 * lane);
        else ef_load_part<8>(r, a, xr, base + part * 128 + 2 * lane);
    } else if (seg * EF_SEG + 16 * lane < a.n_pad) {           // n_pad is a multiple of 64
        ef_load_part<1>(r, a, xr, seg * EF_SEG + 16 * lane);
    }
    return r;
}

// the levels across the NB segments of a block, and the values into the staging rows (one per segment)
template <int NB>
__device__ __forceinline__ void ef_cross(float (&v)[16], float *stg, int pos) {
    constexpr int W = 16 / NB;
#pragma unroll
    for (int h = W; h < 16; h <<= 1) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            if ((j & h) == 0) {
                const float p = v[j], q = v[j | h];
                v[j] = p + q;
                v[j | h] = p - q;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        float *o = stg + k * EF_STG + ef_pad(pos);
        if constexpr (W == 2) *(f32x2 *)o = f32x2{v[2 * k], v[2 * k + 1]};
        else {
#pragma unroll
            for (int w = 0; w < W; w += 4) *(f32x4 *)(o + w) = f32x4{v[W * k + w], v[W * k + w + 1], v[W * k + w + 2], v[W * k + w + 3]};
        }
    }
}

template <int N>
__device__ __forceinline__ float ef_sum(const float *p, int stride) {
    float v[N];
#pragma unroll
    for (int w = 0; w < N; ++w) v[w] = p[w * stride];
#pragma unroll
    for (int w = 1; w < N; ++w) v[0] += v[w];
    return v[0];
}

template <int NS, int TP, bool FUSED>
__global__ void __launch_bounds__(EF_THREADS)
e8_few_kernel(ef_args a) {
    extern __shared__ u32x4 lds[];
    uint32_t *tab = (uint32_t *)lds;
    u32x4 *xs = lds + a.xs_off;                                // (block, token) slots of 8 columns: the whole row, or the K slot
    float *stg = (float *)(lds + a.stg_off);                   // rows of the large blocks' segments
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int WK = 1 << a.lwk, WR = EF_WAVES >> a.lwk, ROWS = 16 * WR;
    const int wr = wave >> a.lwk, wk = wave & (WK - 1);
    const int i = lane & 15, g = lane >> 4;
    const int nblk = a.n_pad >> 3, B = a.B;
    const int RB = (a.m_pad + ROWS - 1) / ROWS, ntiles = RB * a.ksplit;
    const int spt = (a.slot_blks >> 5) >> a.lwk;               // steps per tile
    const int col_tiles = (nblk + 31) >> 5, row_tiles = (a.m_pad + 15) >> 4;
    const uint16_t *q[NS];
    const uint8_t *hi[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) { q[s] = a.q[s]; hi[s] = a.hi[s]; }
    // the wave's steps over all of its workgroup's tiles, in order (everything uniform over the wave)
    struct cursor {
        int tile, st, ct;                                      // ct: the step's column tile of 32 blocks
        int64_t row;                                           // of the wave's row tile: its first index tile
    };
    auto enter = [&](cursor &c, int tile) {
        c.tile = tile;
        c.st = 0;
        c.ct = (tile / RB) * (a.slot_blks >> 5) + wk;
        c.row = (int64_t)min((tile % RB) * WR + wr, row_tiles - 1) * col_tiles;
    };
    auto advance = [&](cursor &c) {
        c.ct += WK;
        if (++c.st == spt) enter(c, c.tile + gridDim.x);
    };
    auto fetch = [&](const cursor &c) { return ef_load_idx<NS>(q, hi, (c.row + min(c.ct, col_tiles - 1)) * 512, lane); };

    // ---- the rows: request the first part, then the first indices, then copy the table
    const int nseg = (a.n_pad + EF_SEG - 1) / EF_SEG, tasks = B * nseg;
    const int rem = a.n_pad & (EF_SEG - 1), big = a.n_pad & ~(2 * EF_SEG - 1);   // blocks under 1024; from 2048 on
    cursor nx;
    enter(nx, blockIdx.x);
    ef_idx<NS> cur;
    if constexpr (!FUSED) cur = fetch(nx);
    // (loads return in order: the table and the activations, which are waited for first, are requested before the
    // indices of the first step, which stay in flight while the rows are transformed)
    const uint32_t n1r = (a.n1 + 1u) & ~1u, tab2_off = a.own2 ? 8u * n1r : 0u;
    u32x2 tw[4];                                               // at most 2048 half codewords per table
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const uint32_t n = u < 2 ? a.n1 : a.n2, j = (uint32_t)(u & 1) * EF_THREADS + threadIdx.x;
        tw[u] = *(const u32x2 *)((u < 2 ? a.t1 : a.t2) + 2 * min(j, n - 1u));
    }
    // transformed rows: one 16-byte LDS slot per (block, token) of the K slot, zero past B and n_pad
    auto x_load = [&](int sb0, int j) -> u32x4 {
        j = min(j, a.slot_blks * TP - 1);
        const int tl = j / a.slot_blks, blk = j % a.slot_blks;
        const u32x4 ld = *(const u32x4 *)((const f16 *)a.x + (int64_t)min(tl, B - 1) * a.n_pad + 8 * min(sb0 + blk, nblk - 1));
        return (tl < B && sb0 + blk < nblk) ? ld : u32x4{0u, 0u, 0u, 0u};
    };
    auto x_store = [&](int j, u32x4 v) {
        if (j < a.slot_blks * TP) xs[(j % a.slot_blks) * TP + j / a.slot_blks] = v;
    };
    auto table_store = [&]() {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t n = u < 2 ? a.n1 : a.n2, j = (uint32_t)(u & 1) * EF_THREADS + threadIdx.x;
            if (j < n && (u < 2 || a.own2)) *(u32x2 *)(tab + (u < 2 ? 0u : 2u * n1r) + 2 * j) = tw[u];
        }
    };
    if constexpr (!FUSED) {
        const int sb0 = ((int)blockIdx.x / RB) * a.slot_blks;
        u32x4 xv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) xv[u] = x_load(sb0, u * EF_THREADS + (int)threadIdx.x);
        table_store();
#pragma unroll
        for (int u = 0; u < 4; ++u) x_store(u * EF_THREADS + (int)threadIdx.x, xv[u]);
    } else {
        for (int j = nblk * TP + (int)threadIdx.x; j < col_tiles * 32 * TP; j += EF_THREADS) xs[j] = u32x4{0u, 0u, 0u, 0u};
    }
    auto finish = [&](float (&v)[16], int tok, int seg, float norm) {   // sixteen columns -> two operand slots
        u32x4 *o = xs + (size_t)(seg * (EF_SEG / 8) + 2 * lane) * TP + tok;
        o[0] = ef_pack8(v, norm);
        o[TP] = ef_pack8(v + 8, norm);
    };
    if constexpr (FUSED) {
    ef_raw raw = {};
    if (wave < tasks) raw = ef_load_raw(a, wave / nseg, wave % nseg, big, lane);
    cur = fetch(nx);
    table_store();
#pragma nounroll
    for (int task = wave; task < tasks; task += EF_WAVES) {
        const int tok = task / nseg, seg = task % nseg;
        float v[16], sf[16];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            ef_unpack8(raw.x[h], a.x_bf16, v + 8 * h);
            ef_unpack8(raw.sv[h], false, sf + 8 * h);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] *= sf[e];
        if (task + EF_WAVES < tasks) raw = ef_load_raw(a, (task + EF_WAVES) / nseg, (task + EF_WAVES) % nseg, big, lane);
        if (seg * EF_SEG < big) {                              // uniform
            const ef_block b = ef_block_of(big, seg);
            float *o = stg + (size_t)(tok * (big / EF_SEG) + b.seg0) * EF_STG;
            const int part = seg - b.seg0;
            if (b.log_nb == 1) ef_cross<2>(v, o, part * 512 + 8 * lane);
            else if (b.log_nb == 2) ef_cross<4>(v, o, part * 256 + 4 * lane);
            else ef_cross<8>(v, o, part * 128 + 2 * lane);
        } else if (seg < nseg - 1 || rem == 0) {               // uniform: a block of 1024 columns
            fht_wave<16>(v, 10, nullptr, lane);
            finish(v, tok, seg, rsqrt_pow2(10));
        } else {                                               // the row's blocks of 512, 256, ... columns side by side
            int off = 0, log_bs = 4;
            for (int l = 9; l >= 4; --l) {
                if (rem >> l & 1) {
                    if (16 * lane >= off && 16 * lane < off + (1 << l)) log_bs = l;
                    off += 1 << l;
                }
            }
            fht_lanes_ragged(v, log_bs, lane);
            if (16 * lane < rem) finish(v, tok, seg, rsqrt_pow2(log_bs));
        }
    }
    if (big) {                                                 // uniform: the segments of the large blocks
        __syncthreads();
        const int bseg = big / EF_SEG;
        for (int task = wave; task < B * bseg; task += EF_WAVES) {
            const int tok = task / bseg, seg = task % bseg;
            const float *src = stg + (size_t)task * EF_STG + ef_pad(16 * lane);
            float v[16];
#pragma unroll
            for (int w = 0; w < 16; w += 4) {
                const f32x4 r = *(const f32x4 *)(src + w);
                v[w] = r[0]; v[w + 1] = r[1]; v[w + 2] = r[2]; v[w + 3] = r[3];
            }
            fht_wave<16>(v, 10, nullptr, lane);
            finish(v, tok, seg, rsqrt_pow2(ef_block_of(big, seg).log_nb + 10));
        }
    }
    }

    // ---- the product
    const bool live = i < TP;                                  // token column of this lane
    const int xi = live ? i : 0;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int slot = tile / RB, rb = tile % RB;
        const int xb0 = FUSED ? 0 : slot * a.slot_blks;        // block of the first operand slot
        const bool first = tile == (int)blockIdx.x;
        if constexpr (!FUSED) {
            if (!first) __syncthreads();                       // the previous tile is done with xs
            for (int j0 = first ? 4 * EF_THREADS : 0; j0 < a.slot_blks * TP; j0 += 4 * EF_THREADS) {
                u32x4 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = x_load(xb0, j0 + u * EF_THREADS + (int)threadIdx.x);
#pragma unroll
                for (int u = 0; u < 4; ++u) x_store(j0 + u * EF_THREADS + (int)threadIdx.x, v[u]);
            }
        }
        if (first || !FUSED) __syncthreads();
        f32x4 acc[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int st = 0; st < spt; ++st) {
            const int b0 = slot * a.slot_blks + (st * WK + wk) * EF_STEP_BLKS;
            // one step ahead only: with more in flight the waves' requests queue up behind each other in the memory
            // system (4096 x 14336, one token, whole call: three steps ahead 16.7 us, two 15.0, one 13.7).  Steps that
            // lie past the row (the last slot of a row that is not a multiple of the step round) request nothing.
            ef_idx<NS> nxt = cur;
            advance(nx);
            if (nx.tile < ntiles && nx.ct < col_tiles) nxt = fetch(nx);   // uniform
            if (b0 < nblk) {                                   // uniform
                const u32x4 *xl = xs + (b0 - xb0 + 8 * g) * TP + xi;
                const char *tb = (const char *)tab;
                constexpr int U = NS <= 2 ? 4 : 2;             // lookups per stage at a time: 32 registers of operands
#pragma unroll
                for (int h = 0; h < 8 / U; ++h) {
                    u32x4 af[NS][U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int t = U * h + u;
#pragma unroll
                        for (int s = 0; s < NS; ++s) {
                            const uint32_t w = cur.v[s][t >> 1], sw = cur.sg[s][t >> 2];
                            // byte offsets 8 * half number: first half from bits 0..10 of the index's 16-bit
                            // word, second from its bits 11..15 and the index's byte
                            const uint32_t lo = t & 1 ? (w >> 13) & 0x3FF8u : (w << 3) & 0x3FF8u;
                            const uint32_t h5 = t & 1 ? (w >> 24) & 0xF8u : (w >> 8) & 0xF8u;
                            const uint32_t b6 = (t & 3) == 0 ? (sw << 8) & 0x3F00u : (t & 3) == 1 ? sw & 0x3F00u
                                              : (t & 3) == 2 ? (sw >> 8) & 0x3F00u : (sw >> 16) & 0x3F00u;
                            const char *tbs = tb + (s == 1 ? tab2_off : 0u);
                            const u32x2 c03 = *(const u32x2 *)(tbs + lo), c47 = *(const u32x2 *)(tbs + (h5 | b6));
                            af[s][u] = u32x4{c03[0], c03[1], c47[0], c47[1]};
                        }
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const f16x8 bf = __builtin_bit_cast(f16x8, xl[(U * h + u) * TP]);
#pragma unroll
                        for (int s = 0; s < NS; ++s)
                            acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, af[s][u]), bf, acc[s], 0, 0, 0);
                    }
                }
            }
            cur = nxt;
        }
        // lane holds rows 4g .. 4g+3 of token i (D layout of the 16x16 MFMA)
        if (WK == 1 && !a.direct) {                            // uniform
            if (live && i < B) {
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int orow = rb * ROWS + wr * 16 + 4 * g + r;
                        if (orow < a.m_pad) a.part[(((int64_t)slot * NS + s) * B + i) * a.m_pad + orow] = a.ps.v[s] * acc[s][r];
                    }
            }
            continue;
        }
        __syncthreads();                                       // the region may be the activations'
        float *red = (float *)(lds + a.red_off);               // [WK][NS][TP][ROWS]
        if (live) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                *(f32x4 *)(red + ((wk * NS + s) * TP + i) * ROWS + wr * 16 + 4 * g) = acc[s];
        }
        __syncthreads();
        const int n = TP * ROWS;                               // values of a stage
        int t0 = threadIdx.x;
        asm volatile("" : "+v"(t0));                           // nothing of what follows is worth registers during the product
        auto sum_parts = [&](int e) -> float {                 // K parts in order
            switch (a.lwk) {
            case 0: return red[e];
            case 1: return ef_sum<2>(red + e, NS * n);
            case 2: return ef_sum<4>(red + e, NS * n);
            case 3: return ef_sum<8>(red + e, NS * n);
            default: return ef_sum<16>(red + e, NS * n);
            }
        };
        if (!a.direct) {
            for (int e = t0; e < NS * n; e += EF_THREADS) {
                const int s = e / n, tl = (e % n) / ROWS, orow = rb * ROWS + e % ROWS;
                if (tl < B && orow < a.m_pad)
                    a.part[(((int64_t)slot * NS + s) * B + tl) * a.m_pad + orow] = a.ps.v[s] * sum_parts(e);
            }
        } else {
            for (int e = t0; e < n; e += EF_THREADS) {
                const int tl = e / ROWS, orow = rb * ROWS + e % ROWS;
                if (tl >= B || orow >= a.m_pad) continue;
                float sum = a.ps.v[0] * sum_parts(e);          // stages in order
#pragma nounroll
                for (int s = 1; s < NS; ++s) sum += a.ps.v[s] * sum_parts(s * n + e);
                a.part[(int64_t)tl * a.m_pad + orow] = sum;
            }
        }
    }
}

struct ef_plan {
    int TP, lwk, slot_blks, ksplit, grid;
    int xs_off, stg_off, red_off;
    size_t lds;
};

// fused: rows up to which a workgroup's own transform is cheaper than a launch of its own, EF_MAX_TASKS segments of
// 1024 columns (sixteen at a time: 0.14 us of vector instructions each on top of about 1.3; two stages of 14336 x 4096 at
// four tokens, 16 segments, 23.1 -> 22.7 us; 2432 x 1152 at sixteen, 32 segments, 17.2 -> 15.9)
constexpr int EF_MAX_TASKS = 32;

int ef_make_plan(int64_t m_pad, int64_t n_pad, int64_t B, int nstages, int64_t tab_words, bool fused, ef_plan *p) {
    if (B < 1 || B > 16 || n_pad < 64 || (n_pad & 63) || m_pad < 1 || m_pad > (1 << 28) || n_pad > (1 << 28)) return 0;
    if (fused && (n_pad >= (1 << 14) || B * ((n_pad + EF_SEG - 1) / EF_SEG) > EF_MAX_TASKS)) return 0;
    const int64_t nblk = n_pad / 8, steps = (nblk + EF_STEP_BLKS - 1) / EF_STEP_BLKS;
    const int cus = glqh_device_cus();
    p->TP = B == 1 ? 1 : B <= 4 ? 4 : 16;
    // K parts of a workgroup.  16-row tiles and all sixteen waves on one row group when they fill the chip at most
    // once and a row fits LDS: no K slot leaves the workgroup (4096 x 14336, whole unfused call at one token: 19.1 ->
    // 15.8 us; at four tokens 20.1 -> 18.8; whole linear 4096 x 4096 at sixteen tokens 25.8 -> 19.6.  Not taken:
    // 14336 x 4096, 896 such tiles, 17.6 -> 21.7 us; 4096 x 14336 at sixteen tokens, a row of 448 KB in four slots,
    // 21.1 -> 39.3).  Otherwise four, or as many as a short row has steps for; at sixteen tokens with rows of more
    // than 1536 blocks one (4096 x 14336 21.1 -> 24.3 with four: every workgroup stages 128 KB for four steps).
    int lwk = 2;
    const int64_t cap16 = p->TP == 16 ? 512 : 2048;             // blocks of a slot: 128 KB / 32 KB (one token) of activations
    if ((m_pad + 15) / 16 <= cus && steps >= 16 && nblk <= cap16) lwk = 4;
    else if (p->TP == 16 && nblk > 1536) lwk = 0;
    while (lwk > 0 && (1 << lwk) > steps) --lwk;
    const int rows = 256 >> lwk;
    const int64_t RB = (m_pad + rows - 1) / rows, unit = (int64_t)EF_STEP_BLKS << lwk, nunits = (nblk + unit - 1) / unit;
    int64_t ks = RB >= cus ? 1 : cus / RB;                      // one tile per workgroup where possible
    if (ks > nunits) ks = nunits;
    int64_t slot_units = (nunits + ks - 1) / ks;
    const int64_t cap = lwk == 4 ? cap16 : p->TP == 16 && lwk == 0 ? 128 : 512;
    if (slot_units * unit > cap) slot_units = cap / unit;
    if (slot_units < 1) slot_units = 1;
    p->lwk = lwk;
    p->slot_blks = (int)(slot_units * unit);
    p->ksplit = (int)((nunits + slot_units - 1) / slot_units);
    const int64_t ntiles = RB * p->ksplit;
    p->grid = (int)(ntiles < cus ? ntiles : cus);
    const int64_t xs = (fused ? steps * EF_STEP_BLKS : p->slot_blks) * p->TP;
    const int64_t stg = fused ? B * (n_pad / (2 * EF_SEG) * 2) * EF_STG / 4 : 0;
    const int64_t red = (int64_t)256 * nstages * p->TP / 4;     // WK * ROWS = 256
    p->xs_off = (int)((tab_words + 3) / 4);
    p->stg_off = p->xs_off + (int)xs;
    p->red_off = fused && ntiles > p->grid ? p->stg_off : p->xs_off;   // fused, several tiles: the activations stay
    const int64_t end1 = p->stg_off + stg, end2 = p->red_off + red;
    p->lds = (size_t)(end1 > end2 ? end1 : end2) * 16;
    return p->lds <= EF_LDS_TOTAL;
}

template <int NS, int TP>
int ef_launch(const ef_plan &p, const ef_args &a, hipStream_t stream) {
    if (a.sv) hipLaunchKernelGGL((e8_few_kernel<NS, TP, true>), dim3((unsigned)p.grid), dim3(EF_THREADS), p.lds, stream, a);
    else hipLaunchKernelGGL((e8_few_kernel<NS, TP, false>), dim3((unsigned)p.grid), dim3(EF_THREADS), p.lds, stream, a);
    GLQH_LAUNCH_CHECK("e8 few-token launch");
    return 0;
}

template <int NS>
int ef_launch_NS(const ef_plan &p, const ef_args &a, hipStream_t stream) {
    if (p.TP == 1) return ef_launch<NS, 1>(p, a, stream);
    if (p.TP == 4) return ef_launch<NS, 4>(p, a, stream);
    return ef_launch<NS, 16>(p, a, stream);
}

template <int NS>
int ef_init_NS() {
    auto set = [](const void *k) {
        return glqh_check_hip(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)EF_LDS_TOTAL),
                              "e8 few-token attribute");
    };
    return set((const void *)e8_few_kernel<NS, 1, false>) || set((const void *)e8_few_kernel<NS, 4, false>) ||
           set((const void *)e8_few_kernel<NS, 16, false>) || set((const void *)e8_few_kernel<NS, 1, true>) ||
           set((const void *)e8_few_kernel<NS, 4, true>) || set((const void *)e8_few_kernel<NS, 16, true>);
}

constexpr int64_t EF_TAB_WORDS_MAX = 2 * 2 * 2048;              // two tables of 2048 half codewords

}  // namespace

int glqh_e8_few_init(void) { return ef_init_NS<1>() || ef_init_NS<2>() || ef_init_NS<3>() || ef_init_NS<4>(); }

// K slots of the call, or 0 when it is not served: up to 16 tokens; fused: of rows that a workgroup can transform itself.
int glqh_e8_few_ksplit(int64_t m_pad, int64_t n_pad, int64_t B, int nstages, int fused) {
    ef_plan p;
    return nstages >= 1 && nstages <= 4 && ef_make_plan(m_pad, n_pad, B, nstages, EF_TAB_WORDS_MAX, fused != 0, &p) ? p.ksplit : 0;
}

// part[((slot * nstages + stage) * B + token) * m_pad + row] = pscale[stage] * (the slot's columns of the transformed
// row . the stage's weights); direct (one K slot): part[token * m_pad + row], the stages added in order.
// sv: the rows are activations (16-bit, x and sv on 16 bytes, x_stride a multiple of 8, in_features even) and transformed here, over
// n_pad's canonical blocks; sv NULL: they are transformed fp16 rows of n_pad.
int glqh_launch_e8_few(const void *x, int x_dtype, int64_t x_stride, const void *sv, int64_t B, int64_t in_features,
                       const glqh_e8_folded *fold, int nstages, int64_t m_pad, int64_t n_pad, const float *pscale, float *part,
                       int direct, hipStream_t stream) {
    glqh_range range("dequant_matmul");
    ef_plan p;
    GLQH_REQUIRE(fold && nstages >= 1 && nstages <= 4, "e8 few tokens: 1..4 folded stages");
    GLQH_REQUIRE(x_dtype == GLQH_F16 || (sv && x_dtype == GLQH_BF16), "e8 few tokens: x must be f16 or bf16");
    GLQH_REQUIRE(!sv || (in_features >= 1 && in_features <= n_pad), "e8 few tokens: in_features exceeds n_pad");
    ef_args a = {};
    a.own2 = nstages >= 2 && fold->halves2 && fold->halves2 != fold->halves1;
    a.t1 = (const uint32_t *)fold->halves1;
    a.t2 = a.own2 ? (const uint32_t *)fold->halves2 : a.t1;
    a.n1 = (uint32_t)fold->n_halves1;
    a.n2 = (uint32_t)(a.own2 ? fold->n_halves2 : fold->n_halves1);
    GLQH_REQUIRE(a.t1 && fold->n_halves1 >= 1 && fold->n_halves1 <= 2048 && a.n2 >= 1 && a.n2 <= 2048,
                 "e8 folded: 1..2048 half codewords per table");
    const int64_t tab_words = 2 * ((a.n1 + 1) & ~1u) + (a.own2 ? 2 * ((a.n2 + 1) & ~1u) : 0);
    if (!ef_make_plan(m_pad, n_pad, B, nstages, tab_words, sv != nullptr, &p)) return glqh_fail("e8 few tokens: shape not eligible");
    GLQH_REQUIRE(!direct || p.ksplit == 1, "e8 few tokens: finished sums need one K slot");
    for (int s = 0; s < 4; ++s) {
        const int j = s < nstages ? s : 0;
        GLQH_REQUIRE(fold->lo16[j] && fold->hi8[j], "e8 folded: stage %d has no folded stream", j + 1);
        a.q[s] = fold->lo16[j];
        a.hi[s] = fold->hi8[j];
        a.ps.v[s] = s >= nstages ? 0.0f : pscale ? pscale[s] : 1.0f;
    }
    a.x = x;
    a.x_stride = x_stride;
    a.sv = (const f16 *)sv;
    a.direct = direct;
    a.x_bf16 = x_dtype == GLQH_BF16;
    a.B = (int)B;
    a.in_features = (int)in_features;
    a.m_pad = (int)m_pad;
    a.n_pad = (int)n_pad;
    a.lwk = p.lwk;
    a.slot_blks = p.slot_blks;
    a.ksplit = p.ksplit;
    a.xs_off = p.xs_off;
    a.stg_off = p.stg_off;
    a.red_off = p.red_off;
    a.part = part;
    switch (nstages) {
    case 1: return ef_launch_NS<1>(p, a, stream);
    case 2: return ef_launch_NS<2>(p, a, stream);
    case 3: return ef_launch_NS<3>(p, a, stream);
    default: return ef_launch_NS<4>(p, a, stream);
    }
}
