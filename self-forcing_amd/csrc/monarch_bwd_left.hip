// Left-factor part of the Monarch backward on gfx950 MFMA (bf16 / fp16, head_dim 64 or 128, block rows b1 <= 128).
//
// Replaces, inside the backward of the two-step attention, the per-(a, j) products and row kernels
//     S2 = q_i . Kbar_r,  dLm = dO_i . Y_r,  L = softmax_r(s S2 - c),  dS2 = L (dLm - sum_r L dLm),
//     dc_r = - sum_i dS2,  dY_r = sum_i L dO_i,  dKbar_r = s sum_i dS2 q_i,  dQ_i = s sum_r dS2 Kbar_r
// (wan/modules/monarch_attn.py:852-886 `_z_bwd_preprocess`, :1034-1222 `_z_bwd`) with one kernel that never writes
// the [i x r] matrices S2, dLm, L, dS2 (dS2 only where the caller forms dQ by a library product).
//
// A wave holds 32 query rows of a column (unit, a, j): they and their dO rows sit in LDS, the r = (k, f) rows of Kbar and
// Y stream through LDS 32 at a time (global_load_lds_dwordx4; all tiles are row-major, 16-byte pieces XOR-swizzled per
// row), twice: pass 1 for the softmax statistics (row maximum, sum, and sum of L dLm, kept per lane and merged across
// lanes once at the end; skipped when the forward's are at hand), pass 2 for the gradients.  Logits are computed as
// S2[i, r] (A = query rows, B = Kbar rows), so that a lane owns one r and holds 16 of the i: the accumulator layout
// is then directly the B operand [n = r, k = i] of dY^T = dO^T L and dKbar^T = s Q^T dS2, whose A operands are
// transposing LDS reads of the dO / Q rows, and dc is an in-lane sum.  dQ^T = Kbar^T dS2^T contracts over r: dS2 goes
// through 2 KB of LDS ([r][i], pitch 72 bytes: both the row writes and the transposing reads are free of conflicts) and
// Kbar^T comes from transposing reads of the chunk.
//
//   TEAM = 1 (b1 <= 32): a wave per column, four to a workgroup that share nothing; the operands of a chunk are in
//       registers (one wave per SIMD), so that the next chunk's loads run beside the whole computation.
//   TEAM = 2..4 (b1 <= 128): a workgroup of up to TEAM query tiles per column shares its chunks; a wave per tile forms L and
//       dS2 of its 32 query rows and hands them to the others through LDS, and the sums over i are split by head-dim blocks,
//       a pair of them of one matrix to each of four waves (head_dim 64: two), so that every Kbar / Y row is read once and
//       every dKbar / dY row written once.
//
// Kbar, Y and the entropy terms are read as the forward arranges them (a column's rows one after the other, (f, k) order) where
// every later part is fused too, so that the forward's own can be handed over; dKbar and dY are written tile after tile, as the
// right factor reads them.
//
// TEAM = 1 is bound by HBM: Kbar, Y read and dKbar, dY written once.  At 12 heads, a = 3, f = 21, b1 = 30, b2 = 52, 1.3 GB
// in 263 us (271 before its rows were fetched at once), where the kernel without dQ took 306 and a second one that read Kbar
// again for dQ 117.  A team is bound by the latency of its own steps, 5200 cycles a chunk of 32 rows, of which 400 wait
// for the rows.  Three frames tied (b1 = 90): against 21 frames 113 us, nine frames block-causal (a = f = 3, a third of the rows
// left out, 565 MB) 143; that was 175 while the column's own rows came a row group after the other (20 000 cycles before the
// first chunk), three waves shared four pairs of head-dim blocks (8400 cycles a chunk; 6600 so) and every request and store
// worked out its row for either arrangement.  A grid slice per 32 query rows, which read the rows three times and wrote partial
// sums, took 352, the kernel that added them 179 and dQ 175.

#include <hip/hip_runtime.h>

#include <type_traits>

#include "sfm_attn.h"
#include "sfm_common.hpp"

namespace sfm {
namespace {

struct LeftArgs {
    const char* q;           // callers' tensors: row i of (unit, a, j) is token qmap.row(a, i) + j; strides batch, token, head
    const char* dout;        // (in elements); out, optional, shares dout's strides
    const char* out;
    int64_t qs[3], os[3];
    TokMap qmap;
    int H;
    // A column's rows x are taken in the order of kbar: with r_pad > 0, the forward's arrangement, x = f * b1 + k at ((u * AJ + aj) *
    // r_pad + x) * D; else x = r = k * nf + f at ((u * RR + r) * AJ + aj) * D
    const uint16_t* kbar;
    const uint16_t* y;
    int r_pad;
    const float* c;          // r_pad > 0: [u][r_pad][AJ], log2 units; else c_rows == 0: [u][aj][RR], natural log units; c_rows == 1:
    int c_rows;              // [(u * RR + r) * AJ + aj], log2 units
    uint16_t* dkbar;         // row r = k * nf + f of (u, aj) at ((u * RR + r) * AJ + aj) * D
    uint16_t* dy;
    float* dc;               // [u][aj][RR], in the order of kbar's rows
    uint16_t* ds2;           // optional: [u][aj][b1][ds2_ld], ds2_ld >= RR
    int ds2_ld;
    float* dq;               // optional: s sum_r dS2 Kbar, in the query's rows with strides dqs (dq_rows), else [u][aj][i][D]
    int64_t dqs[3];
    bool dq_rows;
    const float* stats;      // optional, with out:      // log2-sum-exp of the logits of row (unit, aj, i) at ((unit0 + u) * AJ + aj) * stats_ld + i
    int stats_ld, unit0;
    int b1, b2, AJ, nf, RR, causal;
    float scale;
    int nunits;              // units of this launch
    bool skip;               // only the rows r that a column sees are read and written (block-causal)
};

typedef short bl_s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 bl_read_tr(const char* lds, uint32_t off) {
    bl_s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((bl_s16x4 __attribute__((address_space(3)))*)(lds + off));
    return __builtin_bit_cast(u32x2, v);
}

template <int CPR>
__device__ __forceinline__ int bl_swz(int r) {
    return CPR >= 16 ? (((r & 3) << 2) | ((r >> 2) & 3)) : ((((r >> 1) & 1) << 2) | ((r >> 2) & 3));
}
// (through the caches: teams that read past them gain 1 % where only a new chunk's keys get gradients, and with all keys take up to 2 %
// longer, 12 heads x 128 of 30 x 52 in half-height blocks, three tied, 15 frames: 600, 610 us)
__device__ __forceinline__ void bl_load_lds16(const char* base, uint32_t off, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(base) : "memory", "m0");
}
// the same with the LDS address as a scalar base plus a compile-time offset (one scalar register for all of a chunk's loads), past
// the caches: Kbar and Y are read once here, and what they would displace is read again (training step, 12 heads, three frames
// against 21: 931 -> 899 us; 6 against themselves 335 -> 325)
template <int OFF>
__device__ __forceinline__ void bl_load_lds16_at(const char* base, uint32_t off, uint32_t lds_base) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_base), "v"(off), "s"(base), "n"(OFF) : "memory", "m0", "scc");
}
template <int OFF>
__device__ __forceinline__ void bl_load_lds4_at(const char* base, uint32_t off, uint32_t lds_base) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds_base), "v"(off), "s"(base), "n"(OFF) : "memory", "m0", "scc");
}

template <int D, int TEAM>
struct LeftLds {
    static constexpr int kPitch = 2 * D, kTile = 32 * kPitch;
    static constexpr int kXPitch = 72, kX = 32 * kXPitch;              // a [r][i] matrix
    // TEAM = 1: of a wave, else of the workgroup: q tiles | dO tiles | dO . O | Kbar chunk | Y chunk | c (twice) | per wave
    // dS2 and, in a team, L | the waves' parts of dc
    static constexpr int kDot = 2 * TEAM * kTile;
    static constexpr int kChunk = kDot + TEAM * 128;
    static constexpr int kC = kChunk + 2 * kTile;
    static constexpr int kXs = kC + 256;
    static constexpr int kXWave = TEAM == 1 ? kX : 2 * kX;
    static constexpr int kDc = kXs + TEAM * kXWave;
    static constexpr int kBytes = (kDc + (TEAM == 1 ? 0 : TEAM * 128) + 255) / 256 * 256;
    // a team has a wave per query tile and at least one per pair of head-dim blocks of the two matrices of gradient rows
    static constexpr int kWaves = TEAM == 1 ? 4 : TEAM > D / 32 ? TEAM : D / 32;
    static __host__ __device__ constexpr size_t bytes() { return (size_t)(TEAM == 1 ? 4 : 1) * kBytes; }
};

// FK: Kbar, Y and c are in the forward's arrangement (r_pad > 0), and no dS2 is wanted; the row arithmetic of the other
// arrangement took a quarter of a team's instructions
template <class E, int D, int TEAM, bool FK>
__global__ __launch_bounds__((64 * LeftLds<D, TEAM>::kWaves)) __attribute__((amdgpu_waves_per_eu(TEAM == 1 ? 1 : 2, TEAM == 1 ? 1 : 2)))
void monarch_bwd_left_kernel(LeftArgs p) {
    using L = LeftLds<D, TEAM>;
    constexpr int DS = D / 16, DT = D / 32, CPR = D / 8, NG = CPR / 2;      // NG: 1 KB pieces of a tile
    constexpr int kPitch = L::kPitch, kTile = L::kTile, kXPitch = L::kXPitch;
    constexpr bool SOLO = TEAM == 1;
    constexpr int WAVES = L::kWaves;
    extern __shared__ __attribute__((aligned(256))) char lds[];

    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per_wg = SOLO ? 4 : 1;                      // columns of a workgroup
    const int njg = (p.AJ + per_wg - 1) / per_wg;
    const int item = xcd_item(njg * p.nunits);            // (unit, group of columns), one contiguous range of items per XCD
    if (item >= njg * p.nunits) return;
    const int aj = item % njg * per_wg + (SOLO ? wave : 0);
    if (aj >= p.AJ) return;                               // a lone wave: nothing is shared
    const int u = item / njg;
    const int w = SOLO ? 0 : wave;                        // this wave's query tile
    const bool has_tile = SOLO || WAVES == TEAM || wave < TEAM;        // uniform: the others join for the gradient rows
    const int i0 = 32 * w;
    const int RR = p.RR, b1 = p.b1;
    const int64_t uaj = (int64_t)u * p.AJ + aj;

    char* const base = lds + (SOLO ? wave * L::kBytes : 0);
    char* const qt = base;                                // TEAM query tiles
    char* const qs = qt + w * kTile;
    char* const dos = qs + TEAM * kTile;                  // behind the query tiles TEAM dO tiles
    float* const dls = (float*)(base + L::kDot + w * 128);
    char* const xds = base + L::kXs + w * L::kXWave;      // this wave's dS2
    const bool saved = p.stats != nullptr;                // uniform: the forward's output and row statistics are at hand
    // The column's query, dO (and output) rows: all of a wave's loads on their way at once, and behind them those of the first
    // chunk (one row group after the other waited out the latency of each: 20 000 cycles before the first chunk)
    u32x4 q_in[NG], do_in[NG], out_in[NG];
    const int ch0 = lane % CPR, r0 = lane / CPR;          // piece g of a wave: 16 bytes of row r0 + g (64 / CPR)
    {
        const int unit = p.unit0 + u, bb = unit / p.H, hh = unit % p.H;
        const int a_q = aj / p.b2, j_q = aj % p.b2;
        const char* qg = p.q + ((int64_t)bb * p.qs[0] + (int64_t)hh * p.qs[2]) * 2 + ch0 * 16;
        const char* dg = p.dout + ((int64_t)bb * p.os[0] + (int64_t)hh * p.os[2]) * 2 + ch0 * 16;
        const char* og = saved ? p.out + ((int64_t)bb * p.os[0] + (int64_t)hh * p.os[2]) * 2 + ch0 * 16 : dg;
        const int64_t tok0 = p.qmap.row(a_q, 0) + j_q;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int i = i0 + r0 + g * (64 / CPR);
            q_in[g] = do_in[g] = out_in[g] = u32x4{0u, 0u, 0u, 0u};
            if (i < b1) {                                 // no row of a wave without a tile
                const int64_t tok = tok0 + p.qmap.row_delta(i);
                q_in[g] = *(const u32x4*)(qg + tok * p.qs[1] * 2);
                do_in[g] = *(const u32x4*)(dg + tok * p.os[1] * 2);
                if (saved) out_in[g] = *(const u32x4*)(og + tok * p.os[1] * 2);
            }
        }
    }

    const int a_blk = aj / p.b2;
    const int flim = p.causal ? min(p.nf, (a_blk / p.causal + 1) * p.causal) : p.nf;      // visible kv block-frames
    const int64_t rstride = (int64_t)p.AJ * D;                                           // elements between rows r, r + 1
    const int64_t kbar0 = (FK ? uaj * p.r_pad : (int64_t)u * RR * p.AJ + aj) * D;
    const char* const kbb = (const char*)(p.kbar + kbar0);
    const char* const ybb = (const char*)(p.y + kbar0);
    const char* const cpb = (const char*)(FK ? p.c + (int64_t)u * p.r_pad * p.AJ + aj : p.c_rows ? p.c + (int64_t)u * RR * p.AJ + aj : p.c + uaj * RR);
    const float cmul = FK || p.c_rows ? 1.f : kLog2e;
    const float sc2 = p.scale * kLog2e;
    // The rows of a column, in order: all of them, or (skip) those of its flim visible block-frames, which come first in the
    // forward's arrangement
    const bool skip = p.skip && flim < p.nf;              // uniform
    const int RV = skip ? b1 * flim : RR;
    const int nch = (RV + 31) / 32;
    auto row_of = [&](int x) { return !FK && skip ? x / flim * p.nf + x % flim : x; };       // in Kbar, Y, c, dc
    const float inv_b1 = 1.f / (float)b1;
    auto grad_row = [&](int x) {                          // in dKbar, dY
        if (!FK) return row_of(x);
        const int f = (int)(((float)x + 0.5f) * inv_b1);  // x / b1, exact while x < 2^22
        return (x - f * b1) * p.nf + f;
    };

    // A chunk of 32 rows r goes from global memory into LDS (a row's 2 D bytes by consecutive lanes); there is one chunk
    // buffer.  A lone wave fills its operand registers from it and requests the next chunk at once; a team reads the operands
    // where they are used, and each wave requests its share of the next chunk when all of them are done with this one.
    char* const kt = base + L::kChunk;
    const uint32_t kt0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(size_t)(__attribute__((address_space(3))) char*)kt);
    const uint32_t rsb = FK ? (uint32_t)kPitch : (uint32_t)(rstride * 2), csb = (uint32_t)((FK || p.c_rows ? p.AJ : 1) * 4);
    auto piece_off = [&](int n, int g) {
        const int P = g * 64 + lane;
        const int r = P / CPR, c = (P % CPR) ^ bl_swz<CPR>(r);
        return (uint32_t)row_of(min(32 * n + r, RV - 1)) * rsb + (uint32_t)c * 16;
    };
    auto request_piece = [&](int n, auto g_c) {
        constexpr int g = decltype(g_c)::value;
        const uint32_t off = piece_off(n, g);
        bl_load_lds16_at<g * 1024>(kbb, off, kt0);
        bl_load_lds16_at<kTile + g * 1024>(ybb, off, kt0);
    };
    auto request = [&](int n) {
        if constexpr (SOLO) {
            request_piece(n, std::integral_constant<int, 0>{});
            request_piece(n, std::integral_constant<int, 1>{});
            request_piece(n, std::integral_constant<int, 2>{});
            request_piece(n, std::integral_constant<int, 3>{});
            if constexpr (NG > 4) {
                request_piece(n, std::integral_constant<int, 4>{});
                request_piece(n, std::integral_constant<int, 5>{});
                request_piece(n, std::integral_constant<int, 6>{});
                request_piece(n, std::integral_constant<int, 7>{});
            }
        } else {
#pragma unroll
            for (int q0 = 0; q0 < 2 * NG; q0 += WAVES) {
                const int q = q0 + wave;
                if (2 * NG % WAVES == 0 || q < 2 * NG) bl_load_lds16(q < NG ? kbb : ybb, piece_off(n, q % NG), kt0 + (uint32_t)q * 1024);
            }
        }
        if (SOLO || wave == WAVES - 1) bl_load_lds4_at<2 * kTile>(cpb, (uint32_t)row_of(min(32 * n + m, RV - 1)) * csb, kt0);
    };
    const uint32_t b_off = (uint32_t)m * kPitch + (uint32_t)((hf ^ bl_swz<CPR>(m)) << 4);     // row m of a tile as an operand
    // transposing reads of a tile: lane (m, hf) gets, for head-dim column 32 dt + m, rows 16 ks + 4 hf + {0..3} and + 8 +
    // {0..3}, the order in which the packed accumulators hold them (two reads); for dt: tr[dt & 1] ^ (dt / 2) 128
    uint32_t tr[2][2], trx;
    {
        const int s16 = lane & 15, g16 = lane >> 4;
        const int rl = 4 * hf + (s16 >> 2);
        const int cl = 2 * (g16 & 1) + ((s16 & 3) >> 1);
#pragma unroll
        for (int dl = 0; dl < 2; ++dl)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int r = rl + 8 * half;             // swz depends on r mod 16 only
                tr[dl][half] = (uint32_t)(r * kPitch + (((4 * dl + cl) ^ bl_swz<CPR>(r)) << 4) + (s16 & 1) * 8);
            }
        trx = (uint32_t)(rl * kXPitch + cl * 16 + (s16 & 1) * 8);
    }
    auto read_t = [&](const char* tile, int dl, int dp, int ks) {
        const u32x2 lo = bl_read_tr(tile, (tr[dl][0] ^ (uint32_t)(dp << 7)) + ks * 16 * kPitch);
        const u32x2 hi = bl_read_tr(tile, (tr[dl][1] ^ (uint32_t)(dp << 7)) + ks * 16 * kPitch);
        return u32x4{lo.x, lo.y, hi.x, hi.y};
    };

    u32x4 kcur[SOLO ? DS : 1], ycur[SOLO ? DS : 1], ktr[SOLO ? DT : 1][2];
    float ccur = 0.f;
    // The gradient rows' store instructions that a wave issues behind a request: they may stay in flight when the requested
    // chunk is waited for (vector memory operations complete in order)
    constexpr int kStores = SOLO ? 4 * DT : 4;
    const bool stores = SOLO || wave < DT;                // uniform
    // waits for the chunk requested last (`stored`: gradient rows were stored since); a lone wave fills its registers from it
    // and requests chunk `next`
    auto open_chunk = [&](int next, bool want_t, bool stored) {
        if (stored && stores) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kStores) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if constexpr (SOLO) {
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
                kcur[ds] = *(const u32x4*)(kt + (b_off ^ (uint32_t)(ds << 5)));
                ycur[ds] = *(const u32x4*)(kt + kTile + (b_off ^ (uint32_t)(ds << 5)));
            }
            if (want_t) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks) ktr[dt][ks] = read_t(kt, dt & 1, dt >> 1, ks);
            }
        } else {
            lds_barrier();         // every wave's share is there; every wave is done with what was handed over before
        }
        ccur = *(const float*)(base + L::kC + m * 4) * cmul;
        if constexpr (SOLO) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the registers are filled: the buffer may be overwritten
            if (next >= 0) request(next);
        }
    };
    // a team is done with the chunk (and what it hands over is there): chunk `next` may be requested
    auto close_chunk = [&](int next) {
        if constexpr (!SOLO) {
            lds_barrier();
            if (next >= 0) request(next);
        }
    };
    // logits S2[i, r] and dLm[i, r]: lane -> r = 32 n + m, register v -> i = i0 + 8 (v >> 2) + 4 hf + (v & 3)
    auto products = [&](f32x16& s, f32x16& d) {
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = d[v] = 0.f;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            const uint32_t at = b_off ^ (uint32_t)(ds << 5);
            const u32x4 qb = *(const u32x4*)(qs + at);
            const u32x4 db = *(const u32x4*)(dos + at);
            if constexpr (SOLO) {
                s = E::mfma32(qb, kcur[ds], s);
                d = E::mfma32(db, ycur[ds], d);
            } else {
                s = E::mfma32(qb, *(const u32x4*)(kt + at), s);
                d = E::mfma32(db, *(const u32x4*)(kt + kTile + at), d);
            }
        }
    };
    auto row_ok = [&](int n) {
        const int r = 32 * n + m;
        return FK ? r < b1 * flim : r < RV && (skip || r % p.nf < flim);
    };

    request(0);
    if (has_tile) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int r = r0 + g * (64 / CPR);
            const int at = r * kPitch + ((ch0 ^ bl_swz<CPR>(r)) << 4);
            *(u32x4*)(qs + at) = q_in[g];
            *(u32x4*)(dos + at) = do_in[g];
            if (saved) {                                      // sum_r L dLm of row i is dO_i . O_i
                float dot = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    dot += E::to_float((uint16_t)(do_in[g][e] & 0xffffu)) * E::to_float((uint16_t)(out_in[g][e] & 0xffffu)) +
                           E::to_float((uint16_t)(do_in[g][e] >> 16)) * E::to_float((uint16_t)(out_in[g][e] >> 16));
#pragma unroll
                for (int o = 1; o < CPR; o <<= 1) dot += __shfl_xor(dot, o);
                if (ch0 == 0) dls[r] = dot;
            }
        }
    }
    if (SOLO) lds_wave_sync();
    else lds_barrier();

    float lse[16], delta[16];
    if (saved) {
        const float* st = p.stats + ((int64_t)(p.unit0 + u) * p.AJ + aj) * p.stats_ld;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int i = 8 * (v >> 2) + 4 * hf + (v & 3);
            lse[v] = i0 + i < b1 ? st[i0 + i] : INFINITY;      // no row: its weights are zero
            delta[v] = dls[i];
        }
    } else {
        // ---- pass 1: per lane, for its 16 rows i, the running maximum, sum and sum of L dLm over the lane's own r
        float mloc[16], lloc[16], dloc[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            mloc[v] = -INFINITY;
            lloc[v] = dloc[v] = 0.f;
        }
        for (int n = 0; n < nch; ++n) {
            const int next = n + 1 < nch ? n + 1 : 0;      // after the last chunk the first one, for pass 2
            open_chunk(next, false, false);
            f32x16 s, d;
            if (has_tile) products(s, d);
            const float cl2 = ccur;
            close_chunk(next);
            if (!has_tile) continue;
            const bool ok = row_ok(n);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float z = ok ? s[v] * sc2 - cl2 : -INFINITY;
                const float mnew = fmaxf(mloc[v], z);
                const float mref = mnew == -INFINITY ? 0.f : mnew;
                const float alpha = fast_exp2(mloc[v] - mref), e = fast_exp2(z - mref);
                lloc[v] = lloc[v] * alpha + e;
                dloc[v] = dloc[v] * alpha + e * d[v];
                mloc[v] = mnew;
            }
        }
        // merge over the 32 lanes of a half (they hold the same rows i); every row has at least one visible r
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            float mm = mloc[v], ll = lloc[v], dd = dloc[v];
#pragma unroll
            for (int o = 1; o < 32; o <<= 1) {
                const float m2 = __shfl_xor(mm, o), l2 = __shfl_xor(ll, o), d2 = __shfl_xor(dd, o);
                const float mnew = fmaxf(mm, m2);
                const float mref = mnew == -INFINITY ? 0.f : mnew;
                const float a1 = fast_exp2(mm - mref), a2 = fast_exp2(m2 - mref);
                ll = ll * a1 + l2 * a2;
                dd = dd * a1 + d2 * a2;
                mm = mnew;
            }
            lse[v] = mm + log2f(ll);
            delta[v] = dd / ll;
        }
    }

    // ---- pass 2: gradients
    uint16_t* const dkb = p.dkbar + ((int64_t)u * RR * p.AJ + aj) * D;
    uint16_t* const dyb = p.dy + ((int64_t)u * RR * p.AJ + aj) * D;
    float* const dcp = p.dc + uaj * RR;
    f32x16 dqa[DT];                                       // dQ^T[d = 32 dt + 8 g + 4 hf + e, i = i0 + m] / s
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) dqa[dt][v] = 0.f;

    for (int n = 0; n < nch; ++n) {
        const int next = n + 1 < nch ? n + 1 : -1;
        open_chunk(next, true, n > 0);
        const bool r_in = 32 * n + m < RV;
        const int r = row_of(32 * n + m);
        u32x4 pl[2], pg[2];                              // B operands [n = r, k = i] for the two steps of 16 rows i
        if (has_tile) {
            f32x16 s, d;
            products(s, d);
            const float cl2 = ccur;
            const bool ok = row_ok(n);
            float dsum = 0.f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float pv = ok ? fast_exp2(s[v] * sc2 - cl2 - lse[v]) : 0.f;
                const float gv = pv * (d[v] - delta[v]);
                s[v] = pv;                                   // L[i, r]
                d[v] = gv;                                   // dS2[i, r]
                dsum += gv;
            }
            dsum = xhalf_sum(dsum);
            if (SOLO) {
                if (r_in && hf == 0) dcp[r] = -dsum;
            } else if (hf == 0) {
                *(float*)(base + L::kDc + w * 128 + m * 4) = dsum;
            }
            if (!FK && p.ds2 && r_in) {
                uint16_t* const ds2p = p.ds2 + uaj * b1 * p.ds2_ld;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int i = i0 + 8 * (v >> 2) + 4 * hf + (v & 3);
                    if (i < b1) ds2p[(int64_t)i * p.ds2_ld + r] = E::from_float(d[v]);
                }
            }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                pl[ks].x = pack2<E>(s[8 * ks + 0], s[8 * ks + 1]); pl[ks].y = pack2<E>(s[8 * ks + 2], s[8 * ks + 3]);
                pl[ks].z = pack2<E>(s[8 * ks + 4], s[8 * ks + 5]); pl[ks].w = pack2<E>(s[8 * ks + 6], s[8 * ks + 7]);
                pg[ks].x = pack2<E>(d[8 * ks + 0], d[8 * ks + 1]); pg[ks].y = pack2<E>(d[8 * ks + 2], d[8 * ks + 3]);
                pg[ks].z = pack2<E>(d[8 * ks + 4], d[8 * ks + 5]); pg[ks].w = pack2<E>(d[8 * ks + 6], d[8 * ks + 7]);
                char* const x = xds + m * kXPitch + (16 * ks + 4 * hf) * 2;
                *(u32x2*)x = u32x2{pg[ks].x, pg[ks].y};
                *(u32x2*)(x + 16) = u32x2{pg[ks].z, pg[ks].w};
                if (!SOLO) {
                    *(u32x2*)(x + L::kX) = u32x2{pl[ks].x, pl[ks].y};
                    *(u32x2*)(x + L::kX + 16) = u32x2{pl[ks].z, pl[ks].w};
                }
            }
            lds_wave_sync();
            if (p.dq) {
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    const u32x2 lo = bl_read_tr(xds, trx + ks * 16 * kXPitch);
                    const u32x2 hi = bl_read_tr(xds, trx + (8 + ks * 16) * kXPitch);
                    const u32x4 bop = {lo.x, lo.y, hi.x, hi.y};
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) {
                        if constexpr (SOLO) dqa[dt] = E::mfma32(ktr[dt][ks], bop, dqa[dt]);
                        else dqa[dt] = E::mfma32(read_t(kt, dt & 1, dt >> 1, ks), bop, dqa[dt]);
                    }
                }
            }
        }
        close_chunk(next);
        if (!SOLO && wave == WAVES - 1 && r_in && hf == 0) {
            float t = 0.f;
#pragma unroll
            for (int x = 0; x < TEAM; ++x) t += *(const float*)(base + L::kDc + x * 128 + m * 4);
            dcp[r] = -t;
        }
        // dY^T[d, r] = sum_i dO^T[d, i] L[i, r],  dKbar^T[d, r] = s sum_i Q^T[d, i] dS2[i, r], 64 head-dim rows at a time.
        // A lane (r, hf) holds head-dim 32 dt + 8 g + 4 hf + 0..3 of its row r.  A half swap (v_permlane32_swap) leaves 8
        // consecutive ones per lane; then, over a pair of head-dim blocks, lane bit 4 is traded for the piece pair
        // (v_permlane16_swap) and lane bit 3 for the block within the pair (a rotation by 8 within rows of 16 lanes),
        // after which a lane holds the 16-byte piece 4 (bit 3) + 2 (bit 4) + hf of the rows (r & 7) + 8 rb, rb = 0..3:
        // one store instruction writes 128 contiguous bytes of each of 8 rows.
        uint64_t rowoff[4];                              // bytes
        bool row_in[4];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
            const int rr = 32 * n + (m & 7) + 8 * rb;
            row_in[rb] = rr < RV;
            rowoff[rb] = (uint64_t)(uint32_t)grad_row(min(rr, RV - 1)) * (uint32_t)(rstride * 2) + (4 * ((m >> 3) & 1) + 2 * ((m >> 4) & 1) + hf) * 16;
        }
        // N pairs of head-dim blocks from dp0 on: 2 N independent chains of matrix instructions that share their B operands
        auto half_rows = [&](int which, int dp0, auto n_c) {
            constexpr int N = decltype(n_c)::value;
            const char* const src = qt + (which == 0 ? TEAM * kTile : 0);
            char* const obase = (char*)(which == 0 ? dyb : dkb);
            const float osc = which == 0 ? 1.f : p.scale;
            u32x4 bop[TEAM][2];
#pragma unroll
            for (int t = 0; t < TEAM; ++t)
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    if constexpr (SOLO) {
                        bop[t][ks] = which == 0 ? pl[ks] : pg[ks];
                    } else {
                        const char* x = base + L::kXs + t * L::kXWave + (which == 0 ? L::kX : 0) + m * kXPitch + (16 * ks + 4 * hf) * 2;
                        const u32x2 lo = *(const u32x2*)x, hi = *(const u32x2*)(x + 16);
                        bop[t][ks] = u32x4{lo.x, lo.y, hi.x, hi.y};
                    }
                }
            f32x16 o[2 * N];
#pragma unroll
            for (int x = 0; x < 2 * N; ++x)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[x][v] = 0.f;
#pragma unroll
            for (int t = 0; t < TEAM; ++t)
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int x = 0; x < 2 * N; ++x) o[x] = E::mfma32(read_t(src + t * kTile, x & 1, dp0 + (x >> 1), ks), bop[t][ks], o[x]);
#pragma unroll
            for (int dp = 0; dp < N; ++dp) {
                uint32_t wd[2][2][4];                    // [block in pair][gp][dword]
#pragma unroll
                for (int dl = 0; dl < 2; ++dl) {
                    const f32x16& a = o[2 * dp + dl];
#pragma unroll
                    for (int gp = 0; gp < 2; ++gp) {
                        const int g0 = 2 * gp, g1 = 2 * gp + 1;
                        auto rx = __builtin_amdgcn_permlane32_swap(pack2<E>(a[4 * g0 + 0] * osc, a[4 * g0 + 1] * osc),
                                                                   pack2<E>(a[4 * g1 + 0] * osc, a[4 * g1 + 1] * osc), false, false);
                        auto ry = __builtin_amdgcn_permlane32_swap(pack2<E>(a[4 * g0 + 2] * osc, a[4 * g0 + 3] * osc),
                                                                   pack2<E>(a[4 * g1 + 2] * osc, a[4 * g1 + 3] * osc), false, false);
                        wd[dl][gp][0] = rx[0]; wd[dl][gp][1] = ry[0]; wd[dl][gp][2] = rx[1]; wd[dl][gp][3] = ry[1];
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        auto x = __builtin_amdgcn_permlane16_swap(wd[dl][0][q], wd[dl][1][q], false, false);
                        wd[dl][0][q] = x[0]; wd[dl][1][q] = x[1];
                    }
                }
#pragma unroll
                for (int r4 = 0; r4 < 2; ++r4) {
                    u32x4 lo, hi;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t x0 = wd[0][r4][q], x1 = wd[1][r4][q];
                        // row_ror:8 within 16 lanes; bank mask 0xc writes lanes 8..15 of a row, 0x3 lanes 0..7
                        lo[q] = (uint32_t)__builtin_amdgcn_update_dpp((int)x0, (int)x1, 0x128, 0xf, 0xc, false);
                        hi[q] = (uint32_t)__builtin_amdgcn_update_dpp((int)x1, (int)x0, 0x128, 0xf, 0x3, false);
                    }
                    // non-temporal: the rows are read once, by the right factor's kernel, after this grid has finished.  Before
                    // the last chunk every row exists, and the stores are counted by open_chunk.
                    char* const at_lo = obase + (rowoff[2 * r4 + 0] + 128 * (dp0 + dp));
                    char* const at_hi = obase + (rowoff[2 * r4 + 1] + 128 * (dp0 + dp));
                    if (next >= 0) {
                        __builtin_nontemporal_store(lo, (u32x4*)at_lo);
                        __builtin_nontemporal_store(hi, (u32x4*)at_hi);
                    } else {
                        if (row_in[2 * r4 + 0]) __builtin_nontemporal_store(lo, (u32x4*)at_lo);
                        if (row_in[2 * r4 + 1]) __builtin_nontemporal_store(hi, (u32x4*)at_hi);
                    }
                }
            }
        };
        if constexpr (SOLO) {
            half_rows(0, 0, std::integral_constant<int, DT / 2>{});
            half_rows(1, 0, std::integral_constant<int, DT / 2>{});
        } else if (stores) {
            half_rows(wave / (DT / 2), wave % (DT / 2), std::integral_constant<int, 1>{});
        }
    }
    if (p.dq && i0 + m < b1) {
        float* row;
        if (p.dq_rows) {
            const int unit = p.unit0 + u;
            row = p.dq + (int64_t)(unit / p.H) * p.dqs[0] + (p.qmap.row(a_blk, i0 + m) + aj % p.b2) * p.dqs[1] + (int64_t)(unit % p.H) * p.dqs[2];
        } else {
            row = p.dq + (uaj * b1 + i0 + m) * D;
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *(f32x4*)(row + 32 * dt + 8 * g + 4 * hf) = f32x4{dqa[dt][4 * g] * p.scale, dqa[dt][4 * g + 1] * p.scale,
                                                                  dqa[dt][4 * g + 2] * p.scale, dqa[dt][4 * g + 3] * p.scale};
    }
}

template <class E, int D, int TEAM, bool FK>
int launch_left(const LeftArgs& a, hipStream_t stream) {
    const size_t ldsb = LeftLds<D, TEAM>::bytes();
    const void* fn = (const void*)monarch_bwd_left_kernel<E, D, TEAM, FK>;
    hipError_t e = hipSuccess;
    if (ldsb > 64 * 1024) e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ldsb);
    if (e != hipSuccess) {
        set_error("monarch backward (left factor): cannot reserve %zu bytes of LDS: %s", ldsb, hipGetErrorString(e));
        return SFM_ERR_HIP;
    }
    const int per_wg = TEAM == 1 ? 4 : 1;
    const dim3 grid((unsigned)xcd_grid((a.AJ + per_wg - 1) / per_wg * a.nunits)), block(64 * LeftLds<D, TEAM>::kWaves);
    LeftArgs arg = a;
    void* kargs[] = {&arg};
    e = hipLaunchKernel(fn, grid, block, kargs, ldsb, stream);
    if (e != hipSuccess) {
        set_error("monarch backward (left factor): launch failed: %s", hipGetErrorString(e));
        return SFM_ERR_HIP;
    }
    return SFM_OK;
}

template <class E, int D, int TEAM>
int launch_left(const LeftArgs& a, hipStream_t stream) {
    return a.r_pad > 0 ? launch_left<E, D, TEAM, true>(a, stream) : launch_left<E, D, TEAM, false>(a, stream);
}

template <class E, int D>
int launch_left(const LeftArgs& a, hipStream_t stream) {
    return a.b1 <= 32 ? launch_left<E, D, 1>(a, stream) : a.b1 <= 64 ? launch_left<E, D, 2>(a, stream)
         : a.b1 <= 96 ? launch_left<E, D, 3>(a, stream) : launch_left<E, D, 4>(a, stream);
}

}  // namespace

bool monarch_bwd_left_supported(int dtype, int D, int b1) {
    return (dtype == SFM_BF16 || dtype == SFM_F16) && (D == 64 || D == 128) && b1 >= 1 && b1 <= 128;
}

int launch_monarch_bwd_left(int dtype, int D, int n, int b1, int b2, int AJ, int nf, int causal, float scale, const void* q,
                            const int64_t* qs, const void* dout, const void* out, const int64_t* os, const TokMap& qmap, int H,
                            int unit0, const void* kbar, const void* y, const float* c, int r_pad, int c_rows, void* dkbar, void* dy, float* dc,
                            void* ds2, int ds2_ld, float* dq, const int64_t* dqs, const float* stats, int stats_ld, bool skip_masked,
                            hipStream_t stream) {
    LeftArgs a;
    a.ds2_ld = ds2_ld;
    a.q = (const char*)q; a.dout = (const char*)dout; a.out = (const char*)out;
    for (int i = 0; i < 3; ++i) {
        a.qs[i] = qs[i];
        a.os[i] = os[i];
        a.dqs[i] = dqs ? dqs[i] : 0;
    }
    a.dq = dq;
    a.dq_rows = dqs != nullptr;
    a.qmap = qmap;
    a.H = H;
    a.stats = out ? stats : nullptr; a.stats_ld = stats_ld; a.unit0 = unit0;
    a.c_rows = c_rows;
    a.r_pad = r_pad;
    a.kbar = (const uint16_t*)kbar; a.y = (const uint16_t*)y;
    a.c = c;
    a.dkbar = (uint16_t*)dkbar; a.dy = (uint16_t*)dy;
    a.dc = dc;
    a.ds2 = (uint16_t*)ds2;
    a.b1 = b1; a.b2 = b2; a.AJ = AJ; a.nf = nf; a.RR = nf * b1; a.causal = causal;
    a.scale = scale;
    a.nunits = n;
    a.skip = skip_masked && causal && !ds2;
    if (dtype == SFM_BF16) return D == 128 ? launch_left<BF16, 128>(a, stream) : launch_left<BF16, 64>(a, stream);
    return D == 128 ? launch_left<F16, 128>(a, stream) : launch_left<F16, 64>(a, stream);
}

}  // namespace sfm
