// Right-factor part of the Monarch backward on gfx950 MFMA (bf16 / fp16, head_dim 64 or 128, b2 <= 64).
//
// Replaces, per tile t = (unit, k, f), the small batched products and the row kernel of the GEMM chain
//     dR[aj, l]  = dKbar[aj,:] . K[l,:] + dY[aj,:] . V[l,:]
//     dS1[aj, l] = R (dR + dc ln R - sum_l R (dR + dc ln R))
//     dK[l, :]   = sum_aj R[aj, l] dKbar[aj,:] + s sum_aj dS1[aj, l] q[aj,:]
//     dV[l, :]   = sum_aj R[aj, l] dY[aj,:]
// (wan/modules/monarch_attn.py:403-596 `_al_cl_y_bwd`).  One workgroup per tile: the K and V blocks (read where the callers'
// tensors have them) stay in LDS, the tile's rows of R, dKbar and dY (contiguous in the backward's scratch) come 64
// columns at a time (global_load_lds_dwordx4, 16-byte chunks XOR-swizzled per row as in the dense attention kernel).
//   softmax waves (4): 32 columns aj x 32 key rows l.  dR^T[l, aj] with A = K / V rows, B = dKbar / dY rows, so that a lane
//            owns one column and the softmax backward is in-lane plus one cross-half add and one exchange between the
//            two waves of a column through LDS.  dS1 (16 bit) takes the place of R.
//   gradient waves (4): 32 head-dim rows x 64 (head_dim 64: 32) key rows of dV and of dK, C^T[d, l] with both operands from
//            transposing LDS reads (ds_read_tr16_b64): A = dY^T / dKbar^T / q^T, B = R or dS1, contraction over the columns
//            aj.  The products with R run beside the softmax waves; the query rows of (unit, k) then load over the dY tile.
// dS1 is also written to memory (16 bit) for dQ = s dS1 K, which contracts over f across tiles (monarch_bwd_dqk_kernel
// below).
//
// Bound by HBM and its latency: dKbar, dY, R read and dS1 written once, 0.87 GB at 12 heads x 128, a = 3, f = 21, b1 = 30,
// b2 = 52: 262 us.  64 columns because two workgroups then share a compute unit and one's loads run beside the other's
// products: sixteen waves with 160 columns, which filled the LDS alone, took 336 us there, and as long for 52 columns as for 160.

#include <hip/hip_runtime.h>

#include <type_traits>

#include "sfm_attn.h"
#include "sfm_common.hpp"

namespace sfm {
namespace {

struct RightArgs {
    const char* kk;          // callers' tensors: row kmap.row(f, k) + l, strides (batch, row, head) in elements
    const char* v;
    int64_t ks0, ks1, ks2, vs0, vs1, vs2;
    const char* rb;          // [t][AJ][64]
    const char* dkbar;       // [t][AJ][D]
    const char* dy;
    const float* dc;         // [u][AJ][RR], (k, f) of a column at k * dc_k + f * dc_f
    int dc_k, dc_f;
    const char* q;           // caller's tensor: row (a, j) of (unit, k) is token qmap.row(a, k) + j, strides qs0, qs1, qs2
    int64_t qs0, qs1, qs2;
    TokMap qmap;
    uint16_t* ds1;           // row (a, j) of tile t at u k AJ nf b2p + f ds1_f + aj ds1_aj, b2p = b2 rounded up to 4; the padding is zero
    int64_t ds1_f, ds1_aj;
    uint16_t* dk;            // caller's tensors: row kmap.row(f, k) + l - row0, strides s0 (batch), s1 (row), s2 (head)
    uint16_t* dv;
    int64_t s0, s1, s2, row0;
    TokMap kmap;
    int64_t ntiles;
    int b1, b2, AJ, nf, H, unit0, f0, f1;
    int causal;              // block-causal size: the columns before a tile's first visible one are left out; 0 = none
    float scale;
};

typedef short br_s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 br_read_tr(const char* lds, uint32_t off) {
    br_s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((br_s16x4 __attribute__((address_space(3)))*)(lds + off));
    return __builtin_bit_cast(u32x2, v);
}
__device__ __forceinline__ void br_load_lds16(const char* base, uint32_t off, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(base) : "memory", "m0");
}

// the same past the caches, for rows that are read once: dS1, which the dQ kernel reads next, and the K, V and query rows keep
// their place (forward and backward, three frames against themselves 208 -> 202 us, 21 frames 938 -> 930)
__device__ __forceinline__ void br_load_lds16_nt(const char* base, uint32_t off, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_addr), "v"(off), "s"(base) : "memory", "m0");
}
// chunk c (16 bytes) of row r sits at chunk position c ^ swz(r); rows of CPR chunks (16: 256-byte rows, 8: 128-byte rows)
template <int CPR>
__device__ __forceinline__ int br_swz(int r) {
    return CPR >= 16 ? (((r & 3) << 2) | ((r >> 2) & 3)) : ((((r >> 1) & 1) << 2) | ((r >> 2) & 3));
}

constexpr int kCols = 64;                                  // columns per chunk
constexpr int kWaves = 8, kThreads = 64 * kWaves;

template <int D>
struct RightLds {
    static constexpr int kPitch = 2 * D, kTile = 64 * kPitch;             // K, V, dKbar, dY: 64 rows
    static constexpr int oK = 0, oV = kTile, oG = 2 * kTile, oH = 3 * kTile, oR = 4 * kTile, oDot = oR + kCols * 128;
    static constexpr int kBytes = oDot + 2 * kCols * 4;
};

template <class E, int D>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void monarch_bwd_right_kernel(RightArgs p) {
    using L = RightLds<D>;
    constexpr int DS = D / 16, DT = D / 32;
    constexpr int CPR = D / 8;                            // chunks per row of the D-wide tiles
    constexpr int kPitch = L::kPitch;
    constexpr int LBW = DT / 2;                           // 32-row blocks of key rows that a gradient wave owns
    extern __shared__ __attribute__((aligned(256))) char lds[];
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds;

    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // neighbouring tiles (block-frames of one block row) run on one XCD: their query rows and the lines of their dS1 rows meet in its L2
    const int64_t t = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (t >= p.ntiles) return;
    const int b2 = p.b2, AJ = p.AJ, nf = p.nf;
    const int f = (int)(t % nf);
    const int64_t uk = t / nf;
    const int k = (int)(uk % p.b1);
    const int64_t u = uk / p.b1;
    const int unit = p.unit0 + (int)u;

    // LDS position P (16-byte units) of a tile holds chunk (P % C) ^ swz(row) of row P / C; 64 rows, those past the end repeat
    // the last one.  Key rows past the end land in rows of dK and dV that are not stored; columns are cleared below; a query
    // row that is not finite has made its column's dS1, and with it all of dK, NaN already
    auto stage = [&](const char* src, uint32_t row_bytes, int nrows, uint32_t dst, auto cpr_c, auto once_c) {
        constexpr int C = decltype(cpr_c)::value;
#pragma unroll
        for (int g = 0; g < C / kWaves; ++g) {
            const int P = (wave + g * kWaves) * 64 + lane;
            const int r = P / C, c = (P % C) ^ br_swz<C>(r);
            const uint32_t off = (uint32_t)min(r, nrows - 1) * row_bytes + (uint32_t)(c * 16), to = lds0 + dst + (uint32_t)(wave + g * kWaves) * 1024;
            if constexpr (decltype(once_c)::value) br_load_lds16_nt(src, off, to);
            else br_load_lds16(src, off, to);
        }
    };
    using c_d = std::integral_constant<int, CPR>;
    using c_r = std::integral_constant<int, 8>;
    stage(p.kk + ((int64_t)(unit / p.H) * p.ks0 + (int64_t)(unit % p.H) * p.ks2 + p.kmap.row(f, k) * p.ks1) * 2, (uint32_t)(p.ks1 * 2), b2,
          L::oK, c_d{}, std::false_type{});
    stage(p.v + ((int64_t)(unit / p.H) * p.vs0 + (int64_t)(unit % p.H) * p.vs2 + p.kmap.row(f, k) * p.vs1) * 2, (uint32_t)(p.vs1 * 2), b2,
          L::oV, c_d{}, std::false_type{});
    const bool want = f >= p.f0 && f < p.f1;                             // uniform: dK / dV of this kv block-frame are asked for

    const char* qbase = p.q + ((int64_t)(unit / p.H) * p.qs0 + (int64_t)(unit % p.H) * p.qs2) * 2;
    const uint32_t qrb = (uint32_t)(p.qs1 * 2);
    const int ppr = (b2 + 3) / 4, b2p = 4 * ppr;                         // 8-byte pieces of a dS1 row
    const int cfirst = p.causal ? f / p.causal * p.causal * b2 : 0;      // the first column (a, j) that sees key block-frame f

    // What every wave does in a chunk; the two kinds of waves meet in the same four barriers.
    auto load_g = [&](int c0) { stage(p.dkbar + (t * AJ + c0) * kPitch, kPitch, min(kCols, AJ - c0), L::oG, c_d{}, std::true_type{}); };
    auto load_h = [&](int c0) { stage(p.dy + (t * AJ + c0) * kPitch, kPitch, min(kCols, AJ - c0), L::oH, c_d{}, std::true_type{}); };
    auto load_r = [&](int c0) { stage(p.rb + (t * AJ + c0) * 128, 128, min(kCols, AJ - c0), L::oR, c_r{}, std::true_type{}); };
    // the next chunk's rows are requested as soon as their tiles are free: dKbar (and dY, where no query rows take its place)
    // behind the products, the others at the chunk's end
    auto next_early = [&](int c1) {
        if (c1 >= AJ) return;
        load_g(c1);
        if (!want) load_h(c1);
    };
    auto next_late = [&](int c1) {
        lds_barrier();                                                   // every wave is done with this chunk
        if (c1 >= AJ) return;
        if (want) load_h(c1);
        load_r(c1);
    };
    auto loaded = [&](int nrows) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        if (nrows < kCols) {
            // Columns past the end have no weight, and nothing to weigh: what is loaded there is the last column again, and an
            // infinity of it times a weight of zero would make every row of dV and dK NaN.
            const u32x4 z = {0u, 0u, 0u, 0u};
            for (int i = tid; i < (kCols - nrows) * 8; i += kThreads) *(u32x4*)(lds + L::oR + nrows * 128 + i * 16) = z;
            for (int i = tid; i < (kCols - nrows) * CPR; i += kThreads) {
                *(u32x4*)(lds + L::oG + nrows * kPitch + i * 16) = z;
                *(u32x4*)(lds + L::oH + nrows * kPitch + i * 16) = z;
            }
            lds_barrier();
        }
    };
    auto queries = [&](int c0, int nrows) {                              // the query rows of (unit, k) take the place of the dY tile
        if (!want) return;
#pragma unroll
        for (int g = 0; g < CPR / kWaves; ++g) {
            const int P = (wave + g * kWaves) * 64 + lane;
            const int r = P / CPR, c = (P % CPR) ^ br_swz<CPR>(r);
            const int aj = c0 + min(r, nrows - 1);
            const uint32_t tok = (uint32_t)(p.qmap.row(aj / b2, k) + aj % b2);
            br_load_lds16(qbase, tok * qrb + (uint32_t)(c * 16), lds0 + L::oH + (uint32_t)(wave + g * kWaves) * 1024);
        }
    };
    auto complete = [&](int c0, int nrows) {
        if (want) {                                                      // the query rows have landed (behind them the next dKbar rows)
            if (c0 + kCols < AJ) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CPR / kWaves) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        lds_barrier();                                                   // the dS1 tile is complete
        // dS1 to memory for dQ = s dS1 K: row aj is b2p consecutive elements, 8-byte pieces, consecutive lanes along a row
        uint16_t* out = p.ds1 + uk * AJ * ((int64_t)nf * b2p) + f * p.ds1_f + c0 * p.ds1_aj;
        for (int i = tid; i < nrows * ppr; i += kThreads) {
            const int row = i / ppr, pc = i - row * ppr;
            const u32x2 w = *(const u32x2*)(lds + L::oR + row * 128 + (((pc >> 1) ^ br_swz<8>(row)) << 4) + 8 * (pc & 1));
            *(u32x2*)(out + row * p.ds1_aj + 4 * pc) = w;
        }
    };

    load_g(cfirst);
    load_h(cfirst);
    load_r(cfirst);
    if (wave < 4) {
        // ---- softmax waves: 32 columns x 32 key rows
        const int tl = wave >> 1, col = 32 * (wave & 1) + m;
        const uint32_t a_off = (uint32_t)(32 * tl + m) * kPitch + (uint32_t)((hf ^ br_swz<CPR>(m)) << 4);
        const uint32_t b_off = (uint32_t)col * kPitch + (uint32_t)((hf ^ br_swz<CPR>(m)) << 4);
        for (int c0 = cfirst; c0 < AJ; c0 += kCols) {
            const int nrows = min(kCols, AJ - c0);
            const float dcv = col < nrows ? p.dc[(u * AJ + c0 + col) * ((int64_t)nf * p.b1) + (int64_t)k * p.dc_k + f * p.dc_f] : 0.f;
            loaded(nrows);
            // dR^T[l, aj] = K dKbar^T + V dY^T, then R (16 bit) of the l this lane holds: l = 32 tl + 8 g + 4 hf + 0..3
            f32x16 dr;
            float rv[16];
            float dot = 0.f;
#pragma unroll
            for (int v = 0; v < 16; ++v) dr[v] = 0.f;
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
                const u32x4 bg = *(const u32x4*)(lds + L::oG + (b_off ^ (uint32_t)(ds << 5)));
                const u32x4 bh = *(const u32x4*)(lds + L::oH + (b_off ^ (uint32_t)(ds << 5)));
                const u32x4 ak = *(const u32x4*)(lds + L::oK + (a_off ^ (uint32_t)(ds << 5)));
                const u32x4 av = *(const u32x4*)(lds + L::oV + (a_off ^ (uint32_t)(ds << 5)));
                dr = E::mfma32(ak, bg, dr);
                dr = E::mfma32(av, bh, dr);
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const u32x2 w = *(const u32x2*)(lds + L::oR + col * 128 + (((4 * tl + g) ^ br_swz<8>(m)) << 4) + 8 * hf);
                const float r4[4] = {E::to_float((uint16_t)(w.x & 0xffffu)), E::to_float((uint16_t)(w.x >> 16)),
                                     E::to_float((uint16_t)(w.y & 0xffffu)), E::to_float((uint16_t)(w.y >> 16))};
                const int left = b2 - (32 * tl + 8 * g + 4 * hf);        // rows l of this piece that exist
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int v = 4 * g + e;
                    const float r = e < left ? r4[e] : 0.f;
                    const float gv = r > 0.f ? dr[v] + dcv * __logf(r) : 0.f;        // dR + dc ln R
                    rv[v] = r;
                    dr[v] = gv;
                    dot += r * gv;
                }
            }
            dot = xhalf_sum(dot);
            if (hf == 0) *(float*)(lds + L::oDot + (tl * kCols + col) * 4) = dot;
            lds_barrier();                                               // the dKbar, dY and R tiles are free, the sums complete
            queries(c0, nrows);
            next_early(c0 + kCols);
            // dS1 over the R tile, laid out like it (columns past the end and l >= b2 come out as zeros)
            dot = *(const float*)(lds + L::oDot + col * 4) + *(const float*)(lds + L::oDot + (kCols + col) * 4);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                u32x2 w;
                w.x = pack2<E>(rv[4 * g + 0] * (dr[4 * g + 0] - dot), rv[4 * g + 1] * (dr[4 * g + 1] - dot));
                w.y = pack2<E>(rv[4 * g + 2] * (dr[4 * g + 2] - dot), rv[4 * g + 3] * (dr[4 * g + 3] - dot));
                *(u32x2*)(lds + L::oR + col * 128 + (((4 * tl + g) ^ br_swz<8>(m)) << 4) + 8 * hf) = w;
            }
            complete(c0, nrows);
            next_late(c0 + kCols);
        }
        return;
    }

    // ---- gradient waves: 32 head-dim rows (block dt) x LBW blocks of 32 key rows of dV and of dK, C^T[d, l] = sum_aj A^T[d, aj] B[aj, l]
    const int dt = wave % DT, lb0 = DT == 4 ? 0 : (wave >> 1) & 1;
    uint32_t atr[2], btr[LBW][2];
    {
        const int s16 = lane & 15, g16 = lane >> 4;
        const int rl = 4 * hf + (s16 >> 2);
        const int cl = 2 * (g16 & 1) + ((s16 & 3) >> 1);
        const uint32_t sub = (uint32_t)(s16 & 1) * 8;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int r = rl + 8 * half;                                 // swz depends on r mod 16 only
            atr[half] = (uint32_t)(r * kPitch + (((4 * dt + cl) ^ br_swz<CPR>(r)) << 4)) + sub;
#pragma unroll
            for (int lb = 0; lb < LBW; ++lb)
                btr[lb][half] = (uint32_t)(L::oR + r * 128 + (((4 * (lb0 + lb) + cl) ^ br_swz<8>(r)) << 4)) + sub;
        }
    }
    auto read_a = [&](int tile, int ks) {
        const u32x2 lo = br_read_tr(lds, atr[0] + tile + ks * 16 * kPitch), hi = br_read_tr(lds, atr[1] + tile + ks * 16 * kPitch);
        return u32x4{lo.x, lo.y, hi.x, hi.y};
    };
    auto read_b = [&](int lb, int ks) {
        const u32x2 lo = br_read_tr(lds, btr[lb][0] + ks * 16 * 128), hi = br_read_tr(lds, btr[lb][1] + ks * 16 * 128);
        return u32x4{lo.x, lo.y, hi.x, hi.y};
    };
    f32x16 dva[LBW], dka[LBW];
#pragma unroll
    for (int lb = 0; lb < LBW; ++lb)
#pragma unroll
        for (int v = 0; v < 16; ++v) dva[lb][v] = dka[lb][v] = 0.f;
    for (int c0 = cfirst; c0 < AJ; c0 += kCols) {
        const int nrows = min(kCols, AJ - c0);
        loaded(nrows);
        if (want) {
            // dV += R^T dY, dK += R^T dKbar
#pragma unroll
            for (int ks = 0; ks < kCols / 16; ++ks) {
                const u32x4 ah = read_a(L::oH, ks), ag = read_a(L::oG, ks);
#pragma unroll
                for (int lb = 0; lb < LBW; ++lb) {
                    const u32x4 b = read_b(lb, ks);
                    dva[lb] = E::mfma32(ah, b, dva[lb]);
                    dka[lb] = E::mfma32(ag, b, dka[lb]);
                }
            }
        }
        lds_barrier();                                                   // the dKbar, dY and R tiles are free, the sums complete
        queries(c0, nrows);
        next_early(c0 + kCols);
        complete(c0, nrows);
        if (want) {
            // dK += s dS1^T q
#pragma unroll
            for (int lb = 0; lb < LBW; ++lb) {
                f32x16 x;
#pragma unroll
                for (int v = 0; v < 16; ++v) x[v] = 0.f;
#pragma unroll
                for (int ks = 0; ks < kCols / 16; ++ks) x = E::mfma32(read_a(L::oH, ks), read_b(lb, ks), x);
#pragma unroll
                for (int v = 0; v < 16; ++v) dka[lb][v] = fmaf(p.scale, x[v], dka[lb][v]);
            }
        }
        next_late(c0 + kCols);
    }
    if (!want) return;
    // lane (l, hf) holds head-dim 32 dt + 8 g + 4 hf + 0..3 of key row l; the half swap leaves 8 consecutive ones per lane
    const int64_t obase = (int64_t)(unit / p.H) * p.s0 + (int64_t)(unit % p.H) * p.s2 + (p.kmap.row(f, k) - p.row0) * p.s1;
    auto store = [&](uint16_t* dst, const f32x16& acc, int lb) {
        const int l = 32 * lb + m;
        uint16_t* row = dst + obase + min(l, b2 - 1) * p.s1 + 32 * dt + 8 * hf;
#pragma unroll
        for (int gp = 0; gp < 2; ++gp) {
            const int g0 = 8 * gp, g1 = 8 * gp + 4;
            auto rx = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[g0 + 0], acc[g0 + 1]), pack2<E>(acc[g1 + 0], acc[g1 + 1]), false, false);
            auto ry = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[g0 + 2], acc[g0 + 3]), pack2<E>(acc[g1 + 2], acc[g1 + 3]), false, false);
            const u32x4 w = {(uint32_t)rx[0], (uint32_t)ry[0], (uint32_t)rx[1], (uint32_t)ry[1]};
            if (l < b2) *(u32x4*)(row + 16 * gp) = w;
        }
    };
#pragma unroll
    for (int lb = 0; lb < LBW; ++lb) {
        store(p.dv, dva[lb], lb0 + lb);
        store(p.dk, dka[lb], lb0 + lb);
    }
}


// ---------------------------------------------------------------------------------------------------------------
// dQ of the right factor: dQk[(u, k)][aj, :] = s sum_{f, l} dS1[(u, k)][aj, (f, l)] K[(f, k, l), :], float, added to the left
// factor's part, in the caller's float rows or on the way to 16-bit ones, or written to a scratch matrix.  A workgroup
// takes up to kDqkWaves x 32 columns (a, j) of a (unit, k), a wave 32; the K rows of the nf block-frames stream through LDS 64
// at a time straight from the caller's tensor (global_load_lds_dwordx4, double buffered, chunk swizzle) and come back
// transposed as the A operand [m = d, k = (f, l)]; the B operand is dS1 straight from memory, two 8-byte pieces per step in the
// order in which the transposing reads deliver the rows, so that a lane ends up with four consecutive d of its column.
struct DqkArgs {
    const char* k;           // caller's tensor: row kmap.row(f, k) + l, strides ks0 (batch), ks1 (row), ks2 (head), in elements
    int64_t ks0, ks1, ks2;
    TokMap kmap;
    const uint16_t* ds1;     // [(u, k)][f][AJ][b2p] as the kernel above writes it
    uint32_t b2p_inv;        // 2^32 / b2p, rounded up: x / b2p is the upper half of the product for every x below 2^26
    float* dqk;              // [(u, k)][AJ][D], or (add) the caller's rows to add to: token qmap.row(a, k) + j, strides dqs
    const float* part;       // with dq16: the left factor's part, [u][AJ][b1][D]
    uint16_t* dq16;          // optional: 16-bit rows for the sum, like dqk's with add
    int64_t dqs0, dqs1, dqs2;
    TokMap qmap;
    bool add;
    int causal;              // block-causal size: dS1 beyond a column's visible block-frames is not there; 0 = none
    int b1, b2, AJ, nf, H, unit0;
    int nchunks, total;      // column chunks of a (unit, k), workgroups with work
    float scale;
};

// A (unit, k) of 156 columns as one workgroup of five waves is 360 of them for 256 compute units at 12 heads, b1 = 30: with three
// and two waves 84 -> 73 us (f = 21), and at three frames tied, block-causal (three tiles to a workgroup) 69 -> 61; five waves as
// the kernel is now 79 and 64, two 98 and 64.  Bound by its loads' latency: a tile's K rows and dS1 pieces are one tile ahead.
constexpr int kDqkWaves = 4;

template <class E, int D>
__global__ __launch_bounds__(64 * kDqkWaves) __attribute__((amdgpu_waves_per_eu(4, 4))) void monarch_bwd_dqk_kernel(DqkArgs p) {
    constexpr int DT = D / 32, CPR = D / 8;
    constexpr int kPitch = 2 * D;
    constexpr int kTile = 64 * kPitch;
    extern __shared__ __attribute__((aligned(256))) char lds[];          // two tiles of 64 K rows
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds;

    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nwaves = __builtin_amdgcn_readfirstlane((int)blockDim.x >> 6);
    const int item = xcd_item(p.total);                                  // the chunks of a (unit, k) read the same K rows
    if (item >= p.total) return;
    const int64_t uk = item / p.nchunks;
    const int col0 = (item % p.nchunks) * nwaves * 32;                   // this workgroup's first column
    const int k = (int)(uk % p.b1);
    const int unit = p.unit0 + (int)(uk / p.b1);
    const int b2 = p.b2, b2p = (b2 + 3) & ~3, AJ = p.AJ, NL = p.nf * b2p;
    auto visible = [&](int aj) { return p.causal ? min(p.nf, (aj / b2 / p.causal + 1) * p.causal) * b2p : NL; };      // elements of dS1 row aj
    const int nt = (visible(min(col0 + nwaves * 32, AJ) - 1) + 63) / 64;                       // tiles that the last column sees

    const char* kbase = p.k + ((int64_t)(unit / p.H) * p.ks0 + (int64_t)(unit % p.H) * p.ks2) * 2;
    const uint32_t krb = (uint32_t)(p.ks1 * 2);
    // LDS position P (16-byte units) of a tile holds chunk (P % CPR) ^ swz(row) of row P / CPR; row x of the flat (f, l)
    // axis is token kmap.row(x / b2p, k) + x % b2p (rows past a block's or the whole end repeat its last one; dS1 is zero there)
    auto stage = [&](int t) {
        for (int g = wave; g < CPR; g += nwaves) {
            const int P = g * 64 + lane;
            const int r = P / CPR, c = (P % CPR) ^ br_swz<CPR>(r);
            const int x = min(64 * t + r, NL - 1);
            const int f = (int)__umulhi((uint32_t)x, p.b2p_inv);
            const uint32_t tok = (uint32_t)(p.kmap.row(f, k) + min(x - f * b2p, b2 - 1));
            br_load_lds16(kbase, tok * krb + (uint32_t)(c * 16), lds0 + (uint32_t)(t & 1) * kTile + (uint32_t)g * 1024);
        }
    };
    // dS1 pieces of row aj: x = 64 t + 16 ks + 4 hf + {0..3} and + 8 + {0..3}
    const int aj0 = col0 + 32 * wave;
    const int aj = min(aj0 + m, AJ - 1);
    const uint16_t* arow = p.ds1 + uk * AJ * (int64_t)NL + aj * b2p;
    const uint32_t fstep = (uint32_t)((AJ - 1) * b2p);                  // from a row's end in one block-frame to its start in the next
    auto piece = [&](int x) { return *(const u32x2*)(arow + (uint32_t)x + __umulhi((uint32_t)x, p.b2p_inv) * fstep); };
    const int na = visible(aj);
    // of the wave's longest row; a wave past the last column only fetches tiles
    const int nwave = __builtin_amdgcn_readfirstlane(aj0 < AJ ? visible(min(aj0 + 31, AJ - 1)) : 0);
    auto load_a = [&](int t, u32x4 (&a)[4]) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int x0 = 64 * t + 16 * ks + 4 * hf;
            u32x2 lo = {0u, 0u}, hi = {0u, 0u};
            if (x0 + 4 <= na) lo = piece(x0);                            // a multiple of 4: whole pieces
            if (x0 + 12 <= na) hi = piece(x0 + 8);
            a[ks] = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
    };
    uint32_t tr[DT][2];
    {
        const int s16 = lane & 15, g16 = lane >> 4;
        const int rl = 4 * hf + (s16 >> 2);
        const int cl = 2 * (g16 & 1) + ((s16 & 3) >> 1);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int r = rl + 8 * half;             // swz depends on r mod 16 only
                tr[dt][half] = (uint32_t)(r * kPitch + (((4 * dt + cl) ^ br_swz<CPR>(r)) << 4) + (s16 & 1) * 8);
            }
    }
    f32x16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[dt][v] = 0.f;

    u32x4 acur[4], anext[4];
    stage(0);
    load_a(0, acur);
    for (int t = 0; t < nt; ++t) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();                                   // tile t is in LDS; every wave is done with tile t - 1
        if (t + 1 < nt) {
            stage(t + 1);
            load_a(t + 1, anext);
        }
        const char* tile = lds + (t & 1) * kTile;
        if (64 * t < nwave) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    const u32x2 lo = br_read_tr(tile, tr[dt][0] + ks * 16 * kPitch);
                    const u32x2 hi = br_read_tr(tile, tr[dt][1] + ks * 16 * kPitch);
                    const u32x4 kop = {lo.x, lo.y, hi.x, hi.y};
                    acc[dt] = E::mfma32(kop, acur[ks], acc[dt]);
                }
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) acur[ks] = anext[ks];
    }
    // lane (m, hf) holds d = 32 dt + 8 g + 4 hf + 0..3 of column aj0 + m
    if (aj0 + m >= AJ) return;
    const int64_t tok = p.qmap.row(aj / b2, k) + aj % b2;
    if (p.dq16) {
        const float* const from = p.part + ((uk / p.b1 * AJ + aj) * p.b1 + k) * D + 4 * hf;
        uint16_t* const to = p.dq16 + (int64_t)(unit / p.H) * p.dqs0 + (int64_t)(unit % p.H) * p.dqs2 + tok * p.dqs1 + 8 * hf;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            f32x4 x[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) x[g] = *(const f32x4*)(from + 32 * dt + 8 * g);
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[g][e] += acc[dt][4 * g + e] * p.scale;
            // the half swap leaves 8 consecutive elements per lane (both halves of a column are here)
#pragma unroll
            for (int gp = 0; gp < 2; ++gp) {
                const f32x4 y = x[2 * gp], z = x[2 * gp + 1];
                auto rx = __builtin_amdgcn_permlane32_swap(pack2<E>(y.x, y.y), pack2<E>(z.x, z.y), false, false);
                auto ry = __builtin_amdgcn_permlane32_swap(pack2<E>(y.z, y.w), pack2<E>(z.z, z.w), false, false);
                *(u32x4*)(to + 32 * dt + 16 * gp) = u32x4{(uint32_t)rx[0], (uint32_t)ry[0], (uint32_t)rx[1], (uint32_t)ry[1]};
            }
        }
        return;
    }
    float* const to = (p.add ? p.dqk + (int64_t)(unit / p.H) * p.dqs0 + (int64_t)(unit % p.H) * p.dqs2 + tok * p.dqs1 : p.dqk + (uk * AJ + aj) * D) + 4 * hf;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        f32x4 x[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) x[g] = p.add ? *(const f32x4*)(to + 32 * dt + 8 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *(f32x4*)(to + 32 * dt + 8 * g) = f32x4{x[g].x + acc[dt][4 * g] * p.scale, x[g].y + acc[dt][4 * g + 1] * p.scale,
                                                    x[g].z + acc[dt][4 * g + 2] * p.scale, x[g].w + acc[dt][4 * g + 3] * p.scale};
    }
}

}  // namespace

bool monarch_bwd_right_supported(int dtype, int D, int b2) {
    return (dtype == SFM_BF16 || dtype == SFM_F16) && (D == 64 || D == 128) && b2 >= 1 && b2 <= 64;
}

int launch_monarch_bwd_right(int dtype, int D, int64_t ntiles, int b1, int b2, int AJ, int nf, float scale, const void* kk,
                             const int64_t* ks, const void* v, const int64_t* vs, const void* rb, const void* dkbar, const void* dy, const float* dc,
                             bool dc_fk, const void* q, const int64_t* qs, const TokMap& qmap, void* ds1, bool ds1_tiles, void* dk, void* dv, const int64_t* dks, int64_t row0,
                             const TokMap& kmap, int H, int unit0, int f0, int f1, int skip_causal, hipStream_t stream) {
    if ((dks[0] | dks[1] | dks[2] | vs[0] | vs[1] | vs[2] | ks[0] | ks[1] | ks[2]) % 8 ||
        ((uintptr_t)dk | (uintptr_t)dv | (uintptr_t)v | (uintptr_t)kk) % 16 || (int64_t)(b2 - 1) * vs[1] * 2 + 2 * D > 0xffffffffll ||
        (int64_t)(b2 - 1) * ks[1] * 2 + 2 * D > 0xffffffffll) {
        set_error("monarch backward (right factor): k / v / dk / dv strides must be multiples of 8 elements and the pointers 16-byte aligned");
        return SFM_ERR_STRIDE;
    }
    RightArgs a;
    a.kk = (const char*)kk; a.rb = (const char*)rb;
    a.v = (const char*)v; a.vs0 = vs[0]; a.vs1 = vs[1]; a.vs2 = vs[2];
    a.ks0 = ks[0]; a.ks1 = ks[1]; a.ks2 = ks[2];
    a.dkbar = (const char*)dkbar; a.dy = (const char*)dy;
    a.dc = dc;
    a.dc_k = dc_fk ? 1 : nf;
    a.dc_f = dc_fk ? b1 : 1;
    a.q = (const char*)q; a.qs0 = qs[0]; a.qs1 = qs[1]; a.qs2 = qs[2];
    a.qmap = qmap;
    a.ds1 = (uint16_t*)ds1;
    const int b2p = (b2 + 3) / 4 * 4;
    a.ds1_f = ds1_tiles ? (int64_t)AJ * b2p : b2p;
    a.ds1_aj = ds1_tiles ? b2p : (int64_t)nf * b2p;
    a.dk = (uint16_t*)dk; a.dv = (uint16_t*)dv;
    a.s0 = dks[0]; a.s1 = dks[1]; a.s2 = dks[2]; a.row0 = row0;
    a.kmap = kmap;
    a.b1 = b1; a.b2 = b2; a.AJ = AJ; a.nf = nf; a.H = H; a.unit0 = unit0; a.f0 = f0; a.f1 = f1;
    a.causal = skip_causal;
    a.scale = scale;
    a.ntiles = ntiles;
    const size_t ldsb = D == 128 ? RightLds<128>::kBytes : RightLds<64>::kBytes;
    const void* fn = nullptr;
    if (dtype == SFM_BF16) fn = D == 128 ? (const void*)monarch_bwd_right_kernel<BF16, 128> : (const void*)monarch_bwd_right_kernel<BF16, 64>;
    else fn = D == 128 ? (const void*)monarch_bwd_right_kernel<F16, 128> : (const void*)monarch_bwd_right_kernel<F16, 64>;
    if (ldsb > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ldsb);
        if (e != hipSuccess) {
            set_error("monarch backward (right factor): cannot reserve %zu bytes of LDS: %s", ldsb, hipGetErrorString(e));
            return SFM_ERR_HIP;
        }
    }
    const dim3 grid((unsigned)((ntiles + 7) / 8 * 8));
    void* kargs[] = {(void*)&a};
    hipError_t le = hipLaunchKernel(fn, grid, dim3(kThreads), kargs, ldsb, stream);
    if (le != hipSuccess) {
        set_error("monarch backward (right factor): launch failed: %s", hipGetErrorString(le));
        return SFM_ERR_HIP;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("monarch backward (right factor): launch failed: %s", hipGetErrorString(e));
        return SFM_ERR_HIP;
    }
    return SFM_OK;
}

bool monarch_bwd_dqk_supported(int dtype, int D) {
    return (dtype == SFM_BF16 || dtype == SFM_F16) && (D == 64 || D == 128);
}

int launch_monarch_bwd_dqk(int dtype, int D, int64_t nuk, int b1, int b2, int AJ, int nf, float scale, const void* k, const int64_t* ks,
                           const TokMap& kmap, const void* ds1, float* dqk, void* dq16, const int64_t* dqs, const TokMap& qmap, int H,
                           int unit0, int skip_causal, hipStream_t stream) {
    if ((ks[0] | ks[1] | ks[2]) % 8 || ((uintptr_t)k) % 16 || (int64_t)nf * b1 * b2 * ks[1] * 2 > 0xffffffffll) {
        set_error("monarch backward (dQ of the right factor): k rows must be 16-byte aligned and a (batch, head) slice under 4 GiB");
        return SFM_ERR_STRIDE;
    }
    DqkArgs a;
    a.k = (const char*)k; a.ks0 = ks[0]; a.ks1 = ks[1]; a.ks2 = ks[2];
    a.kmap = kmap;
    a.ds1 = (const uint16_t*)ds1;
    a.b2p_inv = (uint32_t)((((uint64_t)1 << 32) + (b2 + 3) / 4 * 4 - 1) / (uint64_t)((b2 + 3) / 4 * 4));
    a.dqk = dq16 ? nullptr : dqk;
    a.part = dq16 ? dqk : nullptr;
    a.dq16 = (uint16_t*)dq16;
    a.add = dqs != nullptr;
    a.causal = skip_causal;
    a.dqs0 = dqs ? dqs[0] : 0; a.dqs1 = dqs ? dqs[1] : 0; a.dqs2 = dqs ? dqs[2] : 0;
    a.qmap = qmap;
    a.b1 = b1; a.b2 = b2; a.AJ = AJ; a.nf = nf; a.H = H; a.unit0 = unit0;
    a.scale = scale;
    const int waves = (AJ + 31) / 32;
    a.nchunks = (waves + kDqkWaves - 1) / kDqkWaves;
    const int nwaves = (waves + a.nchunks - 1) / a.nchunks;
    a.total = (int)nuk * a.nchunks;
    const size_t ldsb = (size_t)2 * 64 * 2 * D;
    const dim3 grid((unsigned)xcd_grid(a.total)), block((unsigned)(64 * nwaves));
    if (dtype == SFM_BF16) {
        if (D == 128) hipLaunchKernelGGL((monarch_bwd_dqk_kernel<BF16, 128>), grid, block, ldsb, stream, a);
        else hipLaunchKernelGGL((monarch_bwd_dqk_kernel<BF16, 64>), grid, block, ldsb, stream, a);
    } else {
        if (D == 128) hipLaunchKernelGGL((monarch_bwd_dqk_kernel<F16, 128>), grid, block, ldsb, stream, a);
        else hipLaunchKernelGGL((monarch_bwd_dqk_kernel<F16, 64>), grid, block, ldsb, stream, a);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("monarch backward (dQ of the right factor): launch failed: %s", hipGetErrorString(e));
        return SFM_ERR_HIP;
    }
    return SFM_OK;
}

}  // namespace sfm
