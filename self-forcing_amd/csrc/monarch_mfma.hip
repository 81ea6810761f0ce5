// Monarch attention forward on gfx950 MFMA (bf16 / fp16, head_dim 64 or 128, block cols b2 <= 128).
//
// Two kernels per pass over a group of (batch x head) units:
//
//  step 1 (right factor; replaces _al_cl_y_fwd, wan/modules/monarch_attn.py:109-253)
//      work item = tile (unit, key block row k, kv block-frame f) against all (a, j) columns of a chunk of query
//      block-frames; one workgroup per CU, each taking an equal contiguous share of the tile list.
//      per tile: K[f,k,:,:], V[f,k,:,:] go row-major into LDS once, straight from global memory (the contractions
//      take K^T / V^T from transposing LDS reads), and for ALL columns of the chunk
//          S^T[l,(a,j)] = K[f,k,l,:] . Q[a,k,j,:]           (MFMA, wave = 32 (a,j) columns)
//          R = softmax_l(s S)       cl = sum_l R log2 R      (registers + one cross-half shuffle)
//          Kbar^T = K^T R^T,  Y^T = V^T R^T                  (MFMA; R^T is fed straight from the
//                                                             accumulator layout)
//      rows Kbar[a,j,(f,k),:], Y[a,j,(f,k),:] go to the workspace straight from the accumulators: one
//      v_permlane32_swap per dword pair leaves 8 consecutive head-dim elements per lane (16-byte stores).
//
//  step 2 (left factor; replaces _z_fwd, monarch_attn.py:698-842)
//      per (unit, a, j) its contiguous Kbar / Y rows once, 32 rows at a time, through LDS (global_load_lds_dwordx4, one
//      chunk ahead): by one wave that waits for its own loads only (b1 <= 32), by a team of two to four waves with two
//      barriers per chunk (b1 > 32), or, where columns are few, by two or four waves that take the chunks in turn and
//      merge at the end,
//          S2^T[(f,k), i] = Kbar[(f,k),:] . Q[a,i,j,:]  - cl       online softmax over (f,k)
//          O^T[d, i]     += Y^T[d,(f,k)] P^T[(f,k), i]
//      with the Y^T operands from transposing LDS reads and the query rows in registers.
//
// The running output stays in fp32 for the whole KV range (the reference rounds it to 16 bit
// between KV chunks, monarch_attn.py:795,838).

#include "monarch_rules.hpp"
#include "sfm_common.hpp"

#include <algorithm>

namespace sfm {

// ------------------------------------------------------------------------------------------------
// step 1
// ------------------------------------------------------------------------------------------------
// The K and V tiles are staged row-major (64 rows of 2 D bytes, 16-byte chunks XOR-swizzled per row) straight
// from global memory into LDS (global_load_lds_dwordx4, two buffers per wave group) and the K^T / V^T operands of the
// contractions are transposing LDS reads (ds_read_tr16_b64): no staging registers, no transposes written to LDS,
// one barrier per tile.
typedef short s1_s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 s1_read_tr(const char* lds, uint32_t off) {
    s1_s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s1_s16x4 __attribute__((address_space(3)))*)(lds + off));
    return __builtin_bit_cast(u32x2, v);
}
__device__ __forceinline__ void s1_load_lds16(const char* base, uint32_t off, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(base) : "memory", "m0");
}
// past the caches
__device__ __forceinline__ void s1_load_lds16_nt(const char* base, uint32_t off, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_addr), "v"(off), "s"(base) : "memory", "m0");
}
template <int CPR>
__device__ __forceinline__ int s1_swz(int r) {
    return CPR >= 16 ? (((r & 3) << 2) | ((r >> 2) & 3)) : ((((r >> 1) & 1) << 2) | ((r >> 2) & 3));
}
template <int D, int NT, bool KO>
struct S1Lds {
    static constexpr int kPitch = 2 * D, kTile = 32 * NT * kPitch;
    static constexpr int kBuf = (KO ? 1 : 2) * kTile;        // [K tile | V tile]
    static constexpr int kGroup = 2 * kBuf;
};

// NT: 32-row tiles of the key axis l (b2 <= 32 NT).  Up to two tiles a wave has 170 registers and a workgroup is several
//     wave groups: two of 5 waves at 156 columns.  Three and four tiles (b2 up to 128: the 720p and
//     1080p grids) have 256 registers for up to 8 waves, and their tile buffers take 96 / 128 KB of LDS.
// WR: also write the right factor R (16 bit, 64 values per row) to p.rb; the backward uses it.
// IT: a pass of the iterated refinement (wan/modules/monarch_attn.py:1716-1722): the logits are scaled per (a, f, k, j)
//     column and, after the first pass, the query operand of tile (f, k) is the column's representative p.rep[a, j, (f, k)]
//     instead of Q[a, k, j]; the operand is then fetched for every tile.
// KO: Kbar and cl only.  Every refinement pass but the last needs nothing of V: a pass of the refinement at three frames
//     tied (a = 1, f = 7, b1 = 90, b2 = 52, 12 heads) writes 100 MB instead of 200 and takes 93 us instead of 136.
// CS: block-causal without the masked pairs: a wave all of whose columns are masked for a tile forms and stores nothing.  A
//     training clip of three chunks (a = f = 3, b1 = 90, b2 = 52, 12 heads) has a third of its pairs masked: 99 -> 85 us,
//     with R written 119 -> 98.
// NW: a KV-cache call: the tiles of the new chunk come from the chunk and go to their cache rows too.  Its state costs every
//     tile, so that the calls without a chunk have kernels without it: 40 heads x 64, 12 x 36 in half-height blocks, 21 frames
//     275 us with it, 271 without; 19 x 128 of 9 x 95, 15 frames 238, 235.5.
template <class E, int D, int NT, bool WR = false, bool IT = false, bool KO = false, bool CS = false, bool NW = false>
__global__ __launch_bounds__(NT > 2 ? 512 : 768) __attribute__((amdgpu_waves_per_eu(NT > 2 ? 2 : 3, NT > 2 ? 2 : 3)))
void monarch_step1_kernel(MonarchArgs p) {
    using L = S1Lds<D, NT, KO>;
    constexpr int CPR = D / 8;   // 16-byte chunks of a K/V row
    constexpr int DS = D / 16;   // contraction steps of the logits
    extern __shared__ __attribute__((aligned(256))) char lds_s1[];

    // A workgroup is `p.s1_groups` independent wave groups that share nothing but the barriers, each with
    // its own LDS tiles.  Two groups of 5 waves put 3,3,2,2 waves on the four SIMDs, which one group of 5
    // cannot (waves go to SIMDs round-robin).
    const int G = p.s1_groups;
    const int nthreads = blockDim.x / G;                  // threads of one group
    const int nwaves = nthreads >> 6;
    const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x / nthreads);
    const int tid = threadIdx.x - grp * nthreads;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int m = lane & 31;
    const int hf = lane >> 5;
    const uint32_t piece = (uint32_t)(4 * ((m >> 3) & 1) + 2 * ((m >> 4) & 1) + hf) * 16;   // see the output stores below

    char* const lds = lds_s1 + grp * L::kGroup;
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds;

    // Work items are K/V tiles t = ((ul * b1 + k) * n_achunks + ac) * nf + f, i.e. one kv block row (f, k) of
    // one unit against the query rows Q[a, k, :, :] of one chunk of query block-frames.  The launch has one
    // workgroup per CU and every workgroup takes an equal contiguous share of the tile list (its groups
    // alternate within the share), so no round of workgroups is left partly filled.  The query operands
    // stay in registers while consecutive tiles differ in f only.
    const int T = p.s1_total;
    const int t0 = (int)((int64_t)blockIdx.x * T / gridDim.x);
    const int t1 = (int)((int64_t)(blockIdx.x + 1) * T / gridDim.x);
    const int rounds = (t1 - t0 + G - 1) / G;
    const int mine = (t1 - t0 - grp + G - 1) / G;         // tiles of this group: t0 + grp, t0 + grp + G, ...
    if (mine <= 0) {                                      // still joins the barriers of the other group
        for (int r = 0; r < rounds; ++r) lds_barrier();
        return;
    }

    const int b2 = p.b2;
    const uint32_t qs1 = (uint32_t)p.qs[1], ks1 = (uint32_t)p.ks[1];
    const uint32_t fstep = p.ws_f ? p.ws_f : (uint32_t)p.b1 * p.ws_row;     // scratch rows between consecutive f

    struct Tile {
        int f, k, ul, ac, a0, ncols;
    };
    auto decode = [&](int t) {
        Tile x;
        x.f = t % p.nf;
        int r = t / p.nf;
        const int ac = r % p.n_achunks;
        r /= p.n_achunks;
        x.k = r % p.b1;
        x.ul = r / p.b1;
        x.ac = ac;
        x.a0 = ac * p.a_chunk;
        x.ncols = min(p.a_chunk, p.na - x.a0) * b2;
        return x;
    };

    // tile x is of the new chunk, whose rows are not in the cache yet
    auto is_new = [&](const Tile& x) { return NW && x.f >= p.new_f0 && x.f < p.new_f1; };

    // Tile x into buffer `buf`: LDS position P (in 16-byte units) holds chunk (P % CPR) ^ swz(row) of row P / CPR.
    // Rows past the end of a short tile (l >= b2) load row b2 - 1 again; their logits are masked below.  Every wave
    // issues the same number of loads for every tile, which the partial wait at the top of a round relies on.
    auto stage = [&](const Tile& x, int buf) {
        const int unit = p.unit0 + x.ul;
        const int b = unit / p.H, h = unit % p.H;
        const char* kg = (const char*)p.k + ((int64_t)b * p.ks[0] + (int64_t)h * p.ks[2]) * 2;
        const char* vg = (const char*)p.v + ((int64_t)b * p.vs[0] + (int64_t)h * p.vs[2]) * 2;
        uint32_t row0 = (uint32_t)p.kmap.row(x.f, x.k), rs = ks1 * 2;      // uniform
        uint32_t vrow0 = row0, vrs = rs;                                   // V's, where they are not K's
        if (is_new(x)) {               // a refinement's last pass finds K in the cache
            const int64_t n0 = ((int64_t)b * p.ns[0] + (int64_t)h * p.ns[2]) * 2;
            vrow0 = (uint32_t)p.qmap.row(x.f - p.new_f0, x.k);
            vrs = (uint32_t)p.ns[1] * 2;
            if (!IT || KO) {
                kg = (const char*)p.new_k + n0;
                row0 = vrow0;
                rs = vrs;
            }
            vg = (const char*)p.new_v + n0;
        }
        const uint32_t dst = lds0 + (uint32_t)buf * L::kBuf;
        for (int g = wave; g < NT * (CPR / 2); g += nwaves) {         // 1 KB (64 / CPR rows) per step
            const int P = g * 64 + lane;
            const int r = P / CPR, c = (P % CPR) ^ s1_swz<CPR>(r);
            const uint32_t off = (row0 + (uint32_t)min(r, b2 - 1)) * rs + (uint32_t)c * 16;
            s1_load_lds16(kg, off, dst + (uint32_t)g * 1024);
            if (!KO) s1_load_lds16(vg, IT ? (vrow0 + (uint32_t)min(r, b2 - 1)) * vrs + (uint32_t)c * 16 : off, dst + L::kTile + (uint32_t)g * 1024);
        }
    };
    // The new chunk's rows of tile x from LDS to the cache: K and V, or K in a refinement's first pass and V in its last.
    // The write is at the end of a tile's round, behind the stores that the next round's wait leaves in flight, and
    // non-temporal.  Whole call against a write kernel in front (12 heads x 128, 480p): 3 frames against themselves 75.7 -> 63.2
    // us (71.1 with ordinary stores, 74.3 with the write before the next tile's loads), 21 frames 329.8 -> 324.9, 720p 727 ->
    // 716, 2 heads x 64 of 8 x 8 tokens 22.0 -> 18.4.
    auto write_new = [&](const Tile& x, const char* tile) {
        const int unit = p.unit0 + x.ul;
        const int64_t c0 = ((int64_t)(unit / p.H) * p.ks[0] + (int64_t)(unit % p.H) * p.ks[2]) * 2;
        char* kg = (char*)p.k + c0;
        char* vg = (char*)p.v + c0;
        const uint32_t row0 = (uint32_t)p.kmap.row(x.f, x.k);
        for (int g = wave; g < NT * (CPR / 2); g += nwaves) {
            const int P = g * 64 + lane;
            const int r = P / CPR, c = (P % CPR) ^ s1_swz<CPR>(r);
            if (r >= b2) continue;
            const uint32_t off = (row0 + (uint32_t)r) * ks1 * 2 + (uint32_t)c * 16;
            if (!IT || KO) __builtin_nontemporal_store(*(const u32x4*)(tile + P * 16), (u32x4*)(kg + off));
            if (!KO) __builtin_nontemporal_store(*(const u32x4*)(tile + L::kTile + P * 16), (u32x4*)(vg + off));
        }
    };
    // K rows 32 t + m as the logits' A operand
    const uint32_t a_off = (uint32_t)m * L::kPitch + (uint32_t)((hf ^ s1_swz<CPR>(m)) << 4);
    // K^T / V^T as the contractions' A operand: rows = head-dim 32 dt + m, 16 key rows per step in the order the
    // logits' accumulators hold them (two transposing reads of 4 x 4 blocks each)
    uint32_t tr[D / 32][2];
    {
        const int s16 = lane & 15, g16 = lane >> 4;
        const int rl = 4 * hf + (s16 >> 2);
        const int cl = 2 * (g16 & 1) + ((s16 & 3) >> 1);
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int r = rl + 8 * half;
                tr[dt][half] = (uint32_t)(r * L::kPitch + (((4 * dt + cl) ^ s1_swz<CPR>(r)) << 4) + (s16 & 1) * 8);
            }
    }

    const float sc2 = p.scale * kLog2e;
    const f32x16 kZero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    // Everything from the logits to the output stores runs without a branch, and a lane whose column
    // index is past the chunk's last column works on that last column again (same values to the same
    // addresses).  The number of stores after a tile's loads is then the same on every path, so that the
    // wait for the loads can leave those stores in flight instead of draining them.
    u32x4 qb[DS];                                          // logits operand (B): this lane's query row
    u32x4 qn[DS];                                          // the next tile's, requested a tile ahead where it is another one
    float wn = 1.f;                                        // IT: the weight of the next tile's representative (not AH: this tile's factor)
    uint32_t crow[4] = {0, 0, 0, 0};                       // byte offsets in the (f, k) slab of the four scratch rows this lane stores to
    uint32_t cloff = 0;                                    // same for cl
    uint32_t roff[4] = {0, 0, 0, 0};                       // WR: of the four rows of R
    int qkey = -1;
    float wsc = 1.f;                                       // IT: the column's logits factor

    auto scratch_row = [&](const Tile& x) { return (uint32_t)x.ul * p.ws_unit + (uint32_t)x.k * p.ws_row + (uint32_t)x.f * fstep; };
    auto query_key = [&](const Tile& x) { return (x.ul * p.b1 + x.k) * p.n_achunks + x.ac; };     // one value per (unit, k, query chunk)
    // Query rows of tile x.  AH: they are asked for a tile ahead, after the tile's own loads and before this round's stores, and so
    // have landed with them: fetched where they are used, they are waited for behind all the stores of the tile before (3
    // refinement passes at three frames tied, which fetch them for every tile, 547 -> 534 us).  The second copy of the fetch costs
    // calls of few tiles and of short ones more than that: without a new chunk, 1 head x 128 of 22 x 50 in half-width blocks
    // 38.7 us ahead, 37.4 where they are used, 4 heads of 30 x 52, 3 frames 29.0, 28.5; the refinement with one key tile, 6 x 64
    // of 30 x 52 in half-width blocks 388, 373.  With a chunk, 38 x 64 of 30 x 52 in half-height blocks 554, 558.  CS: a wave that
    // skips a tile has no stores to count, and the whole clip's step 1 took 86.3 us ahead, 83.6 where they are used.
    constexpr bool AH = (IT && NT > 1) || NW;
    auto fetch_query = [&](const Tile& x, u32x4* to) {
        const int unit = p.unit0 + x.ul;
        const int b = unit / p.H, h = unit % p.H;
        const uint16_t* qg = (const uint16_t*)p.q + (int64_t)b * p.qs[0] + (int64_t)h * p.qs[2];
        const int cg = min(wave * 32 + m, x.ncols - 1);
        const int ca = cg / b2;
        const uint16_t* qrow = qg + ((uint32_t)(p.qmap.row(x.a0 + ca, x.k) + cg - ca * b2) * qs1 + 8 * hf);
        if (IT && p.iter_mode == 2) {
            const size_t rrow = (size_t)scratch_row(x) + (size_t)(x.a0 * b2 + cg) * p.ws_aj;
            qrow = (const uint16_t*)p.rep + rrow * D + 8 * hf;
            wn = AH ? p.wgt[rrow] : fminf(1.0f / (p.wgt[rrow] + 1e-6f), 1e4f);
        }
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) to[ds] = *(const u32x4*)(qrow + 16 * ds);
    };

    Tile cur = decode(t0 + grp), nxt = cur;
    bool stored = true;                                    // CS: this wave stored rows in the round before
    if (AH) fetch_query(cur, qn);
    stage(cur, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (AH) {                                              // landed: a wait in the loop counts the loop's operations only
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) asm volatile("" : "+v"(qn[ds]));
        if (IT) asm volatile("" : "+v"(wn));
    }
    for (int r = 0; r < rounds; ++r) {
        const bool fresh = r < mine;     // in its last round a group may have no tile left: it repeats its previous one
        // Vector memory operations complete in order: this wave's part of tile r has landed when only the Kbar / Y
        // stores of the round before (8 * D / 64 operations, half as many without Y; a new chunk's cache rows come behind
        // them) are outstanding.
        if (!CS || stored) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((KO ? 4 : 8) * D / 64) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();                   // tile r is in LDS; every wave has finished reading the tile before it
        if (fresh) cur = nxt;
        const char* kt = lds + (r & 1) * L::kBuf;
        const char* vt = kt + L::kTile;
        const uint32_t srow = scratch_row(cur);
        if ((IT && p.iter_mode == 2) || query_key(cur) != qkey) {
            qkey = query_key(cur);
            if (!AH) {
                fetch_query(cur, qb);
#pragma unroll
                for (int ds = 0; ds < DS; ++ds) asm volatile("" : "+v"(qb[ds]));      // waited for here, before the tile loads below
            } else {
#pragma unroll
                for (int ds = 0; ds < DS; ++ds) qb[ds] = qn[ds];
            }
            if (IT) wsc = p.iter_mode != 2 ? 1.0f / (1.0f + 1e-6f) : AH ? fminf(1.0f / (wn + 1e-6f), 1e4f) : wn;
            const int cg = min(wave * 32 + m, cur.ncols - 1);
            cloff = (uint32_t)(cur.a0 * b2 + cg) * p.cl_aj * 4;
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
                const int sg = min(wave * 32 + (m & 7) + 8 * rb, cur.ncols - 1);
                crow[rb] = (uint32_t)(cur.a0 * b2 + sg) * p.ws_aj * (D * 2) + piece;
                if (WR) roff[rb] = (uint32_t)(cur.a0 * b2 + sg) * 128 + piece;
            }
        }
        if (r + 1 < rounds) {
            // the tile after this one; past the end of the share the current tile is loaded again and dropped
            const int tn = t0 + grp + (r + 1) * G;
            nxt = decode(tn < t1 ? tn : t0 + grp + (mine - 1) * G);
            stage(nxt, (r + 1) & 1);
            if (AH && ((IT && p.iter_mode == 2) || query_key(nxt) != qkey)) fetch_query(nxt, qn);
        }

        if (CS) {
            // key block-frame f is seen by query block-frames from f / causal * causal on
            stored = min(wave * 32 + 31, cur.ncols - 1) >= (cur.f / p.causal * p.causal - cur.a0) * b2;
            if (!stored) continue;
        }
        u32x4 pb[2 * NT];                // R^T as B operands, 16 contraction rows per step
        {
            f32x16 s[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int ds = 0; ds < DS; ++ds) {
                    const u32x4 a = *(const u32x4*)(kt + 32 * t * L::kPitch + (a_off ^ (uint32_t)(ds << 5)));
                    s[t] = E::mfma32(a, qb[ds], ds ? s[t] : kZero);
                }
            // block softmax over l (rows of S^T): 16 NT values here, the rest in lane ^ 32
            float mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    int l = 32 * t + 8 * (v >> 2) + 4 * hf + (v & 3);
                    float zz = l < b2 ? (IT ? s[t][v] * sc2 * wsc : s[t][v] * sc2) : kMaskLogit;
                    s[t][v] = zz;
                    mx = fmaxf(mx, zz);
                }
            mx = xhalf_max(mx);
            float sum = 0.f, ent = 0.f;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    float zz = s[t][v];
                    float e = fast_exp2(zz - mx);        // exactly 0 for masked rows
                    sum += e;
                    ent += e * zz;
                    s[t][v] = e;
                }
            sum = xhalf_sum(sum);
            ent = xhalf_sum(ent);
            const float inv_l = 1.f / sum;
            // R = e / sum is rounded to 16 bit once, as the reference's right factor is
#pragma unroll
            for (int st = 0; st < 2 * NT; ++st) {
                const int t = st >> 1, v0 = 8 * (st & 1);
                pb[st].x = pack2<E>(s[t][v0 + 0] * inv_l, s[t][v0 + 1] * inv_l);
                pb[st].y = pack2<E>(s[t][v0 + 2] * inv_l, s[t][v0 + 3] * inv_l);
                pb[st].z = pack2<E>(s[t][v0 + 4] * inv_l, s[t][v0 + 5] * inv_l);
                pb[st].w = pack2<E>(s[t][v0 + 6] * inv_l, s[t][v0 + 7] * inv_l);
            }
            // sum_l R log2 R (both halves of a column hold, and store, the same value)
            {
                const size_t clrow = (size_t)cur.ul * p.cl_unit + (size_t)((uint32_t)cur.k * p.ws_row + (uint32_t)cur.f * fstep) * p.cl_row;
                *(float*)((char*)p.cl + clrow * 4 + cloff) = ent * inv_l - (mx + log2f(sum));
            }
            if (WR) {
                // R[l] for l = 16 st + 0..15: the lower half of the wave holds 0..3 and 8..11, the upper half 4..7 and
                // 12..15; exchanging the lower half's second pair with the upper half's first leaves 8 consecutive values
                const size_t r0 = (size_t)cur.ul * p.rb_unit + (uint32_t)cur.k * p.rb_k + (uint32_t)cur.f * p.rb_f;
                u32x4 w[2 * NT];
#pragma unroll
                for (int st = 0; st < 2 * NT; ++st) {
                    auto rx = __builtin_amdgcn_permlane32_swap(pb[st].x, pb[st].z, false, false);
                    auto ry = __builtin_amdgcn_permlane32_swap(pb[st].y, pb[st].w, false, false);
                    w[st] = u32x4{(uint32_t)rx[0], (uint32_t)ry[0], (uint32_t)rx[1], (uint32_t)ry[1]};
                }
                if constexpr (NT == 2) {
                    // Eight whole rows of 128 bytes per store and past the caches, like the rows of Kbar and Y below and by the
                    // same exchanges: 32-byte pieces of 32 rows, written back under step 2, cost that kernel 18 us (12 heads,
                    // 4680 x 32760: 139 -> 121).
                    char* rbase = (char*)p.rb + r0 * 128;
                    u32x4 row[2][2];
#pragma unroll
                    for (int dl = 0; dl < 2; ++dl)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            auto x = __builtin_amdgcn_permlane16_swap(w[2 * dl][q], w[2 * dl + 1][q], false, false);
                            row[dl][0][q] = x[0];
                            row[dl][1][q] = x[1];
                        }
#pragma unroll
                    for (int r4 = 0; r4 < 2; ++r4) {
                        u32x4 lo, hi;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            lo[q] = (uint32_t)__builtin_amdgcn_update_dpp((int)row[0][r4][q], (int)row[1][r4][q], 0x128, 0xf, 0xc, false);
                            hi[q] = (uint32_t)__builtin_amdgcn_update_dpp((int)row[1][r4][q], (int)row[0][r4][q], 0x128, 0xf, 0x3, false);
                        }
                        __builtin_nontemporal_store(lo, (u32x4*)(rbase + roff[2 * r4 + 0]));
                        __builtin_nontemporal_store(hi, (u32x4*)(rbase + roff[2 * r4 + 1]));
                    }
                } else {
                    char* rrow = (char*)p.rb + (r0 + cloff / 4) * 128 + 16 * hf;
#pragma unroll
                    for (int st = 0; st < 2 * NT; ++st) *(u32x4*)(rrow + 32 * st) = w[st];
                }
            }
        }
        // contractions with K^T then V^T, 32 head-dim columns at a time.  A 32 x 32 accumulator tile holds,
        // per lane (column c, half hf), head-dim 8g + 4hf + 0..3 for g = 0..3; swapping the g-odd dwords of the
        // lower half with the g-even dwords of the upper half (v_permlane32_swap) leaves 8 consecutive
        // elements per lane: the 16-byte piece 4 dt + 2 gp + hf of column c's 2D-byte scratch row.  Two more
        // exchanges, over a pair of head-dim blocks, trade lane bit 4 for gp (v_permlane16_swap) and lane
        // bit 3 for the block within the pair (a rotation by 8 within rows of 16 lanes).  Afterwards a lane
        // holds, for each of the four row groups rb, the piece 4 (dt0 + bit 3) + 2 bit 4 + hf of column
        // (c & 7) + 8 rb, so that one store instruction writes 128 contiguous bytes of each of 8 rows.
        // Past the caches or through them: see step1_through_caches
        auto contract = [&](auto cached) {
#pragma unroll
            for (int which = 0; which < (KO ? 1 : 2); ++which) {
                const char* tbase = which == 0 ? kt : vt;
                char* og = (char*)(which == 0 ? p.kbar : p.y) + (size_t)srow * (D * 2);
#pragma unroll
                for (int dp = 0; dp < D / 64; ++dp) {
                    uint32_t w[2][2][4];             // [block in pair][gp][dword]
#pragma unroll
                    for (int dl = 0; dl < 2; ++dl) {
                        const int dt = 2 * dp + dl;
                        f32x16 acc;
#pragma unroll
                        for (int st = 0; st < 2 * NT; ++st) {
                            const u32x2 lo = s1_read_tr(tbase, tr[dt][0] + st * 16 * L::kPitch);
                            const u32x2 hi = s1_read_tr(tbase, tr[dt][1] + st * 16 * L::kPitch);
                            const u32x4 a = {lo.x, lo.y, hi.x, hi.y};
                            acc = E::mfma32(a, pb[st], st ? acc : kZero);
                        }
#pragma unroll
                        for (int gp = 0; gp < 2; ++gp) {
                            const int g0 = 2 * gp, g1 = 2 * gp + 1;
                            auto rx = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[4 * g0 + 0], acc[4 * g0 + 1]),
                                                                       pack2<E>(acc[4 * g1 + 0], acc[4 * g1 + 1]), false, false);
                            auto ry = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[4 * g0 + 2], acc[4 * g0 + 3]),
                                                                       pack2<E>(acc[4 * g1 + 2], acc[4 * g1 + 3]), false, false);
                            w[dl][gp][0] = rx[0]; w[dl][gp][1] = ry[0]; w[dl][gp][2] = rx[1]; w[dl][gp][3] = ry[1];
                        }
                        // lane bit 4 <-> gp: slot 0 then holds rows (c & 15), slot 1 rows (c & 15) + 16
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            auto x = __builtin_amdgcn_permlane16_swap(w[dl][0][q], w[dl][1][q], false, false);
                            w[dl][0][q] = x[0]; w[dl][1][q] = x[1];
                        }
                    }
                    // lane bit 3 <-> block within the pair
#pragma unroll
                    for (int r4 = 0; r4 < 2; ++r4) {
                        u32x4 lo, hi;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const uint32_t a = w[0][r4][q], b = w[1][r4][q];
                            // row_ror:8 within 16 lanes; bank mask 0xc writes lanes 8..15 of a row, 0x3 lanes 0..7
                            lo[q] = (uint32_t)__builtin_amdgcn_update_dpp((int)a, (int)b, 0x128, 0xf, 0xc, false);
                            hi[q] = (uint32_t)__builtin_amdgcn_update_dpp((int)b, (int)a, 0x128, 0xf, 0x3, false);
                        }
                        if constexpr (decltype(cached)::value) {
                            *(u32x4*)(og + crow[2 * r4 + 0] + 128 * dp) = lo;
                            *(u32x4*)(og + crow[2 * r4 + 1] + 128 * dp) = hi;
                        } else {
                            __builtin_nontemporal_store(lo, (u32x4*)(og + crow[2 * r4 + 0] + 128 * dp));
                            __builtin_nontemporal_store(hi, (u32x4*)(og + crow[2 * r4 + 1] + 128 * dp));
                        }
                    }
                }
            }
        };
        // The empty statement keeps the two ways apart to their ends: without it the compiler made one pair of the last two stores of
        // each, for Kbar alone at head_dim 64, and lost their hint (8 heads x 64 of 30 x 52, 6 frames, three passes 138.2 us, now 134.6).
        if (p.s1_cached) {
            contract(std::true_type{});
            asm volatile("");
        } else {
            contract(std::false_type{});
        }
        if (NW && fresh && cur.ac == 0 && is_new(cur)) write_new(cur, kt);
    }
}

// ------------------------------------------------------------------------------------------------
// step 2
// ------------------------------------------------------------------------------------------------
// Per wave: [Kbar chunk | Y chunk | cl values, two buffers of 256 bytes], a chunk being 32 scratch rows of 2 D bytes,
// row-major with the 16-byte pieces XOR-swizzled per row as in step 1.  One buffer per matrix: the next chunk's Kbar rows
// are requested as soon as the logits have read the current ones, its Y rows as soon as the output products have, which
// keeps a chunk in flight with 17 KB of LDS per wave instead of 33 KB, so that two workgroups share a compute unit
// (two waves per SIMD, and the 1872 waves of the 480p chunk shape in one round instead of two).
template <int D>
struct S2Lds {
    static constexpr int kPitch = 2 * D, kTile = 32 * kPitch;
    static constexpr int kWave = 2 * kTile + 512;
    static __host__ __device__ constexpr size_t bytes() { return 4 * (size_t)kWave; }
    // a team of waves on one column: two chunks of each matrix, and two cl buffers per wave
    static __host__ __device__ constexpr size_t team_bytes(int waves) { return 4 * (size_t)kTile + waves * 512; }
};

__device__ __forceinline__ void s2_load_lds4(const char* base, uint32_t off, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds_addr), "v"(off), "s"(base) : "memory", "m0");
}
// waits until at most N of the wave's vector memory operations are outstanding
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The step is bound by reading the Kbar / Y rows once (604 MB at the 480p chunk shape), so a column's rows are loaded by one
// workgroup whatever the number of its query rows; a wave holds 32 of them (O^T and the query operand are 96 registers):
//   TEAM = 1 (b1 <= 32): a wave per column (a, j), four to a workgroup that share nothing: each streams its column's rows
//       through its own part of LDS (global_load_lds_dwordx4, 1 KB contiguous per instruction) and waits for its own loads
//       only (vector memory operations complete in order, so when only the loads issued after a tile's are outstanding,
//       that tile has landed).
//   TEAM = 2..4 (b1 <= 128 per grid slice): a workgroup of TEAM waves per column; each loads its share of a chunk, two
//       buffers per matrix, one barrier before the logits and one before the output products.  (A pass over the rows for
//       every 32 query rows, as before, took 518 us at the 720p grid, b1 = 45, and 96 us at three frames tied, b1 = 90;
//       this form 299 and 70.  Two query tiles in one wave need 290 registers and spill.)
// A chunk is a chain, barrier to barrier: with the full exp2f and a row mask in every chunk a team's chunk took 1.2 us however
// few columns there were, now 1.0 (2 heads x 30 columns of 1332 rows 50 -> 42 us).  Teams of three and four have three
// waves per SIMD (168 registers, of which a team of three at head_dim 128 spills three), so that the 624 columns of 12 heads with
// three frames tied are one round: 69 -> 60 us, head_dim 64 46 -> 31; a team of two gains nothing from a third wave (head_dim
// 128).  A third chunk pair in LDS: 72.
// SHARE (TEAM = 1): 2 or 4 (p.s2_split) waves of a workgroup share a column's rows, 32-row chunks dealt in turn, and merge
// (maximum, sum, output) through LDS at the end: with few (a, j) columns the chip is otherwise idle and a wave's chain of
// dependent chunks (about 2.5 us each) is the whole time.  A kernel of its own: with the number of waves an argument of one
// kernel for both, a call of three 480p frames against themselves (12 heads), whose columns are not shared, took 76.2 us
// instead of 75.4 (two runs differ by 0.1).
template <class E, int D, int TEAM, bool SHARE = false, bool PAST = false>
__global__ __launch_bounds__(TEAM == 1 ? 256 : 64 * TEAM) __attribute__((amdgpu_waves_per_eu(TEAM >= 3 ? 3 : 2, TEAM >= 3 ? 3 : 2)))
void monarch_step2_kernel(MonarchArgs p) {
    using L = S2Lds<D>;
    constexpr int DS = D / 16, DT = D / 32, CPR = D / 8;
    constexpr int NG = CPR / 2;                            // 1 KB pieces of a chunk
    constexpr int MYG = (NG + TEAM - 1) / TEAM;            // pieces a wave loads (a team of three loads the last ones twice)
    constexpr bool SOLO = TEAM == 1;
    extern __shared__ __attribute__((aligned(256))) char lds_s2[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int m = lane & 31;
    const int hf = lane >> 5;

    const int b2 = p.b2;
    const int split = SHARE ? p.s2_split : 1, lsplit = split >> 1;         // 1, 2 or 4 and its logarithm
    const int per_wg = SOLO ? 4 >> lsplit : 1;             // columns of a workgroup
    const int sp = SHARE ? wave & (split - 1) : 0;
    const int njg = (b2 + per_wg - 1) / per_wg;
    const int a = blockIdx.x / njg;
    const int jraw = (blockIdx.x % njg) * per_wg + (SOLO ? wave >> lsplit : 0);
    const bool j_ok = jraw < b2;
    const int j = j_ok ? jraw : b2 - 1;
    const int ul = blockIdx.y;
    const int unit = p.unit0 + ul;
    const int b = unit / p.H, h = unit % p.H;
    const int i0 = SOLO ? 0 : blockIdx.z * 128 + wave * 32;

    const int f_lim = p.causal ? min(p.nf, (a / p.causal + 1) * p.causal) : p.nf;
    const int r_lim = f_lim * p.b1;
    const int nch = (r_lim + 31) / 32;

    const int64_t blk = (int64_t)ul * p.ws_unit + (int64_t)(a * b2 + j) * p.ws_aj;   // in rows; the rows of one (a, j) are consecutive
    const char* kb = (const char*)p.kbar + blk * (2 * D);
    const char* yb = (const char*)p.y + blk * (2 * D);
    const char* clp = (const char*)(p.cl + (int64_t)ul * p.cl_unit + (int64_t)(a * b2 + j) * p.cl_aj);
    const uint32_t cl_ld = p.cl_row * 4;                  // bytes between the cl values of consecutive rows

    char* const wl = lds_s2 + (SOLO ? wave * L::kWave : 0);
    char* const cll = SOLO ? wl + 2 * L::kTile : lds_s2 + 4 * L::kTile + wave * 512;      // this wave's two cl buffers
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)wl;
    const uint32_t cl0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)cll;

    // logits operand (B): this lane's query row Q[a, i0 + m, j, :] (zero past b1)
    u32x4 qb[DS];
    {
        const uint16_t* qg = (const uint16_t*)p.q + (int64_t)b * p.qs[0] + (int64_t)h * p.qs[2];
        const int i = min(i0 + m, p.b1 - 1);
        const uint16_t* qrow = qg + (p.qmap.row(a, i) + j) * p.qs[1] + 8 * hf;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) qb[ds] = *(const u32x4*)(qrow + 16 * ds);
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) asm volatile("" : "+v"(qb[ds]));       // waited for here, before the first chunk's loads
        if (i0 + m >= p.b1) {
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) qb[ds] = u32x4{0u, 0u, 0u, 0u};
        }
    }

    const uint32_t a_off = (uint32_t)m * L::kPitch + (uint32_t)((hf ^ s1_swz<CPR>(m)) << 4);   // Kbar row m as the logits' A operand
    uint32_t tr[DT][2];            // Y^T as the output's A operand: transposing reads, as in step 1
    {
        const int s16 = lane & 15, g16 = lane >> 4;
        const int rl = 4 * hf + (s16 >> 2);
        const int cl = 2 * (g16 & 1) + ((s16 & 3) >> 1);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int r = rl + 8 * half;
                tr[dt][half] = (uint32_t)(r * L::kPitch + (((4 * dt + cl) ^ s1_swz<CPR>(r)) << 4) + (s16 & 1) * 8);
            }
    }

    const float sc2 = p.scale * kLog2e;
    const f32x16 kZero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    f32x16 oacc[DT];               // O^T[d = 32 dt + 8 g + 4 hf + e, i = i0 + m]
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oacc[dt] = kZero;
    float mrun = -INFINITY, lrun = 0.f;

    auto issue = [&](const char* mat, int n, uint32_t dst) {
#pragma unroll
        for (int g0 = 0; g0 < MYG; ++g0) {
            const int g = SOLO ? g0 : min(wave * MYG + g0, NG - 1);
            const int P = g * 64 + lane;
            const int r = P / CPR, c = (P % CPR) ^ s1_swz<CPR>(r);
            const uint32_t off = (uint32_t)min(32 * n + r, r_lim - 1) * (2 * D) + (uint32_t)c * 16;
            if constexpr (PAST) s1_load_lds16_nt(mat, off, dst + (uint32_t)g * 1024);          // see step2_past_caches
            else s1_load_lds16(mat, off, dst + (uint32_t)g * 1024);
        }
    };
    // buffers of the chunk at position `it` of this wave's sequence: a team alternates between two pairs
    auto buf = [&](int it) { return SOLO ? 0u : (uint32_t)(it & 1) * 2 * L::kTile; };
    auto issue_k = [&](int n, int it) {
        issue(kb, n, lds0 + buf(it));
        s2_load_lds4(clp, (uint32_t)(32 * n + m) * cl_ld, cl0 + (uint32_t)(it & 1) * 256);   // lanes >= 32 repeat
    };
    auto issue_y = [&](int n, int it) { issue(yb, n, lds0 + buf(it) + L::kTile); };
    if (sp < nch) {
        issue_k(sp, 0);
        issue_y(sp, 0);
    }
    for (int n = sp, it = 0; n < nch; n += split, ++it) {
        const bool more = n + split < nch;
        // Kbar and cl of chunk n have landed when only the Y loads issued after them are outstanding
        wait_vm<MYG>();
        if (!SOLO) {
            lds_barrier();         // every wave's share is there, and every wave is done with the chunk before
            if (more) {
                issue_k(n + 1, it + 1);
                issue_y(n + 1, it + 1);
            }
        }
        const char* kt = wl + buf(it);
        const char* yt = kt + L::kTile;
        const char* clt = cll + (it & 1) * 256;

        f32x16 s;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            const u32x4 ak = *(const u32x4*)(kt + (a_off ^ (uint32_t)(ds << 5)));
            s = E::mfma32(ak, qb[ds], ds ? s : kZero);
        }
        f32x4 cc[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) cc[g] = *(const f32x4*)(clt + (8 * g + 4 * hf) * 4);
        if (SOLO) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the Kbar tile has been read: the next chunk's may land on it
            if (more) issue_k(n + split, it + 1);
        }

        float mx = -INFINITY;
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = fmaf(s[v], sc2, -cc[v >> 2][v & 3]);
        if (!more && r_lim % 32) {                 // a column's last chunk: rows past its end
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] = 32 * n + 8 * (v >> 2) + 4 * hf + (v & 3) < r_lim ? s[v] : -INFINITY;
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) mx = fmaxf(mx, s[v]);
        // The sums so far are rescaled only where a row's maximum moves.  (A reference point that may lag behind the maximum, so
        // that this is rare, takes another 3 us of 60 off, but then a row's largest weight is no longer an exact 1: the
        // output's error against float64 grows by 1 %.)
        const bool moves = __any(mx > mrun);
        float alpha = 1.f;
        if (moves) {
            const float mnew = fmaxf(mrun, xhalf_max(mx));       // finite: chunk n has at least one valid row
            alpha = fast_exp2(mrun - mnew);
            lrun *= alpha;
            mrun = mnew;
        }
        float psum = 0.f;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const float e = fast_exp2(s[v] - mrun);
            psum += e;
            s[v] = e;
        }
        lrun += psum;
        u32x4 pb[2];
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            pb[st].x = pack2<E>(s[8 * st + 0], s[8 * st + 1]);
            pb[st].y = pack2<E>(s[8 * st + 2], s[8 * st + 3]);
            pb[st].z = pack2<E>(s[8 * st + 4], s[8 * st + 5]);
            pb[st].w = pack2<E>(s[8 * st + 6], s[8 * st + 7]);
        }
        // Y of chunk n has landed when only the loads issued after it are outstanding
        if (more) wait_vm<SOLO ? MYG + 1 : 2 * MYG + 1>();
        else wait_vm<0>();
        if (!SOLO) lds_barrier();
        if (moves) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int v = 0; v < 16; ++v) oacc[dt][v] *= alpha;
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const u32x2 lo = s1_read_tr(yt, tr[dt][0] + st * 16 * L::kPitch);
                const u32x2 hi = s1_read_tr(yt, tr[dt][1] + st * 16 * L::kPitch);
                const u32x4 ay = {lo.x, lo.y, hi.x, hi.y};
                oacc[dt] = E::mfma32(ay, pb[st], oacc[dt]);
            }
        }
        if (SOLO) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the Y tile has been read
            if (more) issue_y(n + split, it + 1);
        }
    }

    // epilogue: O[i, d] = O^T / l, turned through LDS (the operand buffers are dead: every load has landed)
    uint16_t* const og = (uint16_t*)p.out + (int64_t)b * p.os[0] + (int64_t)h * p.os[2];
    float* const stats = p.stats ? p.stats + ((int64_t)unit * (p.na * b2) + a * b2 + j) * p.stats_ld : nullptr;
    float ltot = xhalf_sum(lrun);
    if constexpr (!SHARE) {
        if (!SOLO) lds_barrier();
        char* const ol = SOLO ? wl : lds_s2 + wave * L::kTile;
        const float inv = 1.f / ltot;
        if (stats && hf == 0 && j_ok && i0 + m < p.b1) stats[i0 + m] = mrun + log2f(ltot);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                u32x2 w;
                w.x = pack2<E>(oacc[dt][4 * g + 0] * inv, oacc[dt][4 * g + 1] * inv);
                w.y = pack2<E>(oacc[dt][4 * g + 2] * inv, oacc[dt][4 * g + 3] * inv);
                *(u32x2*)(ol + m * L::kPitch + (32 * dt + 8 * g + 4 * hf) * 2) = w;
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        for (int c = lane; c < 32 * CPR; c += 64) {
            const int r = c / CPR, ch = c % CPR;
            const int i = i0 + r;
            if (i < p.b1 && j_ok) {
                const u32x4 w = *(const u32x4*)(ol + r * L::kPitch + ch * 16);
                *(u32x4*)(og + (p.qmap.row(a, i) + j) * p.os[1] + ch * 8) = w;
            }
        }
    } else {
        // merge of the `split` waves of a column: statistics through the (dead) cl buffers, outputs through the waves' tile
        // buffers as fp32 rows of 4 D bytes, 16-byte pieces XOR-ed with the row
        char* const col = lds_s2 + (wave - sp) * L::kWave;                // the column's first wave
        if (hf == 0) {
            *(float*)(cll + m * 4) = mrun;
            *(float*)(cll + 128 + m * 4) = ltot;
        }
        lds_barrier();
        float M = -INFINITY, sum = 0.f;
        for (int w = 0; w < split; ++w) M = fmaxf(M, *(const float*)(col + w * L::kWave + 2 * L::kTile + m * 4));
        for (int w = 0; w < split; ++w) {
            const char* c = col + w * L::kWave + 2 * L::kTile + m * 4;
            sum += *(const float*)(c + 128) * exp2f(*(const float*)c - M);           // a wave without chunks: 0 * exp2(-inf)
        }
        const float fac = exp2f(mrun - M) / sum;
        if (stats && sp == 0 && hf == 0 && j_ok && m < p.b1) stats[m] = M + log2f(sum);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 w = {oacc[dt][4 * g + 0] * fac, oacc[dt][4 * g + 1] * fac, oacc[dt][4 * g + 2] * fac, oacc[dt][4 * g + 3] * fac};
                *(f32x4*)(wl + m * (4 * D) + (((8 * dt + 2 * g + hf) ^ m) & (D / 4 - 1)) * 16) = w;
            }
        lds_barrier();
        const int rows = 32 >> lsplit;                                    // this wave's share of the rows
        for (int c = lane; c < rows * CPR; c += 64) {
            const int r = sp * rows + c / CPR, ch = c % CPR;
            f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
            for (int w = 0; w < split; ++w) {
                const char* row = col + w * L::kWave + r * (4 * D);
                lo += *(const f32x4*)(row + (((2 * ch) ^ r) & (D / 4 - 1)) * 16);
                hi += *(const f32x4*)(row + (((2 * ch + 1) ^ r) & (D / 4 - 1)) * 16);
            }
            if (r < p.b1 && j_ok) {
                const u32x4 w = {pack2<E>(lo.x, lo.y), pack2<E>(lo.z, lo.w), pack2<E>(hi.x, hi.y), pack2<E>(hi.z, hi.w)};
                *(u32x4*)(og + (p.qmap.row(a, r) + j) * p.os[1] + ch * 8) = w;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// The left factor's row statistics alone, for the refinement passes whose output is not wanted:
//   stats[i] = log2 sum_r exp2(s log2e <Q_i, Kbar_r> - cl_r)
// Step 2 without Y and the output: bound by reading the Kbar rows once.  The wave arrangements are step 2's; a lone wave
// holds two chunks in its LDS, a team four, of which three are in flight.  At three frames tied (b1 = 90, 21 cached frames
// of 480p, 12 heads) it takes 43 us against 74 us for step 2.
// ------------------------------------------------------------------------------------------------
template <int D, int TEAM>
struct StLds {
    static constexpr int kPitch = 2 * D, kTile = 32 * kPitch;
    static constexpr int kBufs = TEAM == 1 ? 2 : 4;
    static constexpr int kWave = kBufs * (kTile + 256);       // TEAM = 1: a wave's tiles, then its cl values
    static __host__ __device__ constexpr size_t bytes() { return TEAM == 1 ? 4 * (size_t)kWave : kBufs * (kTile + TEAM * 256); }
};

template <class E, int D, int TEAM>
__global__ __launch_bounds__(TEAM == 1 ? 256 : 64 * TEAM)
void monarch_left_stats_kernel(MonarchArgs p) {
    using L = StLds<D, TEAM>;
    constexpr int DS = D / 16, CPR = D / 8;
    constexpr int NG = CPR / 2;                            // 1 KB pieces of a chunk
    constexpr int MYG = (NG + TEAM - 1) / TEAM;            // pieces a wave loads (a team of three loads the last ones twice)
    constexpr int NB = L::kBufs;
    constexpr bool SOLO = TEAM == 1;
    extern __shared__ __attribute__((aligned(256))) char lds_s2[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int m = lane & 31;
    const int hf = lane >> 5;

    const int b2 = p.b2;
    const int split = SOLO ? p.s2_split : 1, lsplit = split >> 1;          // 1, 2 or 4 and its logarithm
    const int per_wg = SOLO ? 4 >> lsplit : 1;             // columns of a workgroup
    const int sp = SOLO ? wave & (split - 1) : 0;
    const int njg = (b2 + per_wg - 1) / per_wg;
    const int a = blockIdx.x / njg;
    const int jraw = (blockIdx.x % njg) * per_wg + (SOLO ? wave >> lsplit : 0);
    const bool j_ok = jraw < b2;
    const int j = j_ok ? jraw : b2 - 1;
    const int ul = blockIdx.y;
    const int unit = p.unit0 + ul;
    const int b = unit / p.H, h = unit % p.H;
    const int i0 = SOLO ? 0 : wave * 32;
    const int r_lim = p.nf * p.b1;
    const int nch = (r_lim + 31) / 32;

    const int64_t blk = (int64_t)ul * p.ws_unit + (int64_t)(a * b2 + j) * p.ws_aj;
    const char* kb = (const char*)p.kbar + blk * (2 * D);
    const char* clp = (const char*)(p.cl + (int64_t)ul * p.cl_unit + (int64_t)(a * b2 + j) * p.cl_aj);
    const uint32_t cl_ld = p.cl_row * 4;

    char* const wl = lds_s2 + (SOLO ? wave * L::kWave : 0);
    char* const cll = SOLO ? wl + NB * L::kTile : lds_s2 + NB * (L::kTile + wave * 256);
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)wl;
    const uint32_t cl0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)cll;

    u32x4 qb[DS];                                          // logits operand (B): this lane's query row (zero past b1)
    {
        const uint16_t* qg = (const uint16_t*)p.q + (int64_t)b * p.qs[0] + (int64_t)h * p.qs[2];
        const uint16_t* qrow = qg + (p.qmap.row(a, min(i0 + m, p.b1 - 1)) + j) * p.qs[1] + 8 * hf;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) qb[ds] = *(const u32x4*)(qrow + 16 * ds);
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) asm volatile("" : "+v"(qb[ds]));       // waited for here, before the first chunk's loads
        if (i0 + m >= p.b1) {
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) qb[ds] = u32x4{0u, 0u, 0u, 0u};
        }
    }
    const uint32_t a_off = (uint32_t)m * L::kPitch + (uint32_t)((hf ^ s1_swz<CPR>(m)) << 4);   // Kbar row m as the logits' A operand
    const float sc2 = p.scale * kLog2e;
    const f32x16 kZero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float mrun = -INFINITY, lrun = 0.f;

    auto issue = [&](int n, int it) {
        const uint32_t dst = lds0 + (uint32_t)(it % NB) * L::kTile;
#pragma unroll
        for (int g0 = 0; g0 < MYG; ++g0) {
            const int g = SOLO ? g0 : min(wave * MYG + g0, NG - 1);
            const int P = g * 64 + lane;
            const int r = P / CPR, c = (P % CPR) ^ s1_swz<CPR>(r);
            const uint32_t off = (uint32_t)min(32 * n + r, r_lim - 1) * (2 * D) + (uint32_t)c * 16;
            s1_load_lds16(kb, off, dst + (uint32_t)g * 1024);
        }
        s2_load_lds4(clp, (uint32_t)(32 * n + m) * cl_ld, cl0 + (uint32_t)(it % NB) * 256);   // lanes >= 32 repeat
    };
#pragma unroll
    for (int it = 0; it < NB - 1; ++it)
        if (sp + it * split < nch) issue(sp + it * split, it);
    for (int n = sp, it = 0; n < nch; n += split, ++it) {
        // vector memory operations complete in order: chunk n has landed when only the chunks requested after it are
        // outstanding.  The buffer of the chunk before is free once its reads have been waited for.
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (SOLO) {
            if (n + split < nch) {
                issue(n + split, it + 1);
                wait_vm<MYG + 1>();
            } else {
                wait_vm<0>();
            }
        } else {
            if (n + 2 < nch) wait_vm<2 * (MYG + 1)>();
            else if (n + 1 < nch) wait_vm<MYG + 1>();
            else wait_vm<0>();
            lds_barrier();         // every wave's share is there, and every wave is done with the chunk before
            if (n + 3 < nch) issue(n + 3, it + 3);
        }
        const char* kt = wl + (it % NB) * L::kTile;
        const char* clt = cll + (it % NB) * 256;
        f32x16 s;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            const u32x4 ak = *(const u32x4*)(kt + (a_off ^ (uint32_t)(ds << 5)));
            s = E::mfma32(ak, qb[ds], ds ? s : kZero);
        }
        f32x4 cc[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) cc[g] = *(const f32x4*)(clt + (8 * g + 4 * hf) * 4);
        float mx = -INFINITY;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int r = 32 * n + 8 * (v >> 2) + 4 * hf + (v & 3);
            const float z = r < r_lim ? s[v] * sc2 - cc[v >> 2][v & 3] : -INFINITY;
            s[v] = z;
            mx = fmaxf(mx, z);
        }
        mx = xhalf_max(mx);
        const float mnew = fmaxf(mrun, mx);        // finite: chunk n has at least one valid row
        float psum = 0.f;
#pragma unroll
        for (int v = 0; v < 16; ++v) psum += exp2f(s[v] - mnew);
        lrun = lrun * exp2f(mrun - mnew) + psum;
        mrun = mnew;
    }

    float* const stats = p.stats + ((int64_t)unit * (p.na * b2) + a * b2 + j) * p.stats_ld;
    float ltot = xhalf_sum(lrun);
    if constexpr (SOLO) {
        if (split > 1) {           // merge of the waves of a column through the (dead) cl buffers, in step 2's order
            if (hf == 0) {
                *(float*)(cll + m * 4) = mrun;
                *(float*)(cll + 128 + m * 4) = ltot;
            }
            lds_barrier();
            const char* col = cll - sp * L::kWave;
            float M = -INFINITY, sum = 0.f;
            for (int w = 0; w < split; ++w) M = fmaxf(M, *(const float*)(col + w * L::kWave + m * 4));
            for (int w = 0; w < split; ++w) {
                const char* c = col + w * L::kWave + m * 4;
                sum += *(const float*)(c + 128) * exp2f(*(const float*)c - M);           // a wave without chunks: 0 * exp2(-inf)
            }
            mrun = M;
            ltot = sum;
        }
    }
    if (sp == 0 && hf == 0 && j_ok && i0 + m < p.b1) stats[i0 + m] = mrun + log2f(ltot);
}

// ------------------------------------------------------------------------------------------------
// iterated refinement: the next pass's query representatives (wan/modules/monarch_attn.py:1741-1744)
//   rep[a, j, r, :] = sum_i L[i, r] Q[a, i, j, :],   wgt[a, j, r] = sum_i L[i, r],   r = (f, k)
// with L[i, r] = exp2(s log2e <Q_i, Kbar_r> - cl_r - stats_i), stats = the left factor's row statistics that step 2 wrote.
// Step 2 with the operands' roles exchanged: one wave per (a, j) streams the column's Kbar rows 32 at a time through its
// LDS; the logits come out as S[i, r] (A = query rows, B = Kbar rows), so that a lane holds a column r, and
// rep^T[d, r] = sum_i Q^T[d, i] L[i, r] takes Q^T from transposing reads of the column's query rows, which sit in the
// wave's LDS for the whole kernel.  NQ = 32-row tiles of the query rows i (b1 <= 32 NQ <= 128: three frames tied per
// block give b1 = 90).  With one tile a wave owns a column and its query rows, and the logits' A operand stays in
// registers; 4 waves to a workgroup.  With more tiles the rows of one column fill the LDS of a wave or two, so a
// workgroup of 8 waves (7 at four tiles) owns one column: one copy of its query rows, chunks of Kbar rows dealt in turn
// (a chunk's representatives need no other chunk's).  A wave per column with its own copy held one workgroup of three
// waves on a compute unit, each with a serial chain of 20 chunks, at b1 = 90, 630 rows: 74 us, now 60.
// ------------------------------------------------------------------------------------------------
template <int D, int NQ>
struct RepLds {
    static constexpr int kPitch = 2 * D, kTile = 32 * kPitch;
    static constexpr int kBuf = kTile + 256;               // [Kbar chunk | cl values]
    static constexpr bool kShared = NQ > 1;                // a workgroup's waves share one column
    static constexpr int kWaves = NQ == 1 ? 4 : NQ < 4 ? 8 : 7;
    static constexpr int kWave = 2 * kBuf + (kShared ? 0 : kTile);      // bytes per wave, its query rows behind its buffers
    static constexpr int kQ = kShared ? kWaves * kWave : 2 * kBuf;      // offset of the query rows (from the workgroup's / the wave's LDS)
    static __host__ __device__ constexpr size_t bytes() { return (size_t)kWaves * kWave + (kShared ? NQ * kTile : 0); }
};

template <class E, int D, int NQ>
__global__ __launch_bounds__(64 * (RepLds<D, NQ>::kWaves)) void monarch_rep_kernel(MonarchArgs p) {
    using L = RepLds<D, NQ>;
    constexpr int DS = D / 16, DT = D / 32, CPR = D / 8;
    extern __shared__ __attribute__((aligned(256))) char lds_s2[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int m = lane & 31;
    const int hf = lane >> 5;

    const int b2 = p.b2;
    const int per_wg = L::kShared ? 1 : L::kWaves;         // columns of a workgroup
    const int njg = (b2 + per_wg - 1) / per_wg;
    const int a = blockIdx.x / njg;
    const int j = (blockIdx.x % njg) * per_wg + (L::kShared ? 0 : wave);
    if (j >= b2) return;                                  // never in a shared workgroup, which has barriers
    constexpr int step = L::kShared ? L::kWaves : 1;       // this wave's chunks: n0, n0 + step, ...
    const int n0 = L::kShared ? wave : 0;
    const int ul = blockIdx.y;
    const int unit = p.unit0 + ul;
    const int b = unit / p.H, h = unit % p.H;

    const int r_lim = p.nf * p.b1;
    const int nch = (r_lim + 31) / 32;
    const int64_t blk = (int64_t)ul * p.ws_unit + (int64_t)(a * b2 + j) * p.ws_aj;
    const char* kb = (const char*)p.kbar + blk * (2 * D);
    const char* clp = (const char*)(p.cl + (int64_t)ul * p.cl_unit + (int64_t)(a * b2 + j) * p.cl_aj);
    const uint32_t cl_ld = p.cl_row * 4;
    char* repb = (char*)p.rep + blk * (2 * D);
    float* wgt = p.wgt + blk;

    char* const wl = lds_s2 + wave * L::kWave;
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)wl;
    char* const qt = (L::kShared ? lds_s2 : wl) + L::kQ;  // the column's query rows, laid out like chunks of scratch rows
    const uint32_t qt0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)qt;

    const uint16_t* qg = (const uint16_t*)p.q + (int64_t)b * p.qs[0] + (int64_t)h * p.qs[2];
    // query rows into LDS (rows past b1 repeat the last one; their weights are zero)
    for (int g = n0; g < NQ * (CPR / 2); g += step) {
        const int P = g * 64 + lane;
        const int r = P / CPR, c = (P % CPR) ^ s1_swz<CPR>(r);
        const uint32_t off = (uint32_t)((p.qmap.row(a, min(r, p.b1 - 1)) + j) * p.qs[1] * 2) + (uint32_t)c * 16;
        s1_load_lds16((const char*)qg, off, qt0 + (uint32_t)g * 1024);
    }
    // one tile: the logits operand (A) is this lane's query row Q[a, m, j, :] (zero past b1), kept in registers
    u32x4 qa[DS];
    if constexpr (NQ == 1) {
        const uint16_t* qrow = qg + (p.qmap.row(a, min(m, p.b1 - 1)) + j) * p.qs[1] + 8 * hf;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) qa[ds] = *(const u32x4*)(qrow + 16 * ds);
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) asm volatile("" : "+v"(qa[ds]));
        if (m >= p.b1) {
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) qa[ds] = u32x4{0u, 0u, 0u, 0u};
        }
    }
    // the statistics of the 16 NQ rows whose logits this lane will hold
    float st[NQ][16];
    {
        const float* sp = p.stats + ((int64_t)unit * (p.na * b2) + a * b2 + j) * p.stats_ld;
#pragma unroll
        for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int i = 32 * qi + 8 * (v >> 2) + 4 * hf + (v & 3);
                st[qi][v] = i < p.b1 ? sp[i] : 0.f;
            }
#pragma unroll
        for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
            for (int v = 0; v < 16; ++v) asm volatile("" : "+v"(st[qi][v]));
    }

    // chunk n of the Kbar rows (and their cl values) into buffer `buf`
    auto issue = [&](int n, int buf) {
        const uint32_t dst = lds0 + (uint32_t)buf * L::kBuf;
#pragma unroll
        for (int g = 0; g < CPR / 2; ++g) {
            const int P = g * 64 + lane;
            const int r = P / CPR, c = (P % CPR) ^ s1_swz<CPR>(r);
            const uint32_t off = (uint32_t)min(32 * n + r, r_lim - 1) * (2 * D) + (uint32_t)c * 16;
            s1_load_lds16(kb, off, dst + (uint32_t)g * 1024);
        }
        s2_load_lds4(clp, (uint32_t)(32 * n + m) * cl_ld, dst + L::kTile);
    };
    const uint32_t b_off = (uint32_t)m * L::kPitch + (uint32_t)((hf ^ s1_swz<CPR>(m)) << 4);   // row m of a 32-row tile as an MFMA operand
    uint32_t tr[DT][2];            // Q^T as the representatives' A operand: transposing reads, as step 2 reads Y^T
    {
        const int s16 = lane & 15, g16 = lane >> 4;
        const int rl = 4 * hf + (s16 >> 2);
        const int cl = 2 * (g16 & 1) + ((s16 & 3) >> 1);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int r = rl + 8 * half;
                tr[dt][half] = (uint32_t)(r * L::kPitch + (((4 * dt + cl) ^ s1_swz<CPR>(r)) << 4) + (s16 & 1) * 8);
            }
    }

    const float sc2 = p.scale * kLog2e;
    const f32x16 kZero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    if (L::kShared) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();             // every wave's share of the query rows is there
    }
    if (n0 < nch) issue(n0, 0);
    for (int n = n0, buf = 0; n < nch; n += step, buf ^= 1) {
        // everything older than the chunk requested last (the stores of the chunk before included) is waited for
        if (n + step < nch) {
            issue(n + step, buf ^ 1);
            if (D == 128) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        const char* kt = wl + buf * L::kBuf;
        const float cc = *(const float*)(kt + L::kTile + m * 4);
        const bool rok = 32 * n + m < r_lim;
        float wsum = 0.f;
        u32x4 pb[NQ][2];
#pragma unroll
        for (int qi = 0; qi < NQ; ++qi) {
            f32x16 s;              // S[i = 32 qi + 8 g + 4 hf + e, r = 32 n + m]
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
                const u32x4 bk = *(const u32x4*)(kt + (b_off ^ (uint32_t)(ds << 5)));
                u32x4 aq;
                if constexpr (NQ == 1) aq = qa[ds];
                else aq = *(const u32x4*)(qt + qi * L::kTile + (b_off ^ (uint32_t)(ds << 5)));
                s = E::mfma32(aq, bk, ds ? s : kZero);
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int i = 32 * qi + 8 * (v >> 2) + 4 * hf + (v & 3);
                const float e = (rok && i < p.b1) ? exp2f(s[v] * sc2 - cc - st[qi][v]) : 0.f;
                s[v] = e;
                wsum += e;
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                pb[qi][q].x = pack2<E>(s[8 * q + 0], s[8 * q + 1]);
                pb[qi][q].y = pack2<E>(s[8 * q + 2], s[8 * q + 3]);
                pb[qi][q].z = pack2<E>(s[8 * q + 4], s[8 * q + 5]);
                pb[qi][q].w = pack2<E>(s[8 * q + 6], s[8 * q + 7]);
            }
        }
        wsum = xhalf_sum(wsum);
        if (hf == 0) wgt[32 * n + m] = wsum;
        char* rrow = repb + (size_t)(32 * n + m) * (2 * D);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            f32x16 acc;
#pragma unroll
            for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const u32x2 lo = s1_read_tr(qt + qi * L::kTile, tr[dt][0] + q * 16 * L::kPitch);
                    const u32x2 hi = s1_read_tr(qt + qi * L::kTile, tr[dt][1] + q * 16 * L::kPitch);
                    const u32x4 aq = {lo.x, lo.y, hi.x, hi.y};
                    acc = E::mfma32(aq, pb[qi][q], (qi | q) ? acc : kZero);
                }
            // rep^T[d = 32 dt + 8 g + 4 hf + e, r]: the half-swap leaves 8 consecutive d per lane
#pragma unroll
            for (int gp = 0; gp < 2; ++gp) {
                const int g0 = 2 * gp, g1 = 2 * gp + 1;
                auto rx = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[4 * g0 + 0], acc[4 * g0 + 1]),
                                                           pack2<E>(acc[4 * g1 + 0], acc[4 * g1 + 1]), false, false);
                auto ry = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[4 * g0 + 2], acc[4 * g0 + 3]),
                                                           pack2<E>(acc[4 * g1 + 2], acc[4 * g1 + 3]), false, false);
                const u32x4 o = {(uint32_t)rx[0], (uint32_t)ry[0], (uint32_t)rx[1], (uint32_t)ry[1]};
                *(u32x4*)(rrow + (32 * dt + 16 * gp + 8 * hf) * 2) = o;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// The two kernels above in one, for columns whose logits fit the registers of the waves that share them: W waves of a
// workgroup deal the column's 32-row chunks of Kbar in turn and keep their logits S[i, r] (C chunks x NQ query tiles x 16
// registers), reduce each row's maximum and sum over their lanes, merge them through LDS and scale:
//   L[i, r] = exp2(z - max_wave) * exp2(max_wave - stats_i),   z = s log2e <Q_i, Kbar_r> - cl_r
// so that Kbar is read, and its logits and exponentials are formed, once.  At one query tile (framewise 480p, 21 frames, 12
// heads x 128: 604 MB) 148 us where the two kernels took 69 + 150, bound by that traffic; at three (three frames tied: 201
// MB) 75 for 46 + 62, where one workgroup fills a compute unit and its loads, logits, reductions and stores follow each
// other.  (98 with every value's maximum and sum reduced in all lanes, and with exp2f.)
// RUN: a workgroup walks a run of columns, the next one's first chunk requested as soon as this one's has been read; the products
// of all chunks share their query rows, and the representatives leave in whole lines, past the caches: 75 -> 70 us at three
// frames tied.  A column's 44 000 cycles there: logits 8500, maxima, exponentials and sums 6500, waiting for the other waves
// 2800, scales and weights 3300, representatives and their stores 10 000, the next column's query rows behind the stores of all
// compute units 12 000.  Held in registers until those rows are requested, the representatives spill (81 us and more).
// ------------------------------------------------------------------------------------------------
template <int D, int NQ, int W>
struct WtLds {
    static constexpr int kPitch = 2 * D, kTile = 32 * kPitch;
    static constexpr int kBuf = kTile + 256;               // [Kbar chunk | cl values]
    static constexpr int kWave = 2 * kBuf;                 // reused: the wave's rows' maxima, sums and scales
    static constexpr int kWaves = W == 1 ? 4 : W;          // waves of a workgroup
    static constexpr int kCols = kWaves / W;               // and its columns
    static __host__ __device__ constexpr size_t bytes() { return (size_t)kWaves * kWave + (size_t)kCols * NQ * kTile; }
};

// Maximum / sum of each of 16 values over the 32 lanes of a half wave: a lane ends with value half_reduce_at(m), and its
// neighbour m ^ 1 with the same.  Lanes trade half of their values at every step, so that it takes 38 operations for the 16.
__device__ __forceinline__ int half_reduce_at(int m) { return 8 * ((m >> 4) & 1) + 4 * ((m >> 3) & 1) + 2 * ((m >> 2) & 1) + ((m >> 1) & 1); }

template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

template <bool MAX>
__device__ __forceinline__ float half_reduce(float* x, int m) {
    auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        auto y = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x[i]), __builtin_bit_cast(uint32_t, x[i + 8]), false, false);
        x[i] = op(__builtin_bit_cast(float, (uint32_t)y[0]), __builtin_bit_cast(float, (uint32_t)y[1]));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bool up = m & 8;
        x[i] = op(up ? x[i + 4] : x[i], dpp_move<0x128>(up ? x[i] : x[i + 4]));          // row_ror:8
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const bool up = m & 4;
        x[i] = op(up ? x[i + 2] : x[i], dpp_move<0x141>(up ? x[i] : x[i + 2]));          // row_half_mirror: lane 7 - l of eight
    }
    const bool up = m & 2;
    x[0] = op(up ? x[1] : x[0], dpp_move<0x4e>(up ? x[0] : x[1]));                       // quad_perm:[2,3,0,1]
    return op(x[0], dpp_move<0xb1>(x[0]));                                               // quad_perm:[1,0,3,2]
}

template <class E, int D, int NQ, int W, int C, bool RUN>
__global__ __launch_bounds__(64 * (WtLds<D, NQ, W>::kWaves)) __attribute__((amdgpu_waves_per_eu(2, 2))) void monarch_weights_kernel(MonarchArgs p, int items) {
    using L = WtLds<D, NQ, W>;
    constexpr int DS = D / 16, DT = D / 32, CPR = D / 8;
    constexpr int NG = CPR / 2;                            // 1 KB pieces of a chunk
    extern __shared__ __attribute__((aligned(256))) char lds_s2[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    const int b2 = p.b2;
    const int njg = (b2 + L::kCols - 1) / L::kCols;
    const int col = W == 1 ? wave : 0;                     // this wave's column of the workgroup's
    const int w = W == 1 ? 0 : wave;                       // its chunks: w, w + W, ...
    // an item is a workgroup's columns (unit, a, kCols of j); RUN: every workgroup takes an equal run of them, else a unit's in x
    int item = RUN ? (int)((int64_t)items * blockIdx.x / gridDim.x) : (int)blockIdx.x;
    const int end = RUN ? (int)((int64_t)items * (blockIdx.x + 1) / gridDim.x) : 0;

    const int r_lim = p.nf * p.b1;
    const int nch = (r_lim + 31) / 32;
    const uint32_t cl_ld = p.cl_row * 4;
    struct Column {
        int ul, a, j;
        int64_t blk;       // its first scratch row
    };
    auto column = [&](int x) {
        Column c;
        const int g = x / njg;
        c.j = min((x - g * njg) * L::kCols + col, b2 - 1);      // past the last column: that one again, with the same results
        c.ul = RUN ? g / p.na : (int)blockIdx.y;
        c.a = RUN ? g - c.ul * p.na : g;
        c.blk = (int64_t)c.ul * p.ws_unit + (int64_t)(c.a * b2 + c.j) * p.ws_aj;
        return c;
    };

    char* const wl = lds_s2 + wave * L::kWave;
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)wl;
    char* const qt = lds_s2 + L::kWaves * L::kWave + col * NQ * L::kTile;     // the column's query rows, laid out like chunks of scratch rows
    const uint32_t qt0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)qt;

    Column cur = column(item);
    for (bool first = true;; ++item, first = false) {
        // what follows from the lane is formed again for every item: kept, it does not fit beside the logits
        int lane = tid & 63;
        if (RUN) asm volatile("" : "+v"(lane));
        const int m = lane & 31;
        const int hf = lane >> 5;
        // query rows into LDS (rows past b1 repeat the last one; their scale is zero)
        auto queries = [&](const Column& x) {
            const int unit = p.unit0 + x.ul;
            const uint16_t* qg = (const uint16_t*)p.q + (int64_t)(unit / p.H) * p.qs[0] + (int64_t)(unit % p.H) * p.qs[2];
            for (int g = w; g < NQ * NG; g += W) {
                const int P = g * 64 + lane;
                const int r = P / CPR, c = (P % CPR) ^ s1_swz<CPR>(r);
                const uint32_t off = (uint32_t)((p.qmap.row(x.a, min(r, p.b1 - 1)) + x.j) * p.qs[1] * 2) + (uint32_t)c * 16;
                s1_load_lds16((const char*)qg, off, qt0 + (uint32_t)g * 1024);
            }
        };
        auto issue = [&](const Column& x, int n, int buf) {
            const char* const kb = (const char*)p.kbar + x.blk * (2 * D);
            const char* const clp = (const char*)(p.cl + (int64_t)x.ul * p.cl_unit + (int64_t)(x.a * b2 + x.j) * p.cl_aj);
            const uint32_t dst = lds0 + (uint32_t)buf * L::kBuf;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const int P = g * 64 + lane;
                const int r = P / CPR, c = (P % CPR) ^ s1_swz<CPR>(r);
                const uint32_t off = (uint32_t)min(32 * n + r, r_lim - 1) * (2 * D) + (uint32_t)c * 16;
                s1_load_lds16(kb, off, dst + (uint32_t)g * 1024);
            }
            s2_load_lds4(clp, (uint32_t)(32 * n + m) * cl_ld, dst + L::kTile);
        };
        const uint32_t b_off = (uint32_t)m * L::kPitch + (uint32_t)((hf ^ s1_swz<CPR>(m)) << 4);   // row m of a 32-row tile as an MFMA operand
        uint32_t tr[DT][2];            // Q^T as the representatives' A operand: transposing reads
        {
            const int s16 = lane & 15, g16 = lane >> 4;
            const int rl = 4 * hf + (s16 >> 2);
            const int cl = 2 * (g16 & 1) + ((s16 & 3) >> 1);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int r = rl + 8 * half;
                    tr[dt][half] = (uint32_t)(r * L::kPitch + (((4 * dt + cl) ^ s1_swz<CPR>(r)) << 4) + (s16 & 1) * 8);
                }
        }
        const float sc2 = p.scale * kLog2e;
        const f32x16 kZero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (first) {
            queries(cur);
            if (w < nch) issue(cur, w, 0);
            if (w + W < nch) issue(cur, w + W, 1);
            // this wave's share of the query rows has landed when only its first two chunks are outstanding
            if (w + W < nch) wait_vm<2 * (NG + 1)>();
            else if (w < nch) wait_vm<NG + 1>();
            else wait_vm<0>();
            lds_barrier();
        }
        const bool more = RUN && item + 1 < end;           // uniform over the workgroup
        const Column next = RUN ? column(more ? item + 1 : item) : cur;
        f32x16 z[C][NQ];               // S[i = 32 qi + 8 g + 4 hf + e, r = 32 n + m], then its exponentials
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int n = w + c * W;
            if (n >= nch) {
#pragma unroll
                for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
                    for (int v = 0; v < 16; ++v) z[c][qi][v] = -INFINITY;
                continue;
            }
            // chunk n has landed when only the one requested after it is outstanding
            if (n + W < nch) wait_vm<NG + 1>();
            else wait_vm<0>();
            const char* kt = wl + (c & 1) * L::kBuf;
            const float cc = *(const float*)(kt + L::kTile + m * 4);
            const bool rok = 32 * n + m < r_lim;
            // a row of Kbar is read once for the query tiles, whose products are independent chains
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
                const u32x4 bk = *(const u32x4*)(kt + (b_off ^ (uint32_t)(ds << 5)));
#pragma unroll
                for (int qi = 0; qi < NQ; ++qi) {
                    const u32x4 aq = *(const u32x4*)(qt + qi * L::kTile + (b_off ^ (uint32_t)(ds << 5)));
                    z[c][qi] = E::mfma32(aq, bk, ds ? z[c][qi] : kZero);
                }
            }
#pragma unroll
            for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
                for (int v = 0; v < 16; ++v) z[c][qi][v] = RUN || rok ? z[c][qi][v] * sc2 - cc : -INFINITY;
            if (RUN && 32 * n + 32 > r_lim) {                // uniform: the last chunk, where it is not a whole one
#pragma unroll
                for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
                    for (int v = 0; v < 16; ++v) z[c][qi][v] = rok ? z[c][qi][v] : -INFINITY;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the chunk has been read: the next but one may land on it
            if (n + 2 * W < nch) issue(cur, n + 2 * W, c & 1);
        }
        if (more && w < nch) issue(next, w, 0);                      // both chunk buffers have been read

        // Rows' maxima and sums over this wave's chunks, to the front of its second chunk buffer: [NQ * 32] maxima, sums
        float* const own = (float*)(wl + L::kBuf);
        const int at = half_reduce_at(m), myrow = 8 * (at >> 2) + 4 * hf + (at & 3);
#pragma unroll
        for (int qi = 0; qi < NQ; ++qi) {
            float t[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                t[v] = z[0][qi][v];
#pragma unroll
                for (int c = 1; c < C; ++c) t[v] = fmaxf(t[v], z[c][qi][v]);
            }
            own[32 * qi + myrow] = half_reduce<true>(t, m);
        }
        lds_wave_sync();
#pragma unroll
        for (int qi = 0; qi < NQ; ++qi) {
            float t[16];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 mx = *(const f32x4*)(own + 32 * qi + 8 * g + 4 * hf);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float base = mx[e] == -INFINITY ? 0.f : mx[e];       // a wave without chunks
                    t[4 * g + e] = 0.f;
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        z[c][qi][4 * g + e] = fast_exp2(z[c][qi][4 * g + e] - base);
                        t[4 * g + e] += z[c][qi][4 * g + e];
                    }
                }
            }
            own[NQ * 32 + 32 * qi + myrow] = half_reduce<false>(t, m);
        }
        if (W > 1) lds_barrier();
        else lds_wave_sync();
        // scale of row i for this wave: exp2(max_wave - max) / sum, behind the maxima and sums that other waves still read
        for (int i = lane; i < NQ * 32; i += 64) {
            float mx[W], sm[W], M = -INFINITY, sum = 0.f;
#pragma unroll
            for (int x = 0; x < W; ++x) {
                const float* o = (const float*)((W == 1 ? wl : lds_s2 + x * L::kWave) + L::kBuf);
                mx[x] = o[i];
                sm[x] = o[NQ * 32 + i];
            }
#pragma unroll
            for (int x = 0; x < W; ++x) M = fmaxf(M, mx[x]);
#pragma unroll
            for (int x = 0; x < W; ++x) sum += sm[x] * fast_exp2(mx[x] - M);          // a wave without chunks: 0 * exp2(-inf)
            own[2 * NQ * 32 + i] = i < p.b1 ? fast_exp2(own[i] - M) / sum : 0.f;
        }
        lds_wave_sync();

#pragma unroll
        for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 fac = *(const f32x4*)(own + 2 * NQ * 32 + 32 * qi + 8 * g + 4 * hf);
#pragma unroll
                for (int c = 0; c < C; ++c)
#pragma unroll
                    for (int e = 0; e < 4; ++e) z[c][qi][4 * g + e] *= fac[e];
            }
        if constexpr (RUN) {
            // weights; the scaled values become the B operands of the representatives
            u32x4 pb[C][NQ][2];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int n = w + c * W;
                float wsum = 0.f;
#pragma unroll
                for (int qi = 0; qi < NQ; ++qi) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) wsum += z[c][qi][v];
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        pb[c][qi][q].x = pack2<E>(z[c][qi][8 * q + 0], z[c][qi][8 * q + 1]);
                        pb[c][qi][q].y = pack2<E>(z[c][qi][8 * q + 2], z[c][qi][8 * q + 3]);
                        pb[c][qi][q].z = pack2<E>(z[c][qi][8 * q + 4], z[c][qi][8 * q + 5]);
                        pb[c][qi][q].w = pack2<E>(z[c][qi][8 * q + 6], z[c][qi][8 * q + 7]);
                    }
                }
                wsum = xhalf_sum(wsum);
                if (n < nch && hf == 0) p.wgt[cur.blk + 32 * n + m] = wsum;
            }
            // rep^T[d = 32 dt + 8 g + 4 hf + e, r], a pair of head-dim blocks at a time: their query rows are read once for all
            // chunks, whose products are independent chains, and the exchanges of step 1 leave whole lines to store, 128 bytes of
            // each of 8 rows an instruction.
            const uint32_t piece = (uint32_t)(4 * ((m >> 3) & 1) + 2 * ((m >> 4) & 1) + hf) * 16;
#pragma unroll
            for (int dp = 0; dp < DT / 2; ++dp) {
                u32x4 aq[2][NQ][2];
#pragma unroll
                for (int dl = 0; dl < 2; ++dl)
#pragma unroll
                    for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            const u32x2 lo = s1_read_tr(qt + qi * L::kTile, tr[2 * dp + dl][0] + q * 16 * L::kPitch);
                            const u32x2 hi = s1_read_tr(qt + qi * L::kTile, tr[2 * dp + dl][1] + q * 16 * L::kPitch);
                            aq[dl][qi][q] = u32x4{lo.x, lo.y, hi.x, hi.y};
                        }
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const int n = w + c * W;
                    if (n >= nch) break;
                    f32x16 acc[2];
#pragma unroll
                    for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
                        for (int q = 0; q < 2; ++q)
#pragma unroll
                            for (int dl = 0; dl < 2; ++dl) acc[dl] = E::mfma32(aq[dl][qi][q], pb[c][qi][q], (qi | q) ? acc[dl] : kZero);
                    uint32_t x[2][2][4];             // [block in pair][gp][dword]
#pragma unroll
                    for (int dl = 0; dl < 2; ++dl) {
#pragma unroll
                        for (int gp = 0; gp < 2; ++gp) {
                            const int g0 = 2 * gp, g1 = 2 * gp + 1;
                            auto rx = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[dl][4 * g0 + 0], acc[dl][4 * g0 + 1]),
                                                                       pack2<E>(acc[dl][4 * g1 + 0], acc[dl][4 * g1 + 1]), false, false);
                            auto ry = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[dl][4 * g0 + 2], acc[dl][4 * g0 + 3]),
                                                                       pack2<E>(acc[dl][4 * g1 + 2], acc[dl][4 * g1 + 3]), false, false);
                            x[dl][gp][0] = rx[0]; x[dl][gp][1] = ry[0]; x[dl][gp][2] = rx[1]; x[dl][gp][3] = ry[1];
                        }
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            auto y = __builtin_amdgcn_permlane16_swap(x[dl][0][q], x[dl][1][q], false, false);
                            x[dl][0][q] = y[0]; x[dl][1][q] = y[1];
                        }
                    }
                    char* const rows = (char*)p.rep + (cur.blk + 32 * n + (m & 7)) * (2 * D) + 128 * dp + piece;
#pragma unroll
                    for (int r4 = 0; r4 < 2; ++r4) {
                        u32x4 lo, hi;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            lo[q] = (uint32_t)__builtin_amdgcn_update_dpp((int)x[0][r4][q], (int)x[1][r4][q], 0x128, 0xf, 0xc, false);
                            hi[q] = (uint32_t)__builtin_amdgcn_update_dpp((int)x[1][r4][q], (int)x[0][r4][q], 0x128, 0xf, 0x3, false);
                        }
                        u32x4* const at = (u32x4*)(rows + 2 * r4 * 8 * (2 * D));
                        u32x4* const at_hi = (u32x4*)(rows + (2 * r4 + 1) * 8 * (2 * D));
                        __builtin_nontemporal_store(lo, at);
                        __builtin_nontemporal_store(hi, at_hi);
                    }
                }
            }
        } else {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int n = w + c * W;
                if (n >= nch) break;
                float wsum = 0.f;
                u32x4 pb[NQ][2];
#pragma unroll
                for (int qi = 0; qi < NQ; ++qi) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) wsum += z[c][qi][v];
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        pb[qi][q].x = pack2<E>(z[c][qi][8 * q + 0], z[c][qi][8 * q + 1]);
                        pb[qi][q].y = pack2<E>(z[c][qi][8 * q + 2], z[c][qi][8 * q + 3]);
                        pb[qi][q].z = pack2<E>(z[c][qi][8 * q + 4], z[c][qi][8 * q + 5]);
                        pb[qi][q].w = pack2<E>(z[c][qi][8 * q + 6], z[c][qi][8 * q + 7]);
                    }
                }
                wsum = xhalf_sum(wsum);
                if (hf == 0) p.wgt[cur.blk + 32 * n + m] = wsum;
                char* rrow = (char*)p.rep + (cur.blk + 32 * n + m) * (2 * D);
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    f32x16 acc;
#pragma unroll
                    for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            const u32x2 lo = s1_read_tr(qt + qi * L::kTile, tr[dt][0] + q * 16 * L::kPitch);
                            const u32x2 hi = s1_read_tr(qt + qi * L::kTile, tr[dt][1] + q * 16 * L::kPitch);
                            const u32x4 aq = {lo.x, lo.y, hi.x, hi.y};
                            acc = E::mfma32(aq, pb[qi][q], (qi | q) ? acc : kZero);
                        }
                    // rep^T[d = 32 dt + 8 g + 4 hf + e, r]: the half-swap leaves 8 consecutive d per lane
#pragma unroll
                    for (int gp = 0; gp < 2; ++gp) {
                        const int g0 = 2 * gp, g1 = 2 * gp + 1;
                        auto rx = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[4 * g0 + 0], acc[4 * g0 + 1]),
                                                                   pack2<E>(acc[4 * g1 + 0], acc[4 * g1 + 1]), false, false);
                        auto ry = __builtin_amdgcn_permlane32_swap(pack2<E>(acc[4 * g0 + 2], acc[4 * g0 + 3]),
                                                                   pack2<E>(acc[4 * g1 + 2], acc[4 * g1 + 3]), false, false);
                        const u32x4 o = {(uint32_t)rx[0], (uint32_t)ry[0], (uint32_t)rx[1], (uint32_t)ry[1]};
                        *(u32x4*)(rrow + (32 * dt + 16 * gp + 8 * hf) * 2) = o;
                    }
                }
            }
        }
        if (!more) return;
        // The next column's first chunk is on its way since its buffer was read; the queries take the place of this one's, and
        // the second chunk that of the maxima and sums, when every wave is done with them.
        lds_barrier();
        cur = next;
        queries(cur);
        if (w + W < nch) {
            issue(cur, w + W, 1);
            wait_vm<NG + 1>();
        } else {
            wait_vm<0>();
        }
        lds_barrier();
    }
}

// ------------------------------------------------------------------------------------------------
// host launch
// ------------------------------------------------------------------------------------------------
bool monarch_mfma_supported(int dtype, int D, int b2) {
    return (dtype == SFM_BF16 || dtype == SFM_F16) && (D == 64 || D == 128) && b2 >= 1 && b2 <= 128;
}

int cu_count() {
    static thread_local int cached_dev = -1, cached = 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (dev != cached_dev) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached = n;
        cached_dev = dev;
    }
    return cached;
}

enum class Step1 { kWhole, kIter, kIterKbar };           // the forward's (or the backward's), a refinement's last pass, its earlier ones

struct Step1Kernel {
    const void* fn;
    size_t group;      // bytes of LDS of a wave group
};

template <class E, int D, int NT>
static Step1Kernel step1_kernel(const MonarchArgs& a, Step1 kind) {
    constexpr size_t whole = S1Lds<D, NT, false>::kGroup;
    if (kind == Step1::kIterKbar)
        return {a.new_kv ? (const void*)monarch_step1_kernel<E, D, NT, false, true, true, false, true> : (const void*)monarch_step1_kernel<E, D, NT, false, true, true>,
                S1Lds<D, NT, true>::kGroup};
    if (kind == Step1::kIter)
        return {a.new_kv ? (const void*)monarch_step1_kernel<E, D, NT, false, true, false, false, true> : (const void*)monarch_step1_kernel<E, D, NT, false, true>, whole};
    if constexpr (NT <= 2) {
        if (a.rb && a.new_kv) return {(const void*)monarch_step1_kernel<E, D, NT, true, false, false, false, true>, whole};
    }
    if (a.new_kv) return {(const void*)monarch_step1_kernel<E, D, NT, false, false, false, false, true>, whole};
    const bool skip = a.causal && a.skip_masked;
    if constexpr (NT <= 2) {
        if (a.rb) return {skip ? (const void*)monarch_step1_kernel<E, D, NT, true, false, false, true> : (const void*)monarch_step1_kernel<E, D, NT, true>, whole};
    }
    return {skip ? (const void*)monarch_step1_kernel<E, D, NT, false, false, false, true> : (const void*)monarch_step1_kernel<E, D, NT, false>, whole};
}

// Enqueues step 1 (with the right factor written too when a.rb is set).
template <class E, int D>
static int enqueue_step1(const MonarchArgs& a, int nunits, hipStream_t stream, Step1 kind = Step1::kWhole) {
    const int ncols = a.a_chunk * a.b2;
    const int nwaves = (ncols + 31) / 32;                 // a wave per 32 (a, j) columns
    if (nwaves < 1 || nwaves > 8) {
        set_error("internal: step-1 launch shape (a_chunk=%d, b2=%d)", a.a_chunk, a.b2);
        return SFM_ERR_UNSUPPORTED;
    }
    const int nt = (a.b2 + 31) / 32;
    if (nt > 2 && a.rb) {
        set_error("internal: the right factor is written for b2 <= 64 only");
        return SFM_ERR_UNSUPPORTED;
    }
    const Step1Kernel k = nt == 4   ? step1_kernel<E, D, 4>(a, kind)
                          : nt == 3 ? step1_kernel<E, D, 3>(a, kind)
                          : nt == 2 ? step1_kernel<E, D, 2>(a, kind)
                                    : step1_kernel<E, D, 1>(a, kind);
    MonarchArgs a1 = a;
    a1.s1_total = a.nf * a.b1 * nunits * a.n_achunks;
    // One workgroup per CU, of as many wave groups as its LDS holds up to 8 waves, or two of 5 (or 6, below; 8 waves in all where one has
    // 256 registers): a group's loads, logits, softmax and stores follow each other, and the other groups fill the gaps.  A
    // group has the waves that its columns need and no more.  With at least four, the others of which formed and stored the last
    // column again and again, and never more than two groups, three refinement passes at three frames tied (52 columns, 12
    // heads x 128, 480p, 21 frames) took 529 us, now 499 (Kbar alone, four groups: 92 -> 73 a pass); one pass 176 -> 164; three
    // tied frames against themselves 50 -> 46; 24 columns of nine 30 x 24 frames 52 -> 39.  Four groups of three waves: 50 us
    // at 7 heads of nine 23 x 31 frames, two 44.5.  Two or four waves for 32 columns, each with its part of the output, took
    // the refinement to 505 and 541 us: they fetch the query rows as often.
    a1.s1_cached = step1_through_caches(a, nunits, kind == Step1::kIterKbar);
    const int cus = a.s1_wgs > 0 ? a.s1_wgs : cu_count();
    // Two groups of six waves are worth it at head_dim 64 only (176 columns of 44 x 44, 12 heads: 161 us, one group 172; head_dim 128
    // 304, 297; 192 columns of 30 x 64 240, 232).
    const int by_waves = nt > 2 ? 8 / nwaves : nwaves == 6 && D == 128 ? 1 : std::min(12 / nwaves, std::max(2, 8 / nwaves));      // within the launch bounds
    const int room = std::min(by_waves, (int)(160 * 1024 / k.group));
    a1.s1_groups = std::max(1, std::min(room, (a1.s1_total + cus - 1) / cus));
    const int wgs = std::min(cus, (a1.s1_total + a1.s1_groups - 1) / a1.s1_groups);
    const size_t lds1 = k.group * a1.s1_groups;
    if (lds1 > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(k.fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds1);
        if (e != hipSuccess) {
            set_error("hipFuncSetAttribute failed: %s", hipGetErrorString(e));
            return SFM_ERR_HIP;
        }
    }
    void* args[] = {&a1};
    hipError_t e = hipLaunchKernel(k.fn, dim3(wgs), dim3(nwaves * 64 * a1.s1_groups), args, lds1, stream);
    if (e != hipSuccess) {
        set_error("hip launch failed: %s", hipGetErrorString(e));
        return SFM_ERR_HIP;
    }
    return SFM_OK;
}

template <class E, int D, int TEAM>
static const void* step2_kernel(bool past) {
    return past ? (const void*)monarch_step2_kernel<E, D, TEAM, false, true> : (const void*)monarch_step2_kernel<E, D, TEAM>;
}

// Enqueues step 2: a wave per column (a, j) of up to 32 query rows, a team of waves for more.  `stats_only` (b1 <= 128):
// the row statistics without the output.
template <class E, int D>
static int enqueue_step2(const MonarchArgs& a, int nunits, hipStream_t stream, bool stats_only = false) {
    const int team = a.b1 > 96 ? 4 : (a.b1 + 31) / 32;
    const bool past = step2_past_caches(a, nunits);
    const void* fn = stats_only ? (team == 4   ? (const void*)monarch_left_stats_kernel<E, D, 4>
                                   : team == 3 ? (const void*)monarch_left_stats_kernel<E, D, 3>
                                   : team == 2 ? (const void*)monarch_left_stats_kernel<E, D, 2>
                                               : (const void*)monarch_left_stats_kernel<E, D, 1>)
                   : team == 4 ? step2_kernel<E, D, 4>(past) : team == 3 ? step2_kernel<E, D, 3>(past)
                   : team == 2 ? step2_kernel<E, D, 2>(past) : step2_kernel<E, D, 1>(past);
    const size_t lds = stats_only ? (team == 4   ? StLds<D, 4>::bytes()
                                     : team == 3 ? StLds<D, 3>::bytes()
                                     : team == 2 ? StLds<D, 2>::bytes()
                                                 : StLds<D, 1>::bytes())
                       : team > 1 ? S2Lds<D>::team_bytes(team) : S2Lds<D>::bytes();
    MonarchArgs a2 = a;
    a2.s2_split = 1;
    if (team == 1) {
        // Up to two columns per compute unit leave most SIMDs idle and four waves share each: 21 cached frames of 480p against
        // one head 60.5 -> 41.9 us for the whole call, 2 heads 75.7 -> 65.4, 8 heads and one query frame (416 columns) 117 ->
        // 108; at 624 columns (4 heads) sharing by two or four loses 2 %.  The rule looks at all units of the call, not at
        // those of this pass, so that the results do not depend on how a call is cut into passes.
        const int64_t columns = (int64_t)a.B * a.H * a.na * a.b2;
        const int nch = (a.nf * a.b1 + 31) / 32;
        if (columns <= 2 * (int64_t)cu_count()) a2.s2_split = nch >= 8 ? 4 : nch >= 4 ? 2 : 1;
        if (!stats_only && a2.s2_split > 1) fn = (const void*)monarch_step2_kernel<E, D, 1, true>;
    }
    const int per_wg = team > 1 ? 1 : 4 / a2.s2_split;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            set_error("hipFuncSetAttribute failed: %s", hipGetErrorString(e));
            return SFM_ERR_HIP;
        }
    }
    const dim3 grid(a.na * ((a.b2 + per_wg - 1) / per_wg), nunits, team > 1 ? (a.b1 + 127) / 128 : 1);
    void* args[] = {&a2};
    hipError_t e = hipLaunchKernel(fn, grid, dim3(team > 1 ? 64 * team : 256), args, lds, stream);
    if (e != hipSuccess) {
        set_error("hip launch failed: %s", hipGetErrorString(e));
        return SFM_ERR_HIP;
    }
    return SFM_OK;
}

template <class E, int D>
static int launch_t(const MonarchArgs& a, int nunits, hipStream_t stream, const StepEvents* ev) {
    if (ev) (void)hipEventRecord(ev->ev[0], stream);
    MonarchArgs a0 = a;
    a0.skip_masked = 1;                                  // step 2 stops at a column's last visible row
    if (int rc = enqueue_step1<E, D>(a0, nunits, stream)) return rc;
    if (ev) (void)hipEventRecord(ev->ev[1], stream);
    if (int rc = enqueue_step2<E, D>(a, nunits, stream)) return rc;
    if (ev) (void)hipEventRecord(ev->ev[2], stream);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        set_error("hip launch failed: %s", hipGetErrorString(err));
        return SFM_ERR_HIP;
    }
    return SFM_OK;
}

template <class E, int D>
static int launch_step1_t(const MonarchArgs& a, int nunits, hipStream_t stream) {
    return enqueue_step1<E, D>(a, nunits, stream);
}

int launch_monarch_step1(const MonarchArgs& a, int dtype, int nunits, hipStream_t stream) {
    if (dtype == SFM_BF16)
        return a.D == 128 ? launch_step1_t<BF16, 128>(a, nunits, stream) : launch_step1_t<BF16, 64>(a, nunits, stream);
    return a.D == 128 ? launch_step1_t<F16, 128>(a, nunits, stream) : launch_step1_t<F16, 64>(a, nunits, stream);
}

bool monarch_iter_mfma_supported(int dtype, int D, int b1, int b2) {
    return monarch_mfma_supported(dtype, D, b2) && b1 >= 1 && b1 <= 128;
}

template <class E, int D, int NQ>
static int launch_rep_t(const MonarchArgs& a, int nunits, hipStream_t stream) {
    using L = RepLds<D, NQ>;
    hipError_t e = hipFuncSetAttribute((const void*)monarch_rep_kernel<E, D, NQ>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::bytes());
    if (e != hipSuccess) {
        set_error("hipFuncSetAttribute failed: %s", hipGetErrorString(e));
        return SFM_ERR_HIP;
    }
    const int njg = L::kShared ? a.b2 : (a.b2 + L::kWaves - 1) / L::kWaves;
    hipLaunchKernelGGL((monarch_rep_kernel<E, D, NQ>), dim3(a.na * njg, nunits), dim3(64 * L::kWaves), L::bytes(), stream, a);
    return SFM_OK;
}

// Representatives and weights in one kernel; false where the logits of a column do not fit its waves' registers (C chunks of
// NQ tiles are 16 C NQ of them, and four query tiles spill at two chunks).  Up to four chunks a wave has a column of its own:
// three passes of 2 heads x 64 over 24 rows took 41.0 us with the two kernels, now 34.0; three frames of 480p 134 -> 123.
template <class E, int D, int NQ, int W, int C>
static bool launch_weights_t(const MonarchArgs& a, int nunits, hipStream_t stream, int* rc) {
    using L = WtLds<D, NQ, W>;
    if ((a.nf * a.b1 + 31) / 32 > W * C) return false;
    int items = nunits * a.na * ((a.b2 + L::kCols - 1) / L::kCols);
    const int room = std::min((int)(160 * 1024 / L::bytes()), 8 / L::kWaves) * cu_count();      // workgroups at a time
    // More columns than the chip holds at a time are taken in runs, unless the representatives are so small that the next pass finds
    // them in the caches, which these kernels store past: three passes at three frames tied (100 MB) 444 us against 471, 5 heads x 64
    // of 23 x 41, 15 frames (9 MB) 137 against 127.  One query tile gains 1 % at most and loses 8 % where columns are few.
    constexpr bool kRun = NQ > 1 && !(D == 64 && NQ == 3);    // (registers)
    const bool run = kRun && items > room && (int64_t)nunits * a.na * a.b2 * a.r_pad * (2 * D) > (int64_t)64 << 20;
    const void* fn = run ? (const void*)monarch_weights_kernel<E, D, NQ, W, C, kRun> : (const void*)monarch_weights_kernel<E, D, NQ, W, C, false>;
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::bytes());
    MonarchArgs a1 = a;
    void* args[] = {&a1, &items};
    if (e == hipSuccess) e = hipLaunchKernel(fn, run ? dim3(room) : dim3(items / nunits, nunits), dim3(64 * L::kWaves), args, L::bytes(), stream);
    if (e != hipSuccess) set_error("hip launch failed: %s", hipGetErrorString(e));
    *rc = e == hipSuccess ? SFM_OK : SFM_ERR_HIP;
    return true;
}

template <class E, int D>
static bool launch_weights(const MonarchArgs& a, int nunits, hipStream_t stream, int* rc) {
    switch ((a.b1 + 31) / 32) {
        case 1: return launch_weights_t<E, D, 1, 1, 4>(a, nunits, stream, rc) || launch_weights_t<E, D, 1, 4, 8>(a, nunits, stream, rc);
        case 2: {
            // Eight waves that get a chunk or none leave compute units, which hold one such workgroup, idle: with many columns the two
            // kernels are faster.  18 heads x 64 of 40 x 44, 6 frames (8 chunks, 2376 columns) 82 us, 29 + 39; two passes of 12 x
            // 64 of 40 x 40, 3 frames (4 chunks, 1440) 103, 91; 36 x 128 of these (4320) 399, 391, 18 x 128 0.97 of the time of two
            // kernels, 2 x 64 of 40 x 16 0.82.
            const int chunks = (a.nf * a.b1 + 31) / 32, cols = nunits * a.na * a.b2;
            if (chunks <= (D == 64 ? 8 : 5) && cols > (D == 64 ? 1 : 10) * cu_count()) return false;
            return launch_weights_t<E, D, 2, 8, 4>(a, nunits, stream, rc);
        }
        case 3: return launch_weights_t<E, D, 3, 8, 3>(a, nunits, stream, rc);
        default: return false;
    }
}

// num_iters - 1 passes of [step 1 with the pass's query operands, Kbar only | row statistics of the left factor |
// representatives for the next pass], then a whole forward with the last representatives.  (With whole forwards in every
// pass a three-pass call at three frames tied took 696 us.)
template <class E, int D>
static int launch_iter_t(const MonarchArgs& a, int nunits, int num_iters, hipStream_t stream) {
    const int nq = (a.b1 + 31) / 32;
    for (int it = 0; it < num_iters; ++it) {
        const bool last = it + 1 == num_iters;
        MonarchArgs a1 = a;
        a1.rb = nullptr;
        a1.iter_mode = it == 0 ? 1 : 2;
        a1.new_kv = it == 0 || last ? a.new_kv : 0;      // K in the first pass, V in the last
        if (int rc = enqueue_step1<E, D>(a1, nunits, stream, last ? Step1::kIter : Step1::kIterKbar)) return rc;
        MonarchArgs a2 = a;
        if (last) a2.stats = nullptr;
        int wrc = SFM_OK;
        if (!last && launch_weights<E, D>(a, nunits, stream, &wrc)) {
            if (wrc) return wrc;
            continue;
        }
        if (int rc = enqueue_step2<E, D>(a2, nunits, stream, !last)) return rc;
        if (!last) {
            const int rc = nq == 1 ? launch_rep_t<E, D, 1>(a, nunits, stream) : nq == 2 ? launch_rep_t<E, D, 2>(a, nunits, stream)
                         : nq == 3 ? launch_rep_t<E, D, 3>(a, nunits, stream) : launch_rep_t<E, D, 4>(a, nunits, stream);
            if (rc) return rc;
        }
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("hip launch failed: %s", hipGetErrorString(e));
        return SFM_ERR_HIP;
    }
    return SFM_OK;
}

int launch_monarch_iter_mfma(const MonarchArgs& a, int dtype, int nunits, int num_iters, hipStream_t stream) {
    if (!monarch_iter_mfma_supported(dtype, a.D, a.b1, a.b2) || a.causal || !a.rep || !a.wgt || !a.stats ||
        (int)a.stats_ld < (a.b1 + 31) / 32 * 32) {
        set_error("internal: iterated MFMA launch");
        return SFM_ERR_UNSUPPORTED;
    }
    if (dtype == SFM_BF16)
        return a.D == 128 ? launch_iter_t<BF16, 128>(a, nunits, num_iters, stream) : launch_iter_t<BF16, 64>(a, nunits, num_iters, stream);
    return a.D == 128 ? launch_iter_t<F16, 128>(a, nunits, num_iters, stream) : launch_iter_t<F16, 64>(a, nunits, num_iters, stream);
}

int launch_monarch_mfma(const MonarchArgs& a, int dtype, int nunits, hipStream_t stream, const StepEvents* ev) {
    if (dtype == SFM_BF16)
        return a.D == 128 ? launch_t<BF16, 128>(a, nunits, stream, ev) : launch_t<BF16, 64>(a, nunits, stream, ev);
    return a.D == 128 ? launch_t<F16, 128>(a, nunits, stream, ev) : launch_t<F16, 64>(a, nunits, stream, ev);
}

}  // namespace sfm
