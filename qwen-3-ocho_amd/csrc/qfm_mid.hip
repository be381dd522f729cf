// qfm_mid.hip -- the forward at a middle number of rows (more than 8, mid_takes):
// weight-streaming grouped MFMA GEMMs.
//
// Reference behaviour: the chunk path (ocho/amd_server/qf8_moe_i8.hip:196-395)
// at the row counts of batched decode and prompt chunks. An expert has a few
// rows here (T K / E on average), so the layer is bound by reading every
// distinct expert's weights once; the 128-row tiles of the prefill GEMMs
// (qfm_prefill.hip) would spend their time on padding rows.
//
// Launches:
//   k_mid_router   exact logits in the canonical fp32 order (8 token rows in
//                  LDS at a time, two experts per wave), the shared-expert
//                  gate, and x as fp16 scaled by 2^k per token with row sums;
//   k_mid_topk     one wave per token (wave_topk);
//   k_mid_plan     one block: the pairs grouped by expert and the work items
//                  {group, first pair, rows <= 16 NT}, or the tiles of the
//                  prefill's GEMMs where a router crowds its rows on few experts
//                  (mid_cost; these then run in place of the next two);
//   k_mid_gateup   hidden = silu(g) * u per item and 64 intermediate rows, as
//                  fp16 scaled by 2^k per pair and those 64;
//   k_mid_down     partials per item and 256 output columns, as fp16 scaled by
//                  2^k per pair and 64 columns (the prefill's form);
//   k_pf_combine_h the K + 1 partials of a token in slot order.
//
// GEMM form: the 16 rows of an MFMA tile are weight rows, its 16 columns the
// item's tokens (NT tiles of 16). A wave reads its weight rows 16 bytes a lane
// along the rows, several chunks in flight in registers, and turns them into
// MFMA fragments through wave-private LDS (fragments loaded straight from
// memory touch 16 rows an instruction, ~64 cycles each). INT8 codes become
// fp16 exactly (1024 + u by v_perm, then - 1152), e2m1 codes fp16 by
// v_cvt_scalef32_pk_f16_fp4 times the block scale (at most 6 significant bits:
// exact). Columns past the item's rows hold whatever LDS held: an MFMA column
// never reaches another one, and they are not stored.
#include "qfm_dev.h"
#include "qfm_internal.h"
#include "qfm_mfma.h"
#include "qfm_prefill_layout.h"

namespace qfm {

// ---- router ---------------------------------------------------------------------
// Blocks [0, ceil(T / 4)): a wave per token writes x as fp16 scaled by 2^k
// (largest magnitude in [2^14, 2^15): bf16 values from 2^-28 of the row's largest
// on exact, smaller ones to 2^-39 of it) and 2^-k. The others:
// 8 router rows (two per wave, held in registers) x tg groups of 8 tokens,
// whose x rows go through LDS; block row E / 8 is the shared-expert gate
// vector. Every dot keeps the canonical order (canon_reduce_rows).
template <int NJ>
__global__ void __launch_bounds__(256, NJ == 8 ? 3 : 2)
k_mid_router(const float *__restrict__ W, const float *__restrict__ bias, const float *__restrict__ g,
             const uint16_t *__restrict__ x, int T, int E, int tg, float *__restrict__ logits,
             float *__restrict__ gam, uint4 *__restrict__ x16, float *__restrict__ x16isc, float *__restrict__ xsum,
             float *__restrict__ x16sum, int *__restrict__ ctr) {
    constexpr int H = NJ * 256;
    __shared__ __align__(16) uint16_t s_x[8 * H];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nxc = (T + 3) / 4;
    if ((int)blockIdx.x < nxc) {
        if (blockIdx.x == 0 && tid < 8) ctr[tid] = 0;          // the selection counts into ctr[0] in a later launch
        const int t = blockIdx.x * 4 + wave;
        if (t >= T) return;
        const uint4 *xr = reinterpret_cast<const uint4 *>(x + (size_t)t * H);
        constexpr int NC = H / 512;
        uint4 v[NC];
#pragma unroll
        for (int q = 0; q < NC; q++) v[q] = xr[q * 64 + lane];
        float amax = 0.0f;
#pragma unroll
        for (int q = 0; q < NC; q++) {
            const uint32_t d[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
#pragma unroll
            for (int u = 0; u < 4; u++) amax = fmaxf(amax, fmaxf(fabsf(bf16_lo(d[u])), fabsf(bf16_hi(d[u]))));
        }
        amax = group_max<64>(amax);
        const int k = amax == 0.0f ? 0 : min(113, max(-113, 141 - (int)(__float_as_uint(amax) >> 23)));
        const float sc = __uint_as_float((uint32_t)(127 + k) << 23);
        uint4 *xo = x16 + (size_t)t * (H / 8);
        float sx = 0.0f, hs = 0.0f;
#pragma unroll
        for (int q = 0; q < NC; q++) {
            const uint32_t d[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
            uint32_t o[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const f16x2_t hp = {(_Float16)(bf16_lo(d[u]) * sc), (_Float16)(bf16_hi(d[u]) * sc)};
                sx += bf16_lo(d[u]) + bf16_hi(d[u]);
                hs += (float)hp.x + (float)hp.y;
                o[u] = __builtin_bit_cast(uint32_t, hp);
            }
            xo[q * 64 + lane] = make_uint4(o[0], o[1], o[2], o[3]);
        }
        sx = group_sum<64>(sx);
        hs = group_sum<64>(hs);
        if (lane == 0) {
            xsum[t] = sx;
            x16sum[t] = hs;
        }
        if (lane == 0) x16isc[t] = __uint_as_float((uint32_t)(127 - k) << 23);
        return;
    }
    const int nx = E / 8 + (g ? 1 : 0), r = (int)blockIdx.x - nxc, xb = r % nx, yb = r / nx;
    const bool is_g = xb == E / 8;
    const int e0 = xb * 8 + wave * 2;
    const int t0 = yb * tg * 8, t1 = min(T, t0 + tg * 8);
    float4 w[2][NJ];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const float *wr = is_g ? g : W + (size_t)(e0 + q) * H;
#pragma unroll
        for (int j = 0; j < NJ; j++) w[q][j] = *reinterpret_cast<const float4 *>(wr + j * 256 + lane * 4);
    }
    u32x4_t xv[NJ];                                            // one group: 8 H / 8 chunks over 256 threads
    auto load = [&](int m0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NJ; i++) {
            const int c = i * 256 + tid, row = c / (H / 8);
            xv[i] = m0 + row < T ? reinterpret_cast<const u32x4_t *>(x + (size_t)(m0 + row) * H)[c - row * (H / 8)]
                                 : u32x4_t{0u, 0u, 0u, 0u};
        }
    };
    load(t0);
    for (int m0 = t0; m0 < t1; m0 += 8) {
        if (m0 > t0) __syncthreads();                          // the previous group is consumed
#pragma unroll
        for (int i = 0; i < NJ; i++) reinterpret_cast<u32x4_t *>(s_x)[i * 256 + tid] = xv[i];
        __syncthreads();
        if (m0 + 8 < t1) load(m0 + 8);
        float a[2][8];
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int i = 0; i < 8; i++) a[q][i] = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint2 p = *reinterpret_cast<const uint2 *>(&s_x[i * H + j * 256 + lane * 4]);
                const float x0 = bf16_lo(p.x), x1 = bf16_hi(p.x), x2 = bf16_lo(p.y), x3 = bf16_hi(p.y);
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    a[q][i] = __fmaf_rn(w[q][j].x, x0, a[q][i]);
                    a[q][i] = __fmaf_rn(w[q][j].y, x1, a[q][i]);
                    a[q][i] = __fmaf_rn(w[q][j].z, x2, a[q][i]);
                    a[q][i] = __fmaf_rn(w[q][j].w, x3, a[q][i]);
                }
            }
        }
        // (the second expert's chains would otherwise sink below the first
        // one's reduction, with every unpacked x value kept for them)
#pragma unroll
        for (int i = 0; i < 8; i++) asm volatile("" : "+v"(a[0][i]), "+v"(a[1][i]));
#pragma unroll
        for (int q = 0; q < 2; q++) {
            float v = canon_reduce_rows<8>(a[q], lane);        // lane r < 8: token m0 + r
            if (lane < 8 && m0 + lane < T) {
                if (is_g) {
                    if (wave == 0 && q == 0) gam[m0 + lane] = sigmoid(v);
                } else {
                    if (bias) v = __fadd_rn(v, bias[e0 + q]);
                    logits[(size_t)(m0 + lane) * E + e0 + q] = v;
                }
            }
        }
    }
}

// One wave per token (wave_topk). n_over counts the tokens with more than 64
// candidates (the exact form of topk_candidates' bound).
template <int EPL>
__global__ void __launch_bounds__(256)
k_mid_topk(const float *__restrict__ logits, int T, int K, int renorm, int *__restrict__ sel, float *__restrict__ wts,
           int *__restrict__ n_over) {
    constexpr int E = EPL * 64;
    __shared__ __align__(16) unsigned long long s_tk[4][kTopkLds];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = blockIdx.x * 4 + wave;
    if (t >= T) return;
    float v[EPL];
#pragma unroll
    for (int i = 0; i < EPL; i++) v[i] = logits[(size_t)t * E + i * 64 + lane];
    int my_i;
    float my_w;
    bool over;
    wave_topk_regs<EPL>(v, K, renorm, lane, s_tk[wave], my_i, my_w, &over);
    if (lane < K) {
        sel[(size_t)t * K + lane] = my_i;
        wts[(size_t)t * K + lane] = my_w;
    }
    if (over && lane == 0) atomicAdd(n_over, 1);
}

// ---- plan -------------------------------------------------------------------------
// A pair is {partial slot t (K + shared) + k, weight bits}: its token is slot / S.
// One block of 1024 threads: pair counts per expert (LDS), offsets, the pairs
// scattered into expert order (the order inside a group is unspecified, as in
// k_pf_scatter), the shared expert's pairs (group E) in token order, and the
// items: the shared group's first, then the experts' in ascending order. The
// selection is read in batches of 16 a thread, and a pair leaves as one 8-byte
// store (scattered stores of three arrays and loads one at a time took 29 us at
// 1021 rows). ctr[3] is the number of items, ctr[4] and ctr[5] those of the tile
// GEMMs (one pair of the three is 0), ctr[1] and ctr[2] the blocks that gate/up
// and down work with (the workspace view's counters; nrb and ncb an item).
constexpr int kPlanBatch = 16;
__global__ void __launch_bounds__(1024)
k_mid_plan(const int *__restrict__ sel, const float *__restrict__ wts, const float *__restrict__ gam, int T, int K,
           int E, int has_sh, int mt, int2 *__restrict__ pairs, int4 *__restrict__ items, int max_items,
           int nrb, int ncb, MidTiles tp, int *__restrict__ ctr) {
    __shared__ int cnt[1024], sa[1024], sb[1024];
    constexpr int BM = kPfTileRows;
    const int g = threadIdx.x, S = K + has_sh, TK = T * K;
    cnt[g] = 0;
    __syncthreads();
    int v[kPlanBatch];
    for (int p0 = g; p0 < TK; p0 += 1024 * kPlanBatch) {
#pragma unroll
        for (int i = 0; i < kPlanBatch; i++) v[i] = p0 + i * 1024 < TK ? sel[p0 + i * 1024] : -1;
#pragma unroll
        for (int i = 0; i < kPlanBatch; i++)
            if (v[i] >= 0) atomicAdd(&cnt[v[i]], 1);
    }
    __syncthreads();
    const int c = g < E ? cnt[g] : 0;
    const int mi = (c + mt - 1) / mt;
    constexpr int kGroup = 1 << 20;                            // (above every pair count)
    sa[g] = c | (c > 0 ? kGroup : 0);                          // pairs, and groups
    sb[g] = mi | ((c + BM - 1) / BM) << 16;                    // items, and 128-row tiles
    __syncthreads();
    for (int st = 1; st < E; st <<= 1) {                       // inclusive scans (packed: neither half carries)
        const int a = g >= st && g < E ? sa[g - st] : 0, b = g >= st && g < E ? sb[g - st] : 0;
        __syncthreads();
        sa[g] += a;
        sb[g] += b;
        __syncthreads();
    }
    const int off = (sa[g] & (kGroup - 1)) - c, shi = has_sh ? (T + mt - 1) / mt : 0;
    cnt[g] = off;                                              // the group's next free pair
    const int n16 = (sb[E - 1] & 0xFFFF) + shi, mtr = sb[E - 1] >> 16, mtot = mtr + (has_sh ? (T + BM - 1) / BM : 0);
    const int ngrp = sa[E - 1] / kGroup + has_sh, gcost = ngrp * tp.cost.group + (n16 - ngrp) * tp.cost.item;
    const bool tiles = mtot <= tp.max_mt && mtot * tp.cost.tile + tp.cost.base < gcost;   // (block-uniform)
    if (tiles) {
        // the work lists of k_pf_gemm, as k_pf_plan stores them: one thread per m-tile
        const int cgu = (mtot + 7) >> 3;
        for (int m = g; m < mtot; m += 1024) {
            int grp = E, row0 = (m - mtr) * BM, rows = min(BM, T - row0), pb = TK + row0;
            if (m < mtr) {
                int lo = 0, hi = E - 1;                        // first group whose tiles end past m
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if ((sb[mid] >> 16) > m) hi = mid; else lo = mid + 1;
                }
                const int end = sa[lo] & (kGroup - 1), cl = end - (lo ? sa[lo - 1] & (kGroup - 1) : 0);
                grp = lo;
                row0 = (m - (lo ? sb[lo - 1] >> 16 : 0)) * BM;
                rows = min(BM, cl - row0);
                pb = end - cl + row0;
            }
            const int xg = m / cgu, mlg = m - xg * cgu;
            for (int n = 0; n < tp.nt_gu; n++) items[((mlg * tp.nt_gu + n) << 3) | xg] = make_int4(grp, pb, rows, n);
            for (int n = 0; n < tp.nt_dn; n++)
                tp.items_dn[(((m >> 3) * tp.nt_dn + n) << 3) | (m & 7)] = make_int4(grp, pb, rows, n);
        }
    }
    auto item = [&](int i, int grp, int first, int rows) __attribute__((always_inline)) {
        if (i < max_items) items[i] = make_int4(grp, first, rows, 0);   // (the host's bound lies below max_items)
    };
    if (!tiles) {
        if (g < E)
            for (int i = 0; i < mi; i++) item(shi + (sb[g] & 0xFFFF) - mi + i, g, off + i * mt, min(mt, c - i * mt));
        for (int i = g; i < shi; i += 1024) item(i, E, TK + i * mt, min(mt, T - i * mt));
    }
    if (g == 0) {
        const int n = tiles ? 0 : min(n16, max_items);
        ctr[1] = tiles ? mtot * tp.nt_gu : n * nrb;
        ctr[2] = tiles ? mtot * tp.nt_dn : n * ncb;
        ctr[3] = n;
        ctr[4] = tiles ? mtot * tp.nt_gu : 0;
        ctr[5] = tiles ? mtot * tp.nt_dn : 0;
    }
    __syncthreads();
    const bool one = TK <= 1024 * kPlanBatch;                  // v still holds every id
    for (int p0 = g; p0 < TK; p0 += 1024 * kPlanBatch) {
        float w[kPlanBatch];
#pragma unroll
        for (int i = 0; i < kPlanBatch; i++) {
            const int p = p0 + i * 1024;
            w[i] = p < TK ? wts[p] : 0.0f;
            if (!one) v[i] = p < TK ? sel[p] : -1;
        }
#pragma unroll
        for (int i = 0; i < kPlanBatch; i++)
            if (v[i] >= 0) {
                const int p = p0 + i * 1024, t = p / K;
                pairs[atomicAdd(&cnt[v[i]], 1)] = make_int2(t * S + p - t * K, __float_as_int(w[i]));
            }
    }
    if (has_sh)
        for (int t = g; t < T; t += 1024) pairs[TK + t] = make_int2(t * S + K, __float_as_int(gam ? gam[t] : 1.0f));
}

// Block b's unit of work of n: the blocks go to the 8 XCDs round-robin (b & 7),
// and each XCD takes a contiguous range of units, so that the items of one
// expert, which read the same weights, share an L2 (2560/640, 1021 rows, where
// ten row blocks an item had spread them: figures at the launcher). -1: none.
__device__ __forceinline__ int xcd_unit(int b, int n) {
    const int c = (n + 7) >> 3, u = (b & 7) * c + (b >> 3);
    return (b >> 3) < c && u < n ? u : -1;
}

// ---- gate/up ------------------------------------------------------------------------
constexpr int mid_kc(int nt) { return nt == 1 ? 256 : 128; }   // k values per chunk
template <int NT>
struct MidGuLds {
    uint8_t x[2][16 * NT * mid_kc(NT) * 2];       // the item's x rows, two chunks
    uint8_t w[4][32 * mid_kc(NT)];                // per wave: 16 gate and 16 up rows of one chunk (NVFP4: codes, then scales)
    float mx[4][16 * NT];
};
// One item, 64 intermediate rows: wave w rows o0 = 64 rb + 16 w .. + 15 of gate
// and up. ag / au: D[row 4 g + i][token l16] per token tile.
template <int H, int I, bool F4, int NT, bool ONCE>
__device__ __forceinline__ void mid_gu_body(const uint8_t *__restrict__ wg, const uint8_t *__restrict__ wu,
                                            const uint8_t *__restrict__ bg, const uint8_t *__restrict__ bu,
                                            const uint16_t *__restrict__ x16, const int2 *__restrict__ pairs, int S, int rows,
                                            MidGuLds<NT> &L, f32x4_t (&ag)[NT], f32x4_t (&au)[NT]) {
    constexpr int KC = mid_kc(NT), NCH = H / KC, MT = 16 * NT;
    constexpr int ROWB = F4 ? H / 2 : H, CB = F4 ? KC / 2 : KC;        // bytes per row, per row and chunk
    constexpr int CPR = CB / 16, RPI = 64 / CPR, NI = 16 / RPI;         // 16-byte chunks per row, rows per load, loads per tile
    constexpr int D = 2;                                                // chunks in flight
    static_assert(NCH % D == 0, "whole rounds of chunks");
    constexpr int XS = KC * 2, XC = XS / 16, XR = 256 / XC, NX = MT / XR; // x row bytes and chunks in LDS, rows and loads per thread
    constexpr int SB = KC / 16;                                         // NVFP4 scale bytes per row and chunk
    typedef uint32_t scv_t __attribute__((ext_vector_type(SB / 4)));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const int lr = lane / CPR, lc = lane % CPR;
    const uint8_t *gp = wg + (size_t)lr * ROWB + lc * 16, *up = wu + (size_t)lr * ROWB + lc * 16;
    // NVFP4 block scales: SB bytes a row and chunk; lanes 0..15 gate rows, 16..31 up rows
    const uint8_t *sp = F4 ? (g == 0 ? bg : bu) + (size_t)l16 * (H / 16) : nullptr;
    u32x4_t buf[D][2 * NI], xr[NX];
    scv_t sc[F4 ? D : 1];
    auto wload = [&](int c, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NI; j++) {
            buf[b][j] = ld_w<ONCE>(gp + (size_t)j * RPI * ROWB + c * CB);
            buf[b][NI + j] = ld_w<ONCE>(up + (size_t)j * RPI * ROWB + c * CB);
        }
        if constexpr (F4)
            if (lane < 32) sc[b] = *reinterpret_cast<const scv_t *>(sp + c * SB);
    };
    const uint16_t *xp[NX];
#pragma unroll
    for (int j = 0; j < NX; j++) {
        const int t = tid / XC + XR * j;
        xp[j] = x16 + (size_t)(t < rows ? pairs[t].x / S : 0) * H + (tid % XC) * 8;
    }
    auto xload = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NX; j++)
            if (tid / XC + XR * j < rows) xr[j] = *reinterpret_cast<const u32x4_t *>(xp[j] + c * KC);
    };
    wload(0, 0);
    xload(0);
    wload(1, 1);
#pragma unroll
    for (int n = 0; n < NT; n++) { ag[n] = f32x4_t{0.f, 0.f, 0.f, 0.f}; au[n] = ag[n]; }
    uint8_t *lw = L.w[wave];
    auto step = [&](int c, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NI; j++) {
            *reinterpret_cast<u32x4_t *>(lw + lds_at<CB>(j * RPI + lr, lc)) = buf[b][j];
            *reinterpret_cast<u32x4_t *>(lw + 16 * CB + lds_at<CB>(j * RPI + lr, lc)) = buf[b][NI + j];
        }
        bool hw = true;                           // every block scale of the chunk below 0x7F
        if constexpr (F4) {
            if (lane < 32) *reinterpret_cast<scv_t *>(lw + 32 * CB + lane * SB) = sc[b];
            hw = __builtin_amdgcn_ballot_w64(lane < 32 && !f4_scales_hw(sc[b])) == 0;
        }
        uint8_t *lx = L.x[b];
#pragma unroll
        for (int j = 0; j < NX; j++)
            if (tid / XC + XR * j < rows) *reinterpret_cast<u32x4_t *>(lx + lds_at<XS>(tid / XC + XR * j, tid % XC)) = xr[j];
        if (c + D < NCH) wload(c + D, b);
        if (c + 1 < NCH) xload(c + 1);
        __syncthreads();                          // (this buffer's readers of two chunks ago passed the last barrier)
        auto xfrag = [&](int n, int ch) __attribute__((always_inline)) {
            return *reinterpret_cast<const f16x8_t *>(lx + lds_at<XS>(n * 16 + l16, ch));
        };
        if constexpr (!F4) {
#pragma unroll
            for (int q = 0; q < KC / 64; q++) {
                f16x8_t g0, g1, u0, u1;
                i8_to_f16(*reinterpret_cast<const u32x4_t *>(lw + lds_at<CB>(l16, 4 * q + g)), g0, g1);
                i8_to_f16(*reinterpret_cast<const u32x4_t *>(lw + 16 * CB + lds_at<CB>(l16, 4 * q + g)), u0, u1);
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    if (NT > 1 && n * 16 >= rows) continue;
                    const f16x8_t x0 = xfrag(n, 8 * q + 2 * g), x1 = xfrag(n, 8 * q + 2 * g + 1);
                    ag[n] = mfma_f16(g0, x0, ag[n]);
                    au[n] = mfma_f16(u0, x0, au[n]);
                    ag[n] = mfma_f16(g1, x1, ag[n]);
                    au[n] = mfma_f16(u1, x1, au[n]);
                }
            }
        } else {
            auto codes = [&](int m, int q) __attribute__((always_inline)) {
                return *reinterpret_cast<const u32x4_t *>(lw + m * 16 * CB + lds_at<CB>(l16, 4 * q + g));
            };
            auto scales = [&](int m, int q) __attribute__((always_inline)) {
                return (uint32_t)*reinterpret_cast<const uint16_t *>(lw + 32 * CB + (m * 16 + l16) * SB + 8 * q + 2 * g);
            };
            if (hw) {
#pragma unroll
                for (int q = 0; q < KC / 128; q++) {
                    const u32x4_t cg = codes(0, q), cu = codes(1, q);
                    const f32x2_t fg = __builtin_amdgcn_cvt_pk_f32_fp8(scales(0, q), false);
                    const f32x2_t fu = __builtin_amdgcn_cvt_pk_f32_fp8(scales(1, q), false);
                    const f16x2_t hg[2] = {{(_Float16)fg.x, (_Float16)fg.x}, {(_Float16)fg.y, (_Float16)fg.y}};
                    const f16x2_t hu[2] = {{(_Float16)fu.x, (_Float16)fu.x}, {(_Float16)fu.y, (_Float16)fu.y}};
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const f16x8_t a = f4_to_f16(cg[m], hg[m >> 1]), b2 = f4_to_f16(cu[m], hu[m >> 1]);
#pragma unroll
                        for (int n = 0; n < NT; n++) {
                            if (NT > 1 && n * 16 >= rows) continue;
                            const f16x8_t xf = xfrag(n, 16 * q + 4 * g + m);
                            ag[n] = mfma_f16(a, xf, ag[n]);
                            au[n] = mfma_f16(b2, xf, au[n]);
                        }
                    }
                }
            } else {                              // a block scale outside the fp16 range: bf16, as the prefill path
#pragma unroll 1
                for (int q = 0; q < KC / 128; q++) {
                    const u32x4_t cg = codes(0, q), cu = codes(1, q);
                    const uint32_t pg = scales(0, q), pu = scales(1, q);
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const bf16x8_t a = f4_to_bf16x8(cg[m], e4m3_scale(m < 2 ? pg & 0xFFu : pg >> 8));
                        const bf16x8_t b2 = f4_to_bf16x8(cu[m], e4m3_scale(m < 2 ? pu & 0xFFu : pu >> 8));
#pragma unroll
                        for (int n = 0; n < NT; n++) {
                            if (NT > 1 && n * 16 >= rows) continue;
                            const bf16x8_t xf = f16_to_bf16x8(xfrag(n, 16 * q + 4 * g + m));
                            ag[n] = mfma_bf16(a, xf, ag[n]);
                            au[n] = mfma_bf16(b2, xf, au[n]);
                        }
                        asm volatile("" ::: "memory");
                    }
                }
            }
        }
        wave_lds_fence();                         // this wave's weight rows are read before they are overwritten
    };
#pragma unroll 1
    for (int c = 0; c < NCH; c += D) {
        step(c, 0);
        step(c + 1, 1);
    }
}

template <int H, int I, bool F4, int NT, bool ONCE>
__global__ void __launch_bounds__(256)
k_mid_gateup(const int4 *__restrict__ items, const int *__restrict__ n_items, const int2 *__restrict__ pairs, int S,
             const uint16_t *__restrict__ x16, const float *__restrict__ x16isc, GroupW g0, GroupW g1, int E,
             uint16_t *__restrict__ hid, int8_t *__restrict__ hk) {
    constexpr int NRB = I / 64;
    __shared__ __align__(16) MidGuLds<NT> L;
    const int u = xcd_unit(blockIdx.x, n_items[0] * NRB);
    if (u < 0) return;
    const int item = u / NRB, rb = u - item * NRB;
    const int4 it = items[item];
    const int grp = it.x, pb = it.y, rows = it.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const int o0 = rb * 64 + wave * 16;
    f32x4_t ag[NT], au[NT];
    f32x4_t sg, su;
    if (F4 && grp < E) {
        const size_t row = (size_t)grp * I + o0;
        const float a = g0.s2[grp], b = g1.s2[grp];
        sg = f32x4_t{a, a, a, a};
        su = f32x4_t{b, b, b, b};
        mid_gu_body<H, I, true, NT, ONCE>(reinterpret_cast<const uint8_t *>(g0.w) + row * (H / 2),
                                    reinterpret_cast<const uint8_t *>(g1.w) + row * (H / 2), g0.sc4 + row * (H / 16),
                                    g1.sc4 + row * (H / 16), x16, pairs + pb, S, rows, L, ag, au);
    } else {
        const size_t row = grp < E ? (size_t)grp * I + o0 : (size_t)o0;
        sg = *reinterpret_cast<const f32x4_t *>((grp < E ? g0.s : g0.s_sh) + row + 4 * g);
        su = *reinterpret_cast<const f32x4_t *>((grp < E ? g1.s : g1.s_sh) + row + 4 * g);
        mid_gu_body<H, I, false, NT, ONCE>(reinterpret_cast<const uint8_t *>(grp < E ? g0.w : g0.w_sh) + row * H,
                                     reinterpret_cast<const uint8_t *>(grp < E ? g1.w : g1.w_sh) + row * H, nullptr,
                                     nullptr, x16, pairs + pb, S, rows, L, ag, au);
    }
    // hidden = silu(g) * u, then fp16 scaled by the power of two of the block's
    // 64 rows of each token
    float m[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const int t = n * 16 + l16;
        const float isc = t < rows ? x16isc[pairs[pb + t].x / S] : 0.0f;
        m[n] = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            ag[n][i] = silu(ag[n][i] * isc * sg[i]) * (au[n][i] * isc * su[i]);
            m[n] = fmaxf(m[n], fabsf(ag[n][i]));
        }
        m[n] = fmaxf(m[n], lane_xor<16>(m[n]));
        m[n] = fmaxf(m[n], lane_xor<32>(m[n]));
        if (g == 0) L.mx[wave][t] = m[n];
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const int t = n * 16 + l16;
        const int k = f16_exp(fmaxf(fmaxf(L.mx[0][t], L.mx[1][t]), fmaxf(L.mx[2][t], L.mx[3][t])));
        if (t < rows) {
            const f16x2_t a = {(_Float16)__builtin_ldexpf(ag[n][0], k), (_Float16)__builtin_ldexpf(ag[n][1], k)};
            const f16x2_t b = {(_Float16)__builtin_ldexpf(ag[n][2], k), (_Float16)__builtin_ldexpf(ag[n][3], k)};
            *reinterpret_cast<u32x2_t *>(hid + (size_t)(pb + t) * I + o0 + 4 * g) =
                u32x2_t{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
            if (wave == 0 && g == 0) hk[(size_t)(pb + t) * NRB + rb] = (int8_t)k;
        }
    }
}

// ---- down ---------------------------------------------------------------------------
// The item's hidden rows (contiguous fp16 rows, exponents hk) into LDS.
template <int I, int NT>
struct MidHidStage {
    static constexpr int NTH = 64 * mid_dn_waves(I, NT), HS = I * 2, HC = HS / 16, NG = I / 64, NX = 16 * NT * HC / NTH;
    static_assert(NX * NTH == 16 * NT * HC, "whole loads per thread");
    const uint16_t *hid;
    const int8_t *hk;
    int rows;
    u32x4_t hr[NX];
    __device__ __forceinline__ void load() {
#pragma unroll
        for (int j = 0; j < NX; j++) {
            const int c = j * NTH + (int)threadIdx.x;
            if (c < rows * HC) hr[j] = reinterpret_cast<const u32x4_t *>(hid)[c];
        }
    }
    __device__ __forceinline__ void store(MidDnLds<I, NT> &L) {
        for (int i = threadIdx.x; i < rows * NG; i += NTH) L.isc[i / NG][i % NG] = exp2i(-(int)hk[i]);
#pragma unroll
        for (int j = 0; j < NX; j++) {
            const int c = j * NTH + (int)threadIdx.x;
            if (c < rows * HC) *reinterpret_cast<u32x4_t *>(L.h + lds_at<HS>(c / HC, c % HC)) = hr[j];
        }
    }
};

template <int H, int I, bool F4, int NT, bool ONCE>
__global__ void __launch_bounds__(64 * mid_dn_waves(I, NT))
k_mid_down(const int4 *__restrict__ items, const int *__restrict__ n_items, const int2 *__restrict__ pairs,
           const uint16_t *__restrict__ hid, const int8_t *__restrict__ hk, GroupW gd,
           int E, uint16_t *__restrict__ part, int8_t *__restrict__ partk) {
    constexpr int CW = 64 * mid_dn_waves(I, NT), NCB = H / CW;    // columns per block, blocks per item
    static_assert(NCB * CW == H, "whole blocks of columns");
    __shared__ __align__(16) MidDnLds<I, NT> L;
    const int u = xcd_unit(blockIdx.x, n_items[0] * NCB);
    if (u < 0) return;
    const int item = u / NCB, cb = u - item * NCB;
    const int4 it = items[item];
    const int grp = it.x, pb = it.y, rows = it.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const int c0 = cb * CW + wave * 64;
    MidHidStage<I, NT> st{hid + (size_t)pb * I, hk + (size_t)pb * (I / 64), rows, {}};
    f32x4_t acc[4][NT], sd[4];
    if (F4 && grp < E) {
        const size_t row = (size_t)grp * H + c0;
        const float a = gd.s2[grp];
#pragma unroll
        for (int rt = 0; rt < 4; rt++) sd[rt] = f32x4_t{a, a, a, a};
        mid_dn_body<I, true, NT, ONCE>(reinterpret_cast<const uint8_t *>(gd.w) + row * (I / 2), gd.sc4 + row * (I / 16), rows,
                                 L, acc, st, tid);
    } else {
        const size_t row = grp < E ? (size_t)grp * H + c0 : (size_t)c0;
#pragma unroll
        for (int rt = 0; rt < 4; rt++)
            sd[rt] = *reinterpret_cast<const f32x4_t *>((grp < E ? gd.s : gd.s_sh) + row + rt * 16 + 4 * g);
        mid_dn_body<I, false, NT, ONCE>(reinterpret_cast<const uint8_t *>(grp < E ? gd.w : gd.w_sh) + row * I, nullptr, rows,
                                  L, acc, st, tid);
    }
    // the wave's 64 columns of each token as fp16 scaled by 2^k (k from the
    // largest finite magnitude; inf and NaN pass through), k to partk
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const int t = n * 16 + l16;
        const bool live = t < rows;
        const int2 pr = live ? pairs[pb + t] : make_int2(0, 0);
        const float w = __int_as_float(pr.y);
        const int slot = pr.x;
        float m = 0.0f;
#pragma unroll
        for (int rt = 0; rt < 4; rt++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float v = w * (acc[rt][n][i] * sd[rt][i]);
                acc[rt][n][i] = v;
                if ((__float_as_uint(v) & 0x7F800000u) != 0x7F800000u) m = fmaxf(m, fabsf(v));
            }
        m = fmaxf(m, lane_xor<16>(m));
        m = fmaxf(m, lane_xor<32>(m));
        const int k = f16_exp(m);
        if (live) {
            uint16_t *dst = part + (size_t)slot * H + c0 + 4 * g;
#pragma unroll
            for (int rt = 0; rt < 4; rt++) {
                const f16x2_t a = {(_Float16)__builtin_ldexpf(acc[rt][n][0], k), (_Float16)__builtin_ldexpf(acc[rt][n][1], k)};
                const f16x2_t b = {(_Float16)__builtin_ldexpf(acc[rt][n][2], k), (_Float16)__builtin_ldexpf(acc[rt][n][3], k)};
                *reinterpret_cast<u32x2_t *>(dst + rt * 16) =
                    u32x2_t{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
            }
            if (g == 0) partk[(size_t)slot * (H / 64) + (c0 >> 6)] = (int8_t)k;
        }
    }
}

// ---- launcher -----------------------------------------------------------------------
int launch_mid(const MidArgs &a, hipStream_t s) {
    const Cfg &c = g_cfg;
    const int T = a.T, E = c.E, K = c.K, H = c.H, I = c.I;
    const int nt = mid_token_tiles(T, E, K, I, a.f4), mt = 16 * nt, max_items = mid_items_bound(T, E, K, a.has_sh, nt);
    if (T <= kMidExactRows) {                                  // (beyond: the caller has launched router and selection)
        const int ng = (T + 7) / 8, nx = E / 8 + (a.g ? 1 : 0);
        const int tg = max(1, ng * nx / 1536);                     // token groups per router block: ~1536 blocks
        const unsigned g_r = (unsigned)((T + 3) / 4 + nx * ((ng + tg - 1) / tg));
        if (H == 2048)
            hipLaunchKernelGGL(k_mid_router<8>, dim3(g_r), dim3(256), 0, s, a.router, a.bias, a.g, a.x, T, E, tg, a.logits,
                               a.gam, a.x16, a.x16isc, a.xsum, a.x16sum, a.ctr);
        else
            hipLaunchKernelGGL(k_mid_router<10>, dim3(g_r), dim3(256), 0, s, a.router, a.bias, a.g, a.x, T, E, tg, a.logits,
                               a.gam, a.x16, a.x16isc, a.xsum, a.x16sum, a.ctr);
        hipLaunchKernelGGL(k_mid_topk<8>, dim3((T + 3) / 4), dim3(256), 0, s, a.logits, T, K, c.renorm, a.sel, a.wts, a.ctr);
    }
    // token tiles per item. With one (16 rows) LDS and registers leave three
    // blocks on a CU (down at 2560/640: two), and an expert's further items find
    // its weights in L2: gate/up + down, us, at 300 / 1021 / 1500 / 2000 rows with
    // one, two and four tiles: INT8 289 / 370 / 443 / 534, 321 / 373 / 466 / 589,
    // 343 / 380 / 425 / 462; NVFP4 198 / 345 / 422 / 500, 278 / 386 / 462 / 580, 436 /
    // 526 / 599 / 688. Two and four tiles also read their weights in chunks half as
    // long (mid_kc), and NVFP4's LDS is sized for the INT8 shared expert's rows: the
    // figures compare these forms, not wider items alone. Four are taken for INT8
    // from 24 rows an expert.
    const int dw = 64 * mid_dn_waves(I, nt);                      // columns, and threads, per down block
    hipLaunchKernelGGL(k_mid_plan, dim3(1), dim3(1024), 0, s, a.sel, a.wts, a.g ? a.gam : nullptr, T, K, E, a.has_sh, mt,
                       a.pairs, a.items, a.max_items, I / 64, H / dw, a.tiles, a.ctr);
    // (xcd_unit wants eight times the largest range: a multiple of 8)
    const dim3 g_gu((unsigned)((max_items * (I / 64) + 7) / 8 * 8)), g_dn((unsigned)((max_items * (H / dw) + 7) / 8 * 8)), b(256), bd((unsigned)dw);
#define QFM_MID(HH, II, F4, NT, ONCE)                                                                               \
    hipLaunchKernelGGL((k_mid_gateup<HH, II, F4, NT, ONCE>), g_gu, b, 0, s, a.items, a.ctr + 3, a.pairs,            \
                       K + a.has_sh, reinterpret_cast<const uint16_t *>(a.x16), a.x16isc, a.gg, a.gu, E, a.hid,     \
                       a.hk);                                                                                       \
    hipLaunchKernelGGL((k_mid_down<HH, II, F4, NT, ONCE>), g_dn, bd, 0, s, a.items, a.ctr + 3, a.pairs, a.hid,      \
                       a.hk, a.gd, E, a.part, a.partk)
#define QFM_MID_ONCE(HH, II, F4)                                                                                    \
    if (mid_reads_once(T, E, K, a.f4)) { QFM_MID(HH, II, F4, 1, true); } else { QFM_MID(HH, II, F4, 1, false); }
    if (shape_2048()) {
        if (a.f4) { QFM_MID_ONCE(2048, 512, true) } else if (nt == 1) { QFM_MID_ONCE(2048, 512, false) } else { QFM_MID(2048, 512, false, 4, false); }
    } else {
        if (a.f4) { QFM_MID_ONCE(2560, 640, true) } else { QFM_MID_ONCE(2560, 640, false) }
    }
#undef QFM_MID_ONCE
#undef QFM_MID
    return 0;
}

}  // namespace qfm
