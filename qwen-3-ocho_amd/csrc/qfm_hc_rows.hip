// qfm_hc_rows.hip -- the hyper-connection pre-mixer over five or more rows
// (contract in include/qf_dense.h; one row and a few rows: qfm_hc.hip).
//
// The two-launch form of a few rows recomputes each row's norm in 162 blocks and
// reads the weights anew from L2 for every row, so its work grows with every row.
// Here, three launches:
//   k_hc_norm  one row per block: the previous mixer's inject, the norm and
//              X8(normed);
//   k_hc_down  the down and inject rows as an int8 MFMA GEMM, 32 rows x 16
//              tokens per block, and X8(hc_d);
//   k_hc_up    the up rows likewise, 4 x 32 rows x 16 tokens per block, the
//              combine and X8(mixed).
// us per call, two launches -> three (H = 2048): T = 2 12.0 -> 18.5, 4 15.1 ->
// 18.8, 5 18.6 -> 18.9, 6 18.8 -> 19.0, 8 23.3 -> 19.1, 16 37.6 -> 19.9, 129
// 252 -> 26.6, 256 497 -> 31.3; H = 2560: T = 4 19.6 -> 21.2, 5 22.6 -> 21.3,
// 129 347 -> 30.1, 256 683 -> 36.6. These calls find the 6.7 or 10.5 MB of weights
// in the caches; over 24 layers, us per layer: H = 2048 T = 4 15.7 (two launches), 5
// 19.4 -> 19.1, 6 19.9 -> 19.1, 8 24.2 -> 19.2, H = 2560 T = 5 23.5 -> 21.8; a call whose
// weights and rows were never read, 129 rows at H = 2560: 376 -> 53. Hence
// kHcFewRows = 4.
#include "qfm_internal.h"
#include "qfm_x8.h"

namespace qfm {

// One row per 1024-thread block: the fused inject of the previous mixer (the
// updated residual stored by the thread that read it), the zero-centred RMS
// norm and X8(normed). Thread c * 256 + t owns elements i * 256 + t of stream
// c and sums them in order, then each wave and the four waves of a stream are
// reduced (the reference's partition and order; hc_slice_body uses the same).
template <int NV>
__global__ void __launch_bounds__(1024)
k_hc_norm(float *__restrict__ R, const uint16_t *__restrict__ wn, const float *__restrict__ y_prev,
          const float *__restrict__ inj_prev, float *__restrict__ normed, int8_t *__restrict__ q,
          float *__restrict__ sc) {
    constexpr int H = NV * 256, RS = 4 * H;
    __shared__ float red[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = tid >> 8, t256 = tid & 255;                  // stream, thread within the stream
    const size_t t = blockIdx.x;
    const size_t base = t * RS + (size_t)c * H;
    float v[NV], yv[NV];
    uint16_t wb[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) {
        v[i] = R[base + i * 256 + t256];
        wb[i] = wn[(size_t)c * H + i * 256 + t256];
    }
    const float sj = y_prev ? inj_prev[t * QF8_HCC + c] : 0.0f;
    if (y_prev) {                                              // uniform
#pragma unroll
        for (int i = 0; i < NV; i++) yv[i] = y_prev[t * H + i * 256 + t256];
#pragma unroll
        for (int i = 0; i < NV; i++) {
            v[i] = fmaf(sj, yv[i], v[i]);
            R[base + i * 256 + t256] = v[i];
        }
    }
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; i++) acc = fmaf(v[i], v[i], acc);
    acc = group_sum<64>(acc);
    if (lane == 0) red[wave] = acc;
    __syncthreads();
    const float rstd = rsqrtf((red[4 * c] + red[4 * c + 1] + red[4 * c + 2] + red[4 * c + 3]) / (float)H + 1e-6f);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int e = c * H + i * 256 + t256;                  // 32 consecutive e per half-wave
        const float nv = v[i] * rstd * (1.0f + bf16_to_f32(wb[i]));
        float s1;
        const int qi = x8_code(nv, s1);
        normed[t * RS + e] = nv;
        q[t * RS + e] = (int8_t)qi;
        if ((tid & 31) == 0) sc[(t * RS + e) >> 5] = s1;
    }
}

// X8 GEMM step on MFMA: D = W (16 rows x 32) . X (32 x 16 tokens) of one X8
// block, exact in int32, scaled by the token's block scale into fp32. Lane l
// holds 8 codes (k = 8 (l >> 4) ..) of weight row l & 15 and of token l & 15;
// D: token l & 15, rows 4 (l >> 4) + i.
typedef float f32x4_t __attribute__((ext_vector_type(4)));
// (the caller's X8 and hcy buffers need no more than their element's alignment)
typedef i32x4 i32x4_u __attribute__((aligned(1)));
typedef f32x4_t f32x4_u __attribute__((aligned(4)));
__device__ __forceinline__ void x8_mfma(long w, long x, float xs, f32x4_t &acc) {
    const i32x4 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(w, x, i32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = fmaf((float)d[i], xs, acc[i]);
}
// LDS written by this wave's other lanes is read next (or read and then
// overwritten): order the accesses, no barrier (LDS serves one wave in order)
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Down / inject GEMM over 16 tokens and 32 rows per block (the 320 down rows
// in ten blocks, the 4 inject rows in one more): 8 waves each take an eighth
// of K = 4H, their partial sums are added in wave order through LDS; X8(hc_d)
// of the block's 32 rows follows in place.
// Bound by the block's 48 code rows (16 tokens, 32 weight rows; 393 KB at H =
// 2048) crossing from L2 to one CU. They are read 16 bytes a lane along the
// rows (4 rows x 256 bytes an instruction, three segments in flight) and turned
// into MFMA fragments through wave-private LDS: fragments loaded straight from
// memory (8 bytes a lane of 16 rows) took ~64 cycles an instruction.
template <int H>
__global__ void __launch_bounds__(512)
k_hc_down(const int8_t *__restrict__ q, const float *__restrict__ sc, const int8_t *__restrict__ Wd,
          const float *__restrict__ Sd, const int8_t *__restrict__ Wi, const float *__restrict__ Si, int T,
          float *__restrict__ hc_d, float *__restrict__ inj, int8_t *__restrict__ d8q, float *__restrict__ d8s) {
    constexpr int L = QF8_HCL, RS = 4 * H, KW = RS / 8, SEG = 256, NSEG = KW / SEG, NBS = SEG / 32, NST = 3;
    static_assert(NSEG * SEG == KW && NSEG >= NST && L % 32 == 0, "whole segments per wave, whole blocks of rows");
    __shared__ __align__(16) int8_t s_t[8][3 * 16 * SEG];      // [wave][W rows 0-15, 16-31, tokens][row][256], swizzled
    __shared__ float s_p[8][32][17];                           // [wave][row][token]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const int r0 = blockIdx.x * 32, t0 = blockIdx.y * 16;
    const bool is_inj = r0 >= L;
    const int8_t *W = is_inj ? Wi : Wd + (size_t)r0 * RS;
    const int rmax = is_inj ? QF8_HCC - 1 : 31;                // rows / tokens past the end repeat the last one, dropped below
    // loads: instruction j of a tile covers rows 4 j + g, chunk l16 of the segment
    const int8_t *src[12];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        src[j] = W + (size_t)min(4 * j + g, rmax) * RS;
        src[4 + j] = W + (size_t)min(16 + 4 * j + g, rmax) * RS;
        src[8 + j] = q + (size_t)min(t0 + 4 * j + g, T - 1) * RS;
    }
    const int k0 = wave * KW;
    const float *sp = sc + (size_t)min(t0 + l16, T - 1) * (RS / 32) + (k0 >> 5);
    i32x4 buf[NST][12];
    f32x4_t xs[NST][2];
    auto load = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 12; j++)
            buf[s % NST][j] = *reinterpret_cast<const i32x4_u *>(src[j] + k0 + s * SEG + l16 * 16);
#pragma unroll
        for (int h = 0; h < 2; h++) xs[s % NST][h] = *reinterpret_cast<const f32x4_u *>(sp + s * NBS + 4 * h);
    };
#pragma unroll
    for (int s = 0; s < NST; s++) load(s);
    f32x4_t a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
    int8_t *lds = s_t[wave];
#pragma unroll
    for (int s = 0; s < NSEG; s++) {
        // chunk c of row r at position c ^ r: the writes and the fragment reads are free of bank conflicts
#pragma unroll
        for (int j = 0; j < 12; j++) {
            const int r = 4 * (j & 3) + g;
            *reinterpret_cast<i32x4 *>(lds + ((j >> 2) * 16 + r) * SEG + ((l16 ^ r) << 4)) = buf[s % NST][j];
        }
        const f32x4_t x0 = xs[s % NST][0], x1 = xs[s % NST][1];
        wave_lds_fence();
        if (s + NST < NSEG) load(s + NST);
#pragma unroll
        for (int b = 0; b < NBS; b++) {
            const int8_t *f = lds + l16 * SEG + (((2 * b + (g >> 1)) ^ l16) << 4) + (g & 1) * 8;
            const long x = *reinterpret_cast<const long *>(f + 2 * 16 * SEG);
            const float xv = b < 4 ? x0[b & 3] : x1[b & 3];
            x8_mfma(*reinterpret_cast<const long *>(f), x, xv, a0);
            x8_mfma(*reinterpret_cast<const long *>(f + 16 * SEG), x, xv, a1);
        }
        wave_lds_fence();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        s_p[wave][4 * g + i][l16] = a0[i];
        s_p[wave][16 + 4 * g + i][l16] = a1[i];
    }
    __syncthreads();
    {                                                          // one (token, row) per thread, a token's 32 rows per half-wave
        const int r = tid & 31, tt = tid >> 5, t = t0 + tt;
        float sum = s_p[0][r][tt];
#pragma unroll
        for (int w = 1; w < 8; w++) sum += s_p[w][r][tt];
        if (is_inj) {
            if (r < QF8_HCC && t < T) inj[(size_t)t * QF8_HCC + r] = gemv_act(sum * Si[r], 2);
        } else {
            const float hv = gemv_act(sum * Sd[r0 + r], 1);
            float s1;
            const int qi = x8_code(hv, s1);
            if (t < T) {
                hc_d[(size_t)t * L + r0 + r] = hv;
                d8q[(size_t)t * L + r0 + r] = (int8_t)qi;
                if (r == 0) d8s[(size_t)t * (L / 32) + blockIdx.x] = s1;
            }
        }
    }
}

// Up GEMM and combine, 16 tokens and 32 outputs j per block (the mix is
// X8-quantized in blocks of 32 values): 8 waves, wave w the 16 up rows
// (w >> 1) * H + j0 + 16 (w & 1) over the 320 codes, then one output per
// thread: the sigmoid-weighted mean over the 4 streams, bf16 and X8 of it.
// The wave's rows and the block's tokens are contiguous: read 16 bytes a lane
// and turned into fragments through LDS, as in k_hc_down. LDS rows of 352
// bytes (24 banks apart modulo 64): two of the 16 rows of a fragment read
// share a bank, as 512 bytes over 64 banks must.
template <int H>
__global__ void __launch_bounds__(512)
k_hc_up(const int8_t *__restrict__ Wu, const float *__restrict__ Su, const int8_t *__restrict__ d8q,
        const float *__restrict__ d8s, const float *__restrict__ normed, int T, float *__restrict__ hcy,
        float *__restrict__ mixed, int8_t *__restrict__ xq_out, float *__restrict__ xs_out,
        uint16_t *__restrict__ xb_out) {
    constexpr int L = QF8_HCL, RS = 4 * H, NB = L / 32, CPR = L / 16, LR = 352, NL = 16 * CPR / 64;
    __shared__ __align__(16) int8_t s_w[8][16 * LR], s_x[16 * LR];
    __shared__ float s_s[16][NB + 1];
    __shared__ float s_h[4][16][33];                           // [stream][token][j]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const int j0 = blockIdx.x * 32, t0 = blockIdx.y * 16;
    const int c = wave >> 1, jh = (wave & 1) * 16;
    const int8_t *wp = Wu + ((size_t)c * H + j0 + jh) * L;
    i32x4 w[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) w[i] = *reinterpret_cast<const i32x4 *>(wp + (i * 64 + lane) * 16);
    if (tid < 16 * CPR) {                                      // tokens past the end repeat the last one, dropped below
        const int r = tid / CPR, ch = tid - r * CPR;
        *reinterpret_cast<i32x4 *>(s_x + r * LR + ch * 16) =
            *reinterpret_cast<const i32x4_u *>(d8q + (size_t)min(t0 + r, T - 1) * L + ch * 16);
    } else if (tid - 16 * CPR < 16 * NB) {
        const int i = tid - 16 * CPR, r = i / NB;
        s_s[r][i - r * NB] = d8s[(size_t)min(t0 + r, T - 1) * NB + i - r * NB];
    }
    // this thread's output and its normed values (the loads overlap the GEMM)
    const int jj = tid & 31, tt = tid >> 5, t = t0 + tt;
    const size_t tc = (size_t)min(t, T - 1);
    float nrm[4];
#pragma unroll
    for (int cc = 0; cc < 4; cc++) nrm[cc] = normed[tc * RS + (size_t)cc * H + j0 + jj];
    const f32x4_t su = *reinterpret_cast<const f32x4_u *>(Su + (size_t)c * H + j0 + jh + 4 * g);
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int k = i * 64 + lane, r = k / CPR;
        *reinterpret_cast<i32x4 *>(s_w[wave] + r * LR + (k - r * CPR) * 16) = w[i];
    }
    static_assert(16 * CPR + 16 * NB <= 512, "one load per thread stages the tokens' codes and scales");
    __syncthreads();
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NB; b++)
        x8_mfma(*reinterpret_cast<const long *>(s_w[wave] + l16 * LR + b * 32 + g * 8),
                *reinterpret_cast<const long *>(s_x + l16 * LR + b * 32 + g * 8), s_s[l16][b], acc);
    const f32x4_t hv = acc * su;
    if (t0 + l16 < T) *reinterpret_cast<f32x4_u *>(hcy + (size_t)(t0 + l16) * RS + (size_t)c * H + j0 + jh + 4 * g) = hv;
    float *sh = &s_h[c][l16][jh + 4 * g];
#pragma unroll
    for (int i = 0; i < 4; i++) sh[i] = hv[i];
    __syncthreads();
    float sum = 0.0f;
#pragma unroll
    for (int cc = 0; cc < 4; cc++) {
        const float m = 1.0f / (1.0f + expf(-s_h[cc][tt][jj]));
        sum = fmaf(m, nrm[cc], sum);
    }
    const float v = sum * 0.25f;
    float s1;
    const int qi = x8_code(v, s1);
    if (t < T) {
        mixed[(size_t)t * H + j0 + jj] = v;
        if (xb_out) xb_out[(size_t)t * H + j0 + jj] = f32_to_bf16(v);   // the fused MoE forward's input row
        xq_out[(size_t)t * H + j0 + jj] = (int8_t)qi;
        if (jj == 0) xs_out[(size_t)t * (H / 32) + blockIdx.x] = s1;
    }
}

void launch_hc_rows(const HcRowsArgs &a, hipStream_t s) {
    const unsigned tt = (unsigned)((a.T + 15) / 16);           // token tiles
    const Qf8I8Mat *in = a.inject;
#define QFM_HC_ROWS(NV)                                                                                             \
    hipLaunchKernelGGL(k_hc_norm<NV>, dim3((unsigned)a.T), dim3(1024), 0, s, a.R, a.wn, a.y_prev, a.inj_prev,       \
                       a.normed, a.n8q, a.n8s);                                                                     \
    hipLaunchKernelGGL(k_hc_down<NV * 256>, dim3(QF8_HCL / 32 + (in ? 1 : 0), tt), dim3(512), 0, s, a.n8q, a.n8s,   \
                       a.down->w, a.down->s, in ? in->w : nullptr, in ? in->s : nullptr, a.T, a.hc_d, a.inj,        \
                       a.d8q, a.d8s);                                                                               \
    hipLaunchKernelGGL(k_hc_up<NV * 256>, dim3(NV * 8, tt), dim3(512), 0, s, a.up->w, a.up->s, a.d8q, a.d8s,        \
                       a.normed, a.T, a.hcy, a.mixed, a.xq_out, a.xs_out, a.xb_out)
    if (g_cfg.H == 2048) { QFM_HC_ROWS(8); } else { QFM_HC_ROWS(10); }
#undef QFM_HC_ROWS
}

}  // namespace qfm
