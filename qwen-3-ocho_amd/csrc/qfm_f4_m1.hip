// qfm_f4_m1.hip -- NVFP4 routed experts + INT8 shared expert for one row (M = 1
// decode), after the router launch.
//
// Reference behaviour: k_nvfp4_gateup_all / k_nvfp4_downacc_all
// (ocho/amd_server/qf_nvfp4_wave64.hip:376-454) and the int8 shared expert
// (ocho/amd_server/qf8_dense_i8.hip:346-358).
//
// The three launches of the INT8 row (qfm_i8_m1.hip): a router launch without a
// selection tail, gate/up whose waves run the top-K themselves, and down with
// one writer per output. The fork-row kernels (qfm_csr.hip), which served this
// row before, rank it in the router launch's tail and pass partials as tagged
// words: two cross-XCD hand-offs, which one row need not pay. Bound by the three
// dependent launches and the selection (~1.3 us), then the weight streams.
// us per layer (8 layers, one graph over and over; with other inputs between the
// passes 2560/640 21.6 -> 19.1), the fork-row kernels -> these: 2048/512 17.3 ->
// 14.3, 2560/640 21.5 -> 18.7 (per launch: router 6.3 -> 3.9, gate/up 8.3 -> 9.5
// with the selection and the shared expert in it, down 7.2 -> 7.2; 2048/512 down
// 4.7).
#include "qfm_dev.h"
#include "qfm_internal.h"

namespace qfm {

// gate/up: grid (I / RPB, K + shared), LPR lanes per row (a row of H / 2 bytes
// is H / 32 16-byte chunks). Job K is the shared expert (INT8 rows, a half-wave
// each; it needs no selection). Block (0, 0) publishes sel / wts and advances
// ctl[0], the workspace's count of one-row-or-more calls. (A half-wave per row at
// H = 2560 too, its third step half empty: 10.6 us against 9.5, twice the waves
// that select.)
template <int H, int I>
__global__ void __launch_bounds__(256)
k_f4_gateup_m1(const uint8_t *__restrict__ Wg, const uint8_t *__restrict__ Wu, const uint8_t *__restrict__ Bg,
               const uint8_t *__restrict__ Bu, const float *__restrict__ s2g, const float *__restrict__ s2u,
               const uint16_t *__restrict__ x, const float *__restrict__ logits, int *__restrict__ sel,
               float *__restrict__ wts, int K, int renorm, float *__restrict__ hidden, ShPtrs sh,
               uint32_t *__restrict__ ctl) {
    constexpr int CPR = H / 32, LPR = lpr_of(CPR), NST = CPR / LPR, RPB = 256 / LPR, EPL = 8;
    __shared__ __align__(16) unsigned long long s_tk[4][kTopkLds];
    const int job = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (job == K) {                               // shared expert: RPB INT8 rows, 8 at a time
        const int l = threadIdx.x & 31;
        float xs[H / 512][16], xsum = 0.0f;
        load_x_slice_bf16<H>(x, l, xs);
#pragma unroll
        for (int st = 0; st < H / 512; st++)
#pragma unroll
            for (int i = 0; i < 16; i++) xsum += xs[st][i];
#pragma unroll
        for (int q = 0; q < RPB / 8; q++) {
            const int row = blockIdx.x * RPB + q * 8 + (threadIdx.x >> 5);
            uint4 wg[H / 512], wu[H / 512];
#pragma unroll
            for (int st = 0; st < H / 512; st++) {
                wg[st] = ld_nt16(sh.qg + (size_t)row * H + st * 512 + l * 16);
                wu[st] = ld_nt16(sh.qu + (size_t)row * H + st * 512 + l * 16);
            }
            const float sg = sh.sg[row], su = sh.su[row];
            float ag = -128.0f * xsum, au = ag;
#pragma unroll
            for (int st = 0; st < H / 512; st++) {
                ag = dot16_u8(wg[st], xs[st], ag);
                au = dot16_u8(wu[st], xs[st], au);
            }
            ag = group_sum<32>(ag);
            au = group_sum<32>(au);
            if (l == 0) hidden[(size_t)K * I + row] = silu(ag * sg) * (au * su);
        }
        return;
    }
    int e;
    if (blockIdx.x == 0 && job == 0 && wave == 0) {
        int my_i;
        float my_w;
        wave_topk<EPL>(logits, K, renorm, lane, s_tk[0], my_i, my_w);
        if (lane < K) {
            sel[lane] = my_i;
            wts[lane] = my_w;
        }
        if (lane == 0) ctl[0] = next_tag(ctl[0]);
        e = __builtin_amdgcn_readfirstlane(my_i);
    } else {
        e = wave_topk_one<EPL>(logits, K, job, lane, s_tk[wave]);
    }
    const int l = threadIdx.x % LPR, row = blockIdx.x * RPB + threadIdx.x / LPR;
    // the x slice after the selection and before the weights (waiting for it never waits for them)
    uint32_t xw[NST][16];
#pragma unroll
    for (int st = 0; st < NST; st++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint4 a = reinterpret_cast<const uint4 *>(x)[(st * LPR + l) * 4 + q];
            xw[st][4 * q] = a.x; xw[st][4 * q + 1] = a.y; xw[st][4 * q + 2] = a.z; xw[st][4 * q + 3] = a.w;
        }
    const size_t roff = ((size_t)e * I + row) * (H / 2), boff = ((size_t)e * I + row) * (H / 16);
    uint4 wg[NST], wu[NST];
    uint32_t bg[NST], bu[NST];
#pragma unroll
    for (int st = 0; st < NST; st++) {
        wg[st] = ld_nt16(Wg + roff + (st * LPR + l) * 16);
        wu[st] = ld_nt16(Wu + roff + (st * LPR + l) * 16);
        bg[st] = *reinterpret_cast<const uint16_t *>(Bg + boff + (st * LPR + l) * 2);
        bu[st] = *reinterpret_cast<const uint16_t *>(Bu + boff + (st * LPR + l) * 2);
    }
    const float fg = s2g[e], fu = s2u[e];
    float ag = 0.0f, au = 0.0f;
#pragma unroll
    for (int st = 0; st < NST; st++) {
        ag += f4_chunk_bx(wg[st], bg[st], xw[st]);
        au += f4_chunk_bx(wu[st], bu[st], xw[st]);
    }
    ag = group_sum<LPR>(ag);
    au = group_sum<LPR>(au);
    if (l == 0) hidden[(size_t)job * I + row] = silu(ag * fg) * (au * fu);
}

// down: one output row per wave, eight per block. The K experts' I / 2-byte rows of one output
// are K I / 32 16-byte chunks, dealt to the 64 lanes in order (NS steps; a chunk's
// expert is its index / (I / 32)), the shared expert's I / 16 INT8 chunks as one
// more step: the sum over experts is linear, so every lane adds its chunks'
// dots times w_k s2 and the wave reduces once. Row groups of a power-of-two
// number of lanes would leave 40 blocks at I = 640 (20 chunks a row).
template <int H, int I, int NS>
__global__ void __launch_bounds__(512)
k_f4_down_m1(const uint8_t *__restrict__ Wd, const uint8_t *__restrict__ Bd, const float *__restrict__ s2d,
             const float *__restrict__ hidden, const float *__restrict__ wts, const int *__restrict__ sel, int K,
             ShPtrs sh, const float *__restrict__ gdot, float *__restrict__ y32, uint16_t *__restrict__ ybf) {
    constexpr int CPR = I / 32, CH = I / 16, RPW = 1, kMaxJobs = 17, NTH = 512;
    constexpr int JOBS = NS * 64 / CPR + 1 < kMaxJobs ? NS * 64 / CPR + 1 : kMaxJobs;   // the most of this NS, the shared one with them
    static_assert(CH <= 64, "the shared row is one step");
    constexpr int CPT = (JOBS * CH + NTH - 1) / NTH;  // hidden chunks per thread
    __shared__ uint4 s_h16[JOBS * CH * 2];        // the hidden rows as scaled fp16 (chunk16_to_f16)
    __shared__ float2 s_hci[JOBS * CH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool has_sh = sh.qd != nullptr;
    const int nch = (K + (has_sh ? 1 : 0)) * CH;
    const int r0 = (blockIdx.x * (NTH / 64) + wave) * RPW;
    // routing first (the weights wait for it), then the hidden chunks, then the
    // weights: every load unconditional, its index clamped (a load under a lane
    // condition made the compiler wait for all before it: 7.5 us a launch)
    int job[NS], ex[NS];
    float wk[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        job[s] = min((s * 64 + lane) / CPR, K - 1);
        ex[s] = sel[job[s]];
        wk[s] = wts[job[s]];
    }
    float hv[CPT][16];
#pragma unroll
    for (int q = 0; q < CPT; q++) {
        const int ch = min(tid + q * NTH, nch - 1);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const float4 f = reinterpret_cast<const float4 *>(hidden)[ch * 4 + v];
            hv[q][4 * v] = f.x; hv[q][4 * v + 1] = f.y; hv[q][4 * v + 2] = f.z; hv[q][4 * v + 3] = f.w;
        }
    }
    uint4 w[RPW][NS], wsh[RPW];
    uint32_t b[RPW * NS];
    float s2[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int c = min(s * 64 + lane - job[s] * CPR, CPR - 1);   // (past the end: a repeat, its weight 0)
        s2[s] = s2d[ex[s]];
#pragma unroll
        for (int r = 0; r < RPW; r++) {
            const size_t row = (size_t)ex[s] * H + r0 + r;
            w[r][s] = ld_nt16(Wd + row * (I / 2) + c * 16);
            b[r * NS + s] = *reinterpret_cast<const uint16_t *>(Bd + row * (I / 16) + c * 2);
        }
    }
    // the shared expert's rows (without one: any readable bytes, weight 0)
    const int8_t *qd = has_sh ? sh.qd : reinterpret_cast<const int8_t *>(Wd);
#pragma unroll
    for (int r = 0; r < RPW; r++) wsh[r] = ld_nt16(qd + (size_t)(r0 + r) * I + min(lane, CH - 1) * 16);
    float sds[RPW] = {}, gd = 0.0f;
    if (has_sh) {                                 // (uniform)
#pragma unroll
        for (int r = 0; r < RPW; r++) sds[r] = sh.sd[r0 + r];
        if (gdot) gd = gdot[0];
    }
#pragma unroll
    for (int q = 0; q < CPT; q++) {
        const int ch = tid + q * NTH;
        if (ch < nch) {
            uint4 ha, hb;
            s_hci[ch] = chunk16_to_f16(hv[q], ha, hb);
            s_h16[2 * ch] = ha;
            s_h16[2 * ch + 1] = hb;
        }
    }
    __syncthreads();
    f32x2_t sc[RPW * NS];
    e4m3_pairs(b, sc);
    float acc[RPW];
#pragma unroll
    for (int r = 0; r < RPW; r++) acc[r] = 0.0f;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int i = s * 64 + lane;
        const bool live = i < K * CPR;
        const int hc = live ? 2 * i : 0;          // its first 16-value hidden chunk (the jobs' rows follow in order)
        const float f = live ? wk[s] * s2[s] : 0.0f;
        uint32_t xw[16];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint4 a = s_h16[2 * hc + q];
            xw[4 * q] = a.x; xw[4 * q + 1] = a.y; xw[4 * q + 2] = a.z; xw[4 * q + 3] = a.w;
        }
        const float i0 = s_hci[hc].y, i1 = s_hci[hc + 1].y;
#pragma unroll
        for (int r = 0; r < RPW; r++) {
            const float d = f4_chunk_h(w[r][s], sc[r * NS + s], xw, i0, i1);
            acc[r] = live ? fmaf(f, d, acc[r]) : acc[r];
        }
    }
    if (has_sh) {
        const int hc = K * CH + min(lane, CH - 1);
        const float2 ci = s_hci[hc];
        const float gm = gdot ? sigmoid(gd) : 1.0f;
#pragma unroll
        for (int r = 0; r < RPW; r++) {
            const float d = dot16_i8h(wsh[r], s_h16[2 * hc], s_h16[2 * hc + 1], ci.x) * ci.y;
            acc[r] = lane < CH ? fmaf(gm * sds[r], d, acc[r]) : acc[r];
        }
    }
#pragma unroll
    for (int r = 0; r < RPW; r++) {
        acc[r] = group_sum<64>(acc[r]);
        if (lane == 0) {
            if (y32) y32[r0 + r] = acc[r];
            else ybf[r0 + r] = f32_to_bf16(acc[r]);
        }
    }
}

int launch_f4_m1(const Qf4ExpCache *a, const ShPtrs *sh, const uint16_t *x, const float *logits, const float *gdot,
                 int *sel, float *wts, float *hidden, uint32_t *ctl, float *y32, uint16_t *ybf, hipStream_t s) {
    const int K = g_cfg.K;
    if (g_cfg.E != 512 || K < 1 || K > 16 || (!y32 && !ybf)) { set_error(-1, "f4_m1: bad arguments"); return -1; }
    ShPtrs sp{};
    if (sh) sp = *sh;
    const unsigned jobs = (unsigned)K + (sh ? 1u : 0u);
#define QFM_F4_DOWN(HH, II, NS)                                                                                     \
    hipLaunchKernelGGL((k_f4_down_m1<HH, II, NS>), dim3(HH / 8), dim3(512), 0, s, a->w_down, a->s_down, a->s2d_dev, \
                       hidden, wts, sel, K, sp, gdot, y32, ybf)
#define QFM_F4_M1(HH, II)                                                                                           \
    hipLaunchKernelGGL((k_f4_gateup_m1<HH, II>), dim3(II / (256 / lpr_of(HH / 32)), jobs), dim3(256), 0, s,         \
                       a->w_gate, a->w_up, a->s_gate, a->s_up, a->s2g_dev, a->s2u_dev, x, logits, sel, wts, K,      \
                       g_cfg.renorm, hidden, sp, ctl);                                                              \
    switch ((K * (II / 32) + 63) / 64) {                                                                            \
    case 1: QFM_F4_DOWN(HH, II, 1); break;                                                                          \
    case 2: QFM_F4_DOWN(HH, II, 2); break;                                                                          \
    case 3: QFM_F4_DOWN(HH, II, 3); break;                                                                          \
    case 4: QFM_F4_DOWN(HH, II, 4); break;                                                                          \
    default: QFM_F4_DOWN(HH, II, 5); break;                                                                         \
    }
    if (shape_2048()) {
        QFM_F4_M1(2048, 512)
    } else if (shape_2560()) {
        QFM_F4_M1(2560, 640)
    } else {
        set_error(-2, "f4_m1: unsupported shape"); return -2;
    }
#undef QFM_F4_M1
#undef QFM_F4_DOWN
    return check_launch("f4_m1");
}

}  // namespace qfm
