// qfm_mfma.h -- weight-streaming MFMA tiles for a few activation rows (gfx950):
// fragment conversions, the LDS layout and the down-projection body shared by
// the middle path (qfm_mid.hip) and the chunk tier (qfm_compat.hip).
#pragma once
#include "qfm_dev.h"

namespace qfm {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// ---- fragments ----------------------------------------------------------------------
// 16 int8 codes -> 16 fp16, exact: 1024 + u (u = q + 128) by v_perm, then - 1152
__device__ __forceinline__ void i8_to_f16(u32x4_t w, f16x8_t &a, f16x8_t &b) {
    const f16x2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
    uint32_t o[8];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint32_t d = w[q] ^ 0x80808080u;
        o[2 * q] = __builtin_bit_cast(uint32_t, as_h2(__builtin_amdgcn_perm(0x64646464u, d, 0x04010400u)) - off);
        o[2 * q + 1] = __builtin_bit_cast(uint32_t, as_h2(__builtin_amdgcn_perm(0x64646464u, d, 0x04030402u)) - off);
    }
    a = __builtin_bit_cast(f16x8_t, u32x4_t{o[0], o[1], o[2], o[3]});
    b = __builtin_bit_cast(f16x8_t, u32x4_t{o[4], o[5], o[6], o[7]});
}
// 8 e2m1 codes (one dword) times a block scale < 0x7F -> fp16, exact
__device__ __forceinline__ f16x8_t f4_to_f16(uint32_t w, f16x2_t s) {
    const u32x4_t o = {__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0) * s),
                       __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1) * s),
                       __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2) * s),
                       __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3) * s)};
    return __builtin_bit_cast(f16x8_t, o);
}
// the same with any scale byte (0x7F: +inf, >= 0x80: up to 2^24) as bf16, exact;
// the activations follow as bf16 (they were bf16 rows times a power of two, or
// are rounded to 8 bits: k_mid_down's hidden rows, as the prefill path holds them)
__device__ __forceinline__ uint32_t pack_bf16_hi(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
__device__ __forceinline__ bf16x8_t f4_to_bf16x8(uint32_t w, float s) {
    const f32x2_t a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 0), b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 1),
                  c = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 2), d = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 3);
    const u32x4_t o = {pack_bf16_hi(a.x * s, a.y * s), pack_bf16_hi(b.x * s, b.y * s), pack_bf16_hi(c.x * s, c.y * s),
                       pack_bf16_hi(d.x * s, d.y * s)};
    return __builtin_bit_cast(bf16x8_t, o);
}
__device__ __forceinline__ bf16x8_t f16_to_bf16x8(f16x8_t h) {
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
        o[i] = (uint32_t)f32_to_bf16((float)h[2 * i]) | ((uint32_t)f32_to_bf16((float)h[2 * i + 1]) << 16);
    return __builtin_bit_cast(bf16x8_t, u32x4_t{o[0], o[1], o[2], o[3]});
}
__device__ __forceinline__ f32x4_t mfma_f16(f16x8_t a, f16x8_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma_bf16(bf16x8_t a, bf16x8_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// no block-scale byte of the vector is 0x7F or more (a carry into a byte can only
// make this false)
template <class V>
__device__ __forceinline__ bool f4_scales_hw(V s) {
    uint32_t bad = 0u;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(V) / 4); i++) bad |= s[i] | (s[i] + 0x01010101u);
    return (bad & 0x80808080u) == 0u;
}
// LDS rows of STRIDE bytes: 16-byte chunk c of row r at chunk position c ^
// lds_rot(r), so that the 16 rows of a fragment read spread over the 64 banks
template <int STRIDE>
__device__ __forceinline__ int lds_rot(int r) {
    static_assert(STRIDE % 256 == 0 || STRIDE % 256 == 128 || STRIDE % 256 == 64, "row strides in use");
    return STRIDE % 256 == 0 ? r & 15 : STRIDE % 256 == 128 ? r & 7 : (r >> 2) & 3;
}
template <int STRIDE>
__device__ __forceinline__ int lds_at(int r, int c) { return r * STRIDE + ((c ^ lds_rot<STRIDE>(r)) << 4); }
// orders this wave's LDS accesses across its lanes (LDS serves one wave in order)
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// 2^k scaling of a group whose largest magnitude is m into [2^14, 2^15)
__device__ __forceinline__ int f16_exp(float m) {
    return m == 0.0f ? 0 : min(113, max(-113, 141 - (int)(__float_as_uint(m) >> 23)));
}
__device__ __forceinline__ float exp2i(int k) { return __uint_as_float((uint32_t)(127 + k) << 23); }

// 16 bytes of weights: nontemporal where (nearly) every byte is read ONCE (INT8
// gate/up + down at 37 / 300 rows 154 -> 136 / 288 -> 262 us, 6.4 TB/s), plain
// where an expert's further items read them again (1021 rows: 264 + 167 us
// nontemporal, 244 + 144 plain; NVFP4 at 2560/640 395 + 255 against 304 + 240;
// at 700 rows no difference; whole calls at 600 rows 2560/640 INT8 evenly spread
// 543 nontemporal, 561 plain, all on ten experts 356 and 270).
template <bool ONCE>
__device__ __forceinline__ u32x4_t ld_w(const uint8_t *p) {
    const u32x4_t *v = reinterpret_cast<const u32x4_t *>(p);
    if constexpr (ONCE) return __builtin_nontemporal_load(v);
    else return *v;
}

// ---- down ---------------------------------------------------------------------------
constexpr int mid_dn_waves(int I, int nt) { return nt == 1 || I * nt > 2048 ? 4 : 8; }
template <int I, int NT>
struct MidDnLds {
    uint8_t h[16 * NT * I * 2];                   // the item's hidden rows (whole K)
    uint8_t w[mid_dn_waves(I, NT)][16 * I];          // per wave: one tile of 16 weight rows (NVFP4: codes, then scales)
    float isc[16 * NT][I / 64 + 1];               // 2^-k of each row and 64 hidden values
};
// 64 output columns per wave as four tiles of 16 weight rows (wd / bd: the
// wave's first row and its block scales) against `rows` activation rows, which
// stage.load() requests and stage.store(L) puts into L.h (fp16, lds_at rows)
// and L.isc; acc[rt][n]: D[row 4 g + i][activation row l16].
template <int I, bool F4, int NT, bool ONCE, class STAGE>
__device__ __forceinline__ void mid_dn_body(const uint8_t *__restrict__ wd, const uint8_t *__restrict__ bd, int rows,
                                            MidDnLds<I, NT> &L, f32x4_t (&acc)[4][NT], STAGE &&stage, int tid) {
    constexpr int NG = I / 64, RT = 4, HS = I * 2;
    constexpr int ROWB = F4 ? I / 2 : I, CPR = ROWB / 16, NL = 16 * CPR / 64;   // bytes, chunks per row, loads per tile
    constexpr int SB = I / 16, SL = 16 * SB / 16;                                // NVFP4 scale bytes per row, 16-byte loads per tile
    constexpr int D = F4 ? 4 : 2;                                                // tiles in flight
    static_assert(NL * 64 == 16 * CPR && SL <= 64, "whole loads per tile");
    static_assert(!F4 || 16 * ROWB + 16 * SB <= 16 * I, "an NVFP4 tile and its scales fit the INT8 tile's LDS");
    const int lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    u32x4_t buf[D][NL], sc[F4 ? D : 1];
    stage.load();                                 // (in L2: ahead of the weights, as loads retire in issue order)
    auto wload = [&](int rt) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NL; j++)
            buf[rt % D][j] = ld_w<ONCE>(wd + (size_t)rt * 16 * ROWB + (j * 64 + lane) * 16);
        if constexpr (F4)
            if (lane < SL) sc[rt % D] = *reinterpret_cast<const u32x4_t *>(bd + (size_t)rt * 16 * SB + lane * 16);
    };
#pragma unroll
    for (int rt = 0; rt < D; rt++) wload(rt);
    stage.store(L);
    __syncthreads();
    uint8_t *lw = L.w[wave];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
#pragma unroll
        for (int j = 0; j < NL; j++) {
            const int c = j * 64 + lane;
            *reinterpret_cast<u32x4_t *>(lw + lds_at<ROWB>(c / CPR, c % CPR)) = buf[rt % D][j];
        }
        // NVFP4: whether every block scale of the tile is below 0x7F (one test, and
        // one branch, per tile: tested per 64 values the branches kept the
        // fragments' LDS reads and conversions from overlapping)
        bool hw = true;
        if constexpr (F4) {
            if (lane < SL) *reinterpret_cast<u32x4_t *>(lw + 16 * ROWB + lane * 16) = sc[rt % D];
            hw = __builtin_amdgcn_ballot_w64(lane < SL && !f4_scales_hw(sc[rt % D])) == 0;
        }
        if (rt + D < RT) wload(rt + D);
        wave_lds_fence();
#pragma unroll
        for (int n = 0; n < NT; n++) acc[rt][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        // 64 values kg: hidden values 64 kg + 16 g .. + 15 of activation row l16, weights of row l16
        auto hfrag = [&](int n, int kg, int h) __attribute__((always_inline)) {
            return *reinterpret_cast<const f16x8_t *>(L.h + lds_at<HS>(n * 16 + l16, 8 * kg + 2 * g + h));
        };
        auto add = [&](int n, int kg, f32x4_t d) __attribute__((always_inline)) {
            const float s = L.isc[n * 16 + l16][kg];
#pragma unroll
            for (int i = 0; i < 4; i++) acc[rt][n][i] = fmaf(d[i], s, acc[rt][n][i]);
        };
        const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
        if constexpr (!F4) {
#pragma unroll 2
            for (int kg = 0; kg < NG; kg++) {
                f16x8_t w0, w1;
                i8_to_f16(*reinterpret_cast<const u32x4_t *>(lw + lds_at<ROWB>(l16, 4 * kg + g)), w0, w1);
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    if (NT > 1 && n * 16 >= rows) continue;
                    add(n, kg, mfma_f16(w1, hfrag(n, kg, 1), mfma_f16(w0, hfrag(n, kg, 0), z)));
                }
            }
        } else {
            auto wfrag = [&](int kg) __attribute__((always_inline)) {
                return *reinterpret_cast<const u32x2_t *>(lw + lds_at<ROWB>(l16, 2 * kg + (g >> 1)) + (g & 1) * 8);
            };
            if (hw) {
#pragma unroll
                for (int kg = 0; kg < NG; kg++) {
                    const u32x2_t w = wfrag(kg);
                    const f32x2_t f = __builtin_amdgcn_cvt_pk_f32_fp8(lw[16 * ROWB + l16 * SB + 4 * kg + g], false);
                    const f16x2_t s = {(_Float16)f.x, (_Float16)f.x};
                    const f16x8_t w0 = f4_to_f16(w[0], s), w1 = f4_to_f16(w[1], s);
#pragma unroll
                    for (int n = 0; n < NT; n++) {
                        if (NT > 1 && n * 16 >= rows) continue;
                        add(n, kg, mfma_f16(w1, hfrag(n, kg, 1), mfma_f16(w0, hfrag(n, kg, 0), z)));
                    }
                }
            } else {
#pragma unroll 1
                for (int kg = 0; kg < NG; kg++) {
                    const u32x2_t w = wfrag(kg);
                    const float s = e4m3_scale(lw[16 * ROWB + l16 * SB + 4 * kg + g]);
                    const bf16x8_t w0 = f4_to_bf16x8(w[0], s), w1 = f4_to_bf16x8(w[1], s);
#pragma unroll
                    for (int n = 0; n < NT; n++) {
                        if (NT > 1 && n * 16 >= rows) continue;
                        add(n, kg, mfma_bf16(w1, f16_to_bf16x8(hfrag(n, kg, 1)),
                                             mfma_bf16(w0, f16_to_bf16x8(hfrag(n, kg, 0)), z)));
                    }
                }
            }
        }
        wave_lds_fence();
    }
}

}  // namespace qfm
