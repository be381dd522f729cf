// qfm_x8.h -- X8 and activation helpers of the dense INT8 kernels.
#pragma once
#include "qfm_dev.h"
#include "../../include/qf_dense.h"

namespace qfm {

typedef int i32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float gemv_act(float v, int act) {
    if (act == 1) {
        const float q = v * 0.25f;
        return q / (1.0f + expf(-q));
    }
    if (act == 2) return 2.0f / (1.0f + expf(-v * 0.25f));
    return v;
}

// X8 of one value per lane over aligned 32-lane groups (qf8_i8_x8's rule)
__device__ __forceinline__ int x8_code(float v, float &scale) {
    const float mx = group_max<32>(fabsf(v));
    scale = mx > 0.0f ? mx * (1.0f / 127.0f) : 1.0f;
    return min(127, max(-127, (int)rintf(v / scale)));
}

// The pre-mixer over more rows than the two-launch form takes (qfm_hc_rows.hip).
struct HcRowsArgs {
    float *R;
    const uint16_t *wn;
    const float *y_prev, *inj_prev;
    const Qf8I8Mat *down, *inject, *up;
    float *normed, *hc_d, *inj, *hcy, *mixed;
    int8_t *n8q, *d8q, *xq_out;
    float *n8s, *d8s, *xs_out;
    uint16_t *xb_out;
    int T;
};
void launch_hc_rows(const HcRowsArgs &a, hipStream_t s);

}  // namespace qfm
