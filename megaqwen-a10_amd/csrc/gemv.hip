// Standalone INT8 weight-only matvec, y[j] = scale[j] * sum_k x[k] * w[j,k]
// (int8_decoder.py:100-115 semantics; fp32 activations as BASELINE config 2): the row
// kernel of gemv_rows.h with sign-extended bytes converted by v_cvt_f32_i32.
#include "gemv_rows.h"

namespace mq {

int device_cu_count() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cached[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev] = n;
    }
    return cached[dev];
}

int launch_int8_gemv_repeat(const float* x, const int8_t* w, int64_t copy_stride, int n_copies, const float* scale,
                            float* y, int M, int K, int reps, hipStream_t stream) {
    return launch_gemv_rows<Int8W>(x, reinterpret_cast<const uint8_t*>(w), copy_stride, n_copies, scale, y, M, K, reps,
                                   stream);
}

int launch_int8_gemv(const float* x, const int8_t* w, const float* scale, float* y, int M, int K,
                     hipStream_t stream) {
    return launch_int8_gemv_repeat(x, w, 0, 1, scale, y, M, K, 1, stream);
}

}  // namespace mq
