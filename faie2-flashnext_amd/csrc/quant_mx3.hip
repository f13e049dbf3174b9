// Matrix-core GEMV instantiations (quant_mx.cuh): Q4_K and Q5_K.
#include "quant_mx.cuh"

namespace fn {

int gemv_mx3(const QLayout &L, const uint8_t *packed, const float *x, int nt, float *y, hipStream_t st) {
    switch (L.type) {
        case QT_Q4_K: return mx_gemv_t<QT_Q4_K>(L, packed, x, nt, y, st);
        case QT_Q5_K: return mx_gemv_t<QT_Q5_K>(L, packed, x, nt, y, st);
        default: FN_FAIL("gemv: unsupported type");
    }
}

}  // namespace fn
