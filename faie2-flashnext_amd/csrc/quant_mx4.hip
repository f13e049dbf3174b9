// Matrix-core GEMV instantiations (quant_mx.cuh): Q6_K and IQ3_S.
#include "quant_mx.cuh"

namespace fn {

int gemv_mx4(const QLayout &L, const uint8_t *packed, const float *x, int nt, float *y, hipStream_t st) {
    switch (L.type) {
        case QT_Q6_K: return mx_gemv_t<QT_Q6_K>(L, packed, x, nt, y, st);
        case QT_IQ3_S: return mx_gemv_t<QT_IQ3_S>(L, packed, x, nt, y, st);
        default: FN_FAIL("gemv: unsupported type");
    }
}

}  // namespace fn
