// Matrix-core GEMV instantiations (quant_mx.cuh): BF16 and Q8_0.
#include "quant_mx.cuh"

namespace fn {

int gemv_mx1(const QLayout &L, const uint8_t *packed, const float *x, int nt, float *y, hipStream_t st) {
    switch (L.type) {
        case QT_BF16: return mx_gemv_t<QT_BF16>(L, packed, x, nt, y, st);
        case QT_Q8_0: return mx_gemv_t<QT_Q8_0>(L, packed, x, nt, y, st);
        default: FN_FAIL("gemv: unsupported type");
    }
}

}  // namespace fn
