// Matrix-core GEMV instantiations (quant_mx.cuh): the IQ4 formats.
#include "quant_mx.cuh"

namespace fn {

int gemv_mx2(const QLayout &L, const uint8_t *packed, const float *x, int nt, float *y, hipStream_t st) {
    switch (L.type) {
        case QT_IQ4_NL: return mx_gemv_t<QT_IQ4_NL>(L, packed, x, nt, y, st);
        case QT_IQ4_XS: return mx_gemv_t<QT_IQ4_XS>(L, packed, x, nt, y, st);
        default: FN_FAIL("gemv: unsupported type");
    }
}

}  // namespace fn
