// Matrix-core GEMV instantiations (quant_mx.cuh): the grouped launches, by the format sets of quant_grp.hip.
#include "quant_mx.cuh"

namespace fn {

int gemv_mx_grp(int kind, const QLayout *const *L, const uint8_t *const *packed, float *const *y, const float *x, int nt,
                hipStream_t st) {
    const int n = kind == 2 ? 4 : 3;
    PP P[4];
    for (int i = 0; i < n; ++i) P[i] = planes(*L[i], packed[i]);
    switch (kind) {
        case 0: return mx_grp<QT_IQ4_XS, QT_IQ3_S, QT_BF16>(L, P, y, x, nt, st);
        case 1: return mx_grp<QT_IQ4_XS, QT_Q6_K, QT_BF16>(L, P, y, x, nt, st);
        default: return mx_grp<QT_IQ4_XS, QT_IQ4_XS, QT_Q6_K, QT_BF16>(L, P, y, x, nt, st);
    }
}

}  // namespace fn
