// What the attention kernels (attn.hip) and the QSA indexer's scoring launch (qsa.hip) share: the attention's
// arguments, the K cache's layout and the query / new key rows' RMSNorm + RoPE.
#pragma once

#include "qsa.h"

namespace fn {

constexpr int HD = 256;     // head dim built (the reference's, faie2fn.cu:49)
constexpr int TILE = 64;    // keys per tile (= wave size)
constexpr int MAXROT = 128;

struct AttnArgs {
    int B, nq, nkv, nt, max_ctx, nsplit, nrot;
    float eps;
    const int32_t *pos;
    const float *qg, *knew, *vnew, *wq, *wk;
    float *Kc, *Vc;
    float *Q;        // [B nt][nkv][HD/4][grp][4]
    float *part_o;   // [B nt][nq][nsplit][HD]
    float *part_ml;  // [B nt][nq][nsplit][2]
    float *og;
    const int32_t *keys;   // visible-key list per query (QSA) or null (dense)
    const int32_t *nkeys;
    int kstride;           // list stride per query
    unsigned *status;      // per-device status word: FN_STATUS_POS when a new token falls outside the cache
    float inv_freq[MAXROT / 2];
};

__device__ __forceinline__ size_t k_index(int max_ctx, int b, int nkv, int g, int p, int d) {
    const size_t tile = ((size_t) b * nkv + g) * (max_ctx / TILE) + p / TILE;
    return ((tile * (HD / 4) + d / 4) * TILE + (p % TILE)) * 4 + (d % 4);
}

// RMSNorm + RoPE of the query heads and the new key (faie2fn.cu:1451-1478), cache append.
// Row j of token bt (the nq query heads, then the nkv keys and values) by HD threads; buf: HD + HD / 64 floats of LDS
__device__ __forceinline__ void attn_prep_row(const AttnArgs &a, int bt, int j, float *buf) {
    float *red = buf + HD;
    const int b = bt / a.nt, t = bt - b * a.nt, d = threadIdx.x;
    const int P = a.pos[b] + t;
    if (P < 0 || P >= a.max_ctx) {  // outside the cache: nothing is written past it; the status word says so
        if (j == 0 && d == 0) atomicOr(a.status, FN_STATUS_POS);
        return;
    }
    const bool isq = j < a.nq;
    const int g = isq ? j / (a.nq / a.nkv) : j - a.nq;
    const float x = isq ? a.qg[((size_t) bt * a.nq + j) * 2 * HD + d] : a.knew[((size_t) bt * a.nkv + g) * HD + d];
    const float ws = wave_sum(x * x);
    if ((d & 63) == 0) red[d >> 6] = ws;
    __syncthreads();
    const float ss = red[0] + red[1] + red[2] + red[3];
    buf[d] = x * rsqrtf(ss / HD + a.eps) * (isq ? a.wq[d] : a.wk[d]);
    __syncthreads();
    float y = buf[d];
    const int half = a.nrot / 2;
    if (d < a.nrot) {
        const int i = d < half ? d : d - half;
        const float x0 = buf[i], x1 = buf[i + half];
        const float ang = (float) P * a.inv_freq[i];  // fp32 angle (faie2fn.cu:1440)
        const float cs = cosf(ang), sn = sinf(ang);
        y = d < half ? x0 * cs - x1 * sn : x1 * cs + x0 * sn;
    }
    if (isq) {
        const int grp = a.nq / a.nkv, hh = j - g * grp;
        a.Q[((((size_t) bt * a.nkv + g) * (HD / 4) + d / 4) * grp + hh) * 4 + (d % 4)] = y;
    } else {
        a.Kc[k_index(a.max_ctx, b, a.nkv, g, P, d)] = y;
        a.Vc[(((size_t) b * a.nkv + g) * a.max_ctx + P) * HD + d] = a.vnew[((size_t) bt * a.nkv + g) * HD + d];
    }
}

}  // namespace fn
