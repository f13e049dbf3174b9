// The walk of k_attn_split_mt on the bf16 matrix cores (included by attn.hip, after its fp32 walk).
//
// Every fp32 operand is the sum of three bf16 values (hi, mid, lo: 8 bits each, rounded to nearest, so the sum is
// exact, down to 2^-110: what lies below is looked after at MX_PUP) and a product takes the six of the nine part products
// that reach fp32's precision: hi hi, hi mid, mid hi, hi lo, lo hi, mid mid.  What is left out, mid lo + lo mid + lo lo,
// is at most 2^-24 of a product (mid reaches 2^-8 of an operand, lo 2^-17), half a unit of its last fp32 place, and about
// 2^-28 in the mean; the sums' error against 64 bits is 8.4e-7 to 8.5e-7 where fp32 products gave 8.9e-7.  On
// v_mfma_f32_16x16x32_bf16 six of them take 96 cycles for 32 contraction slots where v_mfma_f32_16x16x4f32 takes 256.
// What bounds it: per 32 keys and 32 query rows a wave issues 384 products (6,144 cycles) and about as many cycles of
// VALU for the split of K and V (11 instructions for two values), so the two are interleaved by hand: step s of the
// walk issues 12 products on the operand split during step s - 1, and between them the 12 pieces of the split of step
// s + 1's operand.  A step is 32 dims of a 16-key block's scores, or one 16-dim tile of P.V over 32 keys.  By the
// counters of an 8-token step over 16 x 32K the matrix cores are busy 41 % of the time, the vector units 53 %, both at
// once 17 %.
// Contraction slots (free to permute as long as both operands agree), lane l, 8 a lane: of the scores, chunks 4 (2u)
// + l/16 and 4 (2u + 1) + l/16 of the row (the cache's 16-byte chunks); of P.V, keys 4(l/16) + 0..3 of the first and
// of the second 16-key block, which the scores leave in the lane that needs them.
// Order of the steps: scores of the next block's first 16 keys, P.V of this block over dims 0 .. 127, scores of its
// second 16 keys, P.V over dims 128 .. 255, softmax.  A step ends by requesting what takes the place of the operand that
// it split: K of the next 16 keys, V of the other 128 dims; loads are in flight for about 14 steps, in 128 registers
// (with all 256 dims of V held, 192 registers, the walk spills).
// Measured on MI355X, layer step, fp32 walk / this one in us (sequences, keys, tokens, query heads; 2 kv heads): 16, 32K,
// 8, 16: 667 / 520; 16, 32K, 4, 16: 354 / 318; 4, 16K, 6, 24: 185 / 124; 1, 128K, 8, 24: 351 / 218; 1, 4K, 4, 16: 34.0 /
// 29.3; 64, 2K, 3, 16: 119 / 107; 1, 130, 3, 16: 28.3 / 25.6.  Faster at every shape tried, so the rule asks for no more
// than that Q fits.  Up to 16 rows half of the products would be padding and the K/V reads bound the fp32 walk: it stays.

typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int MX_NRW = 2;                       // 16-row blocks a wave
constexpr int MX_QB = 8 * 3 * 64;               // 16-byte Q fragments of a 16-row block: [u][part][lane]
constexpr int MX_MAXCTX = 1 << 21;              // 32-bit byte offsets into a head's cache

// What three bf16 parts hold: a value from 2^-110 on exactly, a smaller one to 2^-134 (bf16 has nothing below 2^-133).
//   P: a probability is 0 or at least fp32's smallest normal number, 2^-126, so its parts are those of MX_PUP p; the
//     sums over V come out scaled by it.
//   Q: an element other than 0 must not be too small, nor so large (2^90) that what K's small elements lose would count in
//     the score (at most 2^-134 2^90 a term).
//   V: what it loses counts only in a small sum: a value loses at most 2^-134, beside a probability of at most 2^28
//     (MX_PUP e^MT_SLACK) and 2^21 keys 2^-85 in all, and products that underflow lose less; so a sum of the split, over
//     its streams, must be 2^-56 or larger, or 0 (rows that see no key, dims that hold none), and finite.  (Looked at in
//     the merge and not in the walk's registers, where it cost 2 us: 128 sums a lane of code that runs once.)
constexpr float MX_PUP = 65536.0f;
struct MxRange {  // the least and largest magnitudes seen other than 0, as bits from bit 1 (least: less 1)
    uint32_t least = ~0u, most = 0u;
    __device__ __forceinline__ void see(float x) {
        const uint32_t u = __float_as_uint(x) << 1;
        least = min(least, u - 1);
        most = max(most, u);
    }
    template <int LO, int HI> __device__ __forceinline__ bool out() const {  // below 2^LO, or 2^HI or larger, or a NaN
        return least < ((127u + LO) << 24) - 1 || most >= (127u + HI) << 24;
    }
};

struct Mx3 {  // 8 values a lane, in three bf16 parts
    v4u p[3];
};

__device__ __forceinline__ uint32_t mx_cvt(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{a, b}), bf16x2));
}
// part PH of values 2k, 2k + 1 of x; r holds their remainder between the parts.  An infinity or NaN (or a value that
// rounds to infinity) leaves a NaN in a later part, which is found in the sums.
__device__ __forceinline__ void mx_split_piece(int k, int ph, const float (&x)[8], float (&r)[2], Mx3 &d) {
    const float a = ph == 0 ? x[2 * k] : r[0], b = ph == 0 ? x[2 * k + 1] : r[1];
    const uint32_t h = mx_cvt(a, b);
    d.p[ph][k] = h;
    if (ph < 2) {
        r[0] = a - __uint_as_float(h << 16);
        r[1] = b - __uint_as_float(h & 0xFFFF0000u);
    }
}
__device__ __forceinline__ void mx_split(const float (&x)[8], Mx3 &d) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float r[2];
#pragma unroll
        for (int ph = 0; ph < 3; ++ph) mx_split_piece(k, ph, x, r, d);
    }
}

__device__ __forceinline__ v4f mx_mma(const v4u &a, const v4u &b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

// One step: A . B[0/1] in six part products each, and the split of the next step's operand x into `nxt` between them.
// hi hi is added to big0/1, the other products to small0/1.  mid() runs once B's hi parts have been used.
template <class Mid>
__device__ __forceinline__ void mx_step(const Mx3 &A, const Mx3 (&B)[MX_NRW], v4f &big0, v4f &big1, v4f &small0,
                                        v4f &small1, const float (&x)[8], Mx3 &nxt, Mid mid) {
    constexpr int PA[6] = {0, 1, 2, 0, 1, 0}, PB[6] = {0, 0, 0, 1, 1, 2};
    float r[2];
#pragma unroll
    for (int s = 0; s < 12; ++s) {
        v4f &acc = s / 2 == 0 ? ((s & 1) ? big1 : big0) : ((s & 1) ? small1 : small0);
        acc = mx_mma(A.p[PA[s / 2]], B[s & 1].p[PB[s / 2]], acc);
        mx_split_piece(s / 3, s % 3, x, r, nxt);
        if (s == 5) mid();
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <bool KEEP>
struct MxWalk {
    const char *Kb, *Vb;
    const v4u *qs;
    int nkmax, lane;
    float4 k[16], v[8][2];  // K of a 16-key block; V of a 32-key block: v[j][c % 2] = dims 64c + 4(l%16) .. +3 of slot j
    v4f o[MX_NRW][16];
    Mx3 A[2], P[MX_NRW];
    float m[MX_NRW], l[MX_NRW], corr[MX_NRW];
    int lim[MX_NRW];
    v4f S[2][MX_NRW];

    __device__ __forceinline__ float4 ld(const char *base, uint32_t off) {
        return mt_ld<KEEP>(reinterpret_cast<const float4 *>(base + off));
    }
    __device__ __forceinline__ uint32_t koff(int kb) const {
        const uint32_t key = min(kb + (lane & 15), nkmax - 1);
        return key / TILE * (TILE * HD * 4) + (key % TILE) * 16 + (lane >> 4) * (TILE * 16);
    }
    __device__ __forceinline__ uint32_t voff(int kb, int j) const {  // key slot j of the lane
        const uint32_t key = min(kb + 16 * (j / 4) + 4 * (lane >> 4) + j % 4, nkmax - 1);
        return key * (HD * 4) + (lane & 15) * 16;
    }
    __device__ __forceinline__ void load_k(int u, uint32_t off) {  // chunks of dim step u: 32 dims
        k[2 * u] = ld(Kb + (size_t) (2 * u) * (4 * TILE * 16), off);
        k[2 * u + 1] = ld(Kb + (size_t) (2 * u + 1) * (4 * TILE * 16), off);
    }
    __device__ __forceinline__ void load_v(int c, int kb) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j][c % 2] = ld(Vb + 256 * c, voff(kb, j));
    }
    __device__ __forceinline__ void raw_k(int u, float (&x)[8]) const {
        const float4 a = k[2 * u], b = k[2 * u + 1];
        x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
    }
    __device__ __forceinline__ void raw_v(int t, float (&x)[8]) const {  // tile t = 4c + e
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float4 a = v[j][t / 4 % 2];
            x[j] = t % 4 == 0 ? a.x : t % 4 == 1 ? a.y : t % 4 == 2 ? a.z : a.w;
        }
    }
    __device__ __forceinline__ void load_q(int u, int p, int qo, Mx3 (&q)[MX_NRW]) const {
#pragma unroll
        for (int j = 0; j < MX_NRW; ++j) q[j].p[p] = qs[j * MX_QB + (u * 3 + p) * 64 + qo];
    }
    // Scores of a 16-key block (its dim step 0 is in A[0]) into S[b]; its registers are requested again at byte offset
    // off (the 16 keys after it), and the operand after it -- V tile t0, or K's next block if t0 < 0 -- is left in A[0].
    __device__ __forceinline__ void qk(int b, uint32_t off, int t0) {
        // the Q offset is made to depend on the block, so that the reads stay in the loop
        int qo = lane;
        asm("" : "+v"(qo) : "v"(off));
        Mx3 q[MX_NRW];  // hi is read half a step ahead, mid and lo at the start of the step (used in its second half)
        load_q(0, 0, qo, q);
        // two sums a row block: hi hi, and the small products (in one sum, every product rounds at the size of the whole
        // score: scores in the hundreds were off by 1.2e-5 where the fp32 walk stays below 1e-5)
        v4f acc[2][MX_NRW];
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][0] = acc[i][1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            float x[8];
            load_q(u, 1, qo, q);
            load_q(u, 2, qo, q);
            if (u < 7) raw_k(u + 1, x);
            else if (t0 < 0) raw_k(0, x);
            else raw_v(t0, x);
            mx_step(A[u & 1], q, acc[0][0], acc[0][1], acc[1][0], acc[1][1], x, A[(u + 1) & 1], [&] {
                if (u < 7) load_q(u + 1, 0, qo, q);
            });
            if (u == 0) load_k(0, off);
            if (u < 7) load_k(u + 1, off);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < MX_NRW; ++j) S[b][j] = acc[0][j] + acc[1][j];
    }
    // P.V of tiles T0 .. T0 + 7 (tile T0 in A[0]) of a block; the other half's V is requested of the block at vkb (T0 = 0:
    // of the same block).  K's dim step 0 is left in A[0] (LAST: V's tile 8, and T0 = 8 requests nothing)
    template <int T0, bool LAST> __device__ __forceinline__ void pv(int vkb) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int t = T0 + i;
            float x[8];
            if (i < 7) raw_v(t + 1, x);
            else if (LAST) raw_v(8, x);
            else raw_k(0, x);
            mx_step(A[i & 1], P, o[0][t], o[1][t], o[0][t], o[1][t], x, A[(i + 1) & 1], [] {});
            if (t % 4 == 2 && !(LAST && T0 == 8)) load_v((t / 4 + 2) % 4, vkb);  // tile t + 1, its group's last, is split
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // the online-softmax step of mt_softmax over 32 keys from kb; P = the probabilities in parts
    __device__ __forceinline__ void softmax(int kb) {
        constexpr float LOG2E = 1.4426950408889634f;
        const float scale = rsqrtf((float) HD);
        const int key = kb + 4 * (lane >> 4);
#pragma unroll
        for (int j = 0; j < MX_NRW; ++j) {
            float sc[8], p[8];
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                sc[i] = key + 16 * (i / 4) + i % 4 < lim[j] ? S[i / 4][j][i % 4] * scale : -INFINITY;
                mx = fmaxf(mx, sc[i]);
            }
            mx = max_x16_x32(mx);
            const bool first = m[j] == -INFINITY, moved = !first && mx > m[j] + MT_SLACK;
            const float mn = first || moved ? mx : m[j];
            corr[j] = moved ? __builtin_amdgcn_exp2f((m[j] - mn) * LOG2E) : 1.0f;
            float ps = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                p[i] = sc[i] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((sc[i] - mn) * LOG2E);
                ps += p[i];
            }
            l[j] = fmaf(l[j], corr[j], ps);
            m[j] = mn;
#pragma unroll
            for (int i = 0; i < 8; ++i) p[i] *= MX_PUP;
            mx_split(p, P[j]);
        }
        mt_rescale<MX_NRW>(o, corr);
        // o stays in AGPRs (left to itself the compiler copies some of it to VGPRs and spills 8 to scratch, whose reloads
        // wait for every load in flight)
#pragma unroll
        for (int t = 0; t < 16; ++t) asm("" : "+a"(o[0][t]), "+a"(o[1][t]));
        __builtin_amdgcn_sched_barrier(0);
    }
    // the nw 32-key blocks from kb0, stride keys apart (loads past the last key are clamped to it: in bounds, unused)
    __device__ __forceinline__ void walk(int kb0, int stride, int nw) {
        float x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) load_k(u, koff(kb0));
        raw_k(0, x);
        mx_split(x, A[0]);
        __builtin_amdgcn_sched_barrier(0);
        qk(0, koff(kb0 + 16), -1);
        qk(1, koff(kb0 + stride), -1);
        // V after K's next block, as in the loop: the loop's waits count loads in the order of both ways into it, and with
        // V ahead of K here they waited for V's latency in every iteration
#pragma unroll
        for (int c = 0; c < 2; ++c) load_v(c, kb0);
        __builtin_amdgcn_sched_barrier(0);
        softmax(kb0);
        int kb = kb0;
        for (int i = 0; i + 1 < nw; ++i) {
            const int kn = kb + stride;  // the block whose scores are taken
            qk(0, koff(kn + 16), 0);
            pv<0, false>(kb);
            qk(1, koff(kn + stride), 8);
            pv<8, false>(kn);
            softmax(kn);
            kb = kn;
        }
        raw_v(0, x);
        mx_split(x, A[0]);
        pv<0, true>(kb);
        pv<8, true>(kb);
    }
};
