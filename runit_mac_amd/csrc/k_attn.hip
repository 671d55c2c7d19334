// k_attn.hip — causal multi-query attention of long prompts: keys and values
// prepared once a call as pairs of f16 (x·2^e = hi + lo, an exponent a row: 22
// bits of the elements down to 2^-18 of the row's largest, 2^-40 of that
// below), both products on the 32x32x16 f16 matrix cores (f16 × f16 products
// exact, f32 sums), the softmax in f32.
//
// k_attn_mq's f32 matrix cores bound it, a sixteenth of the f16 rate, and its
// operand loads, 64 lines of L1 an instruction: 512 queries of 28 heads of 128
// after 1,536 positions ran 182 µs, 13 GFLOP at 72 of 157 TFLOP/s.  Three f16
// products (hi·hi, hi·lo, lo·hi) take 3/16 of the f32 product's matrix time:
// 81 µs here, of which the preparation is 8, the merge of the ranges 8 and
// about 15 the start and end of the main kernel's workgroups: 0.65 µs a record
// and wave are the matrix cores, each wave's softmax hides behind them only in
// part.  (One exponent for all values of a record, put into P before it is
// split, ran 75: it lost the weights of values far below the largest that any
// record held.)  Measured on the way, from 79 µs: expf instead of exp2 95, the
// operands loaded where they are used 82, the sums rescaled at each new
// maximum 80.
#include "rt_attn.h"

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) uint32_t* gptr_t;
typedef __attribute__((address_space(3))) uint32_t* lptr_t;

// Mirrors the host's AttnPfArgs (runtime.cpp).
struct AttnPfArgs {
    const float* q;    // [batch][q_len][H][HD]
    const float* kc;   // [batch][KVH][stride][HD]
    const float* vc;
    float* out;        // [batch][q_len][H][HD]
    u32x4* ops;        // [batch][KVH][tiles] records of 32 positions
    float* part;       // nsp > 1: [batch][KVH][cbs][nsp][128][HD] unnormalised outputs
    float* ml;         //          [batch][KVH][cbs][nsp][128][max, sum]
    uint32_t kv, stride, H, KVH, q_len, q_start;  // kv: positions that some query sees
    uint32_t tiles, cbs, nsp, items;
    float scale;
};

// A record: the key operands [HD/16 steps][hi, lo][64 lanes], the value
// operands [HD/32 blocks][2 steps][hi, lo][64], then 256 words (PfTail on).
template <int HD>
struct PfRec {
    static constexpr uint32_t OPS = HD * 16, LEN = OPS + 64;  // in 16-byte entries
};
enum PfTail {
    kTailK = 0,    // 2^-exponent of the 32 keys
    kTailV = 32,   // of the 32 values, 0 of an all-zero one
    kTailMax = 64, // exponent of the largest value (int)
    kTailBad = 65, // whether a key or value is not finite (int)
};

// x·f as hi + lo
RT_DEV void pf_split(const float (&x)[8], float f, h8_t& hi, h8_t& lo) {
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
        const float v = x[i] * f;
        hi[i] = (_Float16)v;
        lo[i] = (_Float16)(v - (float)hi[i]);
    }
}
// the exponent that takes a row's largest magnitude to [2^14, 2^15): the low
// halves of all elements down to 2^-15 of it stay normal numbers.  At most
// 126, so that 2^-e is a normal number too (f16's last place is then 2^-150).
RT_DEV int pf_exp(float mx) { return mx > 0.0f ? min(126, 15 - __builtin_amdgcn_frexp_expf(mx)) : 0; }
RT_DEV float pf_pow2(int e) { return ldexpf(1.0f, e); }

// One workgroup a record (2·HD threads): every position of the cache is read
// once (its value a second time, from L2) and written in as many bytes, in the
// order that the operands of attn_pf take them, each key and each value scaled
// by an exponent of its own.  Keys: lane l of step s holds d = 16s + 8(l / 32) .. of
// position l % 32.  Values: lane l of (block b, step s) holds d = 32b + l % 32
// at the positions whose scores its half of the wave has in registers 8s ..
// 8s + 7 of the score tile: 16s + 8(i / 4) + 4(l / 32) + i % 4.
template <int HD>
RT_DEV void attn_pf_prep(const AttnPfArgs& a) {
    constexpr uint32_t KS = HD / 16;
    __shared__ float red[16];
    __shared__ float vscale[32];
    const uint32_t t = blockIdx.x, tid = threadIdx.x;
    const size_t seq = (size_t)blockIdx.z * a.KVH + blockIdx.y;
    const float* kb = a.kc + seq * a.stride * HD;
    const float* vb = a.vc + seq * a.stride * HD;
    h8_t* rec = (h8_t*)(a.ops + (seq * a.tiles + t) * PfRec<HD>::LEN);
    float* tail = (float*)(rec + PfRec<HD>::OPS);
    bool bad = false;
    const uint32_t p = tid / KS, s = tid % KS;
    float x[2][8] = {}, vmax = 0.0f, kmax = 0.0f;
    if (t * 32 + p < a.kv) {
        const f32x4* k4 = (const f32x4*)(kb + (size_t)(t * 32 + p) * HD + 16 * s);
        const f32x4* v4 = (const f32x4*)(vb + (size_t)(t * 32 + p) * HD + 16 * s);
#pragma unroll
        for (uint32_t i = 0; i < 16; ++i) {
            x[i / 8][i % 8] = k4[i / 4][i % 4];
            const float av = fabsf(v4[i / 4][i % 4]), ak = fabsf(x[i / 8][i % 8]);
            bad |= !(av < __builtin_huge_valf()) || !(ak < __builtin_huge_valf());
            vmax = fmaxf(vmax, av);
            kmax = fmaxf(kmax, ak);
        }
    }
    for (uint32_t o = 1; o < KS; o *= 2) {
        kmax = fmaxf(kmax, __shfl_xor(kmax, o, 64));
        vmax = fmaxf(vmax, __shfl_xor(vmax, o, 64));
    }
    const int ke = pf_exp(kmax), ve = pf_exp(vmax);
    if (s == 0) {
        vscale[p] = pf_pow2(ve);
        tail[kTailK + p] = pf_pow2(-ke);
        tail[kTailV + p] = vmax > 0.0f ? pf_pow2(-ve) : 0.0f;
    }
    const int vexp = pf_exp(block_max(vmax, red));  // (also the barrier before vscale is read)
    const float any = block_max(bad ? 1.0f : 0.0f, red);
    if (tid == 0) {
        ((int*)tail)[kTailMax] = vexp;
        ((int*)tail)[kTailBad] = any != 0.0f;
    }
    h8_t hi, lo;
#pragma unroll
    for (uint32_t h = 0; h < 2; ++h) {
        pf_split(x[h], pf_pow2(ke), hi, lo);
        rec[2 * s * 64 + p + 32 * h] = hi;
        rec[(2 * s + 1) * 64 + p + 32 * h] = lo;
    }
#pragma unroll
    for (uint32_t r = 0; r < 2; ++r) {
        const uint32_t idx = tid + 2 * HD * r, l = idx & 63, bs = idx >> 6;
        const uint32_t d = 32 * (bs / 2) + (l & 31);
        float v[8];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) {
            const uint32_t pos = 16 * (bs % 2) + 8 * (i / 4) + 4 * (l >> 5) + i % 4;
            v[i] = t * 32 + pos < a.kv ? vb[(size_t)(t * 32 + pos) * HD + d] * vscale[pos] : 0.0f;
        }
        pf_split(v, 1.0f, hi, lo);
        rec[PfRec<HD>::OPS / 2 + 2 * bs * 64 + l] = hi;
        rec[PfRec<HD>::OPS / 2 + (2 * bs + 1) * 64 + l] = lo;
    }
}

// Workgroup: 128 query columns — consecutive (row, head) pairs of one KV
// head's group, row-major — over one of nsp ranges of the records that they
// see; wave w takes columns 32w ...  The next record goes to LDS while this
// one is computed (33 KB each at head size 128: two workgroups a CU).  Per
// record a wave computes Sᵀ = K·Qᵀ (a lane: 16 of the 32 positions of one
// column), the online softmax, and Oᵀ += Vᵀ·Pᵀ.  P is split as the rest after
// the values' scales were put into it: each weight is then as large as what
// its position contributes, the column's largest in [2^14, 2^15), so that a
// value's rounding is measured by its own part of the output, whatever the
// magnitudes of the others, of unseen ones or of ones whose weight is nothing.
// The record's product starts at zero and is added in f32.  A record that holds an
// infinity or NaN is computed in plain f32, from the cache.
template <int HD>
RT_DEV void attn_pf(const AttnPfArgs& a) {
    constexpr uint32_t PF = 3;  // operands loaded two steps ahead
    constexpr uint32_t KS = HD / 16, NB = HD / 32, OPS = PfRec<HD>::OPS, LEN = PfRec<HD>::LEN;
    __shared__ u32x4 lds[2][LEN];
    // the items of one KV head side by side on as few XCDs as they fill: its
    // records are read from their L2
    const uint32_t per = (a.items + 7) / 8, item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (item >= a.items) return;
    const uint32_t lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 31, h = lane >> 5;
    const uint32_t cb = a.cbs - 1 - item % a.cbs, sp = item / a.cbs % a.nsp, seq = item / (a.cbs * a.nsp);
    const uint32_t kvh = seq % a.KVH, bt = seq / a.KVH;
    const uint32_t G = a.H / a.KVH, R = a.q_len * G;
    const uint32_t c = cb * 128 + 32 * w + j, cc = min(c, R - 1);
    const uint32_t row = cc / G, head = kvh * G + cc % G;
    const uint32_t lim = c < R ? min(a.kv, a.q_start + row + 1) : 0;
    auto seen = [&](uint32_t c1) { return min(a.kv, a.q_start + (min(R, c1) - 1) / G + 1); };
    const uint32_t Lw = cb * 128 + 32 * w < R ? seen(cb * 128 + 32 * w + 32) : 0;
    const uint32_t Lf = min(a.kv, a.q_start + min(cb * 128 + 32 * w, R - 1) / G + 1);
    const uint32_t T = (seen(cb * 128 + 128) + 31) / 32;
    const uint32_t t0 = (uint64_t)T * sp / a.nsp, t1 = (uint64_t)T * (sp + 1) / a.nsp;
    const u32x4* recs = a.ops + (size_t)seq * a.tiles * LEN;
    auto copy = [&](uint32_t t, uint32_t b) {
        const u32x4* r = recs + (size_t)t * LEN;
#pragma unroll
        for (uint32_t i = 0; i < OPS / 256; ++i)
            __builtin_amdgcn_global_load_lds((gptr_t)((const uint8_t*)(r + 256 * i + 64 * w) + lane * 16),
                                             (lptr_t)&lds[b][256 * i + 64 * w], 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr_t)((const uint8_t*)(r + OPS + 16 * w) + lane * 4),
                                         (lptr_t)&lds[b][OPS + 16 * w], 4, 0, 0);
    };
    if (t0 < t1) copy(t0, 0);
    // the query operands: d = 16s + 8h .. of column j
    const float* qp = a.q + ((size_t)(bt * a.q_len + row) * a.H + head) * HD;
    h8_t qh[KS], ql[KS];
    int eq;
    {
        float x[KS][8], mx = 0.0f;
#pragma unroll
        for (uint32_t s = 0; s < KS; ++s)
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) {
                x[s][i] = ((const f32x4*)(qp + 16 * s + 8 * h))[i / 4][i % 4];
                mx = fmaxf(mx, fabsf(x[s][i]));
            }
        eq = pf_exp(fmaxf(mx, __shfl_xor(mx, 32, 64)));
#pragma unroll
        for (uint32_t s = 0; s < KS; ++s) pf_split(x[s], pf_pow2(eq), qh[s], ql[s]);
    }
    f16v acc[NB];
#pragma unroll
    for (uint32_t b = 0; b < NB; ++b) acc[b] = f16v{};
    const float NEG = -__builtin_huge_valf();
    // a column's reference, near its largest score so far, in units of log 2,
    // and what is taken off its scores (0 while nothing is seen)
    float m = NEG, md = 0.0f, l = 0.0f;
    const float scale2 = a.scale * 1.44269504f, qf = scale2 * pf_pow2(-eq);
    for (uint32_t t = t0; t < t1; ++t) {
        const uint32_t buf = (t - t0) & 1, p0 = t * 32;
        if (t + 1 < t1) {
            copy(t + 1, buf ^ 1);
            __builtin_amdgcn_s_waitcnt(((OPS / 256 + 1) & 15) | 7 << 4 | 15 << 8);
        } else {
            __builtin_amdgcn_s_waitcnt(0 | 7 << 4 | 15 << 8);
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (p0 < Lw) {
            const h8_t* op = (const h8_t*)lds[buf] + lane;
            const float* tail = (const float*)&lds[buf][OPS];
            const bool plain = __builtin_amdgcn_readfirstlane(((const int*)tail)[kTailBad]) != 0;
            // (values above 2^95 leave the sums no room for weights above 1)
            const float grow = plain || __builtin_amdgcn_readfirstlane(((const int*)tail)[kTailMax]) < -80 ? 0.0f : 8.0f;
            float sv[16], tmax = NEG;
            if (!plain) {
                f16v s0 = {}, s1 = {};
                h8_t k[PF][2];
#pragma unroll
                for (uint32_t s = 0; s < PF - 1; ++s) k[s][0] = op[2 * s * 64], k[s][1] = op[(2 * s + 1) * 64];
#pragma unroll
                for (uint32_t s = 0; s < KS; ++s) {
                    const uint32_t n = s + PF - 1;
                    if (n < KS) k[n % PF][0] = op[2 * n * 64], k[n % PF][1] = op[(2 * n + 1) * 64];
                    __builtin_amdgcn_sched_barrier(0);
                    s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(k[s % PF][1], qh[s], s1, 0, 0, 0);
                    s0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(k[s % PF][0], qh[s], s0, 0, 0, 0);
                    s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(k[s % PF][0], ql[s], s1, 0, 0, 0);
                }
#pragma unroll
                for (uint32_t i = 0; i < 16; ++i) sv[i] = (s0[i] + s1[i]) * (qf * tail[kTailK + 8 * (i / 4) + 4 * h + i % 4]);
            } else {
#pragma unroll
                for (uint32_t i = 0; i < 16; ++i) {
                    const uint32_t p = min(p0 + 8 * (i / 4) + 4 * h + i % 4, a.kv - 1);
                    const float* kp = a.kc + ((size_t)seq * a.stride + p) * HD;
                    float s = 0.0f;
#pragma unroll 1
                    for (uint32_t d = 0; d < HD; ++d) s = fmaf(kp[d], qp[d], s);
                    sv[i] = s * scale2;
                }
            }
            if (p0 + 32 > Lf) {  // (records that every column of the wave sees whole need no mask)
#pragma unroll
                for (uint32_t i = 0; i < 16; ++i) sv[i] = p0 + 8 * (i / 4) + 4 * h + i % 4 < lim ? sv[i] : NEG;
            }
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i) tmax = fmaxf(tmax, sv[i]);
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
            // a new reference only where the largest score has grown by 2^8
            // (the weights then stay below 2^8): the sums are seldom rescaled
            if (__builtin_amdgcn_ballot_w64(tmax > m + grow)) {
                const float m_new = fmaxf(m, tmax), md_new = m_new == NEG ? 0.0f : m_new;
                // (nothing seen yet: the sums are zeros)
                const float alpha = m == NEG ? 0.0f : __builtin_amdgcn_exp2f(md - md_new);
                l *= alpha;
#pragma unroll
                for (uint32_t b = 0; b < NB; ++b) acc[b] *= alpha;
                m = m_new;
                md = md_new;
            }
            float p[16];
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i) {
                p[i] = __builtin_amdgcn_exp2f(sv[i] - md);
                l += p[i];
            }
            if (!plain) {
                const h8_t* vo = op + OPS / 2;
                auto piece = [&](uint32_t n, h8_t (&v)[2]) {
                    v[0] = vo[n * 128];
                    v[1] = vo[n * 128 + 64];
                };
                h8_t v[PF][2], ph[2], pl[2];
#pragma unroll
                for (uint32_t n = 0; n < PF - 1; ++n) piece(n, v[n]);
                float wmax = 0.0f;
#pragma unroll
                for (uint32_t i = 0; i < 16; ++i) {
                    p[i] *= tail[kTailV + 8 * (i / 4) + 4 * h + i % 4];
                    wmax = fmaxf(wmax, p[i]);
                }
                // (at least -111: below, f32 itself has no more bits)
                const int ew = max(-111, __builtin_amdgcn_frexp_expf(fmaxf(wmax, __shfl_xor(wmax, 32, 64))));
                const float pf = pf_pow2(15 - ew), of = pf_pow2(ew - 15);
#pragma unroll
                for (uint32_t s = 0; s < 2; ++s) {
                    float ps[8];
#pragma unroll
                    for (uint32_t i = 0; i < 8; ++i) ps[i] = p[8 * s + i];
                    pf_split(ps, pf, ph[s], pl[s]);
                }
#pragma unroll
                for (uint32_t b = 0; b < NB; ++b) {
                    f16v o = {};
#pragma unroll
                    for (uint32_t s = 0; s < 2; ++s) {
                        const uint32_t n = 2 * b + s;
                        if (n + PF - 1 < 2 * NB) piece(n + PF - 1, v[(n + PF - 1) % PF]);
                        __builtin_amdgcn_sched_barrier(0);
                        o = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[n % PF][1], ph[s], o, 0, 0, 0);
                        o = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[n % PF][0], pl[s], o, 0, 0, 0);
                        o = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[n % PF][0], ph[s], o, 0, 0, 0);
                    }
#pragma unroll
                    for (uint32_t i = 0; i < 16; ++i) acc[b][i] = fmaf(o[i], of, acc[b][i]);
                }
            } else {
#pragma unroll
                for (uint32_t i = 0; i < 16; ++i) {
                    const float mine = p[i], other = __shfl_xor(mine, 32, 64);
#pragma unroll
                    for (uint32_t o = 0; o < 2; ++o) {  // the positions of both halves
                        const uint32_t pos = p0 + 8 * (i / 4) + 4 * o + i % 4;
                        if (pos >= lim) continue;  // (0·inf is none of its column's)
                        const float pp = o == h ? mine : other;
                        const float* vp = a.vc + ((size_t)seq * a.stride + pos) * HD + 4 * h;
#pragma unroll
                        for (uint32_t b = 0; b < NB; ++b)
#pragma unroll
                            for (uint32_t r = 0; r < 16; ++r)
                                acc[b][r] = fmaf(pp, vp[32 * b + 8 * (r / 4) + r % 4], acc[b][r]);
                    }
                }
            }
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0 << 8 | 7 << 4 | 15 | 3 << 14);  // (LDS reads done)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
    l += __shfl_xor(l, 32, 64);
    if (c >= R) return;
    const size_t slot = (((size_t)seq * a.cbs + cb) * a.nsp + sp) * 128 + 32 * w + j;
    float* o = a.nsp == 1 ? a.out + ((size_t)(bt * a.q_len + row) * a.H + head) * HD : a.part + slot * HD;
#pragma unroll
    for (uint32_t b = 0; b < NB; ++b)
#pragma unroll
        for (uint32_t g = 0; g < 4; ++g) {
            f32x4 v;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) v[i] = acc[b][4 * g + i];
            *(f32x4*)(o + 32 * b + 8 * g + 4 * h) = a.nsp == 1 ? v / l : v;
        }
    if (a.nsp > 1 && h == 0) {
        a.ml[slot * 2] = m == NEG ? NEG : md;
        a.ml[slot * 2 + 1] = l;
    }
}

// o = Σ o_s·2^(m_s−M) / Σ l_s·2^(m_s−M) over the ranges, in range order: a
// thread four elements of a column, their loads all in flight
template <int HD>
RT_DEV void attn_pf_merge(const AttnPfArgs& a) {
    const uint32_t G = a.H / a.KVH, R = a.q_len * G;
    const uint32_t e = blockIdx.x * 256 + threadIdx.x, c = e / (HD / 4), d = e % (HD / 4) * 4;
    if (c >= R) return;
    const size_t seq = (size_t)blockIdx.z * a.KVH + blockIdx.y;
    const size_t slot = (seq * a.cbs + c / 128) * a.nsp * 128 + c % 128;
    float mj[RT_ATTN_MQ_NSP_MAX], lj[RT_ATTN_MQ_NSP_MAX], M = -__builtin_huge_valf();
    f32x4 oj[RT_ATTN_MQ_NSP_MAX];
#pragma unroll
    for (uint32_t s = 0; s < RT_ATTN_MQ_NSP_MAX; ++s) {
        const size_t k = slot + 128 * min(s, a.nsp - 1);
        mj[s] = a.ml[2 * k];
        lj[s] = a.ml[2 * k + 1];
        oj[s] = *(const f32x4*)(a.part + k * HD + d);
    }
#pragma unroll
    for (uint32_t s = 0; s < RT_ATTN_MQ_NSP_MAX; ++s) M = fmaxf(M, mj[s]);
    float L = 0.0f;
    f32x4 o = {0, 0, 0, 0};
#pragma unroll
    for (uint32_t s = 0; s < RT_ATTN_MQ_NSP_MAX; ++s) {
        // (an empty range adds zeros; one that the others outweigh its NaN, if it has one)
        const float f = mj[s] == -__builtin_huge_valf() ? 0.0f : __builtin_amdgcn_exp2f(mj[s] - M);
        L += s < a.nsp ? f * lj[s] : 0.0f;
        o += s < a.nsp ? f * oj[s] : f32x4{0, 0, 0, 0};
    }
    const uint32_t row = c / G, head = blockIdx.y * G + c % G;
    *(f32x4*)(a.out + ((size_t)(blockIdx.z * a.q_len + row) * a.H + head) * HD + d) = o / L;
}

#define RT_ATTN_PF_KERNELS(HD)                                                                        \
    extern "C" __global__ void __launch_bounds__(2 * HD) k_attn_pf_prep_hd##HD(AttnPfArgs a) {       \
        attn_pf_prep<HD>(a);                                                                          \
    }                                                                                                 \
    extern "C" __global__ void __launch_bounds__(256, 2) k_attn_pf_f32_hd##HD(AttnPfArgs a) {        \
        attn_pf<HD>(a);                                                                               \
    }                                                                                                 \
    extern "C" __global__ void __launch_bounds__(256) k_attn_pf_merge_hd##HD(AttnPfArgs a) {         \
        attn_pf_merge<HD>(a);                                                                         \
    }
RT_ATTN_PF_KERNELS(64)
RT_ATTN_PF_KERNELS(128)
