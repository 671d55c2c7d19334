// k_gemmw.hip — batched GEMM of more than 32 activation rows (prompts, large
// batches), Y[M,N] = X[M,K]·W[N,K]ᵀ with W in the GGUF block formats (new: the
// reference's only M > 1 path is gemm_f16 on f16-dequantised weights,
// gemm.metal:39-190, called from verify_draft, forward.rs:2193-2271).
//
// A workgroup's tile is 256 weight rows × 64 activation rows: four waves of 64
// weight rows each, all 64 activation rows.  The activations, prepared as f16
// pairs hi + lo in MFMA order (prep_row below), go from memory
// straight to LDS in stages of 64 elements of K; every wave
// reads all of a stage, one read feeding two v_mfma_f32_32x32x16_f16.  The
// weights need no LDS: each lane loads its own weight row's bytes and decodes
// them to the operand it feeds, once per 64 activation rows (the 32-row tiles
// of k_gemm3_* decode them once per 32 and stage both sides through registers
// and LDS).
//
// Bound: matrix cores.  Each product costs two MFMAs (hi and lo), 2·2·M·N·K
// operations; without its weight loads the kernel runs at 1.05-1.13 PFLOP/s of
// them at 512×16384×4096, a large f16 product of the library at 1.2.  With
// them: Q4_K 840 TFLOP/s, Q4_0 870, Q8_0 750, Q6_K 720 (preparation included;
// k_gemm3_*: 350-490).  A lone workgroup on a CU is bound by its waves' own
// chain (1.3 µs a stage), which the loads two stages ahead keep fed: Q8_0
// 64×3584×3584 26.2 → 24.2 µs, Q6_K 37×3584×18944 60.5 → 55.4 against loads
// one stage ahead; with two workgroups on every CU the two are level.
#include <type_traits>
#include "rt_formats.h"
#include "rt_gemm.h"
#include "rt_shared.h"

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

// ───────────────────────────── weight decoding ─────────────────────────────
//
// Lane l of a wave decodes weight row l % 32 of a 32-row tile.  A stage is 64
// elements of K, two records of 32; MFMA p (0, 1) of a record takes its
// elements 16p .. 16p + 15, of which the lanes of half h = l / 32 hold 8h ..
// 8h + 7, in the order 0 2 1 3 4 6 5 7 (the prepared activations have the
// same order): two codes 16 bits apart in a dword then need one and-or to
// become an f16 pair 1024 + code.

RT_DEV h2_t as_h2(uint32_t u) { return __builtin_bit_cast(h2_t, u); }
RT_DEV uint32_t as_u(h2_t h) { return __builtin_bit_cast(uint32_t, h); }
RT_DEV h2_t h2_splat(float f) { return h2_t{(_Float16)f, (_Float16)f}; }
RT_DEV h2_t h2_fma(h2_t a, h2_t b, h2_t c) { return __builtin_elementwise_fma(a, b, c); }
RT_DEV h8_t h8_of(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(h8_t, u32x4{a, b, c, d});
}
constexpr uint32_t K1024 = 0x64006400u;  // f16 pair 1024, 1024 (one unit in the last place = 1)

// The halves of a 16-byte piece (dwords 0, 1 | 2, 3) that two lanes 32 apart
// hold become element groups p = 0 (both lanes' first halves) and p = 1.
RT_DEV void swap_halves(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
RT_DEV void swap_piece(u32x4& q) {
    uint32_t x = q.x, y = q.y, z = q.z, w = q.w;
    swap_halves(x, z);
    swap_halves(y, w);
    q = u32x4{x, y, z, w};
}
// f16 operand of the unsigned byte codes of two dwords, minus `off`
RT_DEV h8_t bytes_to_h8(uint32_t q0, uint32_t q1, float off) {
    const h2_t o = h2_splat(1024.0f + off);
    auto even = [&](uint32_t q) { return as_u(as_h2((q & 0x00FF00FFu) | K1024) - o); };
    auto odd = [&](uint32_t q) { return as_u(as_h2(__builtin_amdgcn_perm(K1024, q, 0x05030501u)) - o); };
    return h8_of(even(q0), odd(q0), even(q1), odd(q1));
}
// f16 operand sc·(code − MID) of the low nibbles of two dwords (HI: the high
// ones), ORed with a fifth bit each in f (at bit 4, or 8 with HI; in dword
// order).  An integer of at most 10 bits, exact.
template <int HI, int MID>
RT_DEV h8_t nibs_to_h8(uint32_t q0, uint32_t q1, h2_t sc, u32x4 f) {
    constexpr uint32_t MASK = HI ? 0x00F000F0u : 0x000F000Fu;
    auto cv = [&](uint32_t q, uint32_t fb) {
        const h2_t v = as_h2((q & MASK) | K1024 | fb);  // 1024 + code (HI: + 16·code)
        const h2_t c = HI ? h2_fma(v, h2_splat(0.0625f), h2_splat(-64.0f - MID)) : v - h2_splat(1024.0f + MID);
        return as_u(c * sc);
    };
    return h8_of(cv(q0, f.x), cv(q0 >> 8, f.y), cv(q1, f.z), cv(q1 >> 8, f.w));
}

// A format's Raw holds what one lane needs of one weight row for one stage.
// Super-block formats with mins (CHAIN): pair<US>() gives the operands sc·(code
// − MID) of stage US, and one MFMA accumulator runs over two stages; y +=
// d·(acc + MID·Σ sc·Σx) − dmin·Σ m·Σx, the sums over the super-block's records
// MFMAs over their activation sums.  The matrix cores drop low bits of a
// growing sum, so its length and size count: chains of 256 over uncentred
// codes were 4.1e-7 off at K = 512 (record by record sums: 2.0e-7).
// Other formats: operands code, scales sc[p] applied per record (per 16
// elements with HALF).
//
// Loads.  What bounds them is the number of load instructions (each touches
// the lines of 32 rows), and misaligned ones cost about twice: formats of
// 2-byte aligned blocks read dword-aligned windows (rows of an even number of
// blocks, OA; a stage is then dword-aligned) and shift in registers, and a
// dword that all lanes of a row need is loaded for the first tile by the
// lanes of half 0 and for the second by half 1 (rowx, Sh).  Q8_0 / Q6_K at
// 512×16384×4096: 262 / 251 µs with misaligned 16-byte loads and 2-byte
// loads of the scales, 131 / 121 µs without any weight loads.
// The lower / upper half-wave's value in all lanes.
RT_DEV void both_halves(uint32_t v, uint32_t& lo, uint32_t& hi) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    lo = r[0];
    hi = r[1];
}
// Of a format: Q, stages of a block (1: blocks of 32); LU, stages that one
// load() covers; LOADS, the fewest load instructions it can compile to.
// A lane's weight row: a wave-uniform base and the lane's 32-bit offset, so
// that the loads take a scalar base and no 64-bit vector arithmetic
struct Row {
    const uint8_t* base;
    uint32_t off;
};
struct NoSh {};
template <bool OA>
struct WQ8_0T {
    static constexpr uint32_t BLK_BYTES = 34, Q = 1, LU = 1, LOADS = OA ? 5 : 8;
    static constexpr bool CHAIN = false, HALF = false, TAIL = false;
    struct Raw {
        u32x4 q[2];
        uint32_t d[2];
    };
    struct Sh {
        uint32_t l;
    };
    RT_DEV static void load(Raw (&r)[2], Sh& s, const Row (&row)[2], const uint8_t* rowx,
                            uint32_t st, uint32_t h, uint32_t nblk) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            if (OA) {
                const uint8_t* b = row[nt].base + (size_t)st * 68;
                const uint32_t o = row[nt].off + 16 * h;
                r[nt].q[0] = *(const u32x4_a4*)(b + o);       // block 0: bytes 16h .. 16h + 15
                r[nt].q[1] = *(const u32x4_a4*)(b + 36 + o);  // block 1's codes
            } else {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const uint8_t* b = row[nt].base + (size_t)min(2 * st + i, nblk - 1) * 34 + row[nt].off;
                    r[nt].q[i] = *(const u32x4_a2*)(b + 2 + 16 * h);
                    r[nt].d[i] = *(const uint16_t*)b;
                }
            }
        }
        if (OA) s.l = *(const uint32_t*)(rowx + (size_t)st * 68 + 32);
    }
    // the codes and scales in place (nt: the lane's tile)
    RT_DEV static void arrange(Raw& r, const Sh& s, int nt, uint32_t, uint32_t h) {
        if (!OA) return;
        uint32_t l0, l1, x0, x1;
        both_halves(s.l, l0, l1);
        const uint32_t l = nt ? l1 : l0;  // codes 30, 31 of block 0 and block 1's scale
        both_halves(r.q[0].x, x0, x1);
        const u32x4 q = r.q[0];
        const uint32_t nx = h ? l : x1;
        r.q[0] = u32x4{alignb(q.y, q.x, 2), alignb(q.z, q.y, 2), alignb(q.w, q.z, 2), alignb(nx, q.w, 2)};
        r.d[0] = x0;
        r.d[1] = l >> 16;
    }
    template <int US>
    RT_DEV static void rec(const Raw& r, int i, uint32_t, h8_t B[2], float sc[2]) {
        u32x4 q = r.q[i] ^ 0x80808080u;
        swap_piece(q);
        B[0] = bytes_to_h8(q.x, q.y, 128.0f);
        B[1] = bytes_to_h8(q.z, q.w, 128.0f);
        sc[0] = h2f(r.d[i]);
    }
};
// 4-bit codes: value d·(q − 8).  ggml layout (G): byte j holds elements j and
// j + 16; reference layout: byte i holds elements 2i and 2i + 1.
template <bool G, bool OA>
struct WQ4_0T {
    static constexpr uint32_t BLK_BYTES = 18, Q = 1, LU = 1, LOADS = OA ? 4 : 8;
    static constexpr bool CHAIN = false, HALF = false, TAIL = false;
    struct Raw {
        uint32_t q[2][2], e;
        uint32_t d[2];
    };
    using Sh = NoSh;
    RT_DEV static void load(Raw (&r)[2], Sh&, const Row (&row)[2], const uint8_t*,
                            uint32_t st, uint32_t h, uint32_t nblk) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            if (OA) {
                const uint32_t* b = (const uint32_t*)(row[nt].base + (size_t)st * 36 + (row[nt].off + 8 * h));
                r[nt].q[0][0] = b[0];
                r[nt].q[0][1] = b[1];
                r[nt].e = b[2];
                r[nt].q[1][0] = b[5];
                r[nt].q[1][1] = b[6];
            } else {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const uint8_t* b = row[nt].base + (size_t)min(2 * st + i, nblk - 1) * 18 + row[nt].off;
                    const u32x2_a2 v = *(const u32x2_a2*)(b + 2 + 8 * h);
                    r[nt].q[i][0] = v.x;
                    r[nt].q[i][1] = v.y;
                    r[nt].d[i] = *(const uint16_t*)b;
                }
            }
        }
    }
    RT_DEV static void arrange(Raw& r, const Sh&, int, uint32_t, uint32_t) {
        if (!OA) return;
        uint32_t x0, x1, e0, e1;
        both_halves(r.q[0][0], x0, x1);  // (half 0: block 0's scale)
        both_halves(r.e, e0, e1);        // (half 1: block 1's scale)
        const uint32_t a = r.q[0][0], b = r.q[0][1];
        r.q[0][0] = alignb(b, a, 2);
        r.q[0][1] = alignb(r.e, b, 2);
        r.d[0] = x0;
        r.d[1] = e1 >> 16;
    }
    template <int US>
    RT_DEV static void rec(const Raw& r, int i, uint32_t, h8_t B[2], float sc[2]) {
        const h2_t ol = h2_splat(1032.0f), oh = h2_splat(-72.0f), s16 = h2_splat(0.0625f);
        auto lo = [&](uint32_t q) { return as_u(as_h2((q & 0x000F000Fu) | K1024) - ol); };
        auto hi = [&](uint32_t q) { return as_u(h2_fma(as_h2((q & 0x00F000F0u) | K1024), s16, oh)); };
        uint32_t a = r.q[i][0], b = r.q[i][1];
        if (G) {
            B[0] = h8_of(lo(a), lo(a >> 8), lo(b), lo(b >> 8));
            B[1] = h8_of(hi(a), hi(a >> 8), hi(b), hi(b >> 8));
        } else {
            swap_halves(a, b);  // the dwords of MFMA 0 / 1
            auto op = [&](uint32_t q) {
                const uint32_t t = __builtin_amdgcn_perm(0u, q, 0x04010400u),
                               u = __builtin_amdgcn_perm(0u, q, 0x04030402u);
                return h8_of(lo(t), hi(t), lo(u), hi(u));
            };
            B[0] = op(a);
            B[1] = op(b);
        }
        sc[0] = h2f(r.d[i]);
    }
};
// bits 0..7 of b as fifth bits of 8 codes in operand order, at bit `at` of
// each 16-bit half
RT_DEV u32x4 spread_bits(uint32_t b, uint32_t at) {
    auto two = [&](uint32_t x, uint32_t lo, uint32_t hi) {
        return ((x >> lo & 1u) << at) | ((x >> hi & 1u) << (at + 16));
    };
    return u32x4{two(b, 0, 2), two(b, 1, 3), two(b, 4, 6), two(b, 5, 7)};
}
template <bool OA>
struct WQ5_0T {  // value d·(q − 16); bit j of qh is the fifth bit of element j
    static constexpr uint32_t BLK_BYTES = 22, Q = 1, LU = 1, LOADS = OA ? 6 : 12;
    static constexpr bool CHAIN = false, HALF = false, TAIL = false;
    struct Raw {
        uint32_t q[2][2], e, f;
        uint32_t qh[2], d[2];
    };
    using Sh = NoSh;
    RT_DEV static void load(Raw (&r)[2], Sh&, const Row (&row)[2], const uint8_t*,
                            uint32_t st, uint32_t h, uint32_t nblk) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            if (OA) {
                const uint8_t* u = row[nt].base + (size_t)st * 44;
                const uint32_t* b = (const uint32_t*)(u + (row[nt].off + 8 * h));
                r[nt].q[0][0] = b[1];
                r[nt].q[0][1] = b[2];
                r[nt].e = b[3];
                r[nt].q[1][0] = b[7];
                r[nt].q[1][1] = b[8];
                r[nt].f = *(const uint32_t*)(u + (row[nt].off + 24 * h));  // dword 0 | dword 6
            } else {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const uint8_t* b = row[nt].base + (size_t)min(2 * st + i, nblk - 1) * 22 + row[nt].off;
                    const u32x2_a2 v = *(const u32x2_a2*)(b + 6 + 8 * h);
                    r[nt].q[i][0] = v.x;
                    r[nt].q[i][1] = v.y;
                    r[nt].qh[i] = *(const u32_a2*)(b + 2);
                    r[nt].d[i] = *(const uint16_t*)b;
                }
            }
        }
    }
    RT_DEV static void arrange(Raw& r, const Sh&, int, uint32_t, uint32_t) {
        if (!OA) return;
        uint32_t x0, x1, e0, e1, f0, f1;
        both_halves(r.q[0][0], x0, x1);  // dword 1 | dword 3
        both_halves(r.e, e0, e1);        // dword 3 | dword 5
        both_halves(r.f, f0, f1);
        const uint32_t a = r.q[0][0], b = r.q[0][1];
        r.q[0][0] = alignb(b, a, 2);
        r.q[0][1] = alignb(r.e, b, 2);
        r.d[0] = f0;
        r.qh[0] = alignb(x0, f0, 2);
        r.d[1] = e1 >> 16;
        r.qh[1] = f1;
    }
    template <int US>
    RT_DEV static void rec(const Raw& r, int i, uint32_t h, h8_t B[2], float sc[2]) {
        const h2_t ol = h2_splat(1040.0f), oh = h2_splat(-80.0f), s16 = h2_splat(0.0625f);
        const uint32_t a = r.q[i][0], b = r.q[i][1];
        const uint32_t hb = r.qh[i] >> (8 * h);
        auto lo = [&](uint32_t v, uint32_t f) { return as_u(as_h2((v & 0x000F000Fu) | K1024 | f) - ol); };
        auto hi = [&](uint32_t v, uint32_t f) {
            return as_u(h2_fma(as_h2((v & 0x00F000F0u) | K1024 | f), s16, oh));
        };
        const u32x4 f0 = spread_bits(hb, 4), f1 = spread_bits(hb >> 16, 8);
        B[0] = h8_of(lo(a, f0.x), lo(a >> 8, f0.y), lo(b, f0.z), lo(b >> 8, f0.w));
        B[1] = h8_of(hi(a, f1.x), hi(a >> 8, f1.y), hi(b, f1.z), hi(b >> 8, f1.w));
        sc[0] = h2f(r.d[i]);
    }
};
// Scale slot of a record of Q4_K / Q5_K: 2j + hi in ggml's layout, j + 4·hi
// in the reference's; sub-block scales / mins as packed 6-bit fields.
template <bool G>
struct KQ {
    template <int R>
    RT_DEV static uint32_t scale(u32x4 hdr) {
        constexpr int SLOT = G ? R : R / 2 + 4 * (R & 1), B = 8 * (SLOT & 3);
        return SLOT < 4 ? (hdr.y >> B) & 63u : ((hdr.w >> B) & 15u) | ((hdr.y >> (B + 2)) & 0x30u);
    }
    template <int R>
    RT_DEV static h2_t scale2(u32x4 hdr) { return as_h2(scale<R>(hdr) * 0x10001u + K1024) - h2_splat(1024.0f); }
    // operands of eight per-record values (bytes of slots 0..3, 4..7), in the
    // order 0 2 1 3 4 6 5 7 of the records: the mins, and the scales times f
    RT_DEV static h8_t by_record(uint32_t a, uint32_t b, float f) {
        const h2_t o = h2_splat(1024.0f), m = h2_splat(f);
        auto pr = [&](uint32_t v, uint32_t sel) { return as_u((as_h2(__builtin_amdgcn_perm(K1024, v, sel)) - o) * m); };
        if (G) return h8_of(pr(a, 0x05020500u), pr(a, 0x05030501u), pr(b, 0x05020500u), pr(b, 0x05030501u));
        return h8_of(pr(a, 0x05010500u), pr(b, 0x05010500u), pr(a, 0x05030502u), pr(b, 0x05030502u));
    }
    RT_DEV static h8_t mins(u32x4 hdr) {
        return by_record(hdr.z & 0x3F3F3F3Fu, ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u), 1.0f);
    }
    RT_DEV static h8_t scales(u32x4 hdr, float f) {
        return by_record(hdr.y & 0x3F3F3F3Fu, (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u), f);
    }
};
template <bool G>
struct WQ4KT {
    static constexpr uint32_t BLK_BYTES = 144, Q = 4, LU = 1, LOADS = 2;
    static constexpr int MID = 8;  // centre of the codes
    static constexpr bool CHAIN = true, HALF = false, TAIL = false;
    struct Raw {
        u32x4 q;
    };
    using Sh = NoSh;
    RT_DEV static void load(Raw (&r)[2], Sh&, const Row (&row)[2], const uint8_t*,
                            uint32_t st, uint32_t h, uint32_t) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
            r[nt].q = *(const u32x4*)(row[nt].base + (size_t)(st / 4) * 144 + 16 + 32 * (st % 4) + (row[nt].off + 16 * h));
    }
    RT_DEV static void arrange(Raw&, const Sh&, int, uint32_t, uint32_t) {}
    // both records of the stage: low nibbles (record 2US) and high (2US + 1)
    template <int US>
    RT_DEV static void pair(const Raw& r, u32x4 hdr, uint32_t, h8_t B[2][2]) {
        u32x4 q = r.q;
        swap_piece(q);
        const h2_t s0 = KQ<G>::template scale2<2 * US>(hdr), s1 = KQ<G>::template scale2<2 * US + 1>(hdr);
        const u32x4 z = {0, 0, 0, 0};
        B[0][0] = nibs_to_h8<0, MID>(q.x, q.y, s0, z);
        B[0][1] = nibs_to_h8<0, MID>(q.z, q.w, s0, z);
        B[1][0] = nibs_to_h8<1, MID>(q.x, q.y, s1, z);
        B[1][1] = nibs_to_h8<1, MID>(q.z, q.w, s1, z);
    }
    using K = KQ<G>;
};
template <bool G>
struct WQ5KT {
    static constexpr uint32_t BLK_BYTES = 176, Q = 4, LU = 1, LOADS = 4;
    static constexpr int MID = 16;  // centre of the codes
    static constexpr bool CHAIN = true, HALF = false, TAIL = false;
    struct Raw {
        u32x4 q, qh;  // (reference layout: two dwords of qh)
    };
    using Sh = NoSh;
    RT_DEV static void load(Raw (&r)[2], Sh&, const Row (&row)[2], const uint8_t*,
                            uint32_t st, uint32_t h, uint32_t) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const uint8_t* b = row[nt].base + (size_t)(st / 4) * 176;
            const uint32_t o = row[nt].off;
            r[nt].q = *(const u32x4*)(b + 48 + 32 * (st % 4) + (o + 16 * h));
            if (G) {
                r[nt].qh = *(const u32x4*)(b + 16 + (o + 16 * h));
            } else {
                const uint2 t = *(const uint2*)(b + 16 + 8 * (st % 4) + o);
                r[nt].qh = u32x4{t.x, t.y, 0, 0};
            }
        }
    }
    RT_DEV static void arrange(Raw&, const Sh&, int, uint32_t, uint32_t) {}
    template <int US>
    RT_DEV static void pair(const Raw& r, u32x4 hdr, uint32_t h, h8_t B[2][2]) {
        u32x4 q = r.q;
        swap_piece(q);
        const h2_t s0 = KQ<G>::template scale2<2 * US>(hdr), s1 = KQ<G>::template scale2<2 * US + 1>(hdr);
        u32x4 f[2][2];
        if (G) {  // bit 2US (+ 1) of byte l for element l of the records
            u32x4 v = r.qh;
            swap_piece(v);
            auto at = [&](uint32_t x, int from, int to) {
                return to >= from ? (x << (to - from)) & (0x00010001u << to) : (x >> (from - to)) & (0x00010001u << to);
            };
            const uint32_t w[2][2] = {{v.x, v.y}, {v.z, v.w}};
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                f[0][p] = u32x4{at(w[p][0], 2 * US, 4), at(w[p][0] >> 8, 2 * US, 4),
                                at(w[p][1], 2 * US, 4), at(w[p][1] >> 8, 2 * US, 4)};
                f[1][p] = u32x4{at(w[p][0], 2 * US + 1, 8), at(w[p][0] >> 8, 2 * US + 1, 8),
                                at(w[p][1], 2 * US + 1, 8), at(w[p][1] >> 8, 2 * US + 1, 8)};
            }
        } else {  // byte 4·record + 2p + h holds the bits of elements 16p + 8h ..
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                f[0][p] = spread_bits(r.qh.x >> (16 * p + 8 * h), 4);
                f[1][p] = spread_bits(r.qh.y >> (16 * p + 8 * h), 8);
            }
        }
        B[0][0] = nibs_to_h8<0, MID>(q.x, q.y, s0, f[0][0]);
        B[0][1] = nibs_to_h8<0, MID>(q.z, q.w, s0, f[0][1]);
        B[1][0] = nibs_to_h8<1, MID>(q.x, q.y, s1, f[1][0]);
        B[1][1] = nibs_to_h8<1, MID>(q.z, q.w, s1, f[1][1]);
    }
    using K = KQ<G>;
};
// Q6_K: record t of half hs holds ((ql[64hs + 32(t & 1) + l] >> 4(t >> 1)) & 15)
// | ((qh[32hs + l] >> 2t) & 3) << 4, minus 32; scale slot 8hs + 2t (+ 1 for
// l ≥ 16 in ggml's layout).  Stage US of a super-block: hs = US / 2, t =
// 2(US & 1), + 1.
// The stages 2i and 2i + 1 of a half read the same bytes: one load for both
// (LU = 2).  A super-block starts at a multiple of 2: where that is none of 4
// (sh = 2) its windows start 2 bytes earlier, and the last 2 bytes of a
// lane's piece come from the next piece's first dword, in the other half's
// register, the last piece's from Sh.
template <bool G, bool OA>
struct WQ6KT {
    static constexpr uint32_t BLK_BYTES = 210, Q = 4, LU = 2, LOADS = OA ? 8 : 6;
    static constexpr bool CHAIN = false, HALF = G, TAIL = true;
    struct Raw {
        u32x4 l[2], h;
    };
    struct Sh {
        uint32_t l, h;
    };
    RT_DEV static void load(Raw (&r)[2], Sh& s, const Row (&row)[2], const uint8_t* rowx,
                            uint32_t st, uint32_t h, uint32_t) {
        const uint32_t sb = st / 4, hs = (st % 4) / 2, sh = OA ? 2 * (sb & 1) : 0;
        const size_t o = (size_t)sb * 210 - sh;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const uint8_t* b = row[nt].base + o;
            const uint32_t ro = row[nt].off + 16 * h;
            if (OA) {
                r[nt].l[0] = *(const u32x4_a4*)(b + 64 * hs + ro);
                r[nt].l[1] = *(const u32x4_a4*)(b + 64 * hs + 32 + ro);
                r[nt].h = *(const u32x4_a4*)(b + 128 + 32 * hs + ro);
            } else {
                r[nt].l[0] = *(const u32x4_a2*)(b + 64 * hs + ro);
                r[nt].l[1] = *(const u32x4_a2*)(b + 64 * hs + 32 + ro);
                r[nt].h = *(const u32x4_a2*)(b + 128 + 32 * hs + ro);
            }
        }
        if (OA) {
            s.l = *(const uint32_t*)(rowx + o + 64 * hs + 64);
            s.h = *(const uint32_t*)(rowx + o + 160 + 32 * hs);
        }
    }
    RT_DEV static void arrange(Raw& r, const Sh& s, int nt, uint32_t st, uint32_t h) {
        if (!OA) return;
        const uint32_t sh = 2 * ((st / 4) & 1);
        uint32_t a0, a1, b0, b1, c0, c1, l[2], g[2];
        both_halves(r.l[0].x, a0, a1);
        both_halves(r.l[1].x, b0, b1);
        both_halves(r.h.x, c0, c1);
        both_halves(s.l, l[0], l[1]);
        both_halves(s.h, g[0], g[1]);
        auto shift = [&](u32x4& q, uint32_t nx) {
            q = u32x4{alignb(q.y, q.x, sh), alignb(q.z, q.y, sh), alignb(q.w, q.z, sh), alignb(nx, q.w, sh)};
        };
        shift(r.l[0], h ? b0 : a1);
        shift(r.l[1], h ? l[nt] : b1);
        shift(r.h, h ? g[nt] : c1);
    }
    // scales and d of a super-block: half h loads those of tile h
    struct Tail {
        u32x4 sc;
        uint32_t d;
    };
    RT_DEV static void load_tail(Tail& t, const uint8_t* rowx, uint32_t st) {
        const uint8_t* b = rowx + (size_t)(st / 4) * 210;
        t.sc = *(const u32x4_a2*)(b + 192);
        t.d = *(const uint16_t*)(b + 208);
    }
    RT_DEV static void spread_tail(const Tail& t, Tail (&x)[2]) {
        uint32_t lo, hi;
        auto two = [&](uint32_t v) { both_halves(v, lo, hi); };
        two(t.sc.x); x[0].sc.x = lo; x[1].sc.x = hi;
        two(t.sc.y); x[0].sc.y = lo; x[1].sc.y = hi;
        two(t.sc.z); x[0].sc.z = lo; x[1].sc.z = hi;
        two(t.sc.w); x[0].sc.w = lo; x[1].sc.w = hi;
        two(t.d); x[0].d = lo; x[1].d = hi;
    }
    template <int US>
    RT_DEV static void rec(const Raw& r, const Tail& tl, int i, h8_t B[2], float sc[2]) {
        constexpr int TP = US & 1;
        u32x4 q = r.l[i], v = r.h;
        if (TP) q = q >> 4;
        // the two high bits to bits 4, 5 of each byte: qh bits 2t, t = 2TP + i
        const int t2 = 2 * (2 * TP + i);
        v = t2 <= 4 ? v << (4 - t2) : v >> (t2 - 4);
        q = (q & 0x0F0F0F0Fu) | (v & 0x30303030u);
        swap_piece(q);
        B[0] = bytes_to_h8(q.x, q.y, 32.0f);
        B[1] = bytes_to_h8(q.z, q.w, 32.0f);
        const float d = h2f(tl.d);
        const uint32_t s4 = US == 0 ? tl.sc.x : US == 1 ? tl.sc.y : US == 2 ? tl.sc.z : tl.sc.w;
        sc[0] = d * (float)(int8_t)(s4 >> (16 * i));
        if (HALF) sc[1] = d * (float)(int8_t)(s4 >> (16 * i + 8));
    }
};

// ───────────────────────────── the GEMM ─────────────────────────────

struct GemmWArgs {
    const uint8_t* w;
    const uint8_t* w2;    // with w as gate and w2 as up: y = silu(x·wᵀ)·(x·w2ᵀ), 128-row tiles
    const u32x4* aops;    // prepared activations, [chunk][stage][1024 entries]
    const int* etab;      // exponent per (padded) activation row
    const u32x4* ssum;    // record sums, [chunk][super-block][128 entries]
    float* y;
    float* part;          // [chunk][split][64][N] partial sums (of w2: part2)
    float* part2;
    uint32_t M, N, nblk, nst, nchunks, splits;  // nst: stages of K
    uint32_t parts_all;   // unsplit tiles too go to part (split 0), as they are
    uint64_t row_bytes;
    const uint16_t* bias;  // other unsplit tiles: y = acc (+ f32(bias[n])) (+ res as res + y)
    const float* res;
};
// Tiles (256 weight rows × 64 activation rows) of up to three matrices, in
// order; the first `full` of them are one workgroup's each, the other `rem`
// have K split over `splits` workgroups of `kst` stages.
struct GemmWMulti {
    GemmWArgs a[3];
    uint32_t t0[4];  // first tile of each matrix
    uint32_t count, full, rem, splits, kst;
};

typedef __attribute__((address_space(1))) const void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

RT_DEV float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// Waits until at most VM of the wave's vector memory operations (they complete
// in order) and none of its LDS operations are under way, then for the
// workgroup.
template <int VM>
RT_DEV void wait_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4) << 14 | 7 << 4);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Pipeline: while stage s is computed, the activations of stage s + 2 go to LDS
// (one of three buffers) and, once the weights of stage s are decoded, those
// of stage s + 2 to their registers; the wait at the end of a stage leaves
// both under way.
template <class P>
RT_DEV void gemmw_tile(const GemmWArgs& a, uint32_t t, uint32_t split, uint32_t st0, uint32_t st1,
                       bool whole, u32x4 (*lds)[1024]) {
    constexpr int NT = 2, MT = 2, LU = P::LU;
    const uint32_t lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 31, h = lane >> 5;
    // chunks fastest: the workgroups of one tile of weights run together
    const uint32_t ch = t % a.nchunks, tile = t / a.nchunks;
    const bool pair = a.w2 != nullptr;
    const uint32_t nb = tile * (pair ? 128 : 256);  // the tile's first weight row
    const uint32_t n0 = nb + wv * (pair ? 32 : 64) + j, n1 = pair ? n0 : n0 + 32;
    const size_t w0 = (size_t)nb * a.row_bytes;
    const Row row[NT] = {  // clamped rows are not stored
        {a.w + w0, (uint32_t)((min(n0, a.N - 1) - nb) * a.row_bytes)},
        {(pair ? a.w2 : a.w) + w0, (uint32_t)((min(n1, a.N - 1) - nb) * a.row_bytes)}};
    const uint8_t* const rowx = h ? row[1].base + row[1].off : row[0].base + row[0].off;
    const u32x4* ap = a.aops + (size_t)ch * a.nst * 1024;

    auto stage_in = [&](uint32_t st, uint32_t buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t e = wv * 256 + i * 64;
            __builtin_amdgcn_global_load_lds((gptr_t)((const uint8_t*)(ap + (size_t)st * 1024 + e) + lane * 16),
                                             (lptr_t)(&lds[buf][e]), 16, 0, 0);
        }
    };
    typename P::Raw raw[2][NT];
    typename P::Sh sh[2];
    f16v acc[NT][MT], C[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[nt][t] = C[nt][t] = f16v{};
    h8_t sm[MT];
    // of the super-block: K-quants' scales and mins, d, dmin; Q6_K's scales and d
    u32x4 hdr[NT], hdr_nx[NT];
    auto load_hdr = [&](u32x4 (&x)[NT], uint32_t st) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) x[nt] = *(const u32x4*)(row[nt].base + (size_t)(st / 4) * P::BLK_BYTES + row[nt].off);
    };
    using PT = typename std::conditional<P::TAIL, P, WQ6KT<false, false>>::type;
    typename PT::Tail tl[NT], tl_nx;

    stage_in(st0, 0);
    if constexpr (P::CHAIN) load_hdr(hdr, st0);
    if constexpr (P::TAIL) PT::load_tail(tl_nx, rowx, st0);
    P::load(raw[0], sh[0], row, rowx, st0, h, a.nblk);
    stage_in(min(st0 + 1, st1 - 1), 1);
    if constexpr (LU == 1) P::load(raw[1], sh[1], row, rowx, min(st0 + 1, st1 - 1), h, a.nblk);
    wait_barrier<0>();
    if constexpr (P::TAIL) PT::spread_tail(tl_nx, tl);
    uint32_t buf = 0;  // of the stage
    auto stage = [&](uint32_t st, auto us_) {
        constexpr int US = decltype(us_)::value, RB = (US / LU) & 1;
        const uint32_t nx = min(st + 2, st1 - 1);
        stage_in(nx, buf == 0 ? 2 : buf - 1);
        if constexpr (LU == 2 && US % 2 == 0) P::load(raw[RB ^ 1], sh[RB ^ 1], row, rowx, nx, h, a.nblk);
        if constexpr (P::CHAIN && US == 1) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
                sm[t] = __builtin_bit_cast(h8_t, a.ssum[((size_t)ch * (a.nst / 4) + st / 4) * 128 + t * 64 + lane]);
        }
        if constexpr (P::CHAIN && US == 2) load_hdr(hdr_nx, nx);
        if constexpr (P::TAIL && US == 2) PT::load_tail(tl_nx, rowx, nx);
        __builtin_amdgcn_sched_barrier(0);  // these loads go out first
        if constexpr (US % LU == 0) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) P::arrange(raw[RB][nt], sh[RB], nt, st, h);
        }
        h8_t B[NT][2][2];
        float sc[NT][2][2];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            if constexpr (P::CHAIN) {
                P::template pair<US>(raw[RB][nt], hdr[nt], h, B[nt]);
                sc[nt][0][0] = h2f(hdr[nt].x);
            } else {
#pragma unroll
                for (int rr = 0; rr < 2; ++rr) {
                    if constexpr (P::TAIL) P::template rec<US>(raw[RB][nt], tl[nt], rr, B[nt][rr], sc[nt][rr]);
                    else P::template rec<US>(raw[RB][nt], rr, h, B[nt][rr], sc[nt][rr]);
                }
            }
        }
        if constexpr (LU == 1) P::load(raw[RB], sh[RB], row, rowx, nx, h, a.nblk);
        // (an odd number of stages: the last is left out, but not its loads and
        // waits, so that every wait counts one path)
        const bool live = P::Q == 4 || US == 0 || st < st1;
        const u32x4* ab = lds[buf];
        auto A = [&](int rr, int p, int t, int hl) {
            return __builtin_bit_cast(h8_t, ab[(((rr * 2 + p) * 2 + t) * 2 + hl) * 64 + lane]);
        };
        if constexpr (P::CHAIN) {
#pragma unroll
            for (int rr = 0; rr < 2; ++rr)
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int hl = 0; hl < 2; ++hl)
#pragma unroll
                        for (int t = 0; t < MT; ++t) {
                            const h8_t av = A(rr, p, t, hl);
#pragma unroll
                            for (int nt = 0; nt < NT; ++nt)
                                C[nt][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, B[nt][rr][p], C[nt][t], 0, 0, 0);
                        }
            if (US == 3) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const h8_t sc = P::K::scales(hdr[nt], 64.0f * P::MID), mn = P::K::mins(hdr[nt]);
                    const float dm = -64.0f * h2f(hdr[nt].x >> 16);
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
                        C[nt][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sm[t], sc, C[nt][t], 0, 0, 0);
                        const f16v S = __builtin_amdgcn_mfma_f32_32x32x16_f16(sm[t], mn, f16v{}, 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[nt][t][i] = __builtin_fmaf(dm, S[i], acc[nt][t][i]);
                    }
                }
            }
            if (US % 2 == 1) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[nt][t][i] = __builtin_fmaf(sc[nt][0][0], C[nt][t][i], acc[nt][t][i]);
                        C[nt][t] = f16v{};
                    }
            }
        } else if (live) {
#pragma unroll
            for (int rr = 0; rr < 2; ++rr)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const h8_t a0 = A(rr, 0, t, 0), a1 = A(rr, 0, t, 1), a2 = A(rr, 1, t, 0), a3 = A(rr, 1, t, 1);
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        const h8_t b0 = B[nt][rr][0], b1 = B[nt][rr][1];
                        f16v c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, b0, f16v{}, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, b0, c, 0, 0, 0);
                        if (P::HALF) {
#pragma unroll
                            for (int i = 0; i < 16; ++i)
                                acc[nt][t][i] = __builtin_fmaf(sc[nt][rr][0], c[i], acc[nt][t][i]);
                            c = f16v{};
                        }
                        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2, b1, c, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a3, b1, c, 0, 0, 0);
                        const float s = sc[nt][rr][P::HALF ? 1 : 0];
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[nt][t][i] = __builtin_fmaf(s, c[i], acc[nt][t][i]);
                    }
                }
        }
        // everything issued before this stage's loads has arrived
        wait_barrier<4 + (LU == 1 || US % 2 == 0 ? (int)P::LOADS : 0)>();
        __builtin_amdgcn_sched_barrier(0);  // (uses of the loads stay behind their wait)
        if constexpr (P::CHAIN && US == 3) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) hdr[nt] = hdr_nx[nt];
        }
        if constexpr (P::TAIL && US == 3) PT::spread_tail(tl_nx, tl);
        buf = buf == 2 ? 0 : buf + 1;
    };
    for (uint32_t st = st0; st < st1; st += P::Q == 4 ? 4 : 2) {
        stage(st, std::integral_constant<int, 0>{});
        stage(st + 1, std::integral_constant<int, 1>{});
        if constexpr (P::Q == 4) {
            stage(st + 2, std::integral_constant<int, 2>{});
            stage(st + 3, std::integral_constant<int, 3>{});
        }
    }
    __builtin_amdgcn_s_waitcnt(0);  // no load to LDS outlives the workgroup
    // lane l holds row 8(i / 4) + 4h + i % 4 of a tile of activation rows for
    // weight row l % 32; the activation rows' exponents scale the sums
    const uint32_t m0 = ch * 64 + 4 * h;
    auto rof = [](int t, int i) { return (uint32_t)(32 * t + 8 * (i / 4) + i % 4); };
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int e = a.etab[m0 + rof(t, i)];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[nt][t][i] = __builtin_amdgcn_ldexpf(acc[nt][t][i], e);
        }
    if (!whole || a.parts_all) {
        const size_t at = (((size_t)ch * a.splits + split) * 64 + 4 * h) * a.N;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const uint32_t n = nt ? n1 : n0;
            if (n >= a.N) continue;
            float* p = (pair && nt ? a.part2 : a.part) + at + n;
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) p[(size_t)rof(t, i) * a.N] = acc[nt][t][i];
        }
        return;
    }
    if (pair) {
        if (n0 >= a.N) return;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const uint32_t m = m0 + rof(t, i);
                if (m < a.M) a.y[(size_t)m * a.N + n0] = silu_mul(acc[0][t][i], acc[1][t][i]);
            }
        return;
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const uint32_t n = nt ? n1 : n0;
        if (n >= a.N) continue;
        const float b = a.bias ? h2f(a.bias[n]) : 0.0f;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const uint32_t m = m0 + rof(t, i);
                if (m >= a.M) continue;
                float v = acc[nt][t][i];
                if (a.bias) v += b;
                if (a.res) v = a.res[(size_t)m * a.N + n] + v;
                a.y[(size_t)m * a.N + n] = v;
            }
    }
}

// Workgroup b runs on XCD b mod 8: each XCD takes consecutive items of a
// range, whose weights and activations its L2 holds.
RT_DEV uint32_t xcd_order(uint32_t b, uint32_t n) {
    const uint32_t x = b % 8, q = n / 8, r = n % 8;
    return x * q + min(x, r) + b / 8;
}
template <class P>
RT_DEV void gemmw_body(const GemmWMulti& m) {
    __shared__ u32x4 lds[3][1024];
    const bool whole = blockIdx.x < m.full;
    uint32_t t, split = 0;
    if (whole) {
        t = xcd_order(blockIdx.x, m.full);
    } else {
        const uint32_t r = xcd_order(blockIdx.x - m.full, m.rem * m.splits);
        t = m.full + r % m.rem;
        split = r / m.rem;
    }
    uint32_t i = 0;
    while (i + 1 < m.count && t >= m.t0[i + 1]) ++i;
    const uint32_t nst = m.a[i].nst;
    const uint32_t st0 = whole ? 0 : split * m.kst, st1 = whole ? nst : min(nst, st0 + m.kst);
    gemmw_tile<P>(m.a[i], t - m.t0[i], split, st0, st1, whole, lds);
}
// ───────────────────────────── activation preparation ─────────────────────────────
//
// A workgroup per (padded) row holds the row in registers, thread u + T·i the
// elements 8u .. 8u + 7, scales it by the power of two e that takes its
// largest |x| into [2^14, 2^15) and writes hi = f16(x·2^-e) and lo =
// f16(x·2^-e − hi): [chunk of 64 rows][stage][record][MFMA p][32-row tile]
// [hi, lo][lane 32h + row] entries of 8 halves, elements 16p + 8h .. + 7 of the
// record in the order 0 2 1 3 4 6 5 7.  Rows past M and a record past K are
// zero.  ssum: the record sums of each super-block as f16 pairs hi + lo of
// Σx·2^-6, [chunk][super-block][tile][32·(hi, lo) + row][8 records, same order].
//
// Bound: memory.  Eight rows share each 128-byte line of the operands, so
// consecutive rows go to one XCD (xcd_order), whose L2 joins their writes.
enum PrepMode { kPrepRows, kPrepNorm, kPrepSumNorm, kPrepAttn };
struct PrepWArgs {
    const float* x;      // rows (kPrepRows, kPrepNorm)
    const float* gamma;  // RMSNorm of the row first (kPrepNorm, kPrepSumNorm): x·rsqrt(mean(x²) + eps)·γ
    float* xn;           // kPrepNorm: the normalised rows, when given
    u32x4* aops;
    int* etab;
    _Float16* ssum;      // or null
    uint32_t M, K;
    float eps;
    PrepSum ps;          // kPrepSumNorm
    PrepAttn pa;         // kPrepAttn
};
template <int T>
RT_DEV float wg_reduce(float v, float* red, bool max) {
    for (int o = 32; o > 0; o >>= 1) {
        const float w = __shfl_xor(v, o, 64);
        v = max ? fmaxf(v, w) : v + w;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for (int w = 1; w < T / 64; ++w) r = max ? fmaxf(r, red[w]) : r + red[w];
    return r;
}
template <int T, int NPT, PrepMode MODE>
RT_DEV void prep_row(const PrepWArgs& a) {
    __shared__ float red[2][T / 64];
    const uint32_t m = xcd_order(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const uint32_t nu = a.K / 8, nup = (a.K / 32 + 1) / 2 * 8;  // with the zero record
    const bool row = m < a.M;
    f32x4 v[NPT][2];
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
        const uint32_t u = tid + T * i;
        v[i][0] = v[i][1] = f32x4{0, 0, 0, 0};
        if (!row || u >= nu) continue;
        if constexpr (MODE == kPrepSumNorm) {
            const PrepSum& ps = a.ps;
            const uint32_t ch = m / 64;
            const size_t off = ((size_t)ch * ps.splits * 64 + m % 64) * a.K + 8 * u, ss = (size_t)64 * a.K;
            const uint32_t nsp = wide_splits(ps.full, ps.splits, 8 * u, 256, ps.nch, ch);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                v[i][q] = *(const f32x4*)(ps.res + (size_t)m * a.K + 8 * u + 4 * q) +
                          split_add(ps.part + off + 4 * q, ss, nsp);
                *(f32x4*)(ps.y + (size_t)m * a.K + 8 * u + 4 * q) = v[i][q];
            }
        } else if constexpr (MODE == kPrepAttn) {
            // element (head, d) of the row, merged over the nsp key ranges as
            // the attention's last workgroup merges them
            const PrepAttn& pa = a.pa;
            const float NEG = -__builtin_huge_valf();
            const uint32_t h = 8 * u / pa.hd, d = 8 * u % pa.hd, kvh = h / pa.G;
            const uint32_t qi = m * pa.G + h % pa.G, cg = qi / 16, col = qi % 16;
            const size_t pair = (size_t)kvh * pa.cgs + cg;
            const float* mlv = pa.ml + (pair * pa.nsp * 16 + col) * 2;
            float mj[RT_ATTN_MQ_NSP_MAX], lj[RT_ATTN_MQ_NSP_MAX];
            f32x4 pj[RT_ATTN_MQ_NSP_MAX][2];
#pragma unroll
            for (uint32_t j = 0; j < RT_ATTN_MQ_NSP_MAX; ++j) {
                const uint32_t jj = j < pa.nsp ? j : 0;
                mj[j] = mlv[32 * jj];
                lj[j] = mlv[32 * jj + 1];
                const f32x4* pp = (const f32x4*)(pa.part + ((pair * pa.nsp + jj) * 16 + col) * pa.hd + d);
                pj[j][0] = pp[0];
                pj[j][1] = pp[1];
            }
            float Mx = NEG, L = 0.0f;
#pragma unroll
            for (uint32_t j = 0; j < RT_ATTN_MQ_NSP_MAX; ++j) Mx = fmaxf(Mx, mj[j]);
            f32x4 o[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (uint32_t j = 0; j < RT_ATTN_MQ_NSP_MAX; ++j) {
                const float w = (j >= pa.nsp || mj[j] == NEG) ? 0.0f : expf(mj[j] - Mx);
                L += w * lj[j];
                o[0] += w * pj[j][0];
                o[1] += w * pj[j][1];
            }
            v[i][0] = o[0] / L;
            v[i][1] = o[1] / L;
        } else {
            const f32x4* xr = (const f32x4*)(a.x + (size_t)m * a.K + 8 * u);
            v[i][0] = xr[0];
            v[i][1] = xr[1];
        }
    }
    if constexpr (MODE == kPrepNorm || MODE == kPrepSumNorm) {
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < NPT; ++i)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f32x4 t = v[i][q];
                ss += t.x * t.x + t.y * t.y + t.z * t.z + t.w * t.w;
            }
        const float rms = rsqrtf(wg_reduce<T>(ss, red[0], false) / (float)a.K + a.eps);
#pragma unroll
        for (int i = 0; i < NPT; ++i) {
            const uint32_t u = tid + T * i;
            if (!row || u >= nu) continue;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f32x4 g = *(const f32x4*)(a.gamma + 8 * u + 4 * q), t = v[i][q];
                v[i][q] = f32x4{t.x * rms * g.x, t.y * rms * g.y, t.z * rms * g.z, t.w * rms * g.w};
                if (MODE == kPrepNorm && a.xn) *(f32x4*)(a.xn + (size_t)m * a.K + 8 * u + 4 * q) = v[i][q];
            }
        }
    }
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < NPT; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const f32x4 t = v[i][q];
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(t.x), fabsf(t.y)), fmaxf(fabsf(t.z), fabsf(t.w))));
        }
    mx = wg_reduce<T>(mx, red[1], true);
    const int e = mx > 0.0f ? __builtin_amdgcn_frexp_expf(mx) - 15 : 0;
    if (tid == 0) a.etab[m] = e;
    const uint32_t ch = m / 64, t32 = m / 32 % 2, mm = m % 32;
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
        const uint32_t u = tid + T * i;
        if (u >= nup) break;  // (the four lanes of a record share this)
        _Float16 h[8], l[8];
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float xs = __builtin_amdgcn_ldexpf(v[i][j / 4][j % 4], -e);
            h[j] = (_Float16)xs;
            l[j] = (_Float16)(xs - (float)h[j]);
            sum += (float)h[j] + (float)l[j];
        }
        const uint32_t rec = u >> 2, p = (u >> 1) & 1, hh = u & 1;
        u32x4* base = a.aops + (((size_t)ch * (nup / 4) + rec) * 2 + p) * 256 + t32 * 128 + 32 * hh + mm;
        auto two = [](_Float16 x, _Float16 y) {
            return (uint32_t)__builtin_bit_cast(uint16_t, x) | ((uint32_t)__builtin_bit_cast(uint16_t, y) << 16);
        };
        base[0] = u32x4{two(h[0], h[2]), two(h[1], h[3]), two(h[4], h[6]), two(h[5], h[7])};
        base[64] = u32x4{two(l[0], l[2]), two(l[1], l[3]), two(l[4], l[6]), two(l[5], l[7])};
        if (a.ssum) {
            // of the operands' own values: their rounding then cancels between a
            // code's products and the min's as far as the weight is small
            sum += __shfl_xor(sum, 1, 64);
            sum += __shfl_xor(sum, 2, 64);
            if ((u & 3) == 0) {
                const float s6 = __builtin_amdgcn_ldexpf(sum, -6);
                const _Float16 sh = (_Float16)s6, sl = (_Float16)(s6 - (float)sh);
                const uint32_t r = rec & 7, pos = (r & 4) | ((r & 1) << 1) | ((r >> 1) & 1);
                _Float16* sp = a.ssum + (((size_t)ch * (nup / 32) + rec / 8) * 128 + t32 * 64 + mm) * 8 + pos;
                sp[0] = sh;
                sp[32 * 8] = sl;
            }
        }
    }
}
// 256 threads up to K = 4096, 1024 up to 20,480 (24,576)
#define RT_GEMMW_PREP(FN, MODE)                                                               \
    extern "C" __global__ void __launch_bounds__(256) k_gemmw_prep##FN(PrepWArgs a) {         \
        prep_row<256, 2, MODE>(a);                                                            \
    }                                                                                         \
    extern "C" __global__ void __launch_bounds__(1024) k_gemmw_prep##FN##_l(PrepWArgs a) {    \
        prep_row<1024, 3, MODE>(a);                                                           \
    }
RT_GEMMW_PREP(, kPrepRows)
RT_GEMMW_PREP(_n, kPrepNorm)
RT_GEMMW_PREP(_sn, kPrepSumNorm)
RT_GEMMW_PREP(_a, kPrepAttn)

#define RT_GEMMW(FN, ...)                                                                     \
    extern "C" __global__ void __launch_bounds__(256, 2) k_gemmw_##FN(GemmWMulti m) {         \
        gemmw_body<__VA_ARGS__>(m);                                                           \
    }
// _o: rows of an odd number of blocks
RT_GEMMW(q8_0, WQ8_0T<true>)
RT_GEMMW(q8_0_o, WQ8_0T<false>)
RT_GEMMW(q4_0, WQ4_0T<false, true>)
RT_GEMMW(q4_0_o, WQ4_0T<false, false>)
RT_GEMMW(q4_0g, WQ4_0T<true, true>)
RT_GEMMW(q4_0g_o, WQ4_0T<true, false>)
RT_GEMMW(q5_0, WQ5_0T<true>)
RT_GEMMW(q5_0_o, WQ5_0T<false>)
RT_GEMMW(q4k, WQ4KT<false>)
RT_GEMMW(q4kg, WQ4KT<true>)
RT_GEMMW(q5k, WQ5KT<false>)
RT_GEMMW(q5kg, WQ5KT<true>)
RT_GEMMW(q6k, WQ6KT<false, true>)
RT_GEMMW(q6k_o, WQ6KT<false, false>)
RT_GEMMW(q6kg, WQ6KT<true, true>)
RT_GEMMW(q6kg_o, WQ6KT<true, false>)
