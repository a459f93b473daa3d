// Expert weights as fp16 matrix operands: the words a lane holds of a weight
// row, their dequantization, their GGUF rows, and the packed copy's fragments
// (moe_mfma.hip: the prefill GEMMs; moe_q8dec.hip: the Q8_0 decode batch).
#pragma once
#include "common.h"
#include "qdecode.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kBK = 64;  // columns of a K step

VH_DEV f16x2 as_h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
VH_DEV f16x2 splat(_Float16 v) { return f16x2{v, v}; }
VH_DEV uint32_t h_bits(float v) { return __builtin_bit_cast(uint16_t, _Float16(v)); }

// (a & m) | e with the operands in registers: the compiler's own form takes at
// most one constant from outside the vector registers and splits in two
VH_DEV uint32_t and_or(uint32_t a, uint32_t m, uint32_t e) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(m), "v"(e));
    return r;
}
// constants that and_or and v_perm_b32 take from vector registers
struct Consts {
    uint32_t lo = 0x000f000fu, hi = 0x00f000f0u, e = 0x64006400u, h0 = 0x00300030u, h1 = 0x03000300u,
             b = 0x64646464u;
    VH_DEV Consts() { asm volatile("" : "+v"(lo), "+v"(hi), "+v"(e), "+v"(h0), "+v"(h1), "+v"(b)); }
};

// ---- operand words --------------------------------------------------------------
// What a lane holds of one weight row r = lane % 32 of a 32-row fragment over
// K step s (64 columns): the 32 weights of its half h = lane / 32 of the step,
// columns 64 s + 32 h + 8 ks + j, of which it supplies j = 0..7 to sub-step ks =
// 0..3 - NW words of quants and a word of their fp16 scales, under the row's
// power of two. (The columns a multiply takes together are free as long as the
// inputs' operand takes the same: the lanes of half h read input chunk 4 h + ks.)
// get() forms sub-step ks's B operand.
template <int T>
struct Op;

template <>
struct Op<VT_Q8_0> {  // src/gguf_compute.c:112-120: y = q d
    // words 2 ks, 2 ks + 1: bytes q_j + 128; scale: the block's d
    static constexpr int NW = 8, scale_bytes = 2;
    static VH_DEV f16x8 get(const uint32_t (&w)[NW], uint32_t sc, int ks, const Consts &c) {
        const f16x2 d = splat(as_h2(sc)[0]);
        f16x8 o;
#pragma unroll
        for (int p = 0; p < 4; p++) {  // fp16 1024 + u is the byte u under the byte 0x64
            const uint32_t v = __builtin_amdgcn_perm(w[2 * ks + (p >> 1)], c.b, (p & 1) ? 0x00070006u : 0x00050004u);
            const f16x2 y = (as_h2(v) - splat(_Float16(1152.0f))) * d;
            o[2 * p] = y[0];
            o[2 * p + 1] = y[1];
        }
        return o;
    }
};

template <>
struct Op<VT_Q4_K> {  // src/gguf_compute.c:52-66: y = d1 q - m1 (d1 = d sc, m1 = dmin m)
    // word ks: nibble j at bit 16 (j % 2) + 4 (j / 2); scales: the sub-block's d1, m1
    static constexpr int NW = 4, scale_bytes = 4;
    static VH_DEV f16x8 get(const uint32_t (&w)[NW], uint32_t sc, int ks, const Consts &c) {
        const f16x2 s = as_h2(sc), d = splat(s[0]), m = splat(s[1]), d16 = d * splat(_Float16(0.0625f));
        const f16x2 k = splat(_Float16(1024.0f));
        const uint32_t a = w[ks], b = a >> 8;
        // bits 0-3 of each half give 1024 + q, bits 4-7 give 1024 + 16 q; both less 1024 are exact
        const f16x2 p0 = __builtin_elementwise_fma(as_h2(and_or(a, c.lo, c.e)) - k, d, -m);
        const f16x2 p1 = __builtin_elementwise_fma(as_h2(and_or(a, c.hi, c.e)) - k, d16, -m);
        const f16x2 p2 = __builtin_elementwise_fma(as_h2(and_or(b, c.lo, c.e)) - k, d, -m);
        const f16x2 p3 = __builtin_elementwise_fma(as_h2(and_or(b, c.hi, c.e)) - k, d16, -m);
        return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    }
};

template <>
struct Op<VT_Q6_K> {  // src/gguf_compute.c:83-103: y = (d sc) (q - 32)
    // word ks: the low nibbles as Q4_K's; words 4, 5: the high 2 bits of
    // sub-steps 0, 1 and 2, 3 - weight j of an even sub-step at bit 16 (j % 2)
    // + {4, 8, 6, 10}[j / 2], of an odd one at 16 (j % 2) + {12, 0, 14, 2}[j / 2];
    // scales: d sc of the two 16-weight sub-blocks (sub-steps 0, 1 and 2, 3)
    static constexpr int NW = 6, scale_bytes = 4;
    static VH_DEV int hi_bit(int ks, int j) {
        const int p = j >> 1;
        return 16 * (j & 1) + ((ks & 1) ? (p == 0 ? 12 : p == 1 ? 0 : p == 2 ? 14 : 2)
                                        : (p == 0 ? 4 : p == 1 ? 8 : p == 2 ? 6 : 10));
    }
    static VH_DEV f16x8 get(const uint32_t (&w)[NW], uint32_t sc, int ks, const Consts &c) {
        const f16x2 d = splat(as_h2(sc)[ks >> 1]), d16 = d * splat(_Float16(0.0625f));
        const f16x2 k0 = splat(_Float16(1056.0f)), k1 = splat(_Float16(1536.0f));
        uint32_t h = w[4 + (ks >> 1)];
        if (ks & 1) h = __builtin_amdgcn_perm(h, h, 0x02030001u);  // the bytes of each half swapped
        const uint32_t a = w[ks], b = a >> 8, g = h >> 2;
        // the 6-bit quant in place: 1024 + q, or 1024 + 16 q from bit 4
        const f16x2 p0 = (as_h2(and_or(h, c.h0, and_or(a, c.lo, c.e))) - k0) * d;
        const f16x2 p1 = (as_h2(and_or(h, c.h1, and_or(a, c.hi, c.e))) - k1) * d16;
        const f16x2 p2 = (as_h2(and_or(g, c.h0, and_or(b, c.lo, c.e))) - k0) * d;
        const f16x2 p3 = (as_h2(and_or(g, c.h1, and_or(b, c.hi, c.e))) - k1) * d16;
        return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    }
};

// The power of two a weight row's scales are multiplied by, as its exponent:
// bound * 2^e lies in [2^13, 2^14) for a bound on the row's magnitudes (0 for
// a row of zeros or with a scale that is not finite). -114 takes the largest
// fp32 number there; below 2^-86 the result is that much smaller.
VH_DEV int exponent_for(float bound) {
    if (!(bound > 0.0f) || !(bound <= 3.4028234663852886e38f)) return 0;
    int ex;
    frexpf(bound, &ex);
    return max(-114, min(100, 14 - ex));
}

// GGUF rows: the loads of one lane and step (raw), their rearrangement into
// operand words, and the row's blocks with the magnitude bound of one.
template <int T>
struct Rows;

// nibbles j = 0..7 (bytes of a, then of b, each below 16) in the order of Op<VT_Q4_K>
VH_DEV uint32_t nibble_word(uint32_t a, uint32_t b) {
    const uint32_t t = a | (b << 4);
    const uint32_t u = __builtin_amdgcn_perm(t, t, 0x01010000u), v = __builtin_amdgcn_perm(t, t, 0x03030202u);
    return (u & 0x000f000fu) | ((u >> 4) & 0x0f000f00u) | ((v << 4) & 0x00f000f0u) | (v & 0xf000f000u);
}

VH_DEV uint32_t u4_at(const uint4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

template <>
struct Rows<VT_Q8_0> {
    struct Raw {
        uint4 q[2];
        uint32_t d;
    };
    static VH_DEV int blocks(int K) { return K / 32; }
    static VH_DEV float bound(gbyte *row, int b) { return fabsf(h2f(ld_u16(row + 34 * b))) * 128.0f; }
    static VH_DEV float step_bound(const Raw &r) { return fabsf(h2f(r.d)) * 128.0f; }
    static VH_DEV void load(gbyte *row, int s, int half, Raw &r) {  // block 2 s + half
        gbyte *p = row + 68 * s + 34 * half;
        r.q[0] = ld_u128(p + 2);
        r.q[1] = ld_u128(p + 18);
        r.d = ld_u16(p);
    }
    static VH_DEV void words(const Raw &r, int, int, float up, uint32_t (&w)[8], uint32_t &sc) {
#pragma unroll
        for (int i = 0; i < 8; i++) w[i] = u4_at(r.q[i >> 2], i & 3) ^ 0x80808080u;
        sc = h_bits(h2f(r.d) * up);
    }
};

template <>
struct Rows<VT_Q4_K> {
    struct Raw {
        uint4 hdr, q[2];
    };
    static VH_DEV int blocks(int K) { return K / 256; }
    static VH_DEV float bound_of(uint32_t h) {
        return fmaxf(fabsf(h2f(h & 0xffffu)) * (63.0f * 15.0f), fabsf(h2f(h >> 16)) * 63.0f);
    }
    static VH_DEV float bound(gbyte *row, int b) { return bound_of(ld_u32(row + 144 * b)); }
    static VH_DEV float step_bound(const Raw &r) { return bound_of(r.hdr.x); }
    // step s: the 32 bytes s % 4 of super-block s / 4, low nibbles (sub-block 2 (s % 4)) for half 0, high for 1
    static VH_DEV void load(gbyte *row, int s, int, Raw &r) {
        gbyte *p = row + 144 * (s >> 2);
        r.hdr = ld_u128(p);
        r.q[0] = ld_u128(p + 16 + 32 * (s & 3));
        r.q[1] = ld_u128(p + 32 + 32 * (s & 3));
    }
    static VH_DEV void words(const Raw &r, int s, int half, float up, uint32_t (&w)[4], uint32_t &sc) {
        const int sh = 4 * half;
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
            w[ks] = nibble_word((u4_at(r.q[ks >> 1], 2 * (ks & 1)) >> sh) & 0x0f0f0f0fu,
                                (u4_at(r.q[ks >> 1], 2 * (ks & 1) + 1) >> sh) & 0x0f0f0f0fu);
        int a0, m0, a1, m1;
        q4k_scale_min(2 * (s & 3), r.hdr.y, r.hdr.z, r.hdr.w, a0, m0);
        q4k_scale_min(2 * (s & 3) + 1, r.hdr.y, r.hdr.z, r.hdr.w, a1, m1);
        sc = h_bits(h2f(r.hdr.x & 0xffffu) * up * float(half ? a1 : a0)) |
             h_bits(h2f(r.hdr.x >> 16) * up * float(half ? m1 : m0)) << 16;
    }
};

template <>
struct Rows<VT_Q6_K> {
    struct Raw {
        uint4 ql[2], qh[2];
        uint32_t sc, d;
    };
    static VH_DEV int blocks(int K) { return K / 256; }
    static VH_DEV float bound(gbyte *row, int b) { return fabsf(h2f(ld_u16(row + 210 * b + 208))) * (128.0f * 32.0f); }
    static VH_DEV float step_bound(const Raw &r) { return fabsf(h2f(r.d)) * (128.0f * 32.0f); }
    // step s: half h = (s % 4) / 2 of super-block s / 4, group g = 2 (s % 2) +
    // `half`: weight l has its low bits in ql[64 h + 32 (g % 2) + l] (low nibbles
    // for g < 2), its high bits 2 g of qh[32 h + l], its scale in scales[8 h + 2 g + l / 16]
    static VH_DEV void load(gbyte *row, int s, int half, Raw &r) {
        gbyte *p = row + 210 * (s >> 2);
        const int h = (s & 3) >> 1;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            r.ql[i] = ld_u128(p + 64 * h + 32 * half + 16 * i);
            r.qh[i] = ld_u128(p + 128 + 32 * h + 16 * i);
        }
        r.sc = ld_u16(p + 192 + 8 * h + 2 * (2 * (s & 1) + half));
        r.d = ld_u16(p + 208);
    }
    static VH_DEV void words(const Raw &r, int s, int half, float up, uint32_t (&w)[6], uint32_t &sc) {
        const int sh = (s & 1) ? 4 : 0, g2 = 2 * (2 * (s & 1) + half);
        w[4] = w[5] = 0;
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            const int i = 2 * (ks & 1);
            w[ks] = nibble_word((u4_at(r.ql[ks >> 1], i) >> sh) & 0x0f0f0f0fu,
                                (u4_at(r.ql[ks >> 1], i + 1) >> sh) & 0x0f0f0f0fu);
            const uint32_t h0 = u4_at(r.qh[ks >> 1], i) >> g2, h1 = u4_at(r.qh[ks >> 1], i + 1) >> g2;
#pragma unroll
            for (int j = 0; j < 8; j++)
                w[4 + (ks >> 1)] |= (((j < 4 ? h0 : h1) >> (8 * (j & 3))) & 3u) << Op<VT_Q6_K>::hi_bit(ks, j);
        }
        const float d = h2f(r.d) * up;
        sc = h_bits(d * float(int(int8_t(r.sc)))) | h_bits(d * float(int(int8_t(r.sc >> 8)))) << 16;
    }
};

// Fragment (group c, step s, j) of a packed matrix: a lane's words together,
// 16 bytes of a lane at a time, then the lanes' scales. Group c of gate/up: rows
// 32 c .. + 31 of gate (j = 0) and of up (j = 1); of down: rows 64 c + 32 j ..
// + 31. It sits at ((c * nk + s) * 2 + j) * bytes; the rows' scales 2^-e follow
// the fragments (gate's rows, then up's).
template <int T>
struct Frag {
    static constexpr int NW = Op<T>::NW, SB = Op<T>::scale_bytes, bytes = 64 * (4 * NW + SB);
    static VH_DEV void load(gbyte *p, int lane, uint32_t (&w)[NW], uint32_t &sc) {
        const uint4 a = ld_u128(p + 16 * lane);
        w[0] = a.x;
        w[1] = a.y;
        w[2] = a.z;
        w[3] = a.w;
        if constexpr (NW == 8) {
            const uint4 b = ld_u128(p + 1024 + 16 * lane);
            w[4] = b.x;
            w[5] = b.y;
            w[6] = b.z;
            w[7] = b.w;
        } else if constexpr (NW == 6) {
            const uint2 b = ld_u64(p + 1024 + 8 * lane);
            w[4] = b.x;
            w[5] = b.y;
        }
        if constexpr (SB == 4) sc = ld_u32(p + 256 * NW + 4 * lane);
        else sc = ld_u16(p + 256 * NW + 2 * lane);
    }
    static VH_DEV void store(uint8_t *p, int lane, const uint32_t (&w)[NW], uint32_t sc) {
        *reinterpret_cast<uint4 *>(p + 16 * lane) = make_uint4(w[0], w[1], w[2], w[3]);
        if constexpr (NW == 8) *reinterpret_cast<uint4 *>(p + 1024 + 16 * lane) = make_uint4(w[4], w[5], w[6], w[7]);
        if constexpr (NW == 6) *reinterpret_cast<uint2 *>(p + 1024 + 8 * lane) = make_uint2(w[4], w[5]);
        if constexpr (SB == 4) *reinterpret_cast<uint32_t *>(p + 256 * NW + 4 * lane) = sc;
        else *reinterpret_cast<uint16_t *>(p + 256 * NW + 2 * lane) = uint16_t(sc);
    }
};

}  // namespace
