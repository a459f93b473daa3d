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

// ---- GGUF rows staged by a wave -----------------------------------------------
// A wave reads its 64 rows (fragment 0's 32, then fragment 1's) a pair of K
// steps (128 columns) at a time, in 16-byte pieces with neighbouring lanes on
// neighbouring bytes of a row, through registers (Regs: the pair in flight) into
// its own part of LDS (Lds: the pair being multiplied), where every lane finds the
// words of its row. A lane per row touched 64 lines with every load instruction,
// and rearranging what it read took more vector instructions than the multiplies
// leave time for: Qwen3 Q4_K_M 2048 tokens gate/up 330 -> 200 us, down 367 -> 151
// (from the packed copy 154 and 107); Q8_0 329 -> 236 and 168 -> 147 (169 and 107).
// Q8_0's pieces are those of the row, 8-byte aligned, not of its 34-byte blocks:
// loads at odd multiples of 2 bytes ran at half the rate.
//   load(r, B, rb, t, lane)  requests pair t of the rows at B[0], B[1] (the
//                            fragments' first rows), rb bytes apart
//   bounds(r, b)             the rows' magnitude bounds in the pair
//   put(l, r, up, lane)      the pair's pieces and its scales (those of Op<T>)
//   fetch(l, p, i, j, ..)    step p's words 4 i .. 4 i + 3 of fragment j (sub-steps
//                            2 i, 2 i + 1): a byte per weight
//   get(w0, w1, sc, ks, c)   the operand of sub-step ks, Op<T>::get's bits
// K-quants: the pieces are swizzled so that 16 lanes' reads and writes take 16 bank
// groups, and a lane per row forms the pair's scales. Q8_0 (PER_STEP): the lanes
// that multiply a row form its scale step by step.
// A row's power of two follows from its first bound (below 2^11 under it) and is
// lowered, with what the row has summed (lower_up), where a later bound would pass
// 2^15 under it: no pass over the row's scales ahead. Powers of two are exact, so
// the results are the packed copy's while no scale is subnormal in fp16 under
// either power: while a row's scales lie within 2^12 of its largest.
template <int T>
struct Staged;

// A lane's offset as a value of its own where it is used: added to a uniform
// base by the load itself. (Hoisted out of the loop as a 64-bit pair, and LDS
// addresses one per store, they take the registers of the loop's operands.)
VH_DEV uint32_t here(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <int N>  // whether any lane's power was lowered (fix is set only then)
VH_DEV bool lower_up(const float (&bound)[N], float (&up)[N], float (&fix)[N]) {
    bool over = false;
#pragma unroll
    for (int i = 0; i < N; i++) over |= bound[i] * up[i] >= 32768.0f;
    if (!__any(over)) return false;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const float to = bound[i] * up[i] >= 32768.0f ? ldexpf(1.0f, exponent_for(bound[i]) - 3) : up[i];
        fix[i] = to / up[i];
        up[i] = to;
    }
    return true;
}
VH_DEV float first_up(float bound) { return ldexpf(1.0f, bound > 0.0f ? exponent_for(bound) - 3 : 14); }
VH_DEV float larger_bound(float a, float b) { return b > a || !(b <= 3.4028234663852886e38f) ? b : a; }

// a byte of w per half of the operand: fp16 1024 + byte, less `zero`
VH_DEV f16x2 byte_pair(uint32_t w, int odd, uint32_t b64, float zero) {
    const uint32_t v = __builtin_amdgcn_perm(w, b64, odd ? 0x00070006u : 0x00050004u);
    return as_h2(v) - splat(_Float16(zero));
}

template <>
struct Staged<VT_Q8_0> {
    // A row's 136 bytes of a pair are staged as they are: the scales lie in them, so
    // the lanes that multiply a row (both halves) keep its power of two.
    static constexpr bool PER_STEP = true;
    static constexpr int NU = 2;  // of the lane's rows of the two fragments
    struct Regs {
        uint4 q[8];
        uint2 tail;
    };
    struct __align__(16) Lds {  // stores of 8 bytes that straddle them take eight times as long
        uint32_t q[64 * 34];
    };
    static VH_DEV void load(Regs &r, gbyte *const (&B)[2], int64_t rb, int t, int lane) {
        const uint32_t o = here(uint32_t(lane >> 3) * uint32_t(rb) + 16u * uint32_t(lane & 7));
#pragma unroll
        for (int q = 0; q < 8; q++) r.q[q] = ld_u128(B[q >> 2] + (8 * (q & 3)) * rb + 136 * t + o);
        r.tail = ld_u64((lane < 32 ? B[0] : B[1]) + 136 * t + 128 + uint32_t(lane & 31) * uint32_t(rb));
    }
    static VH_DEV void put(Lds &l, const Regs &r, int lane) {
        // 8 bytes at a time: two in one store would reach 2 KB from its address register
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        auto *o = reinterpret_cast<volatile __attribute__((address_space(3))) u32x2 *>(
            (__attribute__((address_space(3))) uint32_t *)l.q + 34 * (lane >> 3) + 4 * (lane & 7));
#pragma unroll
        for (int q = 0; q < 8; q++) {
            o[136 * q] = u32x2{r.q[q].x, r.q[q].y};
            o[136 * q + 1] = u32x2{r.q[q].z, r.q[q].w};
        }
        *reinterpret_cast<uint2 *>(l.q + 34 * lane + 32) = r.tail;
    }
    // block `half` of the step lies at byte 34 `half` of its 68: words 0 .. 8, or 8 .. 16
    // with the scale in the upper half of the first
    static VH_DEV void fetch(const Lds &l, int p, int i, int j, int half, int col, uint32_t (&w)[4], uint32_t &d) {
        const uint32_t *x = l.q + 34 * (32 * j + col) + 17 * p + 8 * half + 4 * i;
        const uint32_t sel = half ? 0x07060504u : 0x05040302u;
        uint32_t v[5];
#pragma unroll
        for (int k = 0; k < 5; k++) v[k] = x[k];
#pragma unroll
        for (int k = 0; k < 4; k++) w[k] = __builtin_amdgcn_perm(v[k + 1], v[k], sel) ^ 0x80808080u;
        if (i == 0) d = half ? v[0] >> 16 : v[0] & 0xffffu;
    }
    static VH_DEV float step_bound(uint32_t d) {  // of the row's step: both halves'
        const uint32_t b = __float_as_uint(fabsf(h2f(d)) * 128.0f);
        const auto v = __builtin_amdgcn_permlane32_swap(b, b, false, false);
        return larger_bound(__uint_as_float(v[0]), __uint_as_float(v[1]));
    }
    static VH_DEV float of_row(const float (&v)[NU], int j, int) { return v[j]; }
    static VH_DEV f16x8 get(uint32_t w0, uint32_t w1, uint32_t sc, int, const Consts &c) {
        const f16x2 d = splat(as_h2(sc)[0]);
        const f16x2 p0 = byte_pair(w0, 0, c.b, 1152.0f) * d, p1 = byte_pair(w0, 1, c.b, 1152.0f) * d;
        const f16x2 p2 = byte_pair(w1, 0, c.b, 1152.0f) * d, p3 = byte_pair(w1, 1, c.b, 1152.0f) * d;
        return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    }
};

template <>
struct Staged<VT_Q4_K> {
    static constexpr bool PER_STEP = false;
    static constexpr int NU = 1;  // lane r holds row r's power
    struct Regs {
        uint4 q[4], hdr;
        uint32_t t;  // the pair (uniform)
    };
    struct Lds {
        uint4 q[256];
        uint4 sc[64];
    };
    static VH_DEV void load(Regs &r, gbyte *const (&B)[2], int64_t rb, int t, int lane) {
        const uint32_t oq = here(uint32_t(lane >> 2) * uint32_t(rb) + 16u * uint32_t(lane & 3));
#pragma unroll
        for (int q = 0; q < 4; q++)
            r.q[q] = ld_u128(B[q >> 1] + (16 * (q & 1)) * rb + 144 * (t >> 1) + 16 + 64 * (t & 1) + oq);
        r.hdr = ld_u128((lane < 32 ? B[0] : B[1]) + 144 * (t >> 1) + uint32_t(lane & 31) * uint32_t(rb));
        r.t = uint32_t(t);
    }
    static VH_DEV void bounds(const Regs &r, float (&b)[NU]) { b[0] = Rows<VT_Q4_K>::bound_of(r.hdr.x); }
    static VH_DEV float of_row(const float (&v)[NU], int j, int col) { return __shfl(v[0], 32 * j + col, 64); }
    static VH_DEV void put(Lds &l, const Regs &r, const float (&up)[NU], int lane) {
        const int a = 4 * (lane >> 2) + ((lane & 3) ^ (lane >> 4));
#pragma unroll
        for (int q = 0; q < 4; q++) l.q[64 * q + a] = r.q[q];
        // the scales and minima of sub-blocks 4 (t % 2) .. + 3, a byte each (q4k_scale_min)
        const uint32_t s = (r.t & 1) ? (r.hdr.w & 0x0f0f0f0fu) | ((r.hdr.y >> 2) & 0x30303030u) : r.hdr.y & 0x3f3f3f3fu;
        const uint32_t m = (r.t & 1) ? ((r.hdr.w >> 4) & 0x0f0f0f0fu) | ((r.hdr.z >> 2) & 0x30303030u) : r.hdr.z & 0x3f3f3f3fu;
        const float d = h2f(r.hdr.x & 0xffffu) * up[0], dm = h2f(r.hdr.x >> 16) * up[0];
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
            o[i] = h_bits(d * float((s >> (8 * i)) & 0xffu)) | h_bits(dm * float((m >> (8 * i)) & 0xffu)) << 16;
        l.sc[lane] = make_uint4(o[0], o[1], o[2], o[3]);
    }
    static VH_DEV void fetch(const Lds &l, int p, int i, int j, int half, int col, uint32_t (&w)[4]) {
        const uint4 v = l.q[128 * j + 4 * col + ((2 * p + i) ^ ((col >> 2) & 3))];
        const int sh = 4 * half;
        w[0] = (v.x >> sh) & 0x0f0f0f0fu;
        w[1] = (v.y >> sh) & 0x0f0f0f0fu;
        w[2] = (v.z >> sh) & 0x0f0f0f0fu;
        w[3] = (v.w >> sh) & 0x0f0f0f0fu;
    }
    static VH_DEV f16x8 get(uint32_t w0, uint32_t w1, uint32_t sc, int, const Consts &c) {
        const f16x2 s = as_h2(sc), d = splat(s[0]), m = -splat(s[1]);
        const f16x2 p0 = __builtin_elementwise_fma(byte_pair(w0, 0, c.b, 1024.0f), d, m);
        const f16x2 p1 = __builtin_elementwise_fma(byte_pair(w0, 1, c.b, 1024.0f), d, m);
        const f16x2 p2 = __builtin_elementwise_fma(byte_pair(w1, 0, c.b, 1024.0f), d, m);
        const f16x2 p3 = __builtin_elementwise_fma(byte_pair(w1, 1, c.b, 1024.0f), d, m);
        return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    }
};

template <>
struct Staged<VT_Q6_K> {
    static constexpr bool PER_STEP = false;
    static constexpr int NU = 1;
    struct Regs {
        uint4 ql[4], qh[2];
        uint2 sc;
        uint32_t d;
    };
    struct Lds {
        uint4 ql[256], qh[128];
        uint4 sc[64];
    };
    // pair t: half t % 2 of super-block t / 2 (Rows<VT_Q6_K>)
    static VH_DEV void load(Regs &r, gbyte *const (&B)[2], int64_t rb, int t, int lane) {
        const int sb = 210 * (t >> 1), h = t & 1;
        const uint32_t ol = here(uint32_t(lane >> 2) * uint32_t(rb) + 16u * uint32_t(lane & 3)),
                       oh = here(uint32_t(lane >> 1) * uint32_t(rb) + 16u * uint32_t(lane & 1));
#pragma unroll
        for (int q = 0; q < 4; q++) r.ql[q] = ld_u128(B[q >> 1] + (16 * (q & 1)) * rb + sb + 64 * h + ol);
#pragma unroll
        for (int q = 0; q < 2; q++) r.qh[q] = ld_u128(B[q] + sb + 128 + 32 * h + oh);
        gbyte *p = (lane < 32 ? B[0] : B[1]) + sb + uint32_t(lane & 31) * uint32_t(rb);
        r.sc = ld_u64(p + 192 + 8 * h);
        r.d = ld_u16(p + 208);
    }
    static VH_DEV void bounds(const Regs &r, float (&b)[NU]) { b[0] = fabsf(h2f(r.d)) * (128.0f * 32.0f); }
    static VH_DEV float of_row(const float (&v)[NU], int j, int col) { return __shfl(v[0], 32 * j + col, 64); }
    static VH_DEV void put(Lds &l, const Regs &r, const float (&up)[NU], int lane) {
        const int a = 4 * (lane >> 2) + ((lane & 3) ^ (lane >> 4)), b = 2 * (lane >> 1) + ((lane & 1) ^ ((lane >> 4) & 1));
#pragma unroll
        for (int q = 0; q < 4; q++) l.ql[64 * q + a] = r.ql[q];
#pragma unroll
        for (int q = 0; q < 2; q++) l.qh[64 * q + b] = r.qh[q];
        const float d = h2f(r.d) * up[0];
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v = i < 2 ? r.sc.x : r.sc.y;
            o[i] = h_bits(d * float(int(int8_t(v >> (16 * (i & 1)))))) | h_bits(d * float(int(int8_t(v >> (16 * (i & 1) + 8))))) << 16;
        }
        l.sc[lane] = make_uint4(o[0], o[1], o[2], o[3]);
    }
    static VH_DEV void fetch(const Lds &l, int p, int i, int j, int half, int col, uint32_t (&w)[4]) {
        const uint4 v = l.ql[128 * j + 4 * col + ((2 * half + i) ^ ((col >> 2) & 3))];
        const uint4 h = l.qh[64 * j + 2 * col + (i ^ ((col >> 3) & 1))];
        const int sl = 4 * p, sh = 4 * p + 2 * half;
#pragma unroll
        for (int x = 0; x < 4; x++)
            w[x] = ((u4_at(v, x) >> sl) & 0x0f0f0f0fu) | (((u4_at(h, x) >> sh) & 0x03030303u) << 4);
    }
    static VH_DEV f16x8 get(uint32_t w0, uint32_t w1, uint32_t sc, int ks, const Consts &c) {
        const f16x2 d = splat(as_h2(sc)[ks >> 1]);
        const f16x2 p0 = byte_pair(w0, 0, c.b, 1056.0f) * d, p1 = byte_pair(w0, 1, c.b, 1056.0f) * d;
        const f16x2 p2 = byte_pair(w1, 0, c.b, 1056.0f) * d, p3 = byte_pair(w1, 1, c.b, 1056.0f) * d;
        return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    }
};

}  // namespace
