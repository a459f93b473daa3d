// Decode-batch projections of Q8_0 experts on the matrix cores, for calls of
// kQ8decMinTokens to kMfmaMinCall - 1 tokens. The fp32 kernels (moe_gdec.hip)
// convert and multiply every weight again for each token of its expert and are
// bound by the vector ALUs (23 OLMoE tokens: 104 + 54 us per layer, where reading
// the experts takes 80); here a weight becomes a matrix operand once for up to 32
// tokens: 54 + 43 us, gate/up at 5 TB/s, down at 3 (its arrivals and the combine
// are a tail of round trips).
//
// v_mfma_f32_16x16x32_f16: 16 tokens x 16 weight rows x one block of 32 weights.
// The operand holds the quants themselves (exact in fp16) and each block's sum
// is scaled by its d in fp32 (src/gguf_compute.c:112-120, the sums of :127-157).
// Inputs are split into fp16 parts hi + lo (22 significant bits, under a power
// of two per token: mdec_prep_kernel, natural order), one multiply each; the
// activations h the same way under a power of two per (pair, 32 columns), which
// enters the block's scale in the down projection. Products are exact in fp32, so
// the results differ from the fp32 kernels' by the order of the sums and 2^-23 of
// the inputs, which are no larger than theirs (q8_stream).
//
// A wave owns two 32-row fragments (gate/up: 32 rows of gate and the same of
// up; down: 64 rows) of the layout of mfma_frag.h - the copy the prefill GEMMs
// read, or the GGUF rows: the same words, the same bits - whose lanes hold a
// whole block of their row each. Four lane groups of 16 thus hold the blocks of
// four (16 rows, block) operands, and a 4 x 4 transposition of 8-byte chunks over
// the groups (eight v_permlane swaps) gives every group its quarter of each.
//
// Grid (128 columns of h, or 256 rows of down; expert), four waves; the
// workgroup lists its expert's tokens itself (expert_group.h). The last of a
// token's k experts to write a workgroup's rows adds them into x in selection
// order, as mdec_down_kernel (moe_mdec.hip) does.
#include <hip/hip_runtime.h>
#include <type_traits>
#include "common.h"
#include "expert_group.h"
#include "mfma_frag.h"
#include "route.h"
#include "route_kernels.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr int kTok = 16;                  // tokens per matrix tile; NT of them per pass over the weights

template <bool PK>
struct Q8Lds {
    int list[kGroupMax], wc[4], last[kGroupMax + 1];
    std::conditional_t<PK, int, Staged<VT_Q8_0>::Lds> rows[4];  // a wave's GGUF rows
};

VH_DEV void swap32(uint32_t &a, uint32_t &b) {  // a's upper 32 lanes with b's lower
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
VH_DEV void swap16(uint32_t &a, uint32_t &b) {  // a's odd rows of 16 lanes with b's even ones
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// eight bytes q + 128 as fp16 q
VH_DEV f16x8 q8_operand(uint32_t w0, uint32_t w1, uint32_t kb) {
    f16x8 o;
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const uint32_t v = __builtin_amdgcn_perm(p < 2 ? w0 : w1, kb, (p & 1) ? 0x00070006u : 0x00050004u);
        const f16x2 y = as_h2(v) - splat(_Float16(1152.0f));
        o[2 * p] = y[0];
        o[2 * p + 1] = y[1];
    }
    return o;
}

// acc[j][h][n]: rows 16 h .. + 15 of fragment j times the tokens 16 n .. of the
// pass (lane l: row l % 16, tokens 4 (l / 16) .. + 3). A row of x is K x 4 bytes
// (chunks of 8 inputs: hi parts, then lo); row_of(i) is the pass's token i's.
// hs (down): the scales of h per row and block. A wave reads its inputs' operands
// itself, with its weights (the other waves' reads of the same lines hit the
// L1), so no barrier ties its stream to theirs (inputs staged for the workgroup:
// gate/up 75 us at 23 OLMoE tokens). GGUF rows (rows0, rows1: the fragments' first)
// pass through the wave's own LDS: with a row per lane a load instruction touched
// 64 lines, Qwen3 16 tokens gate/up 166 -> 95 us, down 78 -> 56 (the fp32 kernels
// 101 and 61, from the copy 67 and 48).
template <bool PK, bool DOWN, int NT, class Area, class RowOf>
VH_DEV void q8_stream(gbyte *F, gbyte *rows0, gbyte *rows1, Area &lds, const void *x, const float *hs, int K, int tn,
                      RowOf row_of, f32x4 (&acc)[2][2][NT]) {
    constexpr int SETS = NT == 1 ? 4 : 2;  // K steps of weights in flight; of inputs (from the L2), two
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, half = lane >> 5, nk = K / kBK;
    uint32_t kb = 0x64646464u;
    asm volatile("" : "+v"(kb));
    gbyte *xb = gmem(x), *sb = gmem(hs);
    uint32_t xr[NT], sr[NT][4];  // at most 63 x 64 rows of K x 4 bytes: 32-bit offsets
#pragma unroll
    for (int n = 0; n < NT; n++) {
        xr[n] = uint32_t(row_of(min(16 * n + r, tn - 1))) * uint32_t(K) * 4u + 32u * uint32_t(g);
        if constexpr (DOWN)
#pragma unroll
            for (int i = 0; i < 4; i++)
                sr[n][i] = uint32_t(row_of(min(16 * n + 4 * g + i, tn - 1))) * uint32_t(K / 32) * 4u;
    }
    using S = Staged<VT_Q8_0>;
    struct Set {
        uint32_t w[2][8], d[2];
    } st[PK ? SETS : 1];
    typename S::Regs rg[PK ? 1 : SETS / 2];  // pairs of steps in flight
    gbyte *const B[2] = {rows0, rows1};
    const int64_t rb = int64_t(K / 32) * 34;
    struct In {
        uint4 h[2][NT], l[2][NT];
        uint2 sc[DOWN ? NT : 1][4];
    } in[2];
    auto load = [&](Set &q, int s) {
#pragma unroll
        for (int j = 0; j < 2; j++)
            Frag<VT_Q8_0>::load(F + (size_t(s) * 2 + j) * Frag<VT_Q8_0>::bytes, lane, q.w[j], q.d[j]);
    };
    auto load_in = [&](In &q, int s) {
#pragma unroll
        for (int n = 0; n < NT; n++) {
#pragma unroll
            for (int k = 0; k < 2; k++) {  // block k of the step: chunk 4 k + g
                q.h[k][n] = ld_u128(xb + 256 * s + 128 * k + xr[n]);
                q.l[k][n] = ld_u128(xb + 256 * s + 128 * k + 16 + xr[n]);
            }
            if constexpr (DOWN)
#pragma unroll
                for (int i = 0; i < 4; i++) q.sc[n][i] = ld_u64(sb + 8 * s + sr[n][i]);
        }
    };
#pragma unroll
    for (int i = 0; i < (PK ? SETS : SETS / 2); i++) {
        if constexpr (PK) load(st[i], min(i, nk - 1));
        else S::load(rg[i], B, rb, min(i, nk / 2 - 1), lane);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) load_in(in[i], min(i, nk - 1));
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int n = 0; n < NT; n++) acc[j][h][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Gate/up adds four blocks in fp32 and these sums in fp64, down eight blocks and
    // these sums in fp32. In one fp32 chain of all 2 nk blocks the roundings left the
    // layer 2.9e-7 (2-norm) from 64 bits, the fp32 kernels' many short chains
    // (moe_gdec.hip) 1.86e-7; so it is 1.80e-7 (OLMoE and Qwen3, 9 to 63 tokens), at
    // the same speed.
    f32x4 sub[2][2][NT];
    f64x4 tot[2][2][DOWN ? 1 : NT];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int n = 0; n < (DOWN ? 1 : NT); n++) tot[j][h][n] = f64x4{0., 0., 0., 0.};
    // pair s / 2 of GGUF rows into place; other lanes' reads of the last lie before, those of this one after
    auto place = [&](int s, typename S::Regs &r) {
        if constexpr (!PK) {
            wave_fence();
            S::put(lds, r, lane);
            wave_fence();
        }
    };
    auto request = [&](int s, typename S::Regs &r) {
        if constexpr (!PK) {
            __builtin_amdgcn_sched_barrier(0);
            S::load(r, B, rb, min(s / 2 + SETS / 2, nk / 2 - 1), lane);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto step = [&](int s, Set &t, In &x, bool first) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            uint32_t q[8], dj;
            if constexpr (PK) {
#pragma unroll
                for (int i = 0; i < 8; i++) q[i] = t.w[j][i];
                dj = t.d[j];
            } else {
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    uint32_t w[4];
                    S::fetch(lds, s & 1, i, j, half, lane & 31, w, dj);
#pragma unroll
                    for (int k = 0; k < 4; k++) q[4 * i + k] = w[k];
                }
            }
            swap32(q[0], q[4]);
            swap32(q[1], q[5]);
            swap32(q[2], q[6]);
            swap32(q[3], q[7]);
            swap16(q[0], q[2]);
            swap16(q[1], q[3]);
            swap16(q[4], q[6]);
            swap16(q[5], q[7]);
            uint32_t d0 = dj, d2 = dj;
            swap32(d0, d2);
            uint32_t d1 = d0, d3 = d2;
            swap16(d0, d1);
            swap16(d2, d3);
            const float d[4] = {h2f(d0), h2f(d1), h2f(d2), h2f(d3)};
            // operand m: rows 16 (m % 2) .. of the fragment, block m / 2 of the step
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const f16x8 o = q8_operand(q[2 * m], q[2 * m + 1], kb);
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    f32x4 c = {0.f, 0.f, 0.f, 0.f};
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x.h[m >> 1][n]), o, c, 0, 0, 0);
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x.l[m >> 1][n]), o, c, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float f = DOWN ? d[m] * __uint_as_float(m >> 1 ? x.sc[DOWN ? n : 0][i].y : x.sc[DOWN ? n : 0][i].x) : d[m];
                        sub[j][m & 1][n][i] = first && m < 2 ? f * c[i] : fmaf(f, c[i], sub[j][m & 1][n][i]);
                    }
                    // added here: left for later, every block's products would be held in registers
                    asm volatile("" : "+v"(sub[j][m & 1][n]));
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // the inputs first: loads arrive in order, so the wait for them in two steps
        // would include every load of weights issued before them
        load_in(x, min(s + 2, nk - 1));
        if constexpr (PK) load(t, min(s + SETS, nk - 1));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto add = [&] {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    if constexpr (DOWN) acc[j][h][n] += sub[j][h][n];
                    else tot[j][h][n] += __builtin_convertvector(sub[j][h][n], f64x4);
                }
    };
    // steps s, s + 1 from set 2 `i`: the first of the sum where `first`
    auto pair = [&](int s, auto I, bool first) {
        constexpr int i = SETS == 4 ? decltype(I)::value : 0;
        place(s, rg[PK ? 0 : i]);
        step(s, st[PK ? 2 * i : 0], in[0], first);
        step(s + 1, st[PK ? 2 * i + 1 : 0], in[1], false);
        request(s, rg[PK ? 0 : i]);
        if (!DOWN) add();
    };
    const std::integral_constant<int, 0> i0;
    const std::integral_constant<int, 1> i1;
    for (int s = 0; s < nk; s += 4) {  // nk is even
        pair(s, i0, true);
        if (s + 2 < nk) pair(s + 2, i1, !DOWN);
        if (DOWN) add();
    }
    if constexpr (!DOWN)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int n = 0; n < NT; n++) acc[j][h][n] = __builtin_convertvector(tot[j][h][n], f32x4);
}

struct Q8Args {
    const void *const *table;
    const void *x;        // gate/up: the split inputs [T]; down: the split activations [pairs]
    const float *xsc;     // gate/up: the tokens' scales
    uint16_t *hp;         // gate/up: the activations [pairs x fe x 2]
    float *hs;            // and their block scales [pairs x fe / 32]
    float *y;             // down: [pairs x d]
    int d, fe;
    bool combine;         // down: x += the weighted rows; else rows only, those of the table's experts
    MdecSelf sf;
};

// the largest of v over the 16 lanes of a row of lanes
VH_DEV float row_max(float v) {
    v = fmaxf(v, dpp_keep<0xB1>(v));
    v = fmaxf(v, dpp_keep<0x4E>(v));
    v = fmaxf(v, dpp_keep<0x141>(v));
    return fmaxf(v, dpp_keep<0x140>(v));
}

template <bool PK, int NT>
VH_DEV void gateup_pass(Q8Lds<PK> &L, const Q8Args &a, gbyte *G, gbyte *U, int c, int t0, int tn) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, nk = a.d / kBK;
    const int64_t rb = int64_t(a.d / 32) * 34;
    f32x4 acc[2][2][NT];
    q8_stream<PK, false, NT>(G + size_t(c) * nk * 2 * Frag<VT_Q8_0>::bytes, G + 32 * c * rb, U + 32 * c * rb, L.rows[c & 3],
                             a.x, nullptr, a.d, tn,
                             [&](int i) { return L.list[t0 + i] / a.sf.k; }, acc);
    float rs[2][2] = {{1.0f, 1.0f}, {1.0f, 1.0f}};  // the rows' powers of two in the packed copy
    if constexpr (PK) {
        gbyte *p = G + size_t(2) * a.fe / 32 * nk * Frag<VT_Q8_0>::bytes;
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int h = 0; h < 2; h++) rs[j][h] = __uint_as_float(ld_u32(p + 4 * (j * a.fe + 32 * c + 16 * h + r)));
    }
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int tt = 16 * n + 4 * g + i, pair = L.list[t0 + min(tt, tn - 1)];
            const float sc = a.xsc[pair / a.sf.k];
            float h[2];
#pragma unroll
            for (int x = 0; x < 2; x++)
                h[x] = swiglu(acc[0][x][n][i] * rs[0][x] * sc, acc[1][x][n][i] * rs[1][x] * sc);
            // the block's power of two: |h| < 2^e, kept as h 2^(14 - e) in fp16 parts
            const uint32_t m = __float_as_uint(row_max(fmaxf(fabsf(h[0]), fabsf(h[1]))));
            const int e = m ? max(-100, min(127, int(m >> 23) - 126)) : 0;
            if (tt >= tn) continue;
            const float up = __uint_as_float(uint32_t(127 + 14 - e) << 23);
            if (r == 0) a.hs[size_t(pair) * (a.fe / 32) + c] = ldexpf(1.0f, e - 14);
#pragma unroll
            for (int x = 0; x < 2; x++) {
                const int o = 32 * c + 16 * x + r;
                const float v = h[x] * up;
                const _Float16 hi = _Float16(v);
                uint16_t *p = a.hp + size_t(pair) * a.fe * 2 + (o >> 3) * 16 + (o & 7);
                p[0] = __builtin_bit_cast(uint16_t, hi);
                // no low part of an infinity (h overflowed): it would be a NaN
                p[8] = __builtin_bit_cast(uint16_t, fabsf(v) < 65520.0f ? _Float16(v - float(hi)) : _Float16(0.0f));
            }
        }
}

template <bool PK, int NT>
__global__ void __launch_bounds__(256, 2) q8dec_gateup_kernel(Q8Args a) {
    __shared__ Q8Lds<PK> L;
    if (blockIdx.x == 0 && blockIdx.y == 0)  // the down kernel's counters start at 0
        for (int i = threadIdx.x; i < a.sf.nctr; i += 256) a.sf.ctr[i] = 0u;
    const int e = blockIdx.y, cnt = expert_group<256>(a.sf.idx, a.sf.T * a.sf.k, e, L.list, L.wc);
    if (cnt == 0) return;
    gbyte *G = gmem(a.table[3 * e]), *U = gmem(a.table[3 * e + 1]);
    if (!G || !U) return;  // an unregistered expert: the down kernel writes zeros (src/gguf_run.c:201)
    const int c = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int t0 = 0; t0 < cnt; t0 += NT * kTok) gateup_pass<PK, NT>(L, a, G, U, c, t0, min(NT * kTok, cnt - t0));
}

template <bool PK, int NT>
VH_DEV void down_pass(Q8Lds<PK> &L, const Q8Args &a, gbyte *D, int c, int t0, int tn) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, nk = a.fe / kBK;
    const int64_t rb = int64_t(a.fe / 32) * 34;
    f32x4 acc[2][2][NT];
    if (D) {
        q8_stream<PK, true, NT>(D + size_t(c) * nk * 2 * Frag<VT_Q8_0>::bytes, D + 64 * c * rb, D + (64 * c + 32) * rb,
                                L.rows[c & 3], a.x, a.hs, a.fe, tn,
                                [&](int i) { return L.list[t0 + i]; }, acc);
    } else {  // an unregistered expert's rows are zeros, which the combine adds without changing a bit
#pragma unroll
        for (int x = 0; x < 4 * NT; x++) acc[x / 2 / NT][x / NT % 2][x % NT] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    gbyte *p = D + size_t(a.d) / 32 * nk * Frag<VT_Q8_0>::bytes;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int o = 64 * c + 32 * j + 16 * h + r;
            const float rs = PK && D ? __uint_as_float(ld_u32(p + 4 * o)) : 1.0f;
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int tt = 16 * n + 4 * g + i;
                    if (tt < tn)
                        __hip_atomic_store(&a.y[size_t(L.list[t0 + tt]) * a.d + o], acc[j][h][n][i] * rs,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
        }
}

template <bool PK, int NT>
__global__ void __launch_bounds__(256, 2) q8dec_down_kernel(Q8Args a) {
    __shared__ Q8Lds<PK> L;
    constexpr int CR = 256;  // output rows of one workgroup
    const MdecSelf &sf = a.sf;
    const int tid = threadIdx.x, e = blockIdx.y, k = sf.k, d = a.d;
    const int cnt = expert_group<256>(sf.idx, sf.T * k, e, L.list, L.wc);
    if (cnt == 0) return;
    gbyte *D = gmem(a.table[3 * e + 2]);
    if (!D && !a.combine) return;
    const int c = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int t0 = 0; t0 < cnt; t0 += NT * kTok) down_pass<PK, NT>(L, a, D, c, t0, min(NT * kTok, cnt - t0));
    if (!a.combine) return;
    // the combine (src/gguf_run.c:208-212; see mdec_down_kernel): rows out as
    // agent-scope stores, one arrival per token once they are done, and the
    // workgroup that brings a token's count to k reads its k rows past the L2
    if (tid == 0) L.last[kGroupMax] = 0;
    VH_WAIT_VMCNT(0);
    __syncthreads();
    if (tid < cnt) {
        const int t = L.list[tid] / k;
        const uint32_t n = __hip_atomic_fetch_add(&sf.ctr[blockIdx.x * kGroupMax + t], 1u, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
        if (n == uint32_t(k - 1)) L.last[atomicAdd(&L.last[kGroupMax], 1)] = t;
    }
    __syncthreads();
    const int nl = L.last[kGroupMax], o = blockIdx.x * CR + tid;
    constexpr int KB = 8;  // rows of y in flight per thread and token
    for (int i = 0; i < nl; i++) {
        const int t = L.last[i];
        float s = 0.0f;
        const float xo = sf.x[size_t(t) * d + o];
        for (int j0 = 0; j0 < k; j0 += KB) {
            float yv[KB];
#pragma unroll
            for (int j = 0; j < KB; j++)
                yv[j] = __hip_atomic_load(&a.y[(size_t(t) * k + min(j0 + j, k - 1)) * d + o], __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int j = 0; j < KB; j++)
                if (j0 + j < k) s = add_rn(s, mul_rn(sf.w[size_t(t) * k + j0 + j], yv[j]));
        }
        sf.x[size_t(t) * d + o] = add_rn(xo, s);
    }
}

template <int NT>
void q8dec_launch(Q8Args a, bool packed, int E, const void *hp, hipStream_t s) {
    const dim3 gg(a.fe / 128, E), gd(a.d / 256, E), b(256);
    if (packed) hipLaunchKernelGGL((q8dec_gateup_kernel<true, NT>), gg, b, 0, s, a);
    else hipLaunchKernelGGL((q8dec_gateup_kernel<false, NT>), gg, b, 0, s, a);
    a.x = hp;
    if (packed) hipLaunchKernelGGL((q8dec_down_kernel<true, NT>), gd, b, 0, s, a);
    else hipLaunchKernelGGL((q8dec_down_kernel<false, NT>), gd, b, 0, s, a);
}

}  // namespace

bool vh_q8dec_supported(uint32_t tg, uint32_t td, int d, int fe, int T) {
    return tg == VT_Q8_0 && td == VT_Q8_0 && d % 256 == 0 && fe % 128 == 0 && T <= kGroupMax;
}

int vh_q8dec(const void *const *table, bool packed, const void *xp, const float *xsc, int d, int fe, int E, void *hp,
             float *hs, float *ybuf, const MdecSelf &self, bool combine, hipStream_t s) {
    if (!vh_q8dec_supported(VT_Q8_0, VT_Q8_0, d, fe, self.T) || self.T < 1 || self.k < 1 || !self.x || !self.w ||
        self.nctr < vh_mdec_ctr_words(d))
        return -EINVAL;
    const Q8Args a{table, xp, xsc, static_cast<uint16_t *>(hp), hs, ybuf, d, fe, combine, self};
    // two token tiles per pass where the average expert has more than half a tile (its registers keep two waves
    // per SIMD, one tile's four)
    if (2 * self.T * self.k > kTok * E) q8dec_launch<2>(a, packed, E, hp, s);
    else q8dec_launch<1>(a, packed, E, hp, s);
    return vh_check(hipGetLastError());
}
