// fp16 matrix-core (MFMA) grouped GEMMs for the groups of large calls.
//
// moe_ffn (src/gguf_run.c:193-213) runs every (token, expert) pair as two
// matvecs; when a call carries many tokens, an expert's tokens form a group
// and its projections become GEMMs: H_e = silu(X_e G_e^T) * (X_e U_e^T) and
// Y_e = H_e D_e^T, with X_e the group's rows of hb gathered through the
// dispatch permutation. Every group of a call of at least kMfmaMinCall
// tokens runs here on v_mfma_f32_32x32x16_f16 with fp32 accumulation.
//
// Numbers: both operands are fp16 (11 significant bits) under power-of-two
// scales, which cost nothing in precision and take fp16's narrow range out of
// play: a token's inputs by its largest magnitude (to below 2^14), a weight
// row by a bound on its largest magnitude (row_exponent), the activations h
// per (pair, 32 columns) by the block's largest. A weight is formed from its
// exact quant by packed fp16 operations: Q8_0 and Q6_K (q - 32) times the
// rounded scale, Q4_K one fused d1 q - m1 on the rounded d1 and m1. On the
// benchmark's shapes the layer's output lies 4 to 8 times closer to a 64-bit
// evaluation than with both operands rounded to bf16, and a weight costs 1.5
// (Q8_0), 1.6 (Q4_K) or 2.4 (Q6_K) vector instructions where bf16 rounding
// through fp32 took 2.8 to 4.
//
// Tiles: a workgroup of four waves owns a token tile of 32, 64 or 128 rows of
// one group and 256 weight rows, 64 per wave (gate/up: 32 of gate and the same
// 32 of up; down: 64), and steps over K in kBK = 64 columns. Each wave
// dequantizes its own 64 rows in registers and multiplies all of the tile's
// rows by them, so a weight is converted once per workgroup and an input
// fragment read from LDS feeds two multiplies (with 32 rows per wave the
// operand reads alone took all of the LDS bandwidth). The inputs pass through
// LDS in three buffers (two: TileLds) as 16-byte chunks of 8 consecutive K values
// laid out [K/8][row] (row index XOR-swizzled by the chunk), so a 32-lane group's
// operand read is one contiguous 512-byte run. Two workgroups share a CU:
// 256 registers, two waves per SIMD, one converting while the other multiplies.
//
// Weights: the experts of a pinned layer come from a copy in the operand order
// (Frag, vh_mfma_pack); others are read from their GGUF rows, each wave's through
// its own part of LDS (Staged), into the same operands, so the results do not
// depend on the source. Per layer, GGUF rows / copy: Qwen3 Q4_K_M 101 tokens 233 /
// 178 us, 2048 465 / 396; Q8_0 253 / 198 and 498 / 410 (2048 tokens through the
// kernel that staged bf16 weights for the whole workgroup: 672 and 540).
//
// Order: the workgroups are numbered so that each XCD (hardware dispatch sends
// workgroup b to XCD b mod 8) takes a contiguous run of (token tile, column
// tile) pairs, column tiles fastest: the workgroups sharing a token tile, and
// the consecutive token tiles of one expert that share its weight tiles, meet
// in the same L2. The runs are cut at equal shares of the staged bytes.
//
// Outputs: gate/up writes h as fp16 rows in dispatch order (hs[offs[e] + i])
// with their block exponents (he), so the down GEMM reads its A operand
// contiguously; down writes the fp32 row y[pair] that the combine kernel reads,
// as on the fp32 plan.
#include <hip/hip_runtime.h>
#include <vector>
#include <algorithm>
#include <type_traits>
#include "common.h"
#include "mfma_frag.h"
#include "route_kernels.h"

namespace {

constexpr int kBRows = 256, kWaves = 4, kThreads = 64 * kWaves, kXcds = 8;
constexpr int kChunks = kBK / 8;  // 16-byte chunks per row and K step
constexpr int kBigTile = 128, kSmallTile = 64;  // the largest token tile of the two kernels (tile_rows)

struct GemmArgs {
    const int32_t *tiles, *perm;
    const void *const *table;
    const uint8_t *src;   // A: gate/up: xb [T x K] fp16; down: hs [P x K] fp16
    const float *xsc;     // gate/up: the tokens' scales [T]
    int8_t *he;           // block exponents of hs [P x fe / 32] (gate/up writes, down reads)
    void *out;            // gate/up: hs; down: y [P x rows]
    int K, rows, k;
    int64_t row_bytes;    // GGUF rows
};

// Half of a max-reduction of N pairs of values over lanes: lanes with `hi` set
// keep m[r + N], the others m[r], each the larger of its own and of the lane
// that CTRL reads (one whose `hi` is the other way).
template <int CTRL, int N>
VH_DEV void fold(float (&m)[16], bool hi) {
#pragma unroll
    for (int r = 0; r < N; r++) {
        const float own = hi ? m[r + N] : m[r], other = hi ? m[r] : m[r + N];
        m[r] = fmaxf(own, dpp_keep<CTRL>(other));
    }
}

// 2^n as fp16 bits, n <= 0 (0 below 2^-24)
VH_DEV uint32_t h_pow2(int n) { return n >= -14 ? uint32_t(15 + n) << 10 : n >= -24 ? 1u << (24 + n) : 0u; }

constexpr int kFacBlocks = 32;  // blocks of h whose factors are in LDS at a time

// LDS of a workgroup. The inputs have three buffers (the step's, the next one's
// and the one being written), or two where the staged rows (Staged) leave no room
// for a third in half of a CU's 160 KB.
template <int T, bool GATEUP, int LDB, bool PK>
constexpr int input_bufs() { return !PK && (T == VT_Q8_0 || (LDB == kBigTile && T == VT_Q6_K && !GATEUP)) ? 2 : 3; }
struct NoRows {};

template <int T, bool GATEUP, int LDB, bool PK>
struct TileLds {
    static constexpr int NB = input_bufs<T, GATEUP, LDB, PK>();
    f16x8 As[NB][kChunks][LDB];
    std::conditional_t<PK, NoRows, typename Staged<T>::Lds> rows[kWaves];
    float rsc[LDB];                                  // the rows' scales in the epilogue
    float hsc[GATEUP ? kWaves : 1][32];              // gate/up: a wave's 32 row scales of h
    int prow[GATEUP ? 1 : LDB];                      // down: the rows' y rows
    uint16_t fac[GATEUP ? 1 : kFacBlocks][GATEUP ? 1 : LDB];  // and the factors of their blocks of h (fp16)
};

// One token tile of BM rows against the wave's two 32-row fragments, by the
// kWaves waves of mfma_gemm_kernel. GATEUP: A row i is xb row perm[i] / k, the
// weights gate and up, out = hs row i and its block exponents; else A row i is
// hs row i, scaled to the row's largest block as it is staged, out = y row
// perm[i]. i runs over base + m0 .. + mcnt - 1 (mcnt <= BM) within the group;
// rows of the tile past mcnt repeat the group's last row and are not stored.
//
// K step s: the inputs of step s + 2 (s + 1 with two buffers) go from registers
// into LDS and the next ones are requested; the wave multiplies step s, forming
// its operands from the weights requested two steps ago (GGUF rows: a pair of steps)
// and requests more. Every load is unconditional (steps past the end repeat
// the last one), so the waits count exactly the loads issued after the one needed,
// and the barrier is LDS-only: loads stay in flight across it.
template <int T, bool GATEUP, int BM, int LDB, bool PK>
VH_DEV void gemm_tile(TileLds<T, GATEUP, LDB, PK> &L, const GemmArgs &a, gbyte *M0, gbyte *M1, int base, int m0, int mcnt,
                      int n0) {
    using O = Op<T>;
    constexpr int FI = BM / 32, AQ = BM * kChunks / kThreads;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5;
    const int K = a.K, nk = K / kBK;
    const Consts cst;
    // input staging: slot tid + 256 q holds K chunk kc = tid % 8 of tile row tid / 8 + 32 q
    const int kc = tid & 7, rq = tid >> 3, nblk = K / 32;
    gbyte *abase = gmem(a.src);
    uint32_t aoff[AQ];
#pragma unroll
    for (int q = 0; q < AQ; q++) {
        const int r = rq + 32 * q, i = base + m0 + min(r, mcnt - 1);
        const int t = GATEUP ? a.perm[i] / a.k : i;
        aoff[q] = uint32_t(size_t(t) * K * 2) + 16u * uint32_t(kc);
        if constexpr (GATEUP) {
            if (kc == 0) L.rsc[r] = a.xsc[t];
        }
    }
    // down: the factors 2^(block exponent - row exponent) of kFacBlocks blocks of
    // h, from block b0 on: two threads per row, half of the blocks each
    auto factors = [&](int b0, int e) {
        if (tid < 2 * BM) {
            const int r = tid >> 1;
            gbyte *he = gmem(a.he) + size_t(base + m0 + min(r, mcnt - 1)) * nblk;
            uint32_t w[kFacBlocks / 8];
#pragma unroll
            for (int x = 0; x < kFacBlocks / 8; x++)  // nblk is a multiple of 4; words past the end repeat the last
                w[x] = ld_u32(he + min(b0 + 4 * (kFacBlocks / 8 * (tid & 1) + x), nblk - 4));
            if (b0 == 0) {  // the row's exponent: its largest block's
                e = -128;
#pragma unroll
                for (int x = 0; x < kFacBlocks / 2; x++) e = max(e, int(int8_t(w[x >> 2] >> (8 * (x & 3)))));
                for (int b = kFacBlocks + 4 * (tid & 1); b < nblk; b += 8) {
                    const uint32_t v = ld_u32(he + b);
#pragma unroll
                    for (int x = 0; x < 4; x++) e = max(e, int(int8_t(v >> (8 * x))));
                }
                e = max(e, int(dpp_u<0xB1>(uint32_t(e))));
                if (!(tid & 1)) {
                    L.rsc[r] = ldexpf(1.0f, e - 14);
                    L.prow[r] = a.perm[base + m0 + min(r, mcnt - 1)];
                }
            }
#pragma unroll
            for (int x = 0; x < kFacBlocks / 2; x++)
                L.fac[kFacBlocks / 2 * (tid & 1) + x][r] = uint16_t(h_pow2(int(int8_t(w[x >> 2] >> (8 * (x & 3)))) - e));
        }
        return e;
    };
    uint4 av[AQ];
    auto loadA = [&](int step) {
#pragma unroll
        for (int q = 0; q < AQ; q++) av[q] = ld_u128(abase + 128 * step + (PK ? aoff[q] : here(aoff[q])));
    };
    auto storeA = [&](int buf, int step) {
#pragma unroll
        for (int q = 0; q < AQ; q++) {
            f16x8 v = __builtin_bit_cast(f16x8, av[q]);
            if constexpr (!GATEUP) {
                const _Float16 f = __builtin_bit_cast(_Float16, L.fac[(2 * step + (kc >> 2)) % kFacBlocks][rq + 32 * q]);
                v = v * f16x8{f, f, f, f, f, f, f, f};
            }
            L.As[buf][kc][(rq ^ kc) + 32 * q] = v;
        }
    };

    // the wave's weights: fragment group c of the packed matrix, or the lane's two GGUF rows
    const int c = n0 / (GATEUP ? 32 : 64) + wv, col = lane & 31;
    gbyte *fb = M0 + size_t(c) * nk * 2 * Frag<T>::bytes;
    float rs[2];  // the inverses of the rows' powers of two, for the epilogue
    if constexpr (PK) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int r = GATEUP ? 32 * c + col : 64 * c + 32 * j + col;
            const size_t frags = size_t(GATEUP ? 2 : 1) * a.rows / 32 * nk * Frag<T>::bytes;
            rs[j] = __uint_as_float(ld_u32(M0 + frags + 4 * (GATEUP ? j * a.rows + r : r)));
        }
    }

    f32x16 acc[FI][2];
#pragma unroll
    for (int i = 0; i < FI; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    // The operands of sub-step ks + 1 are formed, and its input fragments read,
    // between the multiplies of sub-step ks (across the step's barrier too where
    // there are three input buffers: the inputs of step s + 1 have been in LDS
    // since the barrier before), so a wave's vector instructions run in the shadow
    // of its own multiplies.
    constexpr int NB = TileLds<T, GATEUP, LDB, PK>::NB, AHEAD = NB - 1;
    int rowe = 0;  // down, threads 2 r and 2 r + 1: row r's exponent
    f16x8 af[FI], b[2], bn[2];
    auto readA = [&](int buf, int ks, int i) {
        const int kg = 4 * half + ks;
        af[i] = L.As[buf][kg][(col ^ kg) + 32 * i];
    };
    // step s's start: the inputs of step s + AHEAD into buffer `buf`, the next ones requested
    auto stage_inputs = [&](int s, int buf) {
        if constexpr (!GATEUP)
            if ((s + AHEAD) % (kFacBlocks / 2) == 0 && s + AHEAD < nk) {  // the next blocks' factors (every 16 steps)
                lds_barrier();
                factors(2 * (s + AHEAD), rowe);
                lds_barrier();
            }
        storeA(buf, s + AHEAD);
        loadA(min(s + AHEAD + 1, nk - 1));
        __builtin_amdgcn_sched_barrier(0);  // the loads stay where they are issued
    };
    // sub-step ks of a step in buffer b0, the next step's in b1
    auto multiply = [&](int ks, int b0, int b1) {
#pragma unroll
        for (int i = 0; i < FI; i++) {
#pragma unroll
            for (int j = 0; j < 2; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], b[j], acc[i][j], 0, 0, 0);
            if (NB == 3 || ks < 3) readA(ks < 3 ? b0 : b1, (ks + 1) & 3, i);
        }
        b[0] = bn[0];
        b[1] = bn[1];
#pragma unroll
        for (int i = 0; i < 2 * FI; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                    // a multiply
            __builtin_amdgcn_sched_group_barrier(0x002, 20 / FI, 0);      // vector instructions
            if (i & 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);         // an LDS read
        }
    };
    auto end_step = [&](int b1) {
        lds_barrier();
        if constexpr (NB == 2)
#pragma unroll
            for (int i = 0; i < FI; i++) readA(b1, 0, i);
    };
    auto first_inputs = [&] {
        loadA(0);
        if constexpr (!GATEUP) {
            rowe = factors(0, 0);
            lds_barrier();
        }
        storeA(0, 0);
        loadA(min(1, nk - 1));
        if constexpr (NB == 3) {
            storeA(1, 1);
            loadA(min(2, nk - 1));
        }
        lds_barrier();
#pragma unroll
        for (int i = 0; i < FI; i++) readA(0, 0, i);
    };
    auto next = [](int buf) { return buf == NB - 1 ? 0 : buf + 1; };
    // K is a multiple of 128 (vh_mfma_supported): an even number of steps
    if constexpr (PK) {
        struct Words {
            uint32_t w[O::NW], sc;
        } st[2][2], wd[2];
        auto loadB = [&](Words (&g)[2], int step) {
#pragma unroll
            for (int j = 0; j < 2; j++) Frag<T>::load(fb + (size_t(step) * 2 + j) * Frag<T>::bytes, lane, g[j].w, g[j].sc);
        };
        auto step = [&](int s, int b0, int b1, int b2, Words (&cur)[2], Words (&nxt)[2]) {
            stage_inputs(s, b2);
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                if (ks == 3) {
                    __builtin_amdgcn_sched_barrier(0);
                    loadB(cur, min(s + 2, nk - 1));
                    __builtin_amdgcn_sched_barrier(0);
                    wd[0] = nxt[0];
                    wd[1] = nxt[1];
                }
#pragma unroll
                for (int j = 0; j < 2; j++) bn[j] = O::get(wd[j].w, wd[j].sc, (ks + 1) & 3, cst);
                multiply(ks, b0, b1);
            }
            end_step(b1);
        };
        loadB(st[0], 0);
        loadB(st[1], min(1, nk - 1));
        first_inputs();
        wd[0] = st[0][0];
        wd[1] = st[0][1];
#pragma unroll
        for (int j = 0; j < 2; j++) b[j] = O::get(wd[j].w, wd[j].sc, 0, cst);
        for (int s = 0, b0 = 0; s < nk; s += 2) {
            const int b1 = next(b0), b2 = next(b1);
            step(s, b0, b1, b2, st[0], st[1]);
            step(s + 1, b1, b2, b0, st[1], st[0]);
            b0 = b2;
        }
    } else {
        using S = Staged<T>;
        typename S::Lds &R = L.rows[wv];
        typename S::Regs g;
        float up[S::NU], fix[S::NU], bnd[S::NU];
        const int64_t r0 = GATEUP ? 32 * c : 64 * c;
        gbyte *const B[2] = {M0 + r0 * a.row_bytes, GATEUP ? M1 + r0 * a.row_bytes : M0 + (r0 + 32) * a.row_bytes};
        uint32_t w[2][2][4], sc[2], d[2];  // [half of the step's words][fragment]; the scales (PER_STEP: of the next d)
        auto put = [&] {  // other lanes' reads of the last pair lie before, those of this one after
            wave_fence();
            if constexpr (S::PER_STEP) S::put(R, g, lane);
            else S::put(R, g, up, lane);
            wave_fence();
        };
        auto fetch = [&](int p, int i) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if constexpr (S::PER_STEP) S::fetch(R, p, i, j, half, col, w[i][j], d[j]);
                else S::fetch(R, p, i, j, half, col, w[i][j]);
            }
        };
        // the scales of step p, whose first words are there: under the rows' powers of two
        auto scales = [&](int p, bool first) {
            bool any = false;
            if constexpr (S::PER_STEP) {
                auto scale = [&](int j) { return h_bits(h2f(d[j]) * up[j]); };
                if (first) {
#pragma unroll
                    for (int j = 0; j < 2; j++) up[j] = first_up(S::step_bound(d[j]));
                }
                sc[0] = scale(0);
                sc[1] = scale(1);
                // fp16 256 or more: 128 times it passes 2^15
                if (!first && __any((sc[0] & 0x7fffu) >= 0x5c00u || (sc[1] & 0x7fffu) >= 0x5c00u)) {
                    bnd[0] = S::step_bound(d[0]);
                    bnd[1] = S::step_bound(d[1]);
                    any = lower_up(bnd, up, fix);
                    sc[0] = scale(0);
                    sc[1] = scale(1);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 2; j++) sc[j] = reinterpret_cast<const uint32_t *>(R.sc)[4 * (32 * j + col) + 2 * p + half];
            }
            return any;
        };
        auto operands = [&](f16x8 (&o)[2], int ks) {
#pragma unroll
            for (int j = 0; j < 2; j++) o[j] = S::get(w[ks >> 1][j][2 * (ks & 1)], w[ks >> 1][j][2 * (ks & 1) + 1], sc[j], ks, cst);
        };
        // step s, step p of its unit: the next step's first words are read (after
        // the next unit is put in place) once its own last operand is formed
        constexpr int N = 2;
        const int units = nk / N;
        auto step = [&](int s, auto P, int b0, int b1, int b2) {
            constexpr int p = decltype(P)::value, q = (p + 1) % N;  // the next step's place in its unit
            stage_inputs(s, b2);
            bool any = false;
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                if (ks == 0) fetch(p, 1);
                if (ks < 3) operands(bn, ks + 1);
                if (ks == 2) {
                    if (q == 0) {
                        if constexpr (!S::PER_STEP) {
                            S::bounds(g, bnd);
                            any = lower_up(bnd, up, fix);
                        }
                        put();
                        __builtin_amdgcn_sched_barrier(0);
                        S::load(g, B, a.row_bytes, min(s / N + 2, units - 1), lane);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    fetch(q, 0);
                }
                if (ks == 3) {
                    any |= scales(q, false);
                    operands(bn, 0);
                }
                multiply(ks, b0, b1);
            }
            if (any) {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const float f = S::of_row(fix, j, col);
#pragma unroll
                    for (int i = 0; i < FI; i++)
#pragma unroll
                        for (int r = 0; r < 16; r++) acc[i][j][r] *= f;
                }
            }
            end_step(b1);
        };
        S::load(g, B, a.row_bytes, 0, lane);
        first_inputs();
        if constexpr (!S::PER_STEP) {
            S::bounds(g, bnd);
            up[0] = first_up(bnd[0]);
        }
        put();
        S::load(g, B, a.row_bytes, min(1, units - 1), lane);
        fetch(0, 0);
        scales(0, true);
        operands(b, 0);
        const std::integral_constant<int, 0> even;
        const std::integral_constant<int, N - 1> odd;
        for (int s = 0, b0 = 0; s < nk; s += 2) {
            if constexpr (NB == 2) {
                step(s, even, 0, 1, 1);
                step(s + 1, odd, 1, 0, 0);
            } else {
                const int b1 = next(b0), b2 = next(b1);
                step(s, even, b0, b1, b2);
                step(s + 1, odd, b1, b2, b0);
                b0 = b2;
            }
        }
#pragma unroll
        for (int j = 0; j < 2; j++) rs[j] = 1.0f / S::of_row(up, j, col);
    }

    // epilogue: the lane holds column `col` of each fragment, rows 8 (r / 4) +
    // 4 half + r % 4 of each 32-row block
    const int r0 = base + m0;
    auto row_of = [&](int r) { return 8 * (r >> 2) + (r & 3); };  // + 4 half
#pragma unroll
    for (int i = 0; i < FI; i++) {
        float sc[16];
#pragma unroll
        for (int r = 0; r < 16; r++) sc[r] = L.rsc[32 * i + row_of(r) + 4 * half];
        if constexpr (GATEUP) {
            float h[16], m[16];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float g = acc[i][0][r] * (rs[0] * sc[r]), u = acc[i][1][r] * (rs[1] * sc[r]);
                h[r] = g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;  // kept to 11 bits below
                m[r] = fabsf(h[r]);
            }
            // each row's largest |h| over the half wave's 32 columns: the rows are
            // folded over the lanes, so that after the steps below lane l holds row
            // r(l) = 8 b4 + 4 b3 + 2 b2 + b1 of the 16 (b: the bits of l)
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const auto v = __builtin_amdgcn_permlane16_swap(__float_as_uint(m[r]), __float_as_uint(m[r + 8]), false, false);
                m[r] = fmaxf(__uint_as_float(v[0]), __uint_as_float(v[1]));
            }
            fold<0x128, 4>(m, (lane & 8) != 0);  // row_ror:8
            fold<0x141, 2>(m, (lane & 4) != 0);  // row_half_mirror: the other four of eight lanes
            fold<0x4E, 1>(m, (lane & 2) != 0);
            m[0] = fmaxf(m[0], dpp_keep<0xB1>(m[0]));
            // the block's exponent: |h| < 2^e, stored as h 2^(14 - e) in fp16
            const uint32_t mb = __float_as_uint(m[0]);
            const int e = mb ? max(-100, min(127, int(mb >> 23) - 126)) : -128;
            const int rl = row_of((lane >> 1) & 15) + 4 * half;
            if (!(lane & 1)) {
                L.hsc[wv][rl] = __uint_as_float(uint32_t(127 + 14 - max(e, -100)) << 23);
                if (32 * i + rl < mcnt) a.he[size_t(r0 + 32 * i + rl) * (a.rows / 32) + c] = int8_t(e);
            }
            wave_fence();
            auto *hs = (__attribute__((address_space(1))) char *)a.out + (size_t(r0 + 32 * i) * a.rows + 32 * c) * 2;
            const uint32_t ho = uint32_t(4 * half * a.rows + col) * 2u;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const _Float16 v = _Float16(h[r] * L.hsc[wv][row_of(r) + 4 * half]);
                if (32 * i + row_of(r) + 4 * half < mcnt)
                    *(__attribute__((address_space(1))) _Float16 *)(hs + size_t(row_of(r)) * a.rows * 2 + ho) = v;
            }
            __builtin_amdgcn_wave_barrier();
        } else {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int tr = 32 * i + row_of(r) + 4 * half;
                if (tr < mcnt) {
                    float *y = static_cast<float *>(a.out) + size_t(L.prow[tr]) * a.rows + 64 * c + col;
                    y[0] = acc[i][0][r] * (rs[0] * sc[r]);
                    y[32] = acc[i][1][r] * (rs[1] * sc[r]);
                }
            }
        }
    }
}

// kXcds x slots workgroups (slots from tile_cost). The plan
// (mfma_plan_kernel) holds n tiles (expert, size, first row of its group)
// and, per launch, where each XCD's run of (tile, column tile) pairs starts:
// workgroup b runs on XCD b mod 8 (hardware dispatch) and takes pair
// start[b mod 8] + b / 8 of that XCD's contiguous run, column tiles fastest.
// BMAX: the plan's largest tile. What bounds it (Qwen3 Q4_K_M, 4093 tokens,
// 128-row tiles): a K step takes 1.5 us of a CU's two workgroups where its
// multiplies need 1.0 at the clock it runs at (2.0 GHz), and a workgroup spends
// 6 us before its first step (a chain of four loads) and 8 (gate/up) or 6
// (down) after its last; gate/up 514 -> 262 us, down 381 -> 182 us against the
// kernel whose waves were split into staging and multiplying ones.
template <int T, bool GATEUP, int BMAX, bool PK>
__global__ void __launch_bounds__(kThreads, BMAX == kBigTile || !PK ? 2 : 3) mfma_gemm_kernel(GemmArgs a) {
    constexpr int NCOL = GATEUP ? kBRows / 2 : kBRows;  // output columns per workgroup
    __shared__ TileLds<T, GATEUP, BMAX, PK> lds;
    const int nct = a.rows / NCOL, xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
    const int32_t *run = a.tiles + (GATEUP ? kPlanRunsGU : kPlanRunsDN);
    const int at = run[xcd] + slot;
    if (at >= run[xcd + 1]) return;
    const int t = at / nct, n0 = (at % nct) * NCOL;
    const int32_t *rec = a.tiles + kPlanHead + 4 * t;
    const int e = rec[0] & 0xffff, bmt = rec[0] >> 16, m0 = rec[1], base = rec[2], mcnt = rec[3];
    gbyte *M0 = gmem(a.table[3 * e + (GATEUP ? 0 : 2)]);
    gbyte *M1 = GATEUP ? gmem(a.table[3 * e + 1]) : M0;
    if (!M0 || !M1) {
        // an unregistered expert contributes nothing (src/gguf_run.c:201): its
        // h rows are zero, and the combine skips its y rows
        if (GATEUP)
            for (int i = threadIdx.x; i < mcnt * NCOL; i += kThreads) {
                const size_t pos = size_t(base + m0 + i / NCOL);
                const int cc = n0 + i % NCOL;
                static_cast<_Float16 *>(a.out)[pos * a.rows + cc] = _Float16(0.0f);
                if (cc % 32 == 0) a.he[pos * (a.rows / 32) + cc / 32] = int8_t(-128);
            }
        return;
    }
    if (bmt == 32) gemm_tile<T, GATEUP, 32, BMAX, PK>(lds, a, M0, M1, base, m0, mcnt, n0);
    else if (bmt == 64) gemm_tile<T, GATEUP, 64, BMAX, PK>(lds, a, M0, M1, base, m0, mcnt, n0);
    else if constexpr (BMAX == 128) gemm_tile<T, GATEUP, 128, BMAX, PK>(lds, a, M0, M1, base, m0, mcnt, n0);
}

// The fp16 copy of hb [T x d] under each token's power of two (its largest
// magnitude brought below 2^14; 1 where that is not finite), a wave per
// token, and the inverse scales xsc [T]; workgroup blk of 256 threads.
VH_DEV void f16_rows(const float *__restrict__ hb, _Float16 *__restrict__ xb, float *__restrict__ xsc, int T, int d,
                     int blk) {
    const int t = blk * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= T) return;
    const float4 *x = reinterpret_cast<const float4 *>(hb + size_t(t) * d);
    f16x4 *y = reinterpret_cast<f16x4 *>(xb + size_t(t) * d);
    float m = 0.0f;
    for (int i = lane; i < d / 4; i += 64) {
        const float4 v = x[i];
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
    const int e = exponent_for(wave_max_f(m));
    const float up = ldexpf(1.0f, e);
    if (lane == 0) xsc[t] = ldexpf(1.0f, -e);
    for (int i = lane; i < d / 4; i += 64) {
        const float4 v = x[i];
        y[i] = f16x4{_Float16(v.x * up), _Float16(v.y * up), _Float16(v.z * up), _Float16(v.w * up)};
    }
}

// The bytes a token tile of bm rows stages per K step (the weights' wb and
// the inputs), in 64-byte units: the cost by which the XCDs' runs are cut.
__host__ __device__ constexpr int tile_step_cost(int wb, int bm) { return (wb + bm * kBK * 2) / 64; }

// A group's token tiles under the largest tile of bm rows (128 or 64): n whole
// ones, then one of rbm (32 or 64) rows if rbm != 0 - the remainder in the
// smallest tile that holds it (above bm / 2 rows, a whole tile).
struct GroupTiles {
    int bm, n, rbm;
    __host__ __device__ GroupTiles(int cnt, int bmax) : bm(bmax), n(cnt / bmax) {
        int r = cnt - bm * n;
        if (2 * r > bm) {
            n++;
            r = 0;
        }
        rbm = r == 0 ? 0 : r <= 32 ? 32 : 64;
    }
    __host__ __device__ int count() const { return n + (rbm ? 1 : 0); }
    __host__ __device__ int rows(int i) const { return i < n ? bm : rbm; }
};

// Workgroup 0 of 256 threads (thread e = expert e, E <= 256): the plan,
//   tiles[0]               n, the number of token tiles
//   tiles[kPlanRunsGU + x]  x = 0..8: where XCD x's run of gate/up (tile,
//                           column tile) pairs starts (x = 8: the end)
//   tiles[kPlanRunsDN + x]  the same for the down launch
//   tiles[kPlanHead + 4 t]  tile t: expert | rows << 16 (32, 64 or 128), the
//                           tile's first row within its group, the group's
//                           first pair (offs), the tile's pairs
// (experts ascending, tiles as GroupTiles). The runs are cut at equal shares
// of the launch's staged bytes (tile_step_cost per pair); a cut that would
// give an XCD more pairs than the launch has slots per XCD falls back to equal
// shares of pairs. The other workgroups: the GEMMs' inputs (f16_rows).
__global__ void __launch_bounds__(256) mfma_plan_kernel(const int32_t *__restrict__ counts,
                                                        const int32_t *__restrict__ offs, int E, int bmax,
                                                        int nct_gu, int wb_gu, int slots_gu, int nct_dn,
                                                        int wb_dn, int slots_dn, int32_t *__restrict__ tiles,
                                                        const float *__restrict__ hb, _Float16 *__restrict__ xb,
                                                        float *__restrict__ xsc, int T, int d) {
    if (blockIdx.x > 0) {
        f16_rows(hb, xb, xsc, T, d, blockIdx.x - 1);
        return;
    }
    __shared__ int wsum[4];
    __shared__ int wcost[4][2];
    __shared__ int runs[2][kXcds + 1];
    __shared__ int total[2];
    __shared__ int ntiles;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int cnt = t < E ? counts[t] : 0;
    const GroupTiles gt(cnt, bmax);
    const int nt = gt.count();
    const int ncts[2] = {nct_gu, nct_dn};
    const int wbs[2] = {wb_gu, wb_dn};
    int c[2];
#pragma unroll
    for (int l = 0; l < 2; l++)
        c[l] = ncts[l] * (gt.n * tile_step_cost(wbs[l], bmax) + (gt.rbm ? tile_step_cost(wbs[l], gt.rbm) : 0));
    int it = nt;
    int ic[2] = {c[0], c[1]};
#pragma unroll
    for (int sh = 1; sh < 64; sh <<= 1) {
        const int ot = __shfl_up(it, sh, 64);
        const int o0 = __shfl_up(ic[0], sh, 64), o1 = __shfl_up(ic[1], sh, 64);
        if (lane >= sh) {
            it += ot;
            ic[0] += o0;
            ic[1] += o1;
        }
    }
    if (lane == 63) {
        wsum[wv] = it;
        wcost[wv][0] = ic[0];
        wcost[wv][1] = ic[1];
    }
    __syncthreads();
    int bt = 0;
    int bc[2] = {0, 0};
    for (int w = 0; w < wv; w++) {
        bt += wsum[w];
        bc[0] += wcost[w][0];
        bc[1] += wcost[w][1];
    }
    const int ex_t = bt + it - nt;
    for (int i = 0; i < nt; i++) {
        int32_t *rec = tiles + kPlanHead + 4 * (ex_t + i);
        rec[0] = t | (gt.rows(i) << 16);
        rec[1] = bmax * i;
        rec[2] = offs[t];
        rec[3] = min(gt.rows(i), cnt - bmax * i);
    }
    if (t == 255) {
        ntiles = ex_t + nt;
        total[0] = bc[0] + ic[0];
        total[1] = bc[1] + ic[1];
        tiles[0] = ex_t + nt;
    }
    __syncthreads();
    // the cuts: XCD x's run starts at the pair holding staged byte x * total / 8
#pragma unroll
    for (int l = 0; l < 2; l++) {
        const int ex_c = bc[l] + ic[l] - c[l];
        for (int x = 1; x < kXcds; x++) {
            const int target = int(int64_t(x) * total[l] / kXcds);
            if (c[l] > 0 && ex_c <= target && target < ex_c + c[l]) {
                // the tile holding the target (a whole tile or the last), then its column
                const int off = target - ex_c, cw = tile_step_cost(wbs[l], bmax), full = gt.n * ncts[l] * cw;
                const int i = off < full ? off / (ncts[l] * cw) : gt.n;
                const int rest = off - i * ncts[l] * cw;
                runs[l][x] = (ex_t + i) * ncts[l] + min(rest / tile_step_cost(wbs[l], gt.rows(i)), ncts[l] - 1);
            }
        }
    }
    if (t == 0) {
        runs[0][0] = runs[1][0] = 0;
        runs[0][kXcds] = ntiles * nct_gu;
        runs[1][kXcds] = ntiles * nct_dn;
        if (total[0] == 0)
            for (int x = 1; x < kXcds; x++) runs[0][x] = 0;
        if (total[1] == 0)
            for (int x = 1; x < kXcds; x++) runs[1][x] = 0;
    }
    __syncthreads();
    if (t < 2) {
        const int slots = t ? slots_dn : slots_gu, live = runs[t][kXcds];
        bool ok = true;
        for (int x = 0; x < kXcds; x++) ok = ok && runs[t][x] <= runs[t][x + 1] && runs[t][x + 1] - runs[t][x] <= slots;
        const int per = (live + kXcds - 1) / kXcds;
        for (int x = 0; x <= kXcds; x++) tiles[(t ? kPlanRunsDN : kPlanRunsGU) + x] = ok ? runs[t][x] : min(x * per, live);
    }
}

// The largest token tile of a call of P pairs over E experts: 128 rows where
// the average group has at least kBigAverage, else 64, whose kernel keeps three
// waves per SIMD instead of two to hide the weights' loads, which bound small
// groups. Measured per layer with tiles of up to 64 / 128 rows: OLMoE Q4_K_M 512
// tokens (64 per expert) 205 / 236 us, Qwen3 Q8_0 2048 tokens (128 per expert,
// Zipf) 424 / 421 us, Qwen3 Q4_K_M 4093 tokens (256 per expert) 705 / 667 us.
// GGUF rows, whose weights cost more to form and whose kernels keep two waves
// either way, from 70: Qwen3 Q8_0 1024 tokens (64 per expert) 382 / 384 us, 1200
// (75) 437 / 420, 1500 (94) 468 / 396; OLMoE Q8_0 512 (64) 274 / 291.
constexpr int kBigAverage = 100, kBigAverageRows = 70;
int tile_rows(int P, int E, bool packed) {
    return P >= (packed ? kBigAverage : kBigAverageRows) * E ? kBigTile : kSmallTile;
}
int max_tiles(int P, int E, bool packed) { return P / tile_rows(P, E, packed) + E; }

// The column tiles, weight bytes per K step and workgroup slots per XCD of a
// launch: an eighth more than an XCD's share of the most pairs there can be
// (mfma_plan_kernel cuts into equal shares of pairs where an XCD would get
// more; a workgroup past its XCD's run costs a round trip).
struct TileCost {
    int nct, wb, slots;
};
TileCost tile_cost(uint32_t type, int K, int rows, bool gateup, int P, int E, bool packed) {
    TileCost c;
    c.nct = rows / (gateup ? kBRows / 2 : kBRows);
    c.wb = int(int64_t(kBRows) * vh_row_bytes(type, K) * kBK / K);  // a multiple of 64 for these types
    const int64_t per = (int64_t(max_tiles(P, E, packed)) * c.nct + kXcds - 1) / kXcds;
    c.slots = int(per + per / 8 + 1);
    return c;
}

template <int T, bool GATEUP>
void launch_gemm(const GemmArgs &a, const dim3 &g, bool big, bool packed, hipStream_t s) {
    const dim3 b(kThreads);
    if (big && packed) hipLaunchKernelGGL((mfma_gemm_kernel<T, GATEUP, kBigTile, true>), g, b, 0, s, a);
    else if (big) hipLaunchKernelGGL((mfma_gemm_kernel<T, GATEUP, kBigTile, false>), g, b, 0, s, a);
    else if (packed) hipLaunchKernelGGL((mfma_gemm_kernel<T, GATEUP, kSmallTile, true>), g, b, 0, s, a);
    else hipLaunchKernelGGL((mfma_gemm_kernel<T, GATEUP, kSmallTile, false>), g, b, 0, s, a);
}

template <bool GATEUP>
int gemm(uint32_t type, int P, int E, bool packed, const GemmArgs &a, hipStream_t s) {
    const dim3 g(unsigned(tile_cost(type, a.K, a.rows, GATEUP, P, E, packed).slots) * kXcds);
    const bool big = tile_rows(P, E, packed) == kBigTile;
    switch (type) {
    case VT_Q8_0: launch_gemm<VT_Q8_0, GATEUP>(a, g, big, packed, s); break;
    case VT_Q4_K: launch_gemm<VT_Q4_K, GATEUP>(a, g, big, packed, s); break;
    case VT_Q6_K: launch_gemm<VT_Q6_K, GATEUP>(a, g, big, packed, s); break;
    default: return -EINVAL;
    }
    return vh_check(hipGetLastError());
}

}  // namespace

bool vh_mfma_supported(uint32_t tg, uint32_t td, int d, int fe, int E) {
    auto ok = [](uint32_t t) { return t == VT_Q8_0 || t == VT_Q4_K || t == VT_Q6_K; };
    auto kq = [](uint32_t t, int n) { return t == VT_Q8_0 ? n % 32 == 0 : n % 256 == 0; };
    return ok(tg) && ok(td) && kq(tg, d) && kq(td, fe) && d % kBRows == 0 && fe % (kBRows / 2) == 0 &&
           d % kBK == 0 && fe % kBK == 0 && E <= 256;
}

int vh_mfma_plan_words(int P, int E) { return kPlanHead + 4 * std::max(max_tiles(P, E, true), max_tiles(P, E, false)); }

int vh_mfma_plan(const int32_t *counts, const int32_t *offs, int E, int T, int k, uint32_t tg, uint32_t td, int d, int fe,
                 bool packed, int32_t *tiles, const float *hb, void *xb, float *xsc, hipStream_t s) {
    if (E > 256 || d % 4 || ((reinterpret_cast<uintptr_t>(hb) | reinterpret_cast<uintptr_t>(xb)) & 15u)) return -EINVAL;
    const int P = T * k, mt = max_tiles(P, E, packed);
    const TileCost gu = tile_cost(tg, d, fe, true, P, E, packed), dn = tile_cost(td, fe, d, false, P, E, packed);
    // the plan's costs are 32-bit sums over every (tile, column tile) pair
    if (int64_t(mt) * std::max(gu.nct, dn.nct) * tile_step_cost(std::max(gu.wb, dn.wb), kBigTile) > INT32_MAX)
        return -E2BIG;
    hipLaunchKernelGGL(mfma_plan_kernel, dim3(1 + unsigned((T + 3) / 4)), dim3(256), 0, s, counts, offs, E, tile_rows(P, E, packed),
                       gu.nct, gu.wb, gu.slots, dn.nct, dn.wb, dn.slots, tiles, hb, static_cast<_Float16 *>(xb), xsc,
                       T, d);
    return vh_check(hipGetLastError());
}

int vh_mfma_gateup(uint32_t type, const int32_t *tiles, int P, int E, const int32_t *perm,
                   const void *const *table, bool packed, const void *xb, const float *xsc, int d,
                   int fe, int k, void *hs, int8_t *he, hipStream_t s) {
    return gemm<true>(type, P, E, packed,
                      GemmArgs{tiles, perm, table, static_cast<const uint8_t *>(xb), xsc, he, hs, d, fe,
                               k, vh_row_bytes(type, d)},
                      s);
}

int vh_mfma_down(uint32_t type, const int32_t *tiles, int P, int E, const int32_t *perm,
                 const void *const *table, bool packed, const void *hs, const int8_t *he, int d,
                 int fe, float *ybuf, hipStream_t s) {
    return gemm<false>(type, P, E, packed,
                       GemmArgs{tiles, perm, table, static_cast<const uint8_t *>(hs), nullptr,
                                const_cast<int8_t *>(he), ybuf, fe, d, 1, vh_row_bytes(type, fe)},
                       s);
}

namespace {
// One workgroup per (fragment row set, expert): the 32 rows of fragment index
// blockIdx.x = 2 c + j (Frag) of the expert's gate/up or down matrix, every K
// step. First the rows' exponents (8 threads scan a row's scales) and their
// scales behind the fragments, then a wave per K step.
template <int T, bool GATEUP>
__global__ void __launch_bounds__(256) frag_pack_kernel(const void *const *__restrict__ src_tab,
                                                        void *const *__restrict__ dst_tab, int K, int rows,
                                                        int64_t row_bytes) {
    __shared__ float up[32];
    const int e = blockIdx.y, c = blockIdx.x >> 1, j = blockIdx.x & 1, tid = threadIdx.x, nk = K / kBK;
    uint8_t *dst = static_cast<uint8_t *>(dst_tab[3 * e + (GATEUP ? 0 : 2)]);
    if (!dst) return;
    gbyte *m = gmem(src_tab[3 * e + (GATEUP ? j : 2)]);
    const int r0 = GATEUP ? 32 * c : 64 * c + 32 * j;
    {
        gbyte *row = m + int64_t(r0 + (tid >> 3)) * row_bytes;
        float b = 0.0f;
        for (int i = tid & 7; i < Rows<T>::blocks(K); i += 8) {
            const float v = Rows<T>::bound(row, i);
            b = v > b || !(v <= 3.4028234663852886e38f) ? v : b;
        }
#pragma unroll
        for (int sh = 1; sh < 8; sh <<= 1) {
            const float o = __shfl_xor(b, sh, 64);
            b = o > b || !(o <= 3.4028234663852886e38f) ? o : b;
        }
        if ((tid & 7) == 0) {
            const int ex = exponent_for(b);
            up[tid >> 3] = ldexpf(1.0f, ex);
            float *rs = reinterpret_cast<float *>(dst + size_t(GATEUP ? 2 : 1) * rows / 32 * nk * Frag<T>::bytes);
            rs[(GATEUP ? j * rows : 0) + r0 + (tid >> 3)] = ldexpf(1.0f, -ex);
        }
    }
    __syncthreads();
    const int lane = tid & 63;
    gbyte *row = m + int64_t(r0 + (lane & 31)) * row_bytes;
    for (int s = tid >> 6; s < nk; s += 4) {
        typename Rows<T>::Raw raw;
        uint32_t w[Op<T>::NW], sc;
        Rows<T>::load(row, s, lane >> 5, raw);
        Rows<T>::words(raw, s, lane >> 5, up[lane & 31], w, sc);
        Frag<T>::store(dst + ((size_t(c) * nk + s) * 2 + j) * Frag<T>::bytes, lane, w, sc);
    }
}

size_t frag_bytes(uint32_t t) {
    return t == VT_Q8_0 ? Frag<VT_Q8_0>::bytes : t == VT_Q4_K ? Frag<VT_Q4_K>::bytes : Frag<VT_Q6_K>::bytes;
}
// an expert's gate/up and down fragments with their rows' scales
size_t pack_gu_bytes(uint32_t tg, int d, int fe) {
    return (size_t(2) * fe / 32 * (d / kBK) * frag_bytes(tg) + size_t(2) * fe * 4 + 255) & ~size_t(255);
}
size_t pack_dn_bytes(uint32_t td, int d, int fe) {
    return (size_t(d) / 32 * (fe / kBK) * frag_bytes(td) + size_t(d) * 4 + 255) & ~size_t(255);
}

template <bool GATEUP>
void pack_launch(uint32_t type, const void *const *table, void *const *dt, int E, int K, int rows, hipStream_t s) {
    const dim3 g(unsigned((GATEUP ? 2 : 1) * rows / 32), unsigned(E)), b(256);
    const int64_t rb = vh_row_bytes(type, K);
    if (type == VT_Q8_0) hipLaunchKernelGGL((frag_pack_kernel<VT_Q8_0, GATEUP>), g, b, 0, s, table, dt, K, rows, rb);
    else if (type == VT_Q4_K) hipLaunchKernelGGL((frag_pack_kernel<VT_Q4_K, GATEUP>), g, b, 0, s, table, dt, K, rows, rb);
    else hipLaunchKernelGGL((frag_pack_kernel<VT_Q6_K, GATEUP>), g, b, 0, s, table, dt, K, rows, rb);
}
}  // namespace

uint64_t vh_mfma_pack_bytes(uint32_t tg, uint32_t td, int E, int d, int fe) {
    if (E < 1 || d < kBRows || fe < kBK || !vh_mfma_supported(tg, td, d, fe, E)) return 0;
    return uint64_t(E) * (pack_gu_bytes(tg, d, fe) + pack_dn_bytes(td, d, fe));
}

int vh_mfma_pack(const void *const *table, uint32_t tg, uint32_t td, int E, int d, int fe, void *buf, void **tab_out,
                 hipStream_t s) {
    *tab_out = nullptr;
    if (!buf || !vh_mfma_pack_bytes(tg, td, E, d, fe)) return -EINVAL;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (int rc = vh_check(hipStreamIsCapturing(s, &cap))) return rc;
    if (cap != hipStreamCaptureStatusNone) return -EBUSY;  // no allocation under capture
    const size_t gb = pack_gu_bytes(tg, d, fe), per = gb + pack_dn_bytes(td, d, fe);
    std::vector<const void *> src(size_t(3) * E), dst(size_t(3) * E, nullptr);
    if (int rc = vh_check(hipMemcpyAsync(src.data(), table, src.size() * sizeof(void *), hipMemcpyDeviceToHost, s)))
        return rc;
    if (int rc = vh_check(hipStreamSynchronize(s))) return rc;
    void *tab = nullptr;
    if (hipMalloc(&tab, src.size() * sizeof(void *)) != hipSuccess) return -ENOMEM;
    char *b = static_cast<char *>(buf);
    for (int e = 0; e < E; e++) {
        if (!src[3 * e] || !src[3 * e + 1] || !src[3 * e + 2]) continue;  // unregistered: stays NULL
        dst[3 * e] = dst[3 * e + 1] = b + per * e;  // gate/up fragments
        dst[3 * e + 2] = b + per * e + gb;           // down fragments
    }
    int rc = vh_check(hipMemcpy(tab, dst.data(), dst.size() * sizeof(void *), hipMemcpyHostToDevice));
    if (!rc) {
        void *const *dt = static_cast<void *const *>(tab);
        pack_launch<true>(tg, table, dt, E, d, fe, s);
        pack_launch<false>(td, table, dt, E, fe, d, s);
        rc = vh_check(hipGetLastError());
    }
    if (rc) {
        (void)hipStreamSynchronize(s);
        (void)hipFree(tab);
        return rc;
    }
    *tab_out = tab;
    return 0;
}
