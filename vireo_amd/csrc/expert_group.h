// The pairs of one expert, found by the workgroups that need them (calls of
// fewer than 64 tokens: no dispatch kernel).
#pragma once
#include "common.h"

namespace {

constexpr int kGroupMax = 64;     // a call's tokens per expert (at most one pair per token; calls < 64 tokens)

// The pairs p < P routed to expert e (idx[p] == e) in ascending order into
// list (at most kGroupMax kept); returns their number. Called by every thread
// of a workgroup of NT threads; the first two rounds' loads are issued
// together, and the function ends with a barrier.
template <int NT>
VH_DEV int expert_group(const int32_t *__restrict__ idx, int P, int e, int *list, int *wc) {
    constexpr int NW = NT / 64;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int v0 = tid < P ? idx[tid] : -1, v1 = tid + NT < P ? idx[tid + NT] : -1;
    int base = 0;
    for (int p0 = 0; p0 < P; p0 += NT) {
        const int p = p0 + tid;
        const int v = p0 == 0 ? v0 : p0 == NT ? v1 : (p < P ? idx[p] : -1);
        const bool hit = v == e;
        const uint64_t m = __ballot(hit);
        if (lane == 0) wc[wv] = __popcll(m);
        __syncthreads();
        int before = base, tot = base;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const int c = wc[w];
            before += w < wv ? c : 0;
            tot += c;
        }
        const int at = before + __popcll(m & ((1ull << lane) - 1ull));
        if (hit && at < kGroupMax) list[at] = p;
        base = tot;
        __syncthreads();  // wc is written again by the next round
    }
    return min(base, kGroupMax);
}

}  // namespace
