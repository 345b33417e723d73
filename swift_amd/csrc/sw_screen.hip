// sw_screen.hip -- the batched path's screen (sw_screen.hpp) as a kernel of its
// own, ahead of the binning: pairs it answers get their outputs here and are
// left out of the bins; or ahead of the one-launch form of a small call and of
// the plain path's packed sweep, which take the list of the pairs it leaves.
#include <algorithm>

#include "sw_screen.hpp"

namespace swift {

namespace {

// Appends the indexes first + lane of every wave's lanes in `left` to the list,
// a workgroup at a time: atomics on one counter come 10 ns apart, which a wave
// of one pair each made 120 us of 12,000 unrelated pairs.  All four waves call.
__device__ __forceinline__ void screen_append(uint64_t left, int first, int32_t *list,
                                              int32_t *count, int32_t *lds) {
    const int lane = threadIdx.x & 63, wv = uni((int)(threadIdx.x >> 6));
    if (lane == 0) lds[wv] = __builtin_popcountll(left);
    __syncthreads();
    if (threadIdx.x == 0) {
        const int n = lds[0] + lds[1] + lds[2] + lds[3];
        lds[4] = n ? atomicAdd(count, n) : 0;
    }
    __syncthreads();
    int at = lds[4];
    for (int w = 0; w < wv; ++w) at += lds[w];
    if ((left >> lane) & 1)
        list[at + __builtin_popcountll(left & ((1ull << lane) - 1))] = first + lane;
}

// A wave takes `per` consecutive pairs: their lengths and offsets a lane each,
// so that the slots of missing pairs (a pipeline's capacity) cost nothing and
// the next pair's addresses are at hand.
__global__ void __launch_bounds__(256) sw_screen_kernel(ScreenArgs a, ScreenConsts sc) {
    __shared__ __attribute__((aligned(16))) uint32_t lds[4][kScreenWords];
    __shared__ int32_t total[5];
    const int lane = threadIdx.x & 63, wv = uni((int)(threadIdx.x >> 6));
    const int first = ((int)blockIdx.x * 4 + wv) * a.per;
    const int mine = first + lane;
    const bool in = lane < a.per && mine < a.npairs;
    int ql = 0, rl = 0;
    if (in) {
        ql = a.qlen[mine];
        rl = a.rlen[mine];
    }
    const bool fits = ql >= kScreenMinQ && ql <= kMaxBatchQ && rl >= kScreenMinR && rl <= kMaxBatchR;
    uint64_t todo = __ballot(fits), left = __ballot(in);
    int64_t qo = 0, ro = 0, co = 0;
    if (fits) {
        qo = a.qoff[mine];
        ro = a.roff[mine];
        co = a.coff[mine];
    }
    auto pick = [](int64_t v, int l) {
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l);
        return (int64_t)(((uint64_t)hi << 32) | lo);
    };
    while (todo) {
        const int l = __builtin_ctzll(todo);
        todo &= todo - 1;
        const char *qs = a.qseq + pick(qo, l), *rs = a.rseq + pick(ro, l);
        Screened s;
        if (!screen_pair<kMaxBatchQ / 32>(sc, qs, __builtin_amdgcn_readlane(ql, l), rs,
                                          __builtin_amdgcn_readlane(rl, l), lds[wv], s))
            continue;
        left &= ~(1ull << l);
        const int64_t c = pick(co, l);
        screen_strings(s, qs, rs, a.qcons + c, a.rcons + c);
        if (lane == 0) {
            const int p = first + l, end = s.row + s.diag + 1;
            a.score_out[p] = s.score;
            a.start_out[p] = end - s.len + 1;
            a.end_out[p] = end;
            a.alen_out[p] = s.len;
            if (a.res) a.res[p] = PairResult{s.score, s.row + 1, end, kScreenedFlag};
        }
    }
    if (a.list) screen_append(left, first, a.list, a.count, total);
}

// The plain path's pairs, [pair0, pair0 + n) of the caller's arrays.
__global__ void __launch_bounds__(256)
sw_screen_plain_kernel(const char *__restrict__ q, const char *__restrict__ r, int qlen, int rlen,
                       int n, int pair0, int per, PlainOut out, int32_t *list, int32_t *count,
                       ScreenConsts sc) {
    __shared__ __attribute__((aligned(16))) uint32_t lds[4][kScreenWords];
    __shared__ int32_t total[5];
    const int lane = threadIdx.x & 63, wv = uni((int)(threadIdx.x >> 6));
    const int first = ((int)blockIdx.x * 4 + wv) * per, m = min(per, n - first);
    uint64_t left = 0;
    for (int l = 0; l < m; ++l) {
        const int64_t gp = pair0 + first + l;
        const char *qs = q + gp * (qlen + 1), *rs = r + gp * (rlen + 1);
        Screened s;
        // (a NUL that ends the reference early is a byte the screen leaves)
        if (!screen_pair<kMaxBatchQ / 32>(sc, qs, qlen, rs, rlen, lds[wv], s)) {
            left |= 1ull << l;
            continue;
        }
        screen_strings(s, qs, rs, out.qcons + gp * out.cstride, out.rcons + gp * out.cstride);
        if (lane == 0) {
            const int end = s.row + s.diag + 1;
            out.score[gp] = (float)s.score;
            out.start[gp] = end - s.len + 1;
            out.end[gp] = end;
            out.alen[gp] = s.len;
        }
    }
    screen_append(left, first, list, count, total);
}

}  // namespace

// sixteen pairs a wave once that still is several waves a SIMD
static int screen_per(int n) { return std::max(1, std::min(16, n / 8192)); }

hipError_t launch_screen(const ScreenArgs &a, const Scoring &s, hipStream_t st) {
    ScreenArgs b = a;
    b.per = screen_per(a.npairs);
    const int waves = (a.npairs + b.per - 1) / b.per;
    hipLaunchKernelGGL(sw_screen_kernel, dim3((waves + 3) / 4), dim3(256), 0, st, b,
                       screen_consts(s));
    return hipGetLastError();
}

hipError_t launch_screen_plain(const char *q, const char *r, const Scoring &s, int qlen, int rlen,
                               int n, int pair0, const PlainOut &out, int32_t *list,
                               int32_t *count, hipStream_t st) {
    const int per = screen_per(n), waves = (n + per - 1) / per;
    hipLaunchKernelGGL(sw_screen_plain_kernel, dim3((waves + 3) / 4), dim3(256), 0, st, q, r, qlen,
                       rlen, n, pair0, per, out, list, count, screen_consts(s));
    return hipGetLastError();
}

}  // namespace swift
