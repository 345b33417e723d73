// sw_screen.hip -- the batched path's screen (sw_screen.hpp) as a kernel of its
// own, ahead of the binning: pairs it answers get their outputs here and are
// left out of the bins.
#include <algorithm>

#include "sw_screen.hpp"

namespace swift {

namespace {

// A wave takes `per` consecutive pairs: their lengths and offsets a lane each,
// so that the slots of missing pairs (a pipeline's capacity) cost nothing and
// the next pair's addresses are at hand.
__global__ void __launch_bounds__(256) sw_screen_kernel(ScreenArgs a, ScreenConsts sc) {
    __shared__ __attribute__((aligned(16))) uint32_t lds[4][kScreenWords];
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
    uint64_t todo = __ballot(fits);
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
        const int64_t c = pick(co, l);
        screen_strings(s, qs, rs, a.qcons + c, a.rcons + c);
        if (lane == 0) {
            const int p = first + l, end = s.row + s.diag + 1;
            a.score_out[p] = s.score;
            a.start_out[p] = end - s.len + 1;
            a.end_out[p] = end;
            a.alen_out[p] = s.len;
            a.res[p] = PairResult{s.score, s.row + 1, end, kScreenedFlag};
        }
    }
}

}  // namespace

hipError_t launch_screen(const ScreenArgs &a, const Scoring &s, hipStream_t st) {
    ScreenArgs b = a;
    // sixteen pairs a wave once that still is several waves a SIMD
    b.per = std::max(1, std::min(16, a.npairs / 8192));
    const int waves = (a.npairs + b.per - 1) / b.per;
    hipLaunchKernelGGL(sw_screen_kernel, dim3((waves + 3) / 4), dim3(256), 0, st, b,
                       screen_consts(s));
    return hipGetLastError();
}

}  // namespace swift
