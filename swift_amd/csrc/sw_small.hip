// sw_small.hip -- the batched path's kernel for small calls: every pair from
// its bytes to its strings in one launch.
//
// A small call is bound by latency: binning, the readback of its sizes, the
// sweep, the walk and the expansion were six kernels, two host round trips and
// their gaps around one task's sweep.  Here a wave takes one or two pairs as
// they come (no binning), sweeps them in the two packed halves of one 64-lane
// group, then walks and expands them from its own trace area, so the host
// waits once.  A pair the packed lanes cannot take (a reference byte outside
// ACGTNacgtn, a score past their limit) is swept again by the same wave in
// 32-bit lanes.  64 pairs of 50-300 bases: 166 -> 95 us
// a call; 1,500 of 100 x 300: 156 -> 59 us; a pipeline of 1,000 reads: 259 ->
// 138 us.
#include <algorithm>

#include "sw_sweep.hpp"

namespace swift {

namespace {

constexpr int kPad = 64;  // LDS words before column 0

__host__ __device__ constexpr int small_cols(int maxr) { return maxr + 2 * kPad + 8; }
__host__ __device__ constexpr int small_qw(int maxq) { return (maxq + 6) / 4; }
__host__ __device__ constexpr int small_rw(int maxr) { return (maxr + 6) / 4; }
__host__ __device__ constexpr int small_mw(int maxq, int maxr) { return (maxq + maxr) / 16 + 1; }

__host__ __device__ constexpr int small_lds_words(int maxq, int maxr) {
    return 2 * small_mw(maxq, maxr) +
           (small_cols(maxr) > 2 * (small_qw(maxq) + small_rw(maxr))
                ? small_cols(maxr) : 2 * (small_qw(maxq) + small_rw(maxr)));
}

// the walk of one pair of the wave's trace area; moves to LDS
__device__ __forceinline__ WalkOut small_walk(const uint32_t *tr, int R, int W, int kl, int bitb,
                                              const GroupResult &gr, int ql, int rl,
                                              uint32_t *moves) {
    LdsMoves mv{moves};
    return walk_wave(reinterpret_cast<const uint4 *>(tr), R, W, kl, bitb, uni(gr.score),
                     uni(gr.row), uni(gr.col), ql, rl, mv);
}

template <int R, int FORM>
__global__ void __launch_bounds__(256) sw_small_kernel(SmallArgs a) {
    using S = Lean<64, R, true, FORM>;
    using S32 = Lean<64, R, false>;
    extern __shared__ uint32_t lds[];
    // every wave works alone, in its own part of the workgroup's LDS
    const int g = threadIdx.x & 63, wv = uni((int)(threadIdx.x >> 6));
    const int wave = (int)blockIdx.x * a.wpb + wv, nwaves = (int)gridDim.x * a.wpb;
    const int mw = small_mw(a.maxq, a.maxr);
    uint32_t *moves = lds + wv * small_lds_words(a.maxq, a.maxr);
    uint32_t *col = moves + 2 * mw;  // the columns, then the expansion's bases
    uint32_t *tr = a.trace + (int64_t)wave * a.wave_words;
    const int npairs = a.nlist ? uni(*a.nlist) : a.npairs;
    // more than a.most: none, and the host takes the general path
    const int ntask = npairs > a.most ? 0 : (npairs + a.ppw - 1) / a.ppw;
    if (ntask == 0 && npairs > 0 && wave == 0 && g == 0) host_flag(a.flags + kSmallMany);
    for (int task = wave; task < ntask; task += nwaves) {
        int pid[2], ql[2], rl[2];
        const char *qs[2], *rs[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int i = task * a.ppw + h;
            int at = min(i, npairs - 1);
            if (a.list) at = uni(a.list[at]);
            pid[h] = h < a.ppw && i < npairs ? at : -1;
            ql[h] = uni(a.qlen[at]);
            rl[h] = uni(a.rlen[at]);
            qs[h] = a.qseq + a.qoff[at];
            rs[h] = a.rseq + a.roff[at];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (pid[h] >= 0 && (ql[h] < 0 || rl[h] < 0 || ql[h] > kMaxBatchQ || rl[h] > kMaxBatchR)) {
                // beyond the batched kernels: left out, and the call reports it
                if (g == 0) host_flag(a.flags + kSmallError);
                pid[h] = -1;
            } else if (pid[h] >= 0 && (ql[h] > min(64 * R, a.maxq) || rl[h] > a.maxr)) {
                // longer than the call said: the host takes the general path
                if (g == 0) host_flag(a.flags + kSmallLonger);
                pid[h] = -1;
            } else if (pid[h] >= 0 && (ql[h] == 0 || rl[h] == 0)) {
                // all-zero matrix: start 0, end -1, length 0 (src/smithWaterman.cu
                // :50,333-334)
                if (g == 0) {
                    a.score_out[pid[h]] = 0;
                    a.start_out[pid[h]] = 0;
                    a.end_out[pid[h]] = -1;
                    a.alen_out[pid[h]] = 0;
                }
                pid[h] = -1;
            }
            if (pid[h] < 0) ql[h] = rl[h] = 0;
        }
        if (pid[0] < 0 && pid[1] < 0) continue;
        const int ncols = max(rl[0], rl[1]);
        GroupResult gr[2];
        uint32_t exotic = 0;
        {
            S sw;
            sw.init(a.kc);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int row = g * R + r;
                    const uint32_t c = row < ql[h] ? (unsigned char)qs[h][row] : 0u;
                    const uint32_t tb = lean_table(c, row >= ql[h], (uint32_t)a.kc.ppm);
                    if (h) sw.q2[r] = tb;
                    else sw.q[r] = tb;
                }
            }
            for (int x = g; x < small_cols(ncols); x += 64) {
                const int j = x - kPad;
                uint32_t v = 0;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint32_t cls = kRefPad;
                    if (j >= 0 && j < rl[h]) {
                        cls = ref_index_bf((unsigned char)rs[h][j]);
                        if (cls == kRefOther) exotic |= 1u << h;
                    }
                    v |= lean_selector(cls, h) << (16 * h);
                }
                col[x] = v;
            }
            wave_lds_sync();
            lean_sweep<S, true>(sw, col + kPad - g, ncols + 63, tr);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t bh;
                int row, t;
                sw.result(h, bh, row, t);
                const bool odd = __ballot((exotic >> h) & 1u) != 0;
                gr[h] = group_best<64>(bh, (uint32_t)(g * R + row + 1), (uint32_t)(t - g + 1), R,
                                       true, a.h_limit, odd ? 1u : 0u);
            }
        }
        wave_store_fence();
        int again = 0;
        WalkOut wo[2] = {{0, -1, 0}, {0, -1, 0}};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (pid[h] < 0) continue;
            if (uni(gr[h].flag)) again |= 1 << h;
            else wo[h] = small_walk(tr, R, S::W, 3, 16 * h, gr[h], ql[h], rl[h], moves + h * mw);
        }
        // the pairs left to 32-bit lanes, one after another; what their
        // columns overwrite in LDS is done with
        if (again) {
            if (g == 0) {
                atomicAdd(a.reruns, __builtin_popcount(again));
                host_flag(a.flags + kSmallRerun);
            }
            for (int h = 0; h < 2; ++h) {
                if (!((again >> h) & 1)) continue;
                S32 sw;
                sw.init(a.kc);
                const int q_n = h ? ql[1] : ql[0], r_n = h ? rl[1] : rl[0];
                const char *q_s = h ? qs[1] : qs[0], *r_s = h ? rs[1] : rs[0];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int row = g * R + r;
                    sw.q[r] = rail_query(row < q_n ? (unsigned char)q_s[row] : 0u, row >= q_n);
                }
                for (int x = g; x < small_cols(r_n); x += 64) {
                    const int j = x - kPad;
                    const bool pad = j < 0 || j >= r_n;
                    col[x] = rail_ref(pad ? 0u : (unsigned char)r_s[j], pad);
                }
                wave_lds_sync();
                lean_sweep<S32, false>(sw, col + kPad - g, r_n + 63, tr);
                uint32_t bh;
                int row, t;
                sw.result(0, bh, row, t);
                const GroupResult r32 = group_best<64>(bh, (uint32_t)(g * R + row + 1),
                                                       (uint32_t)(t - g + 1), R, false, 0, 0);
                wave_store_fence();
                const WalkOut w = small_walk(tr, R, S32::W, 4, 0, r32, q_n, r_n, moves + h * mw);
                if (h) {
                    gr[1] = r32;
                    wo[1] = w;
                } else {
                    gr[0] = r32;
                    wo[0] = w;
                }
            }
        }
        // outputs, and both pairs' strings at once, half a wave each
        const int h = g >> 5;
        ExpandPair e;
        const int p = h ? pid[1] : pid[0];
        if (p >= 0) {
            const GroupResult r = h ? gr[1] : gr[0];
            const WalkOut w = h ? wo[1] : wo[0];
            if ((g & 31) == 0) {
                a.score_out[p] = r.score;
                a.start_out[p] = w.start;
                a.end_out[p] = w.end;
                a.alen_out[p] = w.len;
            }
            const int64_t co = a.coff[p];
            e.live = true;
            e.len = w.len;
            e.row = r.row;
            e.col = r.col;
            e.nq = min(h ? ql[1] : ql[0], r.row);
            e.nr = min(h ? rl[1] : rl[0], r.col);
            e.qsrc = (const unsigned char *)(h ? qs[1] : qs[0]);
            e.rsrc = (const unsigned char *)(h ? rs[1] : rs[0]);
            e.qc = a.qcons + co;
            e.rc = a.rcons + co;
            e.mv = moves + h * mw;
        }
        const int qw = small_qw(a.maxq), rw = small_rw(a.maxr);
        uint32_t *base = col + h * (qw + rw);
        expand_row<32>(e, base, base + qw, g & 31);
    }
}

}  // namespace

int64_t small_wave_words(int maxr) { return (int64_t)((maxr + 63 + 3) & ~3) * 64; }

template <int FORM>
static hipError_t launch_small_as(const SmallArgs &a, int blocks, hipStream_t st) {
    const size_t lds = 4 * (size_t)a.wpb * small_lds_words(a.maxq, a.maxr);
    switch (std::max(1, (a.maxq + 63) / 64)) {
#define SWIFT_S(RR)                                                                          \
    case RR: {                                                                               \
        auto k = sw_small_kernel<RR, FORM>;                                                  \
        hipLaunchKernelGGL(k, dim3(blocks), dim3(64 * a.wpb), lds, st, a);                   \
        break;                                                                               \
    }
        SWIFT_S(1) SWIFT_S(2) SWIFT_S(3) SWIFT_S(4) SWIFT_S(5)
#undef SWIFT_S
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_small(const SmallArgs &a, int blocks, hipStream_t st) {
    return a.form == kLean ? launch_small_as<kLean>(a, blocks, st)
                           : launch_small_as<kLeanWide>(a, blocks, st);
}

}  // namespace swift
