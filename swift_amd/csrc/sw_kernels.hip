// sw_kernels.hip -- Smith-Waterman forward sweep, traceback walk and
// length binning for gfx950 (MI355X, wave64).
//
// Recurrence and tie rules are those of the reference CPU path,
// computeMaxScore_cpu / findArrMax / backtrack_cpu
// (src/smithWaterman.cu:114-335):
//   H(i,j) = first maximum of [diag, up, left, 0]
//   diag = H(i-1,j-1) + (match(q_i, R_j) ? match : mismatch)
//   up   = H(i-1,j) + (dir(i-1,j) == up   ? gapExt : gapOpen)
//   left = H(i,j-1) + (dir(i,j-1) == left ? gapExt : gapOpen)
// with the best cell the first strict maximum in row-major order.
//
// Kernel design (written for CDNA4, not translated from the reference's
// one-thread-per-row block kernel):
//  * A lane group of G lanes (G = 16 via DPP row_shr, or 64 via wave_shr)
//    owns one pair per 32-bit lane slot; lane g holds query rows
//    [g*R, g*R+R) in registers and lane g sweeps column j = t - g at step t
//    (a staggered wavefront).  The last row's exits move one lane down per
//    step with a single DPP mov, no LDS round trip and no barrier.
//  * Every cell works on keys K = 4*H + dir (dir 3 diag, 2 up, 1 left,
//    0 start): max(diagKey, upKey, leftKey, 0) yields both the score and the
//    reference's tie-broken direction.  Exits carried to the neighbours are
//    already keys: EU = 4*(H + gap_up) + 2, EL = 4*(H + gap_left) + 1,
//    DR = 4*H + 4*mismatch + 3 (diagonal, before the match bonus).
//  * Batched form: two pairs per lane in the two 16-bit halves of each
//    register (v_pk_* int16 arithmetic), 4 groups of 16 lanes per wave,
//    8 pairs per wave task; a persistent grid pulls tasks from an atomic
//    counter in length-binned, longest-first order.  Any pair whose best
//    score nears the int16 range is flagged and re-run with int32 lanes.
//  * Direction codes (2 bits/cell) are packed per lane into 32-bit words and
//    stored coalesced ([step][word][lane]); a separate kernel walks them
//    back with one lane per pair.
#include "scan.hpp"
#include "sw_sweep.hpp"

namespace swift {

// ---------------------------------------------------------------------------
// Batched persistent kernels.
// ---------------------------------------------------------------------------
// LDS words per wave: each of the 64 / G groups has its reference columns and
// a tail of G + 2 padding columns (the lanes run up to G - 1 columns past the
// last, and steps are rounded up to whole granules of 4); the G columns before
// a group's column 0 are the end of the tail before it, or the wave's first G
// words; 4 words past the end are read ahead.  31.2 KB a workgroup of the
// 16-lane kernels: five of them fit a CU.
template <int G> constexpr int group_lds_stride() { return kBatchCols + G + 2; }
template <int G> constexpr int wave_lds_words() { return G + 64 / G * group_lds_stride<G>() + 4; }

// One wave task: 64 / G groups of G lanes (G = 16: 4 groups; G = 64, the
// wide form: one); PK -> 2 pairs per group (halves).
template <int G, int R, bool PK, int FORM>
__device__ __forceinline__ void run_task(const BatchArgs &a, const Task &tk, uint32_t *lds) {
    constexpr bool LEAN = FORM != kGeneralForm;
    using S = std::conditional_t<LEAN, Lean<G, R, PK, FORM>,
                                 Sweep<G, R, PK, PK ? kOneHot : kBytes>>;
    constexpr int PPG = PK ? 2 : 1;  // pairs per group
    constexpr int NG = 64 / G;       // groups per wave
    constexpr int TAIL = G + 2;      // padding columns after the last
    const int lane = threadIdx.x & 63;
    const int grp = lane / G, g = lane % G;
    // reference codes at [j], -G <= j < columns + TAIL
    uint32_t *rr_lds = lds + G + grp * group_lds_stride<G>();

    // the group's pairs.  The loads are unconditional (a slot past the
    // task's pairs reads its first pair and is then cleared; byte loads are
    // clamped into the sequence, whose first byte exists for every binned
    // pair) so that each level of the order -> lengths -> bytes chain issues
    // as one batch: one memory round trip per level instead of one per load.
    int pid[PPG], ql[PPG], rl[PPG];
    int64_t qo[PPG], ro[PPG];
#pragma unroll
    for (int h = 0; h < PPG; ++h) {
        const int slot = grp * PPG + h;
        pid[h] = a.order[tk.first + (slot < tk.npairs ? slot : 0)];
    }
#pragma unroll
    for (int h = 0; h < PPG; ++h) {
        const int p = pid[h];
        ql[h] = a.qlen[p];
        rl[h] = a.rlen[p];
        qo[h] = a.qoff[p];
        ro[h] = a.roff[p];
    }
#pragma unroll
    for (int h = 0; h < PPG; ++h) {
        if (grp * PPG + h >= tk.npairs) {
            pid[h] = -1;
            ql[h] = rl[h] = 0;
            qo[h] = ro[h] = 0;
        }
    }
    // the query rows: raw bytes now (in flight during the reference loads
    // below), converted to match tables afterwards
    S sw;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = g * R + r;
        uint32_t v[PPG];
#pragma unroll
        for (int h = 0; h < PPG; ++h) {
            // unconditional load of an in-range byte, then the select: a
            // load under a branch is waited for before the branch joins
            const uint32_t c = (unsigned char)a.qseq[qo[h] + max(0, min(row, ql[h] - 1))];
            v[h] = row < ql[h] ? c : 256u;
        }
        sw.q[r] = v[0];
        if constexpr (PK) sw.q2[r] = v[PPG - 1];
    }
    // reference codes of the group's pairs into LDS (both halves packed),
    // padding up to the last column any lane reaches (ncols + G - 2)
    // and the step-ahead prefetch of it.  Loaded in batches of NB columns
    // per lane, each batch's loads issued together.
    const int ncols = tk.steps - (G - 1);
    constexpr int NB = 8;
    uint32_t exotic = 0;  // bit h: the pair's reference holds a byte outside ACGTNacgtn
    auto ref_word = [](uint32_t cls_or_byte, bool pad, int half) -> uint32_t {
        if constexpr (!PK) return LEAN ? rail_ref(cls_or_byte, pad) : pad ? 0u : byte_rcode((unsigned char)cls_or_byte);
        else return LEAN ? lean_selector(cls_or_byte, half) : column_selector(cls_or_byte, half);
    };
    const uint32_t pad_word = PK ? ref_word(kRefPad, true, 0) | ref_word(kRefPad, true, 1) << 16
                                 : ref_word(0, true, 0);
    for (int j0 = g; j0 < ncols + TAIL; j0 += NB * G) {
        unsigned char cb[NB][PPG];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int j = j0 + i * G;
#pragma unroll
            for (int h = 0; h < PPG; ++h)
                cb[i][h] = (unsigned char)a.rseq[ro[h] + max(0, min(j, rl[h] - 1))];
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int j = j0 + i * G;
            if (j < ncols + TAIL) {
                uint32_t v = 0;
#pragma unroll
                for (int h = 0; h < PPG; ++h) {
                    const bool pad = j >= rl[h];
                    uint32_t code = cb[i][h];
                    if constexpr (PK) {
                        code = pad ? kRefPad : ref_index_bf(cb[i][h]);
                        if (code == kRefOther) exotic |= 1u << h;
                    }
                    v |= ref_word(code, pad, h) << (16 * h);
                }
                rr_lds[j] = v;
            }
        }
    }
    if constexpr (PK) {
#pragma unroll
        for (int s2 = G / 2; s2 >= 1; s2 >>= 1) exotic |= __shfl_xor(exotic, s2, G);
    }
    // the G columns before column 0: the wave's first words, and the end of
    // each group's tail
    if (grp == 0) rr_lds[g - G] = pad_word;
    rr_lds[kBatchCols + 2 + g] = pad_word;
    sw.init(a.kc);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        // 256: a row past the query (no match anywhere)
        auto conv = [&](uint32_t c) -> uint32_t {
            if constexpr (LEAN)
                return PK ? lean_table(c, c > 255u, (uint32_t)a.kc.ppm) : rail_query(c & 255u, c > 255u);
            else
                return c > 255u ? 0u : PK ? query_table(query_mask_bf((unsigned char)c))
                                          : byte_qcode((unsigned char)c);
        };
        sw.q[r] = conv(sw.q[r]);
        if constexpr (PK) sw.q2[r] = conv(sw.q2[r]);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_s_waitcnt(0);  // LDS writes of this wave visible to its lanes
    __builtin_amdgcn_wave_barrier();

    const int T = tk.steps;
    if constexpr (LEAN) {
        lean_sweep<S, PK>(sw, rr_lds - g, T, a.trace + tk.trace_base);
    } else {
        uint32_t *tr = a.trace + tk.trace_base;
        uint32_t rr_next = rr_lds[-g];  // column of step 0
        auto run = [&](auto masked, int t) {
            int j = t - g;
            uint32_t rr = rr_next;
            rr_next = rr_lds[1 + j];  // prefetch the next step's column
            uint32_t vmask = 0;
            if constexpr (decltype(masked)::value) {
#pragma unroll
                for (int h = 0; h < PPG; ++h)
                    if (j >= 0 && j < rl[h]) vmask |= (PK ? 0xFFFFu : 0xFFFFFFFFu) << (16 * h);
            }
            uint32_t a1[S::W];
#pragma unroll
            for (int w = 0; w < S::W; ++w) a1[w] = 0;
            sw.template step<decltype(masked)::value>(rr, j, vmask, splat<PK>(15 - (t & 15)), a1);
#pragma unroll
            for (int w = 0; w < S::W; ++w) tr[trace_word<S::W>(t, w, lane)] = a1[w];
        };
        // int32: masked steps keep the cells outside a pair's columns out of
        // its row maxima.  Packed: no step is masked (see Sweep).
        if constexpr (PK) {
            for (int t = 0; t < T; ++t) {
                run(std::false_type{}, t);
                if ((t & 15) == 15 || t == T - 1) sw.block_end(splat<true>((t >> 4) << 5));
            }
        } else {
            const int lo = min(G - 1, T), hi = max(lo, tk.min_rlen);
            sweep_steps(T, lo, hi, run);
        }
    }

    // per half: the lane's best cell, then the group's
    GroupResult gres[PPG];
#pragma unroll
    for (int h = 0; h < PPG; ++h) {
        uint32_t bh = 0, brow = 0, bcol = 0;
        if constexpr (LEAN) {
            int row, t;
            sw.result(h, bh, row, t);
            brow = (uint32_t)(g * R + row + 1);
            bcol = (uint32_t)(t - g + 1);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                int row = g * R + r;
                uint32_t hv, cv;
                if constexpr (PK) {
                    // block << 5 | (15 - t%16) -> step t -> column t - g (+1)
                    const uint32_t bc = (sw.bcol[r] >> (16 * h)) & 0xFFFFu;
                    hv = ((sw.best[r] >> (16 * h)) & 0xFFFFu) >> 5;
                    cv = ((bc >> 5) << 4) + 15u - (bc & 15u) - (uint32_t)g + 1;
                } else {
                    hv = sw.best[r] >> kColBits;
                    cv = kMaxCols - (sw.best[r] & kMaxCols) + 1;
                }
                if (row < ql[h] && hv > bh) {
                    bh = hv;
                    brow = row + 1;
                    bcol = cv;
                }
            }
        }
        gres[h] = group_best<G>(bh, brow, bcol, R, PK, a.h_limit, (exotic >> h) & 1);
        if (g == 0 && pid[h] >= 0) {
            a.res[pid[h]] = PairResult{gres[h].score, gres[h].row, gres[h].col, gres[h].flag};
            if (gres[h].flag) atomicAdd(a.nflagged, 1);
        }
    }

    const int s = lane;
    const int sg = min(s / PPG, NG - 1), sh = s % PPG;
    if (a.walk_deferred) {
        // record where the pair's trace lives; sw_walk_kernel walks it
        if (s < tk.npairs)
            a.ptr[a.order[tk.first + s]] = PairTrace{tk.trace_base, sg * G, (int16_t)R,
                                                     (int8_t)S::W, (int8_t)(sh | (PK ? 2 : 0))};
        __builtin_amdgcn_wave_barrier();
        return;
    }
    // Traceback of the task's pairs right after the sweep, while the trace
    // is cache-hot: lane s walks slot s.  A flagged pair is left to the int32
    // re-run.  The walk is latency-bound; other waves' sweeps cover it.
    wave_store_fence();
    int w_score = 0, w_row = 0, w_col = 0, w_flag = 1;
#pragma unroll
    for (int h = 0; h < PPG; ++h) {
        int v0 = __shfl(gres[h].score, sg * G, 64);
        int v1 = __shfl(gres[h].row, sg * G, 64);
        int v2 = __shfl(gres[h].col, sg * G, 64);
        int v3 = __shfl(gres[h].flag, sg * G, 64);
        if (h == sh) {
            w_score = v0;
            w_row = v1;
            w_col = v2;
            w_flag = v3;
        }
    }
    if (s < tk.npairs && !w_flag) {
        const int p = a.order[tk.first + s];
        const PairTrace pt{tk.trace_base, sg * G, (int16_t)R, (uint8_t)S::W,
                           (int8_t)(sh | (PK ? 2 : 0))};
        const int64_t co = a.coff[p];
        WalkOut wo = walk_pair(a.trace, w_score, w_row, w_col, pt, a.qseq + a.qoff[p],
                               a.rseq + a.roff[p], a.qlen[p], a.rlen[p], a.qcons + co,
                               a.rcons + co);
        a.score_out[p] = w_score;
        a.start_out[p] = wo.start;
        a.end_out[p] = wo.end;
        a.alen_out[p] = wo.len;
    }
    __builtin_amdgcn_wave_barrier();
}

// Deferred walk-back, in two kernels over the binned pairs after every sweep
// of the call (both passes) has finished.  sw_walk_kernel: one lane per pair
// follows the trace and stores the path as 2-bit moves (16 per word, walk
// order) plus start/end/length; it touches no sequence bytes, so its
// dependent loads are the trace granules alone.  sw_expand_kernel turns the
// moves into the consensus strings, four pairs per wave (below).  A pair
// still flagged for the int32 re-run (none after the re-run pass) is
// skipped.
__global__ void __launch_bounds__(256) sw_walk_kernel(BatchArgs a, const int32_t *order,
                                                      const int32_t *first_p,
                                                      const int32_t *count, uint32_t *moves,
                                                      int move_words) {
    const int n = *count;
    const int32_t *ord = order + (first_p ? *first_p : 0);
    for (int i = blockIdx.x * 256 + (int)threadIdx.x; i < n; i += gridDim.x * 256) {
        const int p = ord[i];
        const PairResult r = a.res[p];
        if (r.flags & 1) continue;
        const PairTrace pt = a.ptr[p];
        uint32_t *mv = moves + (int64_t)p * move_words;
        uint32_t word = 0;
        auto emit = [&](int k, int op, int, int) {
            word |= (uint32_t)op << (2 * (k & 15));
            if ((k & 15) == 15) {
                mv[k >> 4] = word;
                word = 0;
            }
        };
        WalkOut wo = walk_cells<TraceReaderLean>(a.trace, r.score, r.row, r.col, pt, a.qlen[p],
                                                 a.rlen[p], emit);
        if (wo.len & 15) mv[wo.len >> 4] = word;
        a.score_out[p] = r.score;
        a.start_out[p] = wo.start;
        a.end_out[p] = wo.end;
        a.alen_out[p] = wo.len;
    }
}


// sw_walk_kernel's work, one wave per pair (small batches); a path's moves
// fit one word per lane
static_assert((kMaxBatchQ + kMaxBatchR) / 16 + 1 <= 64, "moves of a batched pair");
__global__ void __launch_bounds__(256) sw_walk_wave_kernel(BatchArgs a, const int32_t *order,
                                                           const int32_t *first_p,
                                                           const int32_t *count, uint32_t *moves,
                                                           int move_words) {
    const int n = uni(*count);
    const int32_t *ord = order + (first_p ? uni(*first_p) : 0);
    const int nw = gridDim.x * 4;
    for (int i = uni((int)(blockIdx.x * 4 + (threadIdx.x >> 6))); i < n; i += nw) {
        const int p = uni(ord[i]);
        const PairResult r = a.res[p];
        if (uni(r.flags) & 1) continue;
        const PairTrace pt = a.ptr[p];
        const int half = uni(pt.half), R = uni(pt.rows), W = uni(pt.words);
        const int64_t base = ((int64_t)uni((int)(pt.base >> 32)) << 32) |
                             (uint32_t)uni((int)(uint32_t)pt.base);
        const uint4 *tr = reinterpret_cast<const uint4 *>(a.trace) + base / 4 + uni(pt.lane0);
        const int score = uni(r.score);
        RegMoves<1> mv(moves + (int64_t)p * move_words);
        WalkOut wo = walk_wave(tr, R, W, (half & 2) ? 3 : 4, (half & 1) * 16, score, uni(r.row),
                               uni(r.col), uni(a.qlen[p]), uni(a.rlen[p]), mv);
        if ((threadIdx.x & 63) == 0) {
            a.score_out[p] = score;
            a.start_out[p] = wo.start;
            a.end_out[p] = wo.end;
            a.alen_out[p] = wo.len;
        }
    }
}

// sw_expand_kernel: the batched pass's consensus strings, four pairs per
// wave (one per 16-lane row), 16 pairs per workgroup.
__global__ void __launch_bounds__(256) sw_expand_kernel(BatchArgs a, const int32_t *order,
                                                        const int32_t *first_p,
                                                        const int32_t *count,
                                                        const uint32_t *moves, int move_words) {
    constexpr int kQW = (kMaxBatchQ + 6) / 4, kRW = (kMaxBatchR + 6) / 4;  // dwords staged
    constexpr int kPairs = 16;                                           // per workgroup
    __shared__ uint32_t lq4[kPairs][kQW], lr4[kPairs][kRW];
    const int n = *count;
    const int slot = threadIdx.x >> 4, sl = threadIdx.x & 15;
    const int32_t *ord = order + (first_p ? *first_p : 0);
    for (int i0 = blockIdx.x * kPairs; i0 < n; i0 += gridDim.x * kPairs) {
        const int i = i0 + slot;
        ExpandPair e;
        if (i < n) {
            const int p = ord[i];
            const PairResult r = a.res[p];
            if (!(r.flags & 1)) {  // a flagged pair is left to the int32 pass
                e.live = true;
                e.len = a.alen_out[p];
                e.row = r.row;
                e.col = r.col;
                // the path only visits rows <= row and columns <= col
                e.nq = min(a.qlen[p], r.row);
                e.nr = min(a.rlen[p], r.col);
                const int64_t co = a.coff[p];
                e.qsrc = (const unsigned char *)a.qseq + a.qoff[p];
                e.rsrc = (const unsigned char *)a.rseq + a.roff[p];
                e.qc = a.qcons + co;
                e.rc = a.rcons + co;
                e.mv = moves + (int64_t)p * move_words;
            }
        }
        expand_row<16>(e, lq4[slot], lr4[slot], sl);
    }
}

// Row classes: R per lane with 16-lane groups covers query length 16*R.
// One kernel per R: each gets the register budget its R needs (a single
// kernel switching over all R is allocated for the worst case).
#define SWIFT_R16_CASES(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) \
    X(11) X(12) X(13) X(14) X(15) X(16) X(17) X(18) X(19) X(20)
#define SWIFT_R32_CASES(X) X(2) X(4) X(6) X(8) X(10) X(12) X(14) X(16) X(18) X(20)

// Occupancy floor per row class (waves per SIMD), set where the natural
// register count sits just above an occupancy step.
__host__ __device__ constexpr int batch_waves_per_eu(int R, bool pk, bool lean) {
    return lean ? (R <= 6 ? 5 : R <= 12 ? 4 : 3)
           : pk ? (R <= 7 ? 5 : R <= 12 ? 4 : R <= 16 ? 3 : 2)
                : (R <= 10 ? 5 : R <= 16 ? 4 : 3);
}

template <int R, bool PK, int FORM>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(batch_waves_per_eu(R, PK, FORM != kGeneralForm))))
sw_batch_kernel(BatchArgs a) {
    __shared__ uint32_t lds[4][wave_lds_words<kBatchG>()];
    const int wave = threadIdx.x >> 6;
    const int lo = *a.task_lo, hi = *a.task_hi;
    if (lo >= hi) return;
    for (;;) {
        int tid = 0;
        if ((threadIdx.x & 63) == 0) tid = atomicAdd(a.next_task, 1);
        tid = __builtin_amdgcn_readfirstlane(__shfl(tid, 0, 64)) + lo;
        if (tid >= hi) break;
        const Task tk = a.tasks[tid];
        run_task<kBatchG, R, PK, FORM>(a, tk, lds[wave]);
    }
}

// The wide form for batches too small to fill the chip (scorings outside
// lean_scoring; the others take sw_small.hip's kernel): one 64-lane group
// per wave (the lane shift a wave_shr), kWideRows rows per lane, two packed
// pairs per task.  A 16-lane group sweeps R = 20 rows per lane over rlen + 15
// steps; a 64-lane group 5 rows over rlen + 63, so one task's latency, which
// is all a small batch waits for, drops about 3.5x for the same total work.
template <int R>
__global__ void __launch_bounds__(256) sw_batch_wide_kernel(BatchArgs a) {
    __shared__ uint32_t lds[4][wave_lds_words<kWideG>()];
    const int wave = threadIdx.x >> 6;
    const int lo = *a.task_lo, hi = *a.task_hi;
    if (lo >= hi) return;
    for (;;) {
        int tid = 0;
        if ((threadIdx.x & 63) == 0) tid = atomicAdd(a.next_task, 1);
        tid = __builtin_amdgcn_readfirstlane(__shfl(tid, 0, 64)) + lo;
        if (tid >= hi) break;
        const Task tk = a.tasks[tid];
        run_task<kWideG, R, true, kGeneralForm>(a, tk, lds[wave]);
    }
}

// ---------------------------------------------------------------------------
// Device-side length binning for the batched kernels.
//
// Pass 1 (classify): each pair gets a class -- int16 one-hot (fast path),
// int32 byte semantics (reference bytes outside ACGTN, scores beyond the
// int16 range, or an int16 overflow re-run) -- and a rows-per-lane class R.
// Bins are (class, R, rlen/8) and are visited longest-first, so tasks are
// served in decreasing cost (LPT) from the persistent work queue.
// ---------------------------------------------------------------------------
// pair -> bin (or -1 when the pair takes no part in this pass)
__device__ __forceinline__ int classify_pair(const BinArgs &a, int p) {
    int ql = a.qlen[p], rl = a.rlen[p];
    if (ql < 0 || rl < 0 || ql > kMaxBatchQ || rl > kMaxBatchR) {
        // lengths beyond the batched kernels: the pair is left out (score 0)
        // and the call reports the error
        atomicOr(a.error, 1);
        return -1;
    }
    if (ql == 0 || rl == 0) {
        // all-zero matrix: start 0, end -1, length 0 (src/smithWaterman.cu
        // :50,333-334)
        if (!a.prev) {
            a.score_out[p] = 0;
            a.start_out[p] = 0;
            a.end_out[p] = -1;
            a.alen_out[p] = 0;
        }
        return -1;
    }
    if (a.screened && (a.screened[p].flags & kScreenedFlag)) return -1;
    int cls;
    if (a.prev) {
        if (!(a.prev[p].flags & 1)) return -1;
        cls = 1;
    } else {
        // references with bytes outside ACGTNacgtn are caught by the int16
        // kernel itself and re-run with byte semantics in the int32 pass
        cls = a.force32 ? 1 : 0;
    }
    int R = max(1, (ql + kBatchG - 1) / kBatchG);
    // coarse classes (small batches): fewer class kernels, each a pair's rows
    // spread over fewer lanes of its group; the rows past the query are padding
    // (queries of 100 bases sweep 7 rows a lane, not 10: 20,000 reads' sweep 732
    // -> 527 us)
    if (a.coarse > 0)
        R = max(R, min(a.max_rows, (R + a.coarse - 1) / a.coarse * a.coarse));
    if (cls == 1) R = r32_class(R);
    int lb = min(kLenBins - 1, rl >> 3);
    // bin order: class, then R descending, then rlen descending
    return (cls * kRBins + (kRBins - R)) * kLenBins + (kLenBins - 1 - lb);
}

// Pairs [blockIdx.x * kBinChunk, +kBinChunk) are counted in an LDS
// histogram first, so a bin costs one global atomic per workgroup however
// many pairs share it (uniform reads put every pair in one bin).
constexpr int kBinPer = 8;
constexpr int kBinChunk = 256 * kBinPer;

__global__ void __launch_bounds__(256) sw_bin_classify(BinArgs a) {
    __shared__ int32_t hist[kNumBins];
    for (int b = threadIdx.x; b < kNumBins; b += 256) hist[b] = 0;
    __syncthreads();
    const int base = blockIdx.x * kBinChunk;
#pragma unroll
    for (int i = 0; i < kBinPer; ++i) {
        int p = base + i * 256 + (int)threadIdx.x;
        if (p < a.npairs) {
            int b = classify_pair(a, p);
            a.bin_of[p] = b;
            if (b >= 0) atomicAdd(&hist[b], 1);
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < kNumBins; b += 256)
        if (hist[b]) atomicAdd(&a.bin_count[b], hist[b]);
}

// single workgroup: bin prefix sums and per-(class, R) task counts
__global__ void __launch_bounds__(1024) sw_bin_scan(TaskArgs a) {
    __shared__ int32_t part[1024];
    const int tid = threadIdx.x;
    constexpr int per = (kNumBins + 1023) / 1024;
    int32_t loc[per], s = 0;
#pragma unroll
    for (int i = 0; i < per; ++i) {
        int b = tid * per + i;
        loc[i] = b < kNumBins ? a.bin_count[b] : 0;
        s += loc[i];
    }
    part[tid] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        int32_t v = tid >= off ? part[tid - off] : 0;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    int32_t run = part[tid] - s;
#pragma unroll
    for (int i = 0; i < per; ++i) {
        int b = tid * per + i;
        if (b < kNumBins) a.bin_cursor[b] = run;
        run += loc[i];
    }
    __syncthreads();
    // segment (class, R) lengths in parallel, then their task offsets
    __shared__ int32_t seg_tasks[2 * kRBins];
    if (tid < 2 * kRBins) a.seg_steps[tid] = 0;  // summed by sw_build_tasks
    if (tid < 2 * kRBins) {
        const int seg = tid, cls = seg / kRBins;
        int32_t len = 0;
        for (int lb = 0; lb < kLenBins; ++lb) len += a.bin_count[seg * kLenBins + lb];
        const int slots = cls == 0 ? (a.wide && seg == 0 ? kSlotsWide : kSlots16) : kSlots32;
        a.seg_first[seg] = a.bin_cursor[seg * kLenBins];
        a.seg_len[seg] = len;
        seg_tasks[seg] = (len + slots - 1) / slots;
    }
    __syncthreads();
    if (tid == 0) {
        int32_t t0 = 0;
        for (int seg = 0; seg < 2 * kRBins; ++seg) {
            a.seg_task0[seg] = t0;
            t0 += seg_tasks[seg];
        }
        a.seg_task0[2 * kRBins] = t0;
        *a.ntasks = t0;
        *a.npairs_binned = part[1023];
    }
}

// Same chunks as sw_bin_classify: ranks within the chunk from LDS atomics,
// one global cursor reservation per (chunk, bin).
__global__ void __launch_bounds__(256) sw_bin_scatter(const int32_t *bin_of, int npairs,
                                                      int32_t *bin_cursor, int32_t *order) {
    __shared__ int32_t hist[kNumBins];
    for (int b = threadIdx.x; b < kNumBins; b += 256) hist[b] = 0;
    __syncthreads();
    const int base = blockIdx.x * kBinChunk;
    int bin[kBinPer], rank[kBinPer];
#pragma unroll
    for (int i = 0; i < kBinPer; ++i) {
        int p = base + i * 256 + (int)threadIdx.x;
        bin[i] = p < npairs ? bin_of[p] : -1;
        rank[i] = bin[i] >= 0 ? atomicAdd(&hist[bin[i]], 1) : 0;
    }
    __syncthreads();
    for (int b = threadIdx.x; b < kNumBins; b += 256)
        if (hist[b]) hist[b] = atomicAdd(&bin_cursor[b], hist[b]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kBinPer; ++i)
        if (bin[i] >= 0) order[hist[bin[i]] + rank[i]] = base + i * 256 + (int)threadIdx.x;
}

// task descriptors (trace sizes filled, bases scanned afterwards)
__device__ __forceinline__ void build_task(int t, const int32_t *seg_task0,
                                           const int32_t *seg_first, const int32_t *seg_len,
                                           const int32_t *order, const int32_t *rlen,
                                           Task *tasks, int64_t *task_words,
                                           unsigned long long *steps_acc, int wide) {
    int seg = 0;
    while (seg + 1 < 2 * kRBins && seg_task0[seg + 1] <= t) ++seg;
    int cls = seg / kRBins;
    int R = kRBins - (seg % kRBins);
    int slots = cls == 0 ? kSlots16 : kSlots32;
    int G = kBatchG;
    if (wide && seg == 0) {
        slots = kSlotsWide;
        G = kWideG;
        R = kWideRows;
    }
    int k = t - seg_task0[seg];
    int first = seg_first[seg] + k * slots;
    int n = min(slots, seg_len[seg] - k * slots);
    int mx = 0, mn = 1 << 30;
    for (int i = 0; i < n; ++i) {
        int rl = rlen[order[first + i]];
        mx = max(mx, rl);
        mn = min(mn, rl);
    }
    Task tk;
    tk.trace_base = 0;
    tk.first = first;
    tk.npairs = (int16_t)n;
    tk.rows = (int16_t)R;
    tk.steps = mx + G - 1;
    tk.min_rlen = mn;
    tasks[t] = tk;
    int kpw = cls == 0 ? 8 : 16;
    int W = (R + kpw - 1) / kpw;
    task_words[t] = (int64_t)((tk.steps + 3) & ~3) * W * 64;  // whole 4-step granules
    atomicAdd(&steps_acc[seg], (unsigned long long)tk.steps);
}

__global__ void __launch_bounds__(256)
sw_build_tasks(const int32_t *seg_task0, const int32_t *seg_first, const int32_t *seg_len,
               const int32_t *ntasks_p, const int32_t *order, const int32_t *rlen, Task *tasks,
               int64_t *task_words, unsigned long long *seg_steps, int wide) {
    // per-segment sums of the tasks' sweep steps (the host's cost estimate
    // of each class kernel), reduced in LDS before one atomic per segment
    __shared__ unsigned long long steps_acc[2 * kRBins];
    if (threadIdx.x < 2 * kRBins) steps_acc[threadIdx.x] = 0;
    __syncthreads();
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    int ntasks = *ntasks_p;
    if (t < ntasks) build_task(t, seg_task0, seg_first, seg_len, order, rlen, tasks, task_words,
                               steps_acc, wide);
    __syncthreads();
    if (threadIdx.x < 2 * kRBins && steps_acc[threadIdx.x])
        atomicAdd(&seg_steps[threadIdx.x], steps_acc[threadIdx.x]);
}

// Exclusive scan over one 1,024-thread workgroup (each thread's value v):
// wave scans by shuffles, then the 16 wave totals through LDS.
template <class T>
__device__ __forceinline__ T wg_excl_scan(T v, T *wsum, T *total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    T x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        T o = __shfl_up(x, d, 64);
        if (lane >= d) x += o;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    T before = 0, all = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const T t = wsum[i];
        before += i < w ? t : T(0);
        all += t;
    }
    __syncthreads();
    *total = all;
    return before + x - v;
}

// The whole of pass-1 binning for a batch of up to kBinTinyPairs pairs in
// one workgroup (classify, bin counts, their scan, the segments, the
// scatter, the tasks and their trace bases), with the sizes the host reads
// written straight into its mapped staging block: one launch and no gather
// instead of seven launches.  Same outputs as launch_binning + the gather
// (the order within a bin may differ; nothing depends on it).
__global__ void __launch_bounds__(1024)
sw_bin_tiny(BinArgs a, TaskArgs ta, int32_t *order, Task *tasks, int64_t *task_words,
            int64_t *total_words, const int32_t *counters, TinyStage hs) {
    constexpr int PP = kBinTinyPairs / 1024;           // pairs per thread
    constexpr int BP = (kNumBins + 1023) / 1024;       // bins per thread
    constexpr int TP = (kBinTinyPairs / kSlotsWide + 2 * kRBins + 1023) / 1024;  // tasks per thread
    __shared__ int32_t hist[kNumBins];  // counts, then cursors
    __shared__ int32_t s_task0[2 * kRBins + 1], s_first[2 * kRBins], s_len[2 * kRBins];
    __shared__ unsigned long long steps_acc[2 * kRBins];
    __shared__ int32_t wsum32[16];
    __shared__ int64_t wsum64[16];
    const int tid = threadIdx.x, n = a.npairs;
    for (int i = tid; i < kNumBins; i += 1024) hist[i] = 0;
    if (tid < 2 * kRBins) steps_acc[tid] = 0;
    __syncthreads();
    int bin[PP], rank[PP];
#pragma unroll
    for (int k = 0; k < PP; ++k) {
        const int p = k * 1024 + tid;
        bin[k] = p < n ? classify_pair(a, p) : -1;
        rank[k] = bin[k] >= 0 ? atomicAdd(&hist[bin[k]], 1) : 0;
    }
    __syncthreads();
    if (tid < 2 * kRBins) {
        int32_t len = 0;
        for (int lb = 0; lb < kLenBins; ++lb) len += hist[tid * kLenBins + lb];
        s_len[tid] = len;
    }
    // bin cursors: exclusive scan of the counts
    int32_t loc[BP], sum = 0;
#pragma unroll
    for (int i = 0; i < BP; ++i) {
        const int b = tid * BP + i;
        loc[i] = b < kNumBins ? hist[b] : 0;
        sum += loc[i];
    }
    int32_t binned;
    int32_t run = wg_excl_scan<int32_t>(sum, wsum32, &binned);
#pragma unroll
    for (int i = 0; i < BP; ++i) {
        const int b = tid * BP + i;
        if (b < kNumBins) hist[b] = run;
        run += loc[i];
    }
    __syncthreads();
    if (tid == 0) {
        int32_t t0 = 0;
        for (int seg = 0; seg < 2 * kRBins; ++seg) {
            const int cls = seg / kRBins;
            const int slots = cls == 0 ? (ta.wide && seg == 0 ? kSlotsWide : kSlots16) : kSlots32;
            s_first[seg] = hist[seg * kLenBins];
            s_task0[seg] = t0;
            t0 += (s_len[seg] + slots - 1) / slots;
        }
        s_task0[2 * kRBins] = t0;
    }
#pragma unroll
    for (int k = 0; k < PP; ++k)
        if (bin[k] >= 0) order[hist[bin[k]] + rank[k]] = k * 1024 + tid;
    __syncthreads();  // the order and the segments, for every thread of the group
    const int nt = s_task0[2 * kRBins];
    if (tid <= 2 * kRBins) ta.seg_task0[tid] = s_task0[tid];
    if (tid < 2 * kRBins) {
        ta.seg_first[tid] = s_first[tid];
        ta.seg_len[tid] = s_len[tid];
    }
    if (tid == 0) {
        *ta.ntasks = nt;
        *ta.npairs_binned = binned;
    }
    for (int t = tid; t < nt; t += 1024)
        build_task(t, s_task0, s_first, s_len, order, a.rlen, tasks, task_words, steps_acc,
                   ta.wide);
    __syncthreads();  // the task words
    int64_t tw[TP], tsum = 0;
#pragma unroll
    for (int i = 0; i < TP; ++i) {
        const int t = tid * TP + i;
        tw[i] = t < nt ? task_words[t] : 0;
        tsum += tw[i];
    }
    int64_t words;
    int64_t base = wg_excl_scan<int64_t>(tsum, wsum64, &words);
#pragma unroll
    for (int i = 0; i < TP; ++i) {
        const int t = tid * TP + i;
        if (t < nt) tasks[t].trace_base = base;
        base += tw[i];
    }
    if (tid < 2 * kRBins) {
        ta.seg_steps[tid] = steps_acc[tid];
        hs.steps[tid] = (int64_t)steps_acc[tid];
    }
    if (tid <= 2 * kRBins) hs.seg[tid] = s_task0[tid];
    if (tid == 0) {
        *total_words = words;
        *hs.words = words;
    }
    __syncthreads();  // the counters (the error flag of classify_pair included)
    if (tid < 16)
        hs.cnt[tid] = tid == 0   ? nt
                      : tid == 1 ? binned
                                 : __hip_atomic_load(const_cast<int32_t *>(counters) + tid,
                                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct StoreTaskBase {
    Task *t;
    __device__ void operator()(int i, int64_t v) const { t[i].trace_base = v; }
};

__global__ void fill_i32(int32_t *p, int n, int32_t v) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// zeroes up to four arrays in one launch: blockIdx.y picks the array
__global__ void __launch_bounds__(256) zero_spans(ZeroSpans z) {
    int32_t *p = z.p[blockIdx.y];
    const int n = z.n[blockIdx.y];
    for (int i = blockIdx.x * 256 + (int)threadIdx.x; i < n; i += gridDim.x * 256) p[i] = 0;
}

// Copies a few small device arrays into one host staging block (mapped
// pinned memory), so the host reads them all after a single stream
// synchronisation instead of one copy each.
__global__ void __launch_bounds__(256) gather_words(Gather g) {
    for (int s = 0; s < g.nspans; ++s)
        for (int i = threadIdx.x; i < g.nwords[s]; i += 256) g.out[g.dst[s] + i] = g.src[s][i];
}

// ---------------------------------------------------------------------------
// host-visible launch helpers (used by sw_host.cpp)
// ---------------------------------------------------------------------------
// Persistent grid of one row-class kernel: as many 256-thread blocks as fit
// on every CU at once (cached per kernel); `waves_per_cu` > 0 caps it.
template <class K>
static int full_grid(K kernel, int &cached, int cu_count, int waves_per_cu, int max_tasks) {
    if (cached < 0) {
        int blocks = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, 256, 0) != hipSuccess ||
            blocks < 1)
            blocks = 2;
        cached = blocks;
    }
    int b = cached;
    if (waves_per_cu > 0) b = min(b, max(1, waves_per_cu / 4));
    // with the task count known, no more waves than tasks: every wave of the
    // grid takes at least one turn at the queue's atomic counter, so idle
    // waves lengthen a small class's kernel
    if (max_tasks > 0) return min(b * cu_count, (max_tasks + 3) / 4);
    return b * cu_count;
}

hipError_t launch_batch_wide(const BatchArgs &ba, int cu_count, int max_tasks, hipStream_t st) {
    static int blocks = -1;  // per CU, at full occupancy
    auto k = sw_batch_wide_kernel<kWideRows>;
    hipLaunchKernelGGL(k, dim3(full_grid(k, blocks, cu_count, 0, max_tasks)), dim3(256), 0, st, ba);
    return hipGetLastError();
}

template <int R, bool PK, int FORM>
static void launch_class(const BatchArgs &ba, int cu_count, int waves_per_cu, int max_tasks,
                         hipStream_t st) {
    static int blocks = -1;  // one per row class, lane width and form
    auto k = sw_batch_kernel<R, PK, FORM>;
    hipLaunchKernelGGL(k, dim3(full_grid(k, blocks, cu_count, waves_per_cu, max_tasks)), dim3(256),
                       0, st, ba);
}

template <int FORM>
static hipError_t launch_rows(const BatchArgs &ba, bool int16, int rows, int cu_count,
                              int waves_per_cu, int max_tasks, hipStream_t st) {
    if (int16) {
        switch (rows) {
#define SWIFT_L16(RR)                                                        \
    case RR:                                                                 \
        launch_class<RR, true, FORM>(ba, cu_count, waves_per_cu, max_tasks, st); \
        break;
            SWIFT_R16_CASES(SWIFT_L16)
#undef SWIFT_L16
        default: return hipErrorInvalidValue;
        }
    } else {
        switch (rows) {
#define SWIFT_L32(RR)                                                         \
    case RR:                                                                  \
        launch_class<RR, false, FORM == kLeanWide ? kLean : FORM>(ba, cu_count, waves_per_cu, max_tasks, st); \
        break;
            SWIFT_R32_CASES(SWIFT_L32)
#undef SWIFT_L32
        default: return hipErrorInvalidValue;
        }
    }
    return hipGetLastError();
}

hipError_t launch_batch(const BatchArgs &ba, bool int16, int rows, int cu_count, int waves_per_cu,
                        int max_tasks, hipStream_t st) {
    switch (ba.form) {
    case kLean: return launch_rows<kLean>(ba, int16, rows, cu_count, waves_per_cu, max_tasks, st);
    case kLeanWide:
        return launch_rows<kLeanWide>(ba, int16, rows, cu_count, waves_per_cu, max_tasks, st);
    default:
        return launch_rows<kGeneralForm>(ba, int16, rows, cu_count, waves_per_cu, max_tasks, st);
    }
}

hipError_t launch_walk(const BatchArgs &ba, const int32_t *order, const int32_t *first,
                       const int32_t *count, int max_pairs, uint32_t *moves, int move_words,
                       hipStream_t st) {
    if (max_pairs <= 0) return hipSuccess;
    if (max_pairs < kWaveWalkPairs)
        hipLaunchKernelGGL(sw_walk_wave_kernel, dim3((max_pairs + 3) / 4), dim3(256), 0, st, ba,
                           order, first, count, moves, move_words);
    else
        hipLaunchKernelGGL(sw_walk_kernel, dim3((max_pairs + 255) / 256), dim3(256), 0, st, ba,
                           order, first, count, moves, move_words);
    hipLaunchKernelGGL(sw_expand_kernel, dim3((max_pairs + 15) / 16), dim3(256), 0, st, ba,
                       order, first, count, moves, move_words);
    return hipGetLastError();
}

hipError_t launch_binning_tiny(const BinArgs &bin, const TaskArgs &ta, int32_t *order,
                               Task *tasks, int64_t *task_words, int64_t *total_words,
                               const int32_t *counters, const TinyStage &hs, hipStream_t st) {
    if (bin.npairs > kBinTinyPairs) return hipErrorInvalidValue;
    hipLaunchKernelGGL(sw_bin_tiny, dim3(1), dim3(1024), 0, st, bin, ta, order, tasks, task_words,
                       total_words, counters, hs);
    return hipGetLastError();
}

hipError_t launch_binning(const BinArgs &bin, const TaskArgs &ta, int32_t *order, Task *tasks,
                          int64_t *task_words, const int64_t *base0, int64_t *total_words,
                          int64_t *scan_sums, int max_tasks, hipStream_t st) {
    int n = bin.npairs;
    const int chunks = (n + kBinChunk - 1) / kBinChunk;
    if (n > 0) hipLaunchKernelGGL(sw_bin_classify, dim3(chunks), dim3(256), 0, st, bin);
    hipLaunchKernelGGL(sw_bin_scan, dim3(1), dim3(1024), 0, st, ta);
    if (n > 0)
        hipLaunchKernelGGL(sw_bin_scatter, dim3(chunks), dim3(256), 0, st, bin.bin_of, n,
                           ta.bin_cursor, order);
    if (max_tasks > 0) {
        hipLaunchKernelGGL(sw_build_tasks, dim3((max_tasks + 255) / 256), dim3(256), 0, st,
                           ta.seg_task0, ta.seg_first, ta.seg_len, ta.ntasks, order, bin.rlen,
                           tasks, task_words, ta.seg_steps, ta.wide);
    }
    return launch_scan<int64_t>(LoadArr<int64_t>{task_words}, StoreTaskBase{tasks}, ta.ntasks,
                                max_tasks, scan_sums, base0, total_words, nullptr, st);
}

hipError_t launch_zero(const ZeroSpans &z, hipStream_t st) {
    int most = 0;
    for (int k = 0; k < z.nspans; ++k) most = max(most, z.n[k]);
    if (most <= 0) return hipSuccess;
    const int blocks = min((most + 255) / 256, 2048);
    hipLaunchKernelGGL(zero_spans, dim3(blocks, z.nspans), dim3(256), 0, st, z);
    return hipGetLastError();
}

hipError_t launch_fill(int32_t *p, int n, int32_t v, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_i32, dim3((n + 255) / 256), dim3(256), 0, st, p, n, v);
    return hipGetLastError();
}

hipError_t launch_gather(const Gather &g, hipStream_t st) {
    hipLaunchKernelGGL(gather_words, dim3(1), dim3(256), 0, st, g);
    return hipGetLastError();
}

}  // namespace swift
