// sw_plain.hip -- the plain per-pair path (alignSequences): kernels and
// launches.  Inputs use the reference's layout: pair p's query at
// querySeq + p*(qlen+1) (all qlen bytes are rows, as in smithWaterman_cpu),
// reference at refSeq + p*(rlen+1), columns stopping at its first NUL.
//
// Four routes, by scoring and size (PlainPlan):
//  * packed: the scorings of lean_packed_scoring whose best score stays below the
//    packed limit, from kPlainPackedPairs pairs on: the screen
//    (sw_screen.hpp), then for the pairs it leaves, listed, the batched path's
//    sweep, eight a wave (sw_plain_packed_kernel), walk and expansion.
//    A pair whose reference holds a byte outside ACGTNacgtn is left to the
//    wave kernel.
//  * wave: the other calls under lean_scoring, and those pairs: one wave
//    sweeps, walks and expands a pair in one kernel (sw_plain_wave_kernel),
//    32-bit lanes on any bytes.
//  * general: any other scoring, one wave per pair in 32-bit lanes
//    (sw_plain_kernel), then walk and expansion.
#include <algorithm>

#include "sw_sweep.hpp"

namespace swift {

// ---------------------------------------------------------------------------
// The general kernel: one wave per pair sweeps, G = 64, byte semantics, 32-bit
// lanes, any scoring; walk and expansion follow in kernels of their own.  LDS
// holds the reference codes of the pair.
// ---------------------------------------------------------------------------
constexpr int kPlainPad = 64;  // LDS words before column 0 of the plain kernel's reference

template <int R>
__global__ void __launch_bounds__(64)
sw_plain_kernel(const char *__restrict__ qseq, const char *__restrict__ rseq, int qlen, int rlen_max,
                KeyConsts kc, int npairs, int pair0, uint32_t *__restrict__ trace,
                int64_t trace_words_per_pair, int4 *__restrict__ res) {
    using S = Sweep<64, R, false, kBytes>;
    extern __shared__ uint32_t lds_rr[];
    const int p = blockIdx.x;
    if (p >= npairs) return;
    const int g = threadIdx.x;
    const char *qs = qseq + (int64_t)(pair0 + p) * (qlen + 1);
    const char *rs = rseq + (int64_t)(pair0 + p) * (rlen_max + 1);

    // the column count stops at the first NUL
    int first_nul = rlen_max;
    for (int j = g; j < rlen_max; j += 64)
        if (rs[j] == 0) first_nul = min(first_nul, j);
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) first_nul = min(first_nul, __shfl_xor(first_nul, s, 64));
    const int rlen = first_nul;
    // reference codes into LDS at kPlainPad + j, zero for every column a
    // lane reaches outside [0, rlen) (j from -63 to rlen + 62), so each step
    // reads its column without a branch
    for (int x = g; x < rlen_max + 2 * kPlainPad; x += 64) {
        const int j = x - kPlainPad;
        lds_rr[x] = j >= 0 && j < rlen ? byte_rcode((unsigned char)rs[j]) : 0u;
    }
    __syncthreads();

    S sw;
    sw.init(kc);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int row = g * R + r;
        sw.q[r] = row < qlen ? byte_qcode((unsigned char)qs[row]) : 0u;
    }
    // the pair's trace through a buffer resource: 32-bit byte offsets
    // (a pair's trace is under 2^21 words)
    const __amdgpu_buffer_rsrc_t tr_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        trace + (int64_t)p * trace_words_per_pair, 0, (int)0x7FFFFFFF, 0x00020000);
    const int T = rlen + 63;
    const int main_lo = 63, main_hi = rlen;  // every lane inside [0, rlen)
    auto run = [&](auto masked, int t) {
        int j = t - g;
        uint32_t rr = lds_rr[kPlainPad + j];
        uint32_t vmask = 0;
        if constexpr (decltype(masked)::value) vmask = (j >= 0 && j < rlen) ? ~0u : 0u;
        uint32_t a1[S::W];
#pragma unroll
        for (int w = 0; w < S::W; ++w) a1[w] = 0;
        sw.template step<decltype(masked)::value>(rr, j, vmask, 0u, a1);
        // byte offset of word (t >> 2, w, g, t & 3) of the granule layout
        // (trace_word: 64 lanes x 4 steps = 1 KB per step group and word)
        const uint32_t o = (uint32_t)(t >> 2) * (S::W * 1024u) + (uint32_t)g * 16u +
                           (uint32_t)(t & 3) * 4u;
#pragma unroll
        for (int w = 0; w < S::W; ++w)
            __builtin_amdgcn_raw_buffer_store_b32(a1[w], tr_rsrc, o + (uint32_t)w * 1024u, 0, 0);
    };
    sweep_steps(T, min(main_lo, T), main_hi, run);

    // lane best over its valid rows: row-major first maximum
    uint32_t bh = 0, brow = 0, bcol = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int row = g * R + r;
        uint32_t h = sw.best[r] >> kColBits;
        if (row < qlen && h > bh) {
            bh = h;
            brow = row + 1;
            bcol = kMaxCols - (sw.best[r] & kMaxCols) + 1;
        }
    }
    const GroupResult gr = group_best<64>(bh, brow, bcol, R, false, 0, 0);
    // the walk runs in sw_plain_walk_kernel, one lane per pair
    if (g == 0) res[p] = make_int4(gr.score, gr.row, gr.col, rlen);
}

// The i-th pair of a kernel's work: of n in a row, or of a list (null: none).
struct PlainPairs {
    const int32_t *list, *count;
    int n;
    __device__ __forceinline__ int size() const { return list ? uni(*count) : n; }
    __device__ __forceinline__ int at(int i) const { return list ? list[i] : i; }
};

// Where a pair's trace lies: ppt pairs share a task's area of wpt words (8
// packed pairs, two per 16-lane group; or one pair).
struct PlainTrace {
    const uint32_t *trace;
    int64_t wpt;
    int ppt, R, W;
    __device__ __forceinline__ PairTrace of(int p) const {
        if (ppt == 1) return PairTrace{(int64_t)p * wpt, 0, (int16_t)R, (int8_t)W, 0};
        const int s = p & 7;
        return PairTrace{(int64_t)(p >> 3) * wpt, (s >> 1) * kBatchG, (int16_t)R, (int8_t)W,
                         (int8_t)((s & 1) | 2)};
    }
};

// After a sweep kernel: one lane per pair walks the pair's trace from its
// best cell (res: score, row, col, columns; columns < 0: left to the wave
// kernel) and stores the path as 2-bit moves plus the drop-in's score, start,
// end and length.
__global__ void __launch_bounds__(256) sw_plain_walk_kernel(PlainTrace tr, int qlen,
                                                            PlainPairs pairs, int pair0, const int4 *res,
                                                            uint32_t *moves, int move_words,
                                                            PlainOut out) {
    const int p = blockIdx.x * 256 + (int)threadIdx.x;
    if (p >= pairs.size()) return;
    const int4 r = res[p];
    if (r.w < 0) return;
    uint32_t *mv = moves + (int64_t)p * move_words;
    uint32_t word = 0;
    auto emit = [&](int k, int op, int, int) {
        word |= (uint32_t)op << (2 * (k & 15));
        if ((k & 15) == 15) {
            mv[k >> 4] = word;
            word = 0;
        }
    };
    WalkOut wo = walk_cells<TraceReaderLean>(tr.trace, r.x, r.y, r.z, tr.of(p), qlen, r.w, emit);
    if (wo.len & 15) mv[wo.len >> 4] = word;
    const int gp = pair0 + pairs.at(p);
    out.score[gp] = (float)r.x;
    out.start[gp] = wo.start;
    out.end[gp] = wo.end;
    out.alen[gp] = wo.len;
}

// sw_plain_walk_kernel's work, one wave per pair (small calls); NMV: move
// words per lane (a path's moves fit NMV * 64 words)
template <int NMV>
__global__ void __launch_bounds__(256)
sw_plain_walk_wave_kernel(PlainTrace tr, int qlen, PlainPairs pairs, int pair0,
                          const int4 *res, uint32_t *moves, int move_words, PlainOut out) {
    const int p = uni((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    if (p >= pairs.size()) return;
    const int4 r = res[p];
    const int score = uni(r.x);
    if (uni(r.w) < 0) return;
    const PairTrace pt = tr.of(p);
    RegMoves<NMV> mv(moves + (int64_t)p * move_words);
    WalkOut wo = walk_wave(reinterpret_cast<const uint4 *>(tr.trace) + pt.base / 4 + pt.lane0,
                           tr.R, tr.W, (pt.half & 2) ? 3 : 4, (pt.half & 1) * 16, score, uni(r.y),
                           uni(r.z), qlen, uni(r.w), mv);
    if ((threadIdx.x & 63) == 0) {
        const int gp = pair0 + pairs.at(p);
        out.score[gp] = (float)score;
        out.start[gp] = wo.start;
        out.end[gp] = wo.end;
        out.alen[gp] = wo.len;
    }
}

// The expansion of pair gp's moves `mv`, from its best cell (row, col).
__device__ __forceinline__ ExpandPair plain_expand(const char *qseq, const char *rseq, int qlen,
                                                   int rlen_max, int gp, int len, int row, int col,
                                                   int rlen, const uint32_t *mv,
                                                   const PlainOut &out) {
    ExpandPair e;
    e.live = true;
    e.len = len;
    e.row = row;
    e.col = col;
    e.nq = min(qlen, row);
    e.nr = min(rlen, col);
    e.qsrc = (const unsigned char *)qseq + (int64_t)gp * (qlen + 1);
    e.rsrc = (const unsigned char *)rseq + (int64_t)gp * (rlen_max + 1);
    e.qc = out.qcons + (int64_t)gp * out.cstride;
    e.rc = out.rcons + (int64_t)gp * out.cstride;
    e.mv = mv;
    return e;
}

// The consensus strings from the walks' moves, four pairs per one-wave
// workgroup (dynamic LDS: 4 x (qw + rw) dwords).
__global__ void __launch_bounds__(64) sw_plain_expand_kernel(const char *qseq, const char *rseq,
                                                             int qlen, int rlen_max,
                                                             PlainPairs pairs, int pair0,
                                                             const int4 *res,
                                                             const uint32_t *moves,
                                                             int move_words, int qw, int rw,
                                                             PlainOut out) {
    extern __shared__ uint32_t lds_x[];
    const int slot = threadIdx.x >> 4, sl = threadIdx.x & 15;
    const int p = blockIdx.x * 4 + slot;
    const int npairs = pairs.size();
    if ((int)blockIdx.x * 4 >= npairs) return;
    ExpandPair e;
    if (p < npairs) {
        const int4 r = res[p];
        const int gp = pair0 + pairs.at(p);
        if (r.w >= 0)
            e = plain_expand(qseq, rseq, qlen, rlen_max, gp, out.alen[gp], r.y, r.z, r.w,
                             moves + (int64_t)p * move_words, out);
    }
    expand_row<16>(e, lds_x + slot * (qw + rw), lds_x + slot * (qw + rw) + qw, sl);
}

// columns of a reference at rs[0, rlen_max): up to its first NUL; lane g of G
// lanes looks at every G-th byte
template <int G>
__device__ __forceinline__ int ref_columns(const char *rs, int rlen_max, int g) {
    constexpr int NB = 8;  // loads in flight
    int first = rlen_max;
    for (int j0 = g; j0 < rlen_max; j0 += NB * G) {
        char c[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) c[i] = rs[min(j0 + i * G, rlen_max - 1)];
#pragma unroll
        for (int i = 0; i < NB; ++i)
            if (c[i] == 0) first = min(first, min(j0 + i * G, rlen_max - 1));
    }
#pragma unroll
    for (int s = G / 2; s >= 1; s >>= 1) first = min(first, __shfl_xor(first, s, G));
    return first;
}

// The packed sweep: eight pairs a wave, two per 16-lane group, R = ceil(qlen /
// 16) rows a lane.  Against one wave per pair in 32-bit lanes (64 columns of
// ramp instead of 16, one cell a lane and instruction instead of two):
// 100,000 pairs of 100 x 300 3.37 -> 0.93 ms, and 0.32 where the screen takes
// four in five.  Dynamic LDS: plain_packed_lds().
constexpr int kPackedTail = kBatchG + 2;  // padding columns after the last
__host__ __device__ constexpr int plain_packed_stride(int rlen_max) { return rlen_max + kPackedTail; }
static int plain_packed_lds(int rlen_max) {
    return 4 * (kBatchG + 4 * plain_packed_stride(rlen_max) + 4);
}

template <int R, int FORM>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(R <= 6 ? 5 : R <= 12 ? 4 : 3)))
sw_plain_packed_kernel(const char *__restrict__ qseq, const char *__restrict__ rseq, int qlen,
                       int rlen_max, KeyConsts kc, PlainPairs pairs, int pair0,
                       uint32_t *__restrict__ trace, int64_t wpt, int4 *__restrict__ res) {
    using S = Lean<kBatchG, R, true, FORM>;
    constexpr int G = kBatchG;
    extern __shared__ uint32_t lds_p[];
    const int lane = threadIdx.x, grp = lane / G, g = lane % G;
    uint32_t *col = lds_p + G + grp * plain_packed_stride(rlen_max);
    const int npairs = pairs.size();
    if ((int)blockIdx.x * kSlots16 >= npairs) return;
    const int p0 = (int)blockIdx.x * kSlots16 + grp * 2;
    S sw;
    sw.init(kc);
    int rl[2];
    const char *rs[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        // a slot past the last pair reads that pair and is cleared
        const int64_t gp = pair0 + pairs.at(min(p0 + h, npairs - 1));
        const char *qs = qseq + gp * (qlen + 1);
        rs[h] = rseq + gp * (rlen_max + 1);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int row = g * R + r;
            const uint32_t c = row < qlen ? (unsigned char)qs[row] : 0u;
            const uint32_t tb = lean_table(c, row >= qlen, (uint32_t)kc.ppm);
            if (h) sw.q2[r] = tb;
            else sw.q[r] = tb;
        }
        rl[h] = rlen_max > 0 ? ref_columns<G>(rs[h], rlen_max, g) : 0;
        if (p0 + h >= npairs) rl[h] = 0;
    }
    int ncols = max(rl[0], rl[1]);  // of the wave's pairs
#pragma unroll
    for (int s = 32; s >= G; s >>= 1) ncols = max(ncols, __shfl_xor(ncols, s, 64));
    ncols = uni(ncols);
    const uint32_t pad = lean_selector(kRefPad, 0) | lean_selector(kRefPad, 1) << 16;
    uint32_t exotic = 0;
    for (int j = g; j < rlen_max + kPackedTail; j += G) {
        uint32_t v = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t cls = kRefPad;
            if (j < rl[h]) {
                cls = ref_index_bf((unsigned char)rs[h][j]);
                if (cls == kRefOther) exotic |= 1u << h;
            }
            v |= lean_selector(cls, h) << (16 * h);
        }
        col[j] = v;
    }
    if (grp == 0) col[g - G] = pad;  // before column 0 of the first group
#pragma unroll
    for (int s = G / 2; s >= 1; s >>= 1) exotic |= __shfl_xor(exotic, s, G);
    wave_lds_sync();
    lean_sweep<S, true>(sw, col - g, ncols + G - 1, trace + (int64_t)blockIdx.x * wpt);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t bh;
        int row, t;
        sw.result(h, bh, row, t);
        const GroupResult gr = group_best<G>(bh, (uint32_t)(g * R + row + 1),
                                             (uint32_t)(t - g + 1), R, false, 0, 0);
        if (g == 0 && p0 + h < npairs)
            res[p0 + h] = make_int4(gr.score, gr.row, gr.col, (exotic >> h) & 1 ? -1 : rl[h]);
    }
}

// One wave takes a pair from its bytes to its strings: the sweep in 32-bit
// lanes (dual-rail bytes, so any byte compares as the reference's), the walk
// over its own trace area, the moves in LDS, the expansion.  For small calls,
// where every launch and every kernel's tail counts, and for calls whose
// scores pass the packed lanes' range.  Each wave takes pairs in turn; with
// `flagged` (res of a packed sweep over `pairs`) only those that sweep left,
// `per` at a time.  256 pairs of 143 x 253 81 -> 45 us.  Dynamic LDS: plain_wave_lds().
static int plain_wave_lds(int qlen, int rlen_max, int move_words) {
    return 4 * (std::max(rlen_max + 2 * kPlainPad + 8, (qlen + 6) / 4 + (rlen_max + 6) / 4) +
                move_words);
}

template <int R>
__global__ void __launch_bounds__(64)
sw_plain_wave_kernel(const char *__restrict__ qseq, const char *__restrict__ rseq, int qlen,
                     int rlen_max, KeyConsts kc, PlainPairs pairs, int pair0, uint32_t *trace,
                     int64_t wpp, const int4 *flagged, int per, int move_words, PlainOut out) {
    using S = Lean<64, R, false>;
    extern __shared__ uint32_t lds_w[];
    const int g = threadIdx.x;
    uint32_t *mvs = lds_w, *col = lds_w + move_words;  // the columns, then the expansion's bases
    uint32_t *tr = trace + (int64_t)blockIdx.x * wpp;
    const int npairs = pairs.size();
    auto pair = [&](int p) {
        const int gp = pair0 + p;
        const char *qs = qseq + (int64_t)gp * (qlen + 1);
        const char *rs = rseq + (int64_t)gp * (rlen_max + 1);
        S sw;
        sw.init(kc);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int row = g * R + r;
            sw.q[r] = rail_query(row < qlen ? (unsigned char)qs[row] : 0u, row >= qlen);
        }
        const int rlen = rlen_max > 0 ? uni(ref_columns<64>(rs, rlen_max, g)) : 0;
        const int n = rlen + 2 * kPlainPad + 8;
        for (int x = g; x < n; x += 64) {
            const int j = x - kPlainPad;
            const bool pad = j < 0 || j >= rlen;
            col[x] = rail_ref(pad ? 0u : (unsigned char)rs[j], pad);
        }
        wave_lds_sync();
        lean_sweep<S, false>(sw, col + kPlainPad - g, rlen + 63, tr);
        uint32_t bh;
        int row, t;
        sw.result(0, bh, row, t);
        const GroupResult gr =
            group_best<64>(bh, (uint32_t)(g * R + row + 1), (uint32_t)(t - g + 1), R, false, 0, 0);
        const int score = uni(gr.score), brow = uni(gr.row), bcol = uni(gr.col);
        wave_store_fence();
        LdsMoves mv{mvs};
        const WalkOut wo = walk_wave(reinterpret_cast<const uint4 *>(tr), R, S::W, 4, 0, score,
                                     brow, bcol, qlen, rlen, mv);
        if (g == 0) {
            out.score[gp] = (float)score;
            out.start[gp] = wo.start;
            out.end[gp] = wo.end;
            out.alen[gp] = wo.len;
        }
        expand_row<64>(plain_expand(qseq, rseq, qlen, rlen_max, gp, wo.len, brow, bcol, rlen, mvs,
                                    out),
                       col, col + (qlen + 6) / 4, g);
    };
    if (!flagged) {
        for (int p = blockIdx.x; p < npairs; p += gridDim.x) pair(p);
        return;
    }
    for (int p0 = (int)blockIdx.x * per; p0 < npairs; p0 += (int)gridDim.x * per) {
        const int p = p0 + g;
        uint64_t left = __ballot(g < per && p < npairs && flagged[min(p, npairs - 1)].w < 0);
        while (left) {
            pair(uni(pairs.at(p0 + (int)__builtin_ctzll(left))));
            left &= left - 1;
        }
    }
}

// ---------------------------------------------------------------------------
// Plans and launches
// ---------------------------------------------------------------------------
int plain_rows_for(int qlen) {
    int R = (qlen + 63) / 64;
    if (R < 1) R = 1;
    if (R <= 8) return R;
    if (R <= 10) return 10;
    if (R <= 12) return 12;
    if (R <= 16) return 16;
    return -1;
}

// trace words of a pair swept by a whole wave: whole 4-step granules of
// (rlen + 63) steps, one word a lane and step (R <= 16)
static int64_t wave_trace_words(int rlen) { return (int64_t)((rlen + 63 + 3) & ~3) * 64; }
// ... of eight packed pairs
static int64_t packed_trace_words(int R, int rlen) {
    return (int64_t)((rlen + kBatchG - 1 + 3) & ~3) * ((R + 7) / 8) * 64;
}

// Waves of the wave kernel (each keeps a trace area): four to a SIMD
constexpr int kPlainWaves = 4096;
// Calls of at least this many pairs take the packed route, whose sixteen-lane
// groups need eight times the pairs to fill the chip.  Packed (without the
// screen) against wave route, us: 100 x 300 bases, 2,048 pairs 90 against 61,
// 4,096 94 against 104, 8,192 98 against 208; 250 x 450, 231 against 133, 238
// against 237, 256 against 462.  Past 16 rows a lane (three trace words a step)
// the chunks have to be as large: in a small scratch one is a task a wave on a
// part of the chip, and lasts as long as that task.  With the screen, in 64 MiB,
// 4,200 related (unrelated) pairs: 320 x 480, chunks of 1,048, 1,467 against 825
// (1,495; 838); 300 x 200, 2,432, 308 against 256 (315; 254).  Of fewer rows the
// packed route comes out even or ahead: 250 x 450, 1,664, 699 against 680 (725;
// 672); 150 x 450, 1,664, 477 against 547 (497; 548); 120 x 1000, 1,528, 793
// against 1,564 (802; 1,549).
constexpr int kPlainPackedPairs = 4096;
// Calls under this many pairs walk a wave a pair, others a lane.  The packed
// route's line against the general one's, us, related pairs, of which most are
// the screen's (pairs that are all left to the sweep): 40,000 of 100 x 300 242
// -> 202 (433 -> 396), of 250 x 400 747 -> 628 (1,041 -> 970), 100,000 of 100 x
// 300 353 -> 322 (898, 905), 130,000 447 -> 404 (1,089, 1,110).
constexpr int kPackedWalkPairs = 131072;
constexpr int kGeneralWalkPairs = 16384;
// longest references of the packed route (four groups' columns in LDS)
constexpr int kPlainPackedCols = 1024;

PlainPlan plain_plan(const Scoring &sc, int qlen, int rlen, int npairs, int64_t budget) {
    PlainPlan pl{};
    pl.qlen = qlen;
    pl.rlen = rlen;
    pl.move_words = (qlen + rlen) / 16 + 1;  // a path has at most qlen + rlen moves
    pl.wave_rows = plain_rows_for(qlen);
    pl.wave_words = wave_trace_words(rlen);
    if (!lean_scoring(sc)) {
        pl.route = PlainPlan::kGeneral;
        return pl;
    }
    const bool packed = npairs >= kPlainPackedPairs && qlen <= kMaxBatchQ &&
                        rlen <= kPlainPackedCols &&
                        packed_form(sc, qlen) != kGeneralForm;
    pl.form = packed_form(sc, qlen);
    pl.route = packed ? PlainPlan::kPacked : PlainPlan::kWave;
    pl.packed_rows = std::max(1, (qlen + kBatchG - 1) / kBatchG);
    pl.task_words = packed_trace_words(pl.packed_rows, rlen);
    int chunk, waves;
    plain_chunk(pl, npairs, budget, &chunk, &waves);
    if (packed && pl.packed_rows > 16 && chunk < kPlainPackedPairs) pl.route = PlainPlan::kWave;
    return pl;
}

// waves of the wave kernel over n pairs with room for `words` of trace
static int plain_waves(const PlainPlan &pl, int n, int64_t words) {
    return (int)std::max<int64_t>(
        1, std::min<int64_t>(std::min(n, kPlainWaves), words / pl.wave_words));
}

// Scratch of a chunk of n pairs: general [n traces][n best cells][n moves];
// packed [tasks' traces][n best cells][n moves][waves' traces][the list's
// count, the list]; wave [waves'
// traces].  Every part is a multiple of 4 words, so the best cells are 16-byte
// aligned.
int64_t plain_words(const PlainPlan &pl, int n, int waves) {
    const int64_t cells = (int64_t)n * 4 + (((int64_t)n * pl.move_words + 3) & ~(int64_t)3);
    switch (pl.route) {
    case PlainPlan::kGeneral: return (int64_t)n * pl.wave_words + cells;
    case PlainPlan::kPacked:
        return (int64_t)((n + kSlots16 - 1) / kSlots16) * pl.task_words + cells +
               (int64_t)waves * pl.wave_words + 4 + ((n + 3) & ~3);
    default: return (int64_t)waves * pl.wave_words;
    }
}

// The largest chunk of at most npairs pairs whose scratch fits `budget` words
// (at least one pair), and its waves.
void plain_chunk(const PlainPlan &pl, int npairs, int64_t budget, int *chunk, int *waves) {
    // a quarter of the scratch at most for the waves of a packed chunk's
    // left-over pairs
    *waves = plain_waves(pl, npairs, pl.route == PlainPlan::kWave ? budget : budget / 4);
    *chunk = npairs;
    if (pl.route == PlainPlan::kWave) return;
    const int64_t left = budget - (pl.route == PlainPlan::kPacked ? *waves * pl.wave_words : 0);
    const int64_t per8 = plain_words(pl, kSlots16, 0);
    *chunk = (int)std::max<int64_t>(1, std::min<int64_t>(npairs, left / per8 * kSlots16));
}

template <int R>
static void launch_general(const char *q, const char *r, const PlainPlan &pl, const KeyConsts &kc,
                           int n, int pair0, uint32_t *trace, int4 *res, hipStream_t st) {
    const size_t lds = sizeof(uint32_t) * (size_t)(pl.rlen + 2 * kPlainPad);
    hipLaunchKernelGGL(sw_plain_kernel<R>, dim3(n), dim3(64), lds, st, q, r, pl.qlen, pl.rlen, kc,
                       n, pair0, trace, pl.wave_words, res);
}

template <int R>
static void launch_wave(const char *q, const char *r, const PlainPlan &pl, const KeyConsts &kc,
                        PlainPairs pairs, int pair0, uint32_t *trace, int waves,
                        const int4 *flagged, const PlainOut &out, hipStream_t st) {
    const int n = pairs.n;
    const int per = flagged ? std::min(64, (n + waves - 1) / waves) : 1;
    hipLaunchKernelGGL(sw_plain_wave_kernel<R>, dim3(std::min(waves, (n + per - 1) / per)),
                       dim3(64), plain_wave_lds(pl.qlen, pl.rlen, pl.move_words), st, q, r,
                       pl.qlen, pl.rlen, kc, pairs, pair0, trace, pl.wave_words, flagged, per,
                       pl.move_words, out);
}

template <int R, int FORM>
static void launch_packed_as(const char *q, const char *r, const PlainPlan &pl, const KeyConsts &kc,
                          PlainPairs pairs, int pair0, uint32_t *trace, int4 *res, hipStream_t st) {
    auto k = sw_plain_packed_kernel<R, FORM>;
    hipLaunchKernelGGL(k, dim3((pairs.n + kSlots16 - 1) / kSlots16), dim3(64),
                       plain_packed_lds(pl.rlen), st, q, r, pl.qlen, pl.rlen, kc, pairs, pair0, trace, pl.task_words, res);
}
template <int R>
static void launch_packed(const char *q, const char *r, const PlainPlan &pl, const KeyConsts &kc,
                          PlainPairs pairs, int pair0, uint32_t *trace, int4 *res,
                          hipStream_t st) {
    if (pl.form == kLean) launch_packed_as<R, kLean>(q, r, pl, kc, pairs, pair0, trace, res, st);
    else launch_packed_as<R, kLeanWide>(q, r, pl, kc, pairs, pair0, trace, res, st);
}

#define SWIFT_PLAIN_ROWS(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(10) X(12) X(16)
#define SWIFT_PACKED_ROWS(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) \
    X(13) X(14) X(15) X(16) X(17) X(18) X(19) X(20)

hipError_t launch_plain(const PlainPlan &pl, const char *q, const char *r, const Scoring &sc,
                        int n, int pair0, uint32_t *scratch, int waves, const PlainOut &out,
                        hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const KeyConsts kc = make_consts(sc, kBytes);
    PlainPairs pairs{nullptr, nullptr, n};
    auto wave = [&](uint32_t *trace, const int4 *flagged) -> bool {
        switch (pl.wave_rows) {
#define SWIFT_W(RR) \
    case RR: launch_wave<RR>(q, r, pl, kc, pairs, pair0, trace, waves, flagged, out, st); return true;
            SWIFT_PLAIN_ROWS(SWIFT_W)
#undef SWIFT_W
        default: return false;
        }
    };
    if (pl.route == PlainPlan::kWave)
        return wave(scratch, nullptr) ? hipGetLastError() : hipErrorInvalidValue;
    const bool packed = pl.route == PlainPlan::kPacked;
    const int64_t tw = packed ? (int64_t)((n + kSlots16 - 1) / kSlots16) * pl.task_words
                              : (int64_t)n * pl.wave_words;
    int4 *res = reinterpret_cast<int4 *>(scratch + tw);
    uint32_t *moves = scratch + tw + (int64_t)n * 4;
    PlainTrace tr{scratch, pl.wave_words, 1, pl.wave_rows, 1};
    uint32_t *area = moves + (((int64_t)n * pl.move_words + 3) & ~(int64_t)3);
    if (packed) {
        int32_t *count = reinterpret_cast<int32_t *>(area + waves * pl.wave_words);
        pairs.list = count + 4;
        pairs.count = count;
        ZeroSpans z{};
        z.p[0] = count;
        z.n[0] = 1;
        z.nspans = 1;
        hipError_t e = launch_zero(z, st);
        if (e == hipSuccess)
            e = launch_screen_plain(q, r, sc, pl.qlen, pl.rlen, n, pair0, out, count + 4, count,
                                    st);
        if (e != hipSuccess) return e;
        tr = PlainTrace{scratch, pl.task_words, kSlots16, pl.packed_rows, (pl.packed_rows + 7) / 8};
        switch (pl.packed_rows) {
#define SWIFT_P(RR) \
    case RR: launch_packed<RR>(q, r, pl, kc, pairs, pair0, scratch, res, st); break;
            SWIFT_PACKED_ROWS(SWIFT_P)
#undef SWIFT_P
        default: return hipErrorInvalidValue;
        }
    } else {
        switch (pl.wave_rows) {
#define SWIFT_G(RR) \
    case RR: launch_general<RR>(q, r, pl, kc, n, pair0, scratch, res, st); break;
            SWIFT_PLAIN_ROWS(SWIFT_G)
#undef SWIFT_G
        default: return hipErrorInvalidValue;
        }
    }
    const int mw = pl.move_words, nmv = (mw + 63) / 64;
    if (n < (packed ? kPackedWalkPairs : kGeneralWalkPairs) && nmv <= 5) {
        auto k = nmv <= 1 ? sw_plain_walk_wave_kernel<1>
                 : nmv == 2 ? sw_plain_walk_wave_kernel<2>
                 : nmv == 3 ? sw_plain_walk_wave_kernel<3>
                 : nmv == 4 ? sw_plain_walk_wave_kernel<4>
                            : sw_plain_walk_wave_kernel<5>;
        hipLaunchKernelGGL(k, dim3((n + 3) / 4), dim3(256), 0, st, tr, pl.qlen, pairs,
                           pair0, res, moves, mw, out);
    } else {
        hipLaunchKernelGGL(sw_plain_walk_kernel, dim3((n + 255) / 256), dim3(256), 0, st, tr,
                           pl.qlen, pairs, pair0, res, moves, mw, out);
    }
    const int qw = (pl.qlen + 6) / 4, rw = (pl.rlen + 6) / 4;
    hipLaunchKernelGGL(sw_plain_expand_kernel, dim3((n + 3) / 4), dim3(64),
                       sizeof(uint32_t) * 4 * (size_t)(qw + rw), st, q, r, pl.qlen, pl.rlen, pairs,
                       pair0, res, moves, mw, qw, rw, out);
    if (packed && !wave(area, res)) return hipErrorInvalidValue;  // the pairs the packed sweep left
    return hipGetLastError();
}

}  // namespace swift
