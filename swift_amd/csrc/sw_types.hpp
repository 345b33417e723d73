// sw_types.hpp -- kernel argument structures and layout constants shared by
// sw_kernels.hip and the host code.
#pragma once

#include "swift_common.hpp"

namespace swift {

// per-launch constants in key space (key = 4*H + direction)
struct KeyConsts {
    int dr;    // added to 4H to form the diagonal-ready value
    int dsub;  // added when the substitution flag is set
    int eo2;   // 4*gapOpen + 2 (up exit, open)
    int eo1;   // 4*gapOpen + 1 (left exit, open)
    int de;    // 4*(gapExt - gapOpen)
    // 15, passed at run time: an arithmetic shift by it leaves the optimiser
    // no sign-splat to turn a masked merge of packed halves into per-half
    // compares and selects
    int sign;
    // lean sweeps (see Lean): the diagonal-ready value of H = 0, u*match + 3, the
    // mismatch penalty u*(match - mismatch), and the exits' penalties, one byte
    // each; u = 4 in 32-bit lanes, by the cell's direction code, and 8 in packed
    // ones (p...), by 3 less the code
    int x, pm;
    uint32_t tab_u, tab_l;
    int px, ppm;
    uint32_t ptab_u, ptab_l;
};

// ONEHOT: flag = match,    dr = 4*mismatch + 3, dsub = 4*(match - mismatch)
// BYTES : flag = mismatch, dr = 4*match + 3,    dsub = 4*(mismatch - match)
enum Policy { kOneHot = 0, kBytes = 1 };

inline KeyConsts make_consts(const Scoring &s, int policy) {
    KeyConsts k;
    if (policy == kOneHot) {
        k.dr = 4 * s.mismatch + 3;
        k.dsub = 4 * (s.match - s.mismatch);
    } else {
        k.dr = 4 * s.match + 3;
        k.dsub = 4 * (s.mismatch - s.match);
    }
    k.eo2 = 4 * s.gap_open + 2;
    k.eo1 = 4 * s.gap_open + 1;
    k.de = 4 * (s.gap_ext - s.gap_open);
    k.sign = 15;
    k.x = 4 * s.match + 3;
    k.pm = 4 * (s.match - s.mismatch);
    // exit = key - penalty: 4*(H + gap) + 2 (up) or + 1 (left) from 4*H + d;
    // d = 0 (a start, key 0) saturates whatever is subtracted
    k.tab_u = k.tab_l = k.ptab_u = k.ptab_l = 0;
    for (int d = 1; d <= 3; ++d) {
        const int up = d == 2 ? s.gap_ext : s.gap_open, left = d == 1 ? s.gap_ext : s.gap_open;
        k.tab_u |= (uint32_t)((d - 2 - 4 * up) & 0xFF) << (8 * d);
        k.tab_l |= (uint32_t)((d - 1 - 4 * left) & 0xFF) << (8 * d);
        k.ptab_u |= (uint32_t)((d - 2 - 8 * up) & 0xFF) << (8 * (3 - d));
        k.ptab_l |= (uint32_t)((d - 1 - 8 * left) & 0xFF) << (8 * (3 - d));
    }
    k.px = 8 * s.match + 3;
    k.ppm = 8 * (s.match - s.mismatch);
    return k;
}

// Scorings of the lean sweeps: mismatch and gap moves all lose score (their
// steps run unmasked), the exits' penalties fit a byte, and the mismatch
// penalty 7 bits (bit 7 of a match table marks padding rows).
inline bool lean_scoring(const Scoring &s) {
    return s.match >= 1 && s.mismatch < 0 && s.match - s.mismatch <= 31 && s.gap_open <= -1 &&
           s.gap_open >= -63 && s.gap_ext <= -1 && s.gap_ext >= -63;
}
// ... of the packed ones, whose keys are 8*H + code
inline bool lean_packed_scoring(const Scoring &s) {
    return lean_scoring(s) && s.match - s.mismatch <= 15 && s.gap_open >= -31 && s.gap_ext >= -31;
}
// Forms of a sweep.  The packed lean ones keep best-cell keys 32*H + 32*match +
// row code in 16 bits: kLean takes their maxima three at a time as
// half-precision numbers (keys below the infinity's bit pattern, 0x7C00: H +
// match <= 990), kLeanWide two at a time as unsigned ones (below 65536: H +
// match <= 2046).  A pair whose best reaches the form's limit is flagged: H
// rises by at most match (<= 30) a cell, so a pair with any larger cell has one
// between the limit and the exact range's end.
enum SweepForm { kGeneralForm = 0, kLean = 1, kLeanWide = 2 };
inline int lean_limit(int form, int match) { return (form == kLean ? 960 : 2016) - match; }
// the packed form for queries of at most maxq bases (larger scores would be
// re-run in 32-bit lanes)
inline SweepForm packed_form(const Scoring &s, int maxq) {
    if (!lean_packed_scoring(s)) return kGeneralForm;
    const int64_t most = (int64_t)maxq * s.match;
    return most < lean_limit(kLean, s.match) ? kLean
           : most < lean_limit(kLeanWide, s.match) ? kLeanWide : kGeneralForm;
}

constexpr int kColBits = 12;                   // int32 best key: H << 12 | (4095 - j)
constexpr int kMaxCols = (1 << kColBits) - 1;  // longest reference window (plain kernel)
constexpr int kMaxScore32 = 1 << 19;           // scores must stay below this
constexpr int kBatchG = 16;                    // lanes per pair group (batched kernels)
constexpr int kBatchCols = 480;                // reference columns per group (LDS)
constexpr int kRBins = 20;                     // R = 1..20 rows per lane (query <= 320)
constexpr int kLenBins = kBatchCols / 8;       // bins of 8 reference columns
constexpr int kNumBins = 2 * kRBins * kLenBins;
constexpr int kMaxBatchQ = kBatchG * kRBins;   // 320
constexpr int kMaxBatchR = kBatchCols;         // 480
constexpr int kSlots16 = 8;                    // pairs per wave task, int16 packed
constexpr int kSlots32 = 4;                    // pairs per wave task, int32
// wide form (small batches): one 64-lane group per wave, packed int16
constexpr int kWideG = 64;
constexpr int kWideRows = kMaxBatchQ / kWideG;  // 5
constexpr int kSlotsWide = 2;

__host__ __device__ inline int r32_class(int r) { return r <= 2 ? 2 : (r + 1) & ~1; }

struct Task {
    int64_t trace_base;  // word offset
    int32_t first;       // index of the task's first pair in the sorted order
    int16_t npairs;      // pairs in the task (<= slots per wave)
    int16_t rows;        // R
    int32_t steps;       // max rlen + G - 1
    int32_t min_rlen;    // smallest rlen among the task's pairs
};

struct BatchArgs {
    const char *qseq;
    const int64_t *qoff;
    const int32_t *qlen;
    const char *rseq;
    const int64_t *roff;
    const int32_t *rlen;
    const int32_t *order;     // sorted pair order
    const Task *tasks;
    const int32_t *task_lo;   // device: first task of this kernel's class
    const int32_t *task_hi;   // device: one past its last task
    int32_t *next_task;       // work-queue cursor (zeroed before launch)
    uint32_t *trace;
    PairResult *res;
    PairTrace *ptr;
    KeyConsts kc;
    uint32_t h_limit;         // 4*H at or above this flags an int16 overflow risk
    // traceback outputs, written by the fused walk
    int32_t *score_out, *start_out, *end_out, *alen_out;
    char *qcons, *rcons;
    const int64_t *coff;
    int form;                 // SweepForm
    int walk_deferred;        // 1: record PairTrace descriptors, walk in sw_walk_kernel
    int32_t *nflagged;        // counts the pairs flagged for the int32 re-run
};

// One-launch form of a small batched call (sw_small.hip).  flags: mapped host
// words, cleared by the host where it reads them.
enum SmallFlag { kSmallError = 0, kSmallLonger = 1, kSmallRerun = 2, kSmallMany = 3, kSmallFlags = 4 };
struct SmallArgs {
    const char *qseq;
    const int64_t *qoff;
    const int32_t *qlen;
    const char *rseq;
    const int64_t *roff;
    const int32_t *rlen;
    const int32_t *list, *nlist;  // or null: the pairs to take (of npairs at most)
    int most;                 // with more than that on the list, none is taken
    int npairs, ppw, wpb;     // pairs, pairs a wave (1 or 2), waves a workgroup (<= 4)
    int maxq, maxr;
    int form;                 // kLean or kLeanWide
    KeyConsts kc;
    uint32_t h_limit;         // 4*H at or above this: swept again in 32-bit lanes
    uint32_t *trace;          // wave_words for each wave of the grid
    int64_t wave_words;
    int32_t *score_out, *start_out, *end_out, *alen_out;
    char *qcons, *rcons;
    const int64_t *coff;
    int32_t *flags;
    int32_t *reruns;          // device: pairs swept again, counted on from call to call
};
int64_t small_wave_words(int maxr);
hipError_t launch_small(const SmallArgs &a, int blocks, hipStream_t st);

// The screen ahead of the batched path's binning (sw_screen.hip).  A pair it
// answers has kScreenedFlag in its result's flags.
constexpr int32_t kScreenedFlag = 2;
struct ScreenArgs {
    const char *qseq;
    const int64_t *qoff;
    const int32_t *qlen;
    const char *rseq;
    const int64_t *roff;
    const int32_t *rlen;
    int npairs, per;          // pairs; pairs a wave (set by the launch)
    int32_t *score_out, *start_out, *end_out, *alen_out;
    char *qcons, *rcons;
    const int64_t *coff;
    PairResult *res;          // or null
    int32_t *list, *count;    // or null: the pairs left, counted on from *count
};
hipError_t launch_screen(const ScreenArgs &a, const Scoring &s, hipStream_t st);

// outputs of the plain (alignSequences) kernel: reference layout
struct PlainOut {
    float *score;
    int32_t *start, *end, *alen;
    char *qcons, *rcons;
    int64_t cstride;
};
// list: the pairs (from 0) the screen leaves, counted on from *count
hipError_t launch_screen_plain(const char *q, const char *r, const Scoring &s, int qlen, int rlen,
                               int n, int pair0, const PlainOut &out, int32_t *list,
                               int32_t *count, hipStream_t st);


struct BinArgs {
    const char *rseq;
    const int64_t *roff;
    const int32_t *qlen;
    const int32_t *rlen;
    const PairResult *prev;   // rerun pass: only flagged pairs take part
    int npairs;
    int force32;              // scoring outside the int16 range: all pairs int32
    int32_t *bin_of;          // per pair bin (or -1 when not in this pass)
    int32_t *bin_count;       // kNumBins
    int32_t *error;           // set to nonzero when a pair's lengths are out of range
    // empty pairs (query or reference of length 0) get their all-zero result
    // here and take no part in the kernels
    int32_t *score_out, *start_out, *end_out, *alen_out;
    // > 0: rows per lane rounded up to a multiple of `coarse` (kCoarseRows,
    // or kCoarseRowsSmall for the smallest batches: at most kRBins / coarse
    // classes; exact, the extra rows are padding) but not past max_rows, what
    // the call's longest query takes; 0: every R its own class
    int coarse;
    int max_rows;
    const PairResult *screened;  // null, or results in which kScreenedFlag leaves a pair out
};

constexpr int kCoarseRows = 5;
constexpr int kCoarseRowsSmall = 10;

struct TaskArgs {
    const int32_t *bin_count;
    int32_t *bin_cursor;      // exclusive prefix of bin_count (scatter cursor)
    int32_t *seg_task0;       // first task of each (class, R) segment (+1 sentinel)
    int32_t *seg_first;       // first sorted pair of each segment
    int32_t *seg_len;         // pairs in each segment
    int32_t *ntasks;
    int32_t *npairs_binned;
    unsigned long long *seg_steps;  // sweep steps summed over each segment's tasks
    // 1: segment 0 (int16, R = kRBins) runs the wide form: kSlotsWide pairs
    // per task, kWideRows rows per lane, rlen + kWideG - 1 steps
    int wide;
};

// launch helpers (sw_kernels.hip)
// max_tasks > 0: the class's task count, known on the host (the grid then
// has no more waves than tasks); 0: a full persistent grid
hipError_t launch_batch(const BatchArgs &ba, bool int16, int rows, int cu_count, int waves_per_cu,
                        int max_tasks, hipStream_t st);
// the wide form's kernel (int16, kWideRows rows per lane)
hipError_t launch_batch_wide(const BatchArgs &ba, int cu_count, int max_tasks, hipStream_t st);
// deferred walk-back over pairs order[*first .. *first + *count) (first may
// be null: 0; max_pairs bounds *count); moves holds move_words words per pair
// id, move_words >= (kMaxBatchQ + kMaxBatchR) / 16 + 1.  Under
// kWaveWalkPairs pairs a wave walks each pair, else a lane.
// A lane's walk waits for one granule after another, whatever the pairs beside
// it; a class of the pairs the screen leaves is 10,000 to 40,000.  16,384 -> 40,960:
// 1.0M uneven pairs 4.77 -> 4.64 ms, 100,000 with ambiguity codes 2.18 -> 2.08,
// 100,000 of 130-150 bases 672 -> 606 us; of unrelated pairs, all of them left,
// 1.0M 9.74 and 9.75 ms, 400,000 of 50-300 bases 5.75 -> 5.42.  131,072 gave no
// more.
constexpr int kWaveWalkPairs = 40960;
hipError_t launch_walk(const BatchArgs &ba, const int32_t *order, const int32_t *first,
                       const int32_t *count, int max_pairs, uint32_t *moves, int move_words,
                       hipStream_t st);
// pass-1 binning in one workgroup for batches up to kBinTinyPairs pairs,
// the sizes written into the host's mapped staging block (TinyStage)
constexpr int kBinTinyPairs = 4096;
struct TinyStage {
    int64_t *words;   // total trace words
    int64_t *steps;   // 2 * kRBins: sweep steps per segment
    int32_t *seg;     // 2 * kRBins + 1: first task of each segment
    int32_t *cnt;     // 16: the counters (ntasks, binned pairs, error flag, ...)
};
hipError_t launch_binning_tiny(const BinArgs &bin, const TaskArgs &ta, int32_t *order,
                               Task *tasks, int64_t *task_words, int64_t *total_words,
                               const int32_t *counters, const TinyStage &hs, hipStream_t st);
// scan_sums: room for max_tasks / 2048 + 1 int64 values; bin.bin_count
// must be zero on entry
hipError_t launch_binning(const BinArgs &bin, const TaskArgs &ta, int32_t *order, Task *tasks,
                          int64_t *task_words, const int64_t *base0, int64_t *total_words,
                          int64_t *scan_sums, int max_tasks, hipStream_t st);

}  // namespace swift
