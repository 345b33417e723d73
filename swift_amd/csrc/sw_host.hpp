// sw_host.hpp -- declarations shared by the host-side translation units.
#pragma once

#include "swift_common.hpp"

namespace swift {

struct KeyConsts;
struct Task;
struct BatchArgs;
struct BinArgs;
struct TaskArgs;

// The plain path's route for a call, and its sizes in 32-bit words
// (sw_plain.hip)
struct PlainPlan {
    enum Route { kGeneral, kPacked, kWave } route;
    int qlen, rlen, move_words;
    int form;                     // of the packed sweep (SweepForm)
    int wave_rows, packed_rows;   // rows a lane of the whole-wave and the packed sweeps
    int64_t wave_words;           // trace of a pair swept by a whole wave
    int64_t task_words;           // trace of eight packed pairs
};
struct PlainOut;
// budget: the words of scratch the call's chunks may take
PlainPlan plain_plan(const Scoring &sc, int qlen, int rlen, int npairs, int64_t budget);
// the largest chunk of at most npairs pairs that fits `budget` words of
// scratch (one pair at least), with its waves of the wave kernel
void plain_chunk(const PlainPlan &pl, int npairs, int64_t budget, int *chunk, int *waves);
int64_t plain_words(const PlainPlan &pl, int npairs, int waves);
// Plain path over pairs [pair0, pair0 + npairs) of the caller's arrays: sweep,
// walk and consensus expansion.  scratch holds plain_words(pl, npairs, waves)
// words, 16-byte aligned.
hipError_t launch_plain(const PlainPlan &pl, const char *q, const char *r, const Scoring &sc,
                        int npairs, int pair0, uint32_t *scratch, int waves, const PlainOut &out,
                        hipStream_t st);
int plain_rows_for(int qlen);
void set_plain_chunk_pairs(int pairs);             // 0: chunks by the scratch budget alone
hipError_t launch_fill(int32_t *p, int n, int32_t v, hipStream_t st);
// up to four int32 arrays zeroed by one kernel launch
struct ZeroSpans {
    int32_t *p[4];
    int n[4];
    int nspans;
};
hipError_t launch_zero(const ZeroSpans &z, hipStream_t st);

// up to four device arrays of 32-bit words -> one host staging block
struct Gather {
    const uint32_t *src[4];
    int nwords[4];
    int dst[4];      // word offset of each array in `out`
    uint32_t *out;   // mapped pinned host memory
    int nspans;
};
hipError_t launch_gather(const Gather &g, hipStream_t st);

// Device buffer that only grows.
struct DevBuf {
    void *ptr = nullptr;
    size_t bytes = 0;
    int ensure(size_t want);
    template <class T> T *as() const { return static_cast<T *>(ptr); }
    ~DevBuf();
};

// Batched SW over pairs already resident on the device.  Lengths live on
// the device; maxq/maxr bound them (host-side validation and buffer sizing).
// Results: int32 score/start/end/alen and reversed consensus strings at
// cons_off[p] (capacity qlen + rlen + 2 each).  When `sync_sizes` is false
// the call allocates nothing and relies on `reserve_batch` having sized the
// workspace for (npairs, maxq, maxr); that form is graph-capturable.
struct BatchIO {
    const char *qseq;
    const int64_t *qoff;
    const int32_t *qlen;
    const char *rseq;
    const int64_t *roff;
    const int32_t *rlen;
    int npairs, maxq, maxr;
    int32_t *score, *start, *end, *alen;
    char *qcons, *rcons;
    const int64_t *cons_off;
    // 1: every reference byte is one of ACGTNacgtn (the caller knows it, as
    // the pipeline does from its index); with scores that cannot reach the
    // int16 limit either, no pair can take the int32 re-run
    int refs_plain = 0;
    // 1: npairs is a capacity and pairs may be missing (length 0), as in the
    // pipeline
    int sparse = 0;
};

int validate_scoring(const Scoring &s, int maxq, int maxr, bool *force32);
// float scores of the reference's interfaces -> integers (each must be integral)
int scoring_from_floats(float match, float mismatch, float gap_open, float gap_ext, Scoring *sc);
int sw_batch_run(const BatchIO &io, const Scoring &sc, hipStream_t st, bool sync_sizes);
int reserve_batch(int npairs, int maxq, int maxr);

// Private batched-SW workspaces (device buffers, side streams), so that
// several batches can be in flight at once, each driven by its own host
// thread on its own stream.  sw_batch_run_in sizes the trace on the device
// (it synchronises `st`) and reports lengths beyond the batched limits; a small
// call does neither, and the caller asks sw_batch_status_in once it has
// waited for `st`: an error too where a pair is longer than maxq or maxr.
struct Workspace;
// side_streams: row-class kernels spread over that many private streams
// (0..3); 0 runs them one after another on the caller's stream
Workspace *workspace_new(int side_streams = 3);
void workspace_free(Workspace *w);
// persistent waves per CU of this workspace's row-class kernels, in place of
// the process-wide tuning (-1: follow it)
void workspace_set_waves(Workspace *w, int waves_per_cu);
int64_t workspace_bytes(const Workspace *w);
int sw_batch_run_in(Workspace *w, const BatchIO &io, const Scoring &sc, hipStream_t st);
int sw_batch_status_in(Workspace *w);
// Capturable form: no host synchronisation, no allocation (reserve_batch_in
// first, for at least this npairs / maxq / maxr); every row class is launched
// and empty ones exit at once.  sw_batch_check_in reads the length-error flags
// afterwards (it synchronises `st`): of the last run and, of small calls, of
// every one since the last check.
int reserve_batch_in(Workspace *w, int npairs, int maxq, int maxr);
int sw_batch_enqueue_in(Workspace *w, const BatchIO &io, const Scoring &sc, hipStream_t st);
int sw_batch_check_in(Workspace *w, hipStream_t st);
int64_t batch_bytes_estimate(int npairs, int maxq, int maxr);

// statistics of the last batched run (for tests and the bench)
struct BatchStats {
    int ntasks16, ntasks32, nrerun;
    int64_t trace_words;
};
BatchStats last_batch_stats();

// HIP-event phase timing of swift_sw_batch (binning, int16/int32 forward
// sweep, re-run pass, walk-back), in ms, recorded on the call's stream
void set_batch_timing(bool on);
const float *batch_timing_ms();

// tuning knobs set by the autotuner (see tune.cpp)
struct Tuning {
    int waves_per_cu = 0;       // cap on persistent waves per CU (0: occupancy limit)
    int int16 = 1;              // allow the int16 packed path
    int walk_deferred = 1;      // 1: walk-back kernels after each class's sweep (moves,
                                // then strings); 0: the walk fused into each wave task
    int coarse_rows = -1;       // 1: rows per lane rounded up to a multiple of 5 (at most
                                // 4 row classes); 0: every R its own class; -1: per call
};
// batches below this many pairs take the coarse row classes under coarse_rows -1
constexpr int kCoarsePairs = 131072;
constexpr int kCoarseSmallPairs = 16384;  // ... rounded to kCoarseRowsSmall below this
constexpr int kCoarseTinyPairs = 4096;    // ... and to one class (R = kRBins) below this
// ... but from this many pairs only when some query needs more than
// kCoarseRowsSmall rows per 16-lane group
constexpr int kWideShortPairs = 2048;
// One-launch form (sw_small.hip): a pair a wave up to kSmallSingles pairs (one
// wave a SIMD), then two.
constexpr int kSmallSingles = 1024;
constexpr int kSmallWaves = 4096;   // each keeps a trace area
// From this many pairs on the screen goes first (sw_screen.hip) and the one
// launch takes what it leaves: two launches more, against the related pairs'
// sweeps.  us a call without -> with, queries of 50-300 bases beside their places
// (unrelated pairs, all left to the sweep): 2,048 114 -> 124 (111 -> 126); 4,000
// 163 -> 133 (161 -> 185); 8,000 269 -> 198 (270 -> 301); 16,000 495 -> 294 (496 ->
// 547); of 100 bases 2,048 59 -> 67 (58 -> 72); 4,000 77 -> 74 (76 -> 96); 16,000
// 217 -> 115 (209 -> 261).  Not where slots may be missing: most of a pipeline's
// pairs are unrelated, and its small calls wait for launches.
constexpr int kSmallScreen = 4000;
// The one launch's waves take pairs unsorted, 64 lanes of ceil(maxq / 64) rows
// each, against the general path's binning, readback and 16-lane groups: taken
// up to kSmallWork = pairs x rows a lane, and of those the screen leaves, which
// only the device knows, up to kSmallLeft: with more the kernel's waves leave at
// once and the host goes on to the general path, 30 us later than it would have.
// us a call, general path -> one launch without that line, of pairs that are all
// related, three in four of them unrelated, all unrelated:
//   50-300 bases: 12,000 386 -> 256, 414 -> 397, 415 -> 433; 20,000 524 -> 323,
//     607 -> 569, 617 -> 633; 26,000 575 -> 378, 634 -> 693, 639 -> 793
//   100: 20,000 194 -> 115, 256 -> 250, 291 -> 287; 30,000 208 -> 142, 318 -> 356,
//     362 -> 399; 60,000 275 -> 226, 526 -> 639, 586 -> 753
//   150: 30,000 306 -> 241, 473 -> 485, 520 -> 536; 43,000 343 -> 314, 595 -> 645,
//     703 -> 747
//   300: 14,000 558 -> 407, 615 -> 519, 627 -> 604; 26,000 684 -> 621, 913 -> 870,
//     1,002 -> 946
// three rounds of the waves' pairs, two each, lie between the sides.
// A pipeline's capacity counts slots of which a half or fewer hold records:
// 5,000 reads of 300 bases (capacity 30,000) 1,052 -> 816 us, 13,000 of 100
// 1,039 -> 995.
constexpr int kSmallWork = 130000;
constexpr int kSmallWorkSparse = 160000;
constexpr int kSmallLeft = 3 * 2 * kSmallWaves;
inline bool small_call(int npairs, int maxq, bool sparse) {
    const int64_t rows = maxq > 64 ? (maxq + 63) / 64 : 1;
    return npairs * rows <= (sparse ? kSmallWorkSparse : kSmallWork);
}
Tuning &tuning();

}  // namespace swift
