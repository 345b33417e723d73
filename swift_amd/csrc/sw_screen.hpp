// sw_screen.hpp -- device code that answers a pair from its bytes alone when
// its best alignment provably has no gap: no matrix, no trace, no walk.
//
// Most pairs a mapper makes are a read beside the place it came from, a few
// substitutions apart.  Their matrix holds one diagonal that matters.  The
// screen compares the query with the reference along every diagonal, 32 bases
// an instruction (two bit planes of 2-bit bases: xor, or, population count),
// and takes a pair out of the sweep when the counts prove what the sweep would
// have found.
//
// The proof.  Cut the query into words of 16 to 47 rows.  Let m be the match
// score, -x the mismatch, -g what opening a gap costs (extending only adds to
// it), K = ceil(g / m).  Suppose that
//   (a) on one diagonal d0 every word has e mismatches (rows outside the
//       reference among them) with (m + x) * e < g, and
//   (b) on every other diagonal every word has at least K mismatches.
// Let P be any path with a gap, J its rows, S(J) the score of J's rows on d0.
// Each stretch of P off d0 costs a gap at each end that joins d0 (the
// diagonal changes there), or one inside it.  What such a stretch gains over
// the same rows of d0 is, in a word it fills: nothing, as off d0 a word scores
// at most m (rows - K) <= m rows - g on one diagonal, and at most m rows - g
// with a gap in it, and (a) puts d0's word above both; in a word it fills in
// part: at most (m + x) e < g, the mismatches it avoids, which the gap at
// that end outweighs.  Where the path itself begins or ends off d0, the rows
// of that word which J leaves out score on d0 what makes up the word, and all
// whole words of d0 score more than 0.  So P scores strictly less than the
// best stretch of d0, and by (b) so does every path on another diagonal alone.
// H of a cell is the score of the path its directions trace, and H never
// falls below what the cell's own diagonal gives: so the largest H is d0's best stretch,
// its first cell in row-major order the first row that reaches it, and the
// traced path stays on d0 until the running score falls below 0 or a border
// (a path that left it would have a gap and the best score).
//
// Rows past the reference's ends match nothing on d0 and count as an arbitrary
// base elsewhere, which can only make (b) fail.  Pairs with another
// byte than ACGT in the query or ACGTacgt in the reference are left to the
// sweep.
//
// Cost: a wave's 64 lanes take 64 diagonals at once; their words come out of a
// ring of shifted ones (two 64-bit shifts and two LDS reads a plane and turn),
// then 4 instructions each.  Bound by issue: 0.64 us of a SIMD a pair of 150 x
// 300 (7 turns of 5 words), where the sweep takes 9; of 143 x 253 on average 314
// vector instructions a pair, 57 % of the SIMDs' cycles, beside 278 scalar ones.
// Measured without the screen and with it, 1.0M such pairs of uneven lengths, a
// quarter with a gap: 10.1 -> 4.9 ms a call, 0.92 of it the screen.
// Where three pairs in four are of unrelated sequences (every candidate place
// of 250,000 reads): 10.9 -> 9.1.
#pragma once

#include "sw_sweep.hpp"

namespace swift {

struct ScreenConsts {
    int match, delta, gap, mis, k;  // m, m + x, g, x, K
};
// for scorings of lean_scoring (match >= 1, the others < 0)
inline ScreenConsts screen_consts(const Scoring &s) {
    return ScreenConsts{s.match, s.match - s.mismatch, -s.gap_open, -s.mismatch,
                        (-s.gap_open + s.match - 1) / s.match};
}
constexpr int kScreenMinQ = 16;    // a word has 16 rows at least
constexpr int kScreenMinR = 8;     // the shortest reference a lane can load of
// a wave's LDS words: the planes of the reference, then the query's
constexpr int kScreenPlane = 48, kScreenQuery = 2 * kScreenPlane, kScreenQPlane = 16;
constexpr int kScreenWords = kScreenQuery + 2 * kScreenQPlane;

// the alignment of a pair the screen answers: `len` cells down a diagonal to
// (row, row + diag), 0-based
struct Screened {
    int score, row, diag, len;
};

// A lane's eight of n bytes at s (n >= 8; those past the end 0) as bits of two
// planes, a base's code being (b >> 1) & 3 (A 0, C 1, T 2, G 3); `odd` where a
// byte, its bits of FOLD cleared, is not that code's letter.
template <uint32_t FOLD>
__device__ __forceinline__ void screen_load(const char *s, int n, uint8_t *p0, uint8_t *p1,
                                            uint32_t &odd) {
    const int k = 8 * (int)(threadIdx.x & 63), at = min(k, n - 8);
    uint64_t x;
    __builtin_memcpy(&x, s + at, 8);
    const uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    const uint32_t l0 = __builtin_amdgcn_perm(0u, 0x47544341u, (lo >> 1) & 0x03030303u);
    const uint32_t l1 = __builtin_amdgcn_perm(0u, 0x47544341u, (hi >> 1) & 0x03030303u);
    odd |= (l0 ^ (lo & ~(FOLD * 0x01010101u))) | (l1 ^ (hi & ~(FOLD * 0x01010101u)));
    x >>= 8 * min(k - at, 7);
    const uint32_t a = (uint32_t)x, b = (uint32_t)(x >> 32);
    auto plane = [&](uint32_t m) {
        return __builtin_amdgcn_udot4(b & m, 0x80402010u,
                                      __builtin_amdgcn_udot4(a & m, 0x08040201u, 0u, false), false);
    };
    const uint32_t v0 = plane(0x02020202u) >> 1, v1 = plane(0x04040404u) >> 2;
    if (k < n) {
        p0[k >> 3] = (uint8_t)v0;
        p1[k >> 3] = (uint8_t)v1;
    }
}
__device__ __forceinline__ uint32_t low_bits(int n) {  // 0 <= n <= 32
    return n >= 32 ? ~0u : (1u << n) - 1u;
}

// One wave, one pair of 1 <= ql <= 32 * NW rows (more than 32 * (NW - 1)).
// lds: kScreenWords words of this wave's own, 8-byte aligned; free once it returns.
template <int NW>
__device__ __forceinline__ bool screen_words(const ScreenConsts &sc, const char *qs, int ql,
                                             const char *rs, int rl, uint32_t *lds, Screened &out) {
    constexpr int kTurns = (kMaxBatchR + 32 * NW) / 64 + 1;
    static_assert(2 * kTurns + NW + 2 <= kScreenPlane, "words read of the staged reference");
    const int lane = threadIdx.x & 63;
    // a last word of under 16 rows is counted with the one before it
    const int rem = ql - 32 * (NW - 1);
    const bool merge = NW > 1 && rem < 16;
    const int last = merge ? 32 + rem : rem;
    const int first = NW == 1 || (NW == 2 && merge) ? last : 32;
    // the diagonals on which some word may have fewer than K mismatches: its
    // rows inside the reference are more than its rows less K (from a whole
    // staged byte on)
    const int d_lo = min((last - sc.k + 1 - ql) & ~7, 0), d_n = rl - first + sc.k - d_lo;
    if (d_n <= 0) return false;
    const int turns = (d_n + 63) >> 6;
    if (turns > kTurns) return false;

    // bit b of the staged words is column d_lo + b; bits outside the reference 0
    reinterpret_cast<uint2 *>(lds)[lane] = make_uint2(0u, 0u);
    uint32_t odd = 0;
    uint8_t *ref = reinterpret_cast<uint8_t *>(lds) + (-d_lo >> 3);
    screen_load<0x20u>(rs, rl, ref, ref + 4 * kScreenPlane, odd);
    uint8_t *qry = reinterpret_cast<uint8_t *>(lds + kScreenQuery);
    screen_load<0u>(qs, ql, qry, qry + 4 * kScreenQPlane, odd);
    if (__ballot(odd != 0)) return false;
    wave_lds_sync();
    const uint32_t *q0 = lds + kScreenQuery, *q1 = q0 + kScreenQPlane;

    // every diagonal: the least mismatches of its words
    const uint32_t *w0 = lds + (lane >> 5), *w1 = w0 + kScreenPlane;
    const uint32_t sh = (uint32_t)lane & 31u;
    const uint32_t lmask = low_bits(rem);
    const uint32_t m_add = merge ? 64u : 0u, m_sel = merge ? ~0u : 0u;
    uint32_t qa[NW], qb[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        qa[w] = (uint32_t)uni((int)q0[w]);
        qb[w] = (uint32_t)uni((int)q1[w]);
    }
    // word w of turn t is staged word 2t + w, shifted: a ring of registers, as
    // many turns unrolled as it takes to come round
    constexpr int RING = (NW + 1) & ~1;
    uint32_t s0[RING], s1[RING];
    uint32_t a0 = w0[0], a1 = w1[0];
    auto word = [&](int slot, uint32_t b0, uint32_t b1) {
        s0[slot] = __builtin_amdgcn_alignbit(b0, a0, sh);
        s1[slot] = __builtin_amdgcn_alignbit(b1, a1, sh);
        a0 = b0;
        a1 = b1;
    };
#pragma unroll
    for (int i = 0; i < NW - 2; ++i) word(i, w0[i + 1], w1[i + 1]);
    int live = 0, at = 0;
    for (int t0 = 0; t0 < turns && live < 2; t0 += RING / 2, w0 += RING, w1 += RING) {
#pragma unroll
        for (int u = 0; u < RING / 2; ++u) {
            const int t = t0 + u;
            if (t >= turns) break;
            if constexpr (NW == 1) {  // a word is passed over between turns
                a0 = w0[2 * u];
                a1 = w1[2 * u];
            }
#pragma unroll
            for (int i = max(2 * u + NW - 2, 0); i < 2 * u + NW; ++i)
                word(i % RING, w0[i + 1], w1[i + 1]);
            uint32_t least = 64, before = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int i = (2 * u + w) % RING;
                const uint32_t x = (s0[i] ^ qa[w]) | (s1[i] ^ qb[w]);
                if (w < NW - 1) {
                    const uint32_t n = (uint32_t)__builtin_popcount(x);
                    if (w == NW - 2) {
                        before = n;
                        least = min(least, n + m_add);
                    } else {
                        least = min(least, n);
                    }
                } else {
                    const uint32_t n = (uint32_t)__builtin_popcount(x & lmask) + (before & m_sel);
                    least = min(least, n);
                }
            }
            const uint64_t b = __ballot((int)least < sc.k && 64 * t + lane < d_n);
            if (b) {
                live += __builtin_popcountll(b);
                at = 64 * t + __builtin_ctzll(b);
            }
        }
    }
    if (live != 1) return false;

    // the diagonal's mismatches, word w in lane w
    const int diag = d_lo + at;
    const int wl = min(lane, NW - 1), wr = (at >> 5) + wl;
    const uint32_t ds = (uint32_t)at & 31u;
    uint32_t mm = (__builtin_amdgcn_alignbit(lds[wr + 1], lds[wr], ds) ^ q0[wl]) |
                  (__builtin_amdgcn_alignbit(lds[kScreenPlane + wr + 1], lds[kScreenPlane + wr], ds) ^
                   q1[wl]);
    auto rows = [&](int n) { return low_bits(max(0, min(n - 32 * wl, 32))); };
    mm = (mm | ~(rows(rl - diag) & ~rows(-diag))) & rows(ql);

    // its best stretch, the first cell of the largest score
    int score = 0, best_row = 0, best_from = 0, e_before = 0;
    int run = 0, from_row = 0, pos = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)mm, w);
        const int e = __builtin_popcount(x);
        if (sc.delta * (e + (w == NW - 1 && merge ? e_before : 0)) >= sc.gap) return false;
        e_before = e;
        while (x) {
            const int row = 32 * w + __builtin_ctz(x);
            x &= x - 1;
            run += sc.match * (row - pos);
            if (run > score) {
                score = run;
                best_row = row - 1;
                best_from = from_row;
            }
            run -= sc.mis;
            pos = row + 1;
            if (run < 0) {
                run = 0;
                from_row = pos;
            }
        }
    }
    run += sc.match * (ql - pos);
    if (run > score) {
        score = run;
        best_row = ql - 1;
        best_from = from_row;
    }
    wave_lds_sync();  // before the next pair's planes
    out = Screened{score, best_row, diag, best_row - best_from + 1};
    return out.len >= 4;  // what screen_strings takes
}

// ql <= 32 * MAXW
template <int MAXW>
__device__ __forceinline__ bool screen_pair(const ScreenConsts &sc, const char *qs, int ql,
                                            const char *rs, int rl, uint32_t *lds, Screened &out) {
    if (ql < kScreenMinQ || rl < kScreenMinR || rl > kMaxBatchR) return false;
    switch ((ql + 31) >> 5) {
#define SWIFT_W(N) \
    case N:        \
        if constexpr (N <= MAXW) return screen_words<N>(sc, qs, ql, rs, rl, lds, out); \
        return false;
        SWIFT_W(1) SWIFT_W(2) SWIFT_W(3) SWIFT_W(4) SWIFT_W(5)
        SWIFT_W(6) SWIFT_W(7) SWIFT_W(8) SWIFT_W(9) SWIFT_W(10)
#undef SWIFT_W
    default: return false;
    }
}

// the reversed strings of a screened pair, 4 bytes a lane
__device__ __forceinline__ void screen_strings(const Screened &s, const char *qs, const char *rs,
                                               char *qc, char *rc) {
    const char *qe = qs + s.row, *re = rs + s.row + s.diag;  // the last cell's bases
    for (int k = 4 * (int)(threadIdx.x & 63); k <= s.len; k += 256) {
        if (k + 4 <= s.len) {
            uint32_t q, r;
            __builtin_memcpy(&q, qe - k - 3, 4);
            __builtin_memcpy(&r, re - k - 3, 4);
            q = __builtin_bswap32(q);
            r = __builtin_bswap32(r);
            __builtin_memcpy(qc + k, &q, 4);
            __builtin_memcpy(rc + k, &r, 4);
        } else {
            for (int i = k; i < s.len; ++i) {
                qc[i] = qe[-i];
                rc[i] = re[-i];
            }
            qc[s.len] = 0;
            rc[s.len] = 0;
        }
    }
}

}  // namespace swift
