// sw_sweep.hpp -- device code shared by the batched and the plain
// Smith-Waterman kernels: the sweeps of a lane group, the best cell, the
// traceback walks over the packed direction codes and the consensus
// expansion.
#pragma once

#include <type_traits>

#include "sw_host.hpp"
#include "sw_types.hpp"

namespace swift {

// ---------------------------------------------------------------------------
// lane arithmetic: PK = packed 2 x int16 in a uint32, else one int32
// ---------------------------------------------------------------------------
typedef short v2s __attribute__((ext_vector_type(2)));
typedef unsigned short v2u __attribute__((ext_vector_type(2)));

__device__ __forceinline__ v2s as_s(uint32_t x) { return __builtin_bit_cast(v2s, x); }
__device__ __forceinline__ v2u as_us(uint32_t x) { return __builtin_bit_cast(v2u, x); }
__device__ __forceinline__ uint32_t as_u(v2s x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ uint32_t as_u(v2u x) { return __builtin_bit_cast(uint32_t, x); }

template <bool PK> __host__ __device__ constexpr uint32_t splat(int x) {
    return PK ? ((uint32_t)(x & 0xFFFF) | ((uint32_t)(x & 0xFFFF) << 16)) : (uint32_t)x;
}
template <bool PK> __device__ __forceinline__ uint32_t vadd(uint32_t a, uint32_t b) {
    if constexpr (PK) return as_u(as_s(a) + as_s(b));
    else return a + b;
}
template <bool PK> __device__ __forceinline__ uint32_t vsub(uint32_t a, uint32_t b) {
    if constexpr (PK) return as_u(as_s(a) - as_s(b));
    else return a - b;
}
template <bool PK> __device__ __forceinline__ uint32_t vmax(uint32_t a, uint32_t b) {
    if constexpr (PK) return as_u(__builtin_elementwise_max(as_s(a), as_s(b)));
    else return (uint32_t)max((int)a, (int)b);
}
// a * b + c, a in {0, 1}
template <bool PK> __device__ __forceinline__ uint32_t vmad(uint32_t a, uint32_t b, uint32_t c) {
    if constexpr (PK) return as_u(as_s(a) * as_s(b) + as_s(c));
    else return (uint32_t)((int)a * (int)b + (int)c);
}
template <bool PK> __device__ __forceinline__ uint32_t vmin1(uint32_t a) {
    if constexpr (PK) return as_u(__builtin_elementwise_min(as_us(a), (v2u){1, 1}));
    else return min(a, 1u);
}
// per element (k >> s) & 1 for a constant bit pattern k
template <bool PK> __device__ __forceinline__ uint32_t vbit(uint32_t k, uint32_t s) {
    if constexpr (PK) return as_u(as_us(splat<true>(k)) >> as_us(s)) & 0x00010001u;
    else return (k >> s) & 1u;
}

// Hides a value's range from the optimiser (no instruction is emitted), so
// that products by 0/1 flags and masked merges stay packed v_pk_* /
// v_bitop3 arithmetic instead of being rewritten into per-half compares and
// selects (there is no packed select).
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
    asm("" : "+v"(x));
    return x;
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_shift(uint32_t old, uint32_t src) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, CTRL, 0xF, 0xF, false);
}
constexpr int kRowShr1 = 0x111;   // lane l <- lane l-1 within each row of 16
constexpr int kWaveShr1 = 0x138;  // lane l <- lane l-1 across the wave

// Byte policy codes: low byte = byte value (reference byte upper-cased),
// bits 8..15 = 0xFF unless the byte is 'N' (the wildcard of isMatch_cpu).
__device__ __forceinline__ uint32_t byte_qcode(unsigned char c) {
    return (uint32_t)c | (c == 'N' ? 0u : 0xFF00u);
}
__device__ __forceinline__ uint32_t byte_rcode(unsigned char c) {
    int u = upper_byte(c) & 0xFF;
    return (uint32_t)u | (u == 'N' ? 0u : 0xFF00u);
}

// Byte policy (int32 lanes): 1 = mismatch.
__device__ __forceinline__ uint32_t byte_mismatch(uint32_t q, uint32_t r) {
    uint32_t x = (q ^ r) & ((q & r) >> 8) & 0xFFu;
    return min(x, 1u);
}

// Packed one-hot policy: the match flag of both halves from one v_perm_b32.
// A row holds the query's match table over the reference classes A C G T
// (0-3): 4 bytes per half, 0xFF where the query byte matches the class
// (query N: all four; any other query byte: none).  A column's word holds,
// per half, a perm selector in both bytes: class k -> k (half 0, table in
// bytes 0-3) or 4 + k (half 1, bytes 4-7); reference N -> 13 (0xFF, it
// matches every query byte); a padding column or another byte -> 12 (0x00).
// perm(table half 1, table half 0, selector) is 0xFFFF per matching half.
__host__ __device__ constexpr uint32_t query_table(uint32_t mask) {
    uint32_t t = 0;
    for (int k = 0; k < 4; ++k)
        if ((mask >> k) & 1u) t |= 0xFFu << (8 * k);
    return t;
}
__host__ __device__ constexpr uint32_t column_selector(uint32_t cls, int half) {
    const uint32_t s = cls < 4 ? cls + 4u * (uint32_t)half : cls == 4 ? 13u : 12u;
    return s * 0x0101u;
}

// ---------------------------------------------------------------------------
// The staggered sweep of one lane group.  G lanes, R rows per lane.
// Each lane slot carries PK ? 2 : 1 pairs.
// ---------------------------------------------------------------------------
//
// The packed kernels (PK) run every step unmasked: they take only scorings
// whose mismatch and gap moves all lose score (mismatch < 0, gaps <= -1), so
// cells left of column 1 stay in the column-0 state and cells right of a
// pair's last column (padding selectors: never a match) score strictly below
// the pair's best real cell.  The left exit is kept >= 0 by a saturating
// subtract, which makes the zero candidate of the max implicit.
template <int G, int R, bool PK, int POL>
struct Sweep {
    static_assert(PK == (POL == kOneHot), "packed lanes use the one-hot policy, int32 the bytes");
    static constexpr int KPW = PK ? 8 : 16;          // rows per trace word
    static constexpr int W = (R + KPW - 1) / KPW;     // trace words per step
    static constexpr uint32_t H4MASK = PK ? 0xFFFCFFFCu : ~3u;
    static constexpr uint32_t CMASK = PK ? 0x00030003u : 3u;
    static constexpr int CTRL = G == 16 ? kRowShr1 : kWaveShr1;

    uint32_t q[R];             // int32: query byte codes; PK: match tables of half 0
    uint32_t q2[PK ? R : 1];   // PK: match tables of half 1
    uint32_t dr[R];       // DR of (row, j-1)
    uint32_t el[R];       // EL of (row, j-1)
    // int32: best[r] = max over the row of H<<12 | (4095-j).
    // PK: best[r] = running max of the key 32H + (15 - t%16) (unsigned),
    // sealed to 32H + 31 at each block end; bcol[r] = block << 5 | key code
    // of the row's first strict maximum (see block_end).
    uint32_t best[R];
    uint32_t bcol[R];
    uint32_t eu_last, dr_last, dr_top;

    uint32_t c_dr, c_dsub, c_eo2, c_eo1, c_de, c_sign, c_eight;
    // PK: 16-bit tables indexed by direction code, laid out for v_perm_b32
    // (entry of code c in bytes 2c, 2c+1): the up exit, and the left exit's
    // penalty (subtracted with saturation at 0)
    uint32_t lut_u_lo, lut_u_hi, pen_l_lo, pen_l_hi;

    static __device__ __forceinline__ void lut(int v0, int v1, int v2, int v3, uint32_t &lo,
                                               uint32_t &hi) {
        lo = (uint32_t)(v0 & 0xFFFF) | ((uint32_t)(v1 & 0xFFFF) << 16);
        hi = (uint32_t)(v2 & 0xFFFF) | ((uint32_t)(v3 & 0xFFFF) << 16);
    }

    __device__ __forceinline__ void init(const KeyConsts &k) {
        c_dr = splat<PK>(k.dr);
        c_dsub = splat<PK>(PK ? -k.dsub : k.dsub);  // PK: times a 0xFFFF flag
        c_eo2 = splat<PK>(k.eo2);
        c_eo1 = splat<PK>(k.eo1);
        c_de = splat<PK>(k.de);
        c_sign = splat<PK>(k.sign);
        c_eight = opaque(splat<PK>(8));  // kept a multiplier: one v_pk_mad per key
        // up exit: open unless the cell came from above (code 2); left exit:
        // open unless it came from the left (code 1)
        lut(k.eo2, k.eo2, k.eo2 + k.de, k.eo2, lut_u_lo, lut_u_hi);
        lut(-k.eo1, -(k.eo1 + k.de), -k.eo1, -k.eo1, pen_l_lo, pen_l_hi);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            dr[r] = c_dr;   // column 0: H = 0, start
            // column 0 is not a left move -> open; PK: clamped at 0
            el[r] = PK ? 0u : c_eo1;
            best[r] = PK ? 0x001F001Fu : 0u;  // PK: H = 0, sealed
            bcol[r] = 0;
        }
        eu_last = c_eo2;
        dr_last = c_dr;
        dr_top = c_dr;
    }

    // One step.  rr: reference code(s) of column j; j = t - g; vmask: per
    // element all-ones where column j is inside the pair (MASKED only);
    // code (PK): 15 - t%16 in both halves.
    template <bool MASKED>
    __device__ __forceinline__ void step(uint32_t rr, int j, uint32_t vmask, uint32_t code,
                                         uint32_t *acc) {
        // row 0 of this lane takes the lane above's last row: its up exit at
        // column j (computed last step) and its diagonal value at column j-1
        // (received last step).  Lane 0 of the group sees matrix row 0.
        const uint32_t eu_in = dpp_shift<CTRL>(c_eo2, eu_last);
        const uint32_t dr_next = dpp_shift<CTRL>(c_dr, dr_last);
        const uint32_t diag0 = dr_top;
        dr_top = dr_next;
        if (MASKED && j < 0) return;  // left of column 1: keep column-0 state

        uint32_t colterm = 0;
        if constexpr (!PK) colterm = (uint32_t)(kMaxCols - j);
        // The diagonal, left and zero candidates depend only on column j-1:
        // fold them for every row first, so the row-to-row chain through the
        // up exit eu is just max -> code -> exit per row, with the rows'
        // independent work free to fill its gaps (max is order-free: the
        // direction code in the key's low bits breaks ties).
        uint32_t pre[R];
        if constexpr (PK) {
            // all diagonal candidates first, then the maxes: a packed result
            // read by the very next instruction costs a wait state
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t diag = r == 0 ? diag0 : dr[r - 1];
                const uint32_t f = __builtin_amdgcn_perm(q2[r], q[r], rr);  // 0xFFFF: match
                pre[r] = vmad<true>(f, c_dsub, diag);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) pre[r] = vmax<true>(pre[r], el[r]);  // el >= 0
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t diag = r == 0 ? diag0 : dr[r - 1];
                const uint32_t dk = vmad<false>(byte_mismatch(q[r], rr), c_dsub, diag);
                pre[r] = vmax<false>(vmax<false>(dk, el[r]), 0u);
            }
        }
        uint32_t eu = eu_in;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            uint32_t K = vmax<PK>(pre[r], eu);
            uint32_t h4 = K & H4MASK;
            uint32_t c = K & CMASK;
            acc[r / KPW] |= c << (2 * (r % KPW));
            dr[r] = vadd<PK>(h4, c_dr);
            if constexpr (PK) {
                // per-half gap exits from the 16-bit tables
                const uint32_t sel = c * 0x0202u + 0x01000100u;
                eu = vadd<true>(h4, __builtin_amdgcn_perm(lut_u_hi, lut_u_lo, sel));
                el[r] = as_u(__builtin_elementwise_sub_sat(
                    as_us(h4), as_us(__builtin_amdgcn_perm(pen_l_hi, pen_l_lo, sel))));
            } else {
                // int32: a select of the extension delta (a 32-bit multiply
                // by the 0/1 flag would be a quarter-rate v_mul_lo_u32)
                eu = h4 + c_eo2 + (c == 2u ? c_de : 0u);
                el[r] = h4 + c_eo1 + (c == 1u ? c_de : 0u);
            }
            if constexpr (PK) {
                static_assert(!(PK && MASKED), "packed steps are never masked");
                // key = 32H + code: within a block of 16 steps the largest
                // key is the row's largest H at its earliest step
                best[r] = as_u(__builtin_elementwise_max(
                    as_us(best[r]), as_us(vmad<true>(h4, c_eight, code))));
            } else {
                uint32_t key = (h4 << (kColBits - 2)) | colterm;
                if (MASKED) key &= vmask;
                best[r] = max(best[r], key);
            }
        }
        eu_last = eu;
        dr_last = dr[R - 1];
    }

    // PK, after the last step of a block of 16 (and after the sweep's last
    // step).  The previous block end sealed the running maximum to 32H + 31,
    // which every later key of the same H (code <= 15) leaves in place; a key
    // of larger H replaces it.  So a row's maximum rose in this block exactly
    // where the low 5 bits are no longer 31, and the row's first strict
    // maximum is then in this block, at the key's code.  blk32 = block index
    // << 5 in both halves.
    __device__ __forceinline__ void block_end(uint32_t blk32) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t lo = best[r] & 0x001F001Fu;
            const uint32_t m = as_u(as_s(vsub<true>(lo, 0x001F001Fu)) >> as_s(c_sign));
            bcol[r] = (m & (lo | blk32)) | (~m & bcol[r]);
            best[r] |= 0x001F001Fu;
        }
    }
};

// ---------------------------------------------------------------------------
// The lean sweep, for the scorings of lean_scoring (packed lanes:
// lean_packed_scoring): the same staggered recurrence and trace codes as Sweep in
// fewer instructions.
//
// What bounds a sweep is VALU issue, about 4 SIMD cycles an instruction
// whichever it is (a form with 32-bit subtracts for the packed ones, 2.3 cycles
// alone, and one more maximum a row took 7 % more).  A step of 10 rows of two
// packed cells takes 125 instructions here, 166 in Sweep:
//  * A cell's key is one v_pk_maximum3_f16 (v_max3_u32 in 32-bit lanes) of its
//    three candidates.  Every candidate is kept >= 0 by saturating subtracts,
//    which makes the zero candidate implicit, and non-negative keys below
//    0x7C00 order as half-precision bit patterns exactly as integers do.
//  * Exits are key - penalty[direction], the penalty a byte picked by
//    v_perm_b32 with the direction code itself as selector: the selector's
//    high bytes pick a 0.  A start's key and penalty are 0.
//  * Packed keys are 8H + direction, and c = 4 + (3 - direction), one v_bitop3,
//    is both that selector (the table in the perm's upper word) and, as key ^ c
//    is 8H + 7, all it takes to make x in one v_xad: an instruction a row less
//    than keys of 4H, whose bits are masked and added to.  The trace word sums
//    the rows' c and is put right once a step.
//  * The match test's v_perm_b32 yields the mismatch penalty (0 or pm), so the
//    diagonal candidate is one saturating subtract from x.
//  * The best cell is kept per lane, not per row: each step's maximum over
//    the rows of 32H + row code (smaller rows larger codes), and the first
//    step at which it rose.  That is the lane's first maximum in row-major
//    order, in 2 registers instead of 2R, which also lets another wave of the
//    larger classes onto a SIMD.
//  * Four steps a loop turn: their columns read together, their trace words
//    stored 16 bytes a lane.
// Sweep kernels, Sweep -> keys of 4H -> 8H: 1.0M pairs of 150 x 300 (R = 10) 11.8
// -> 9.4 ms, 768,000 of them 7.05 -> 6.65; 323,000 of 100 x 300 (R = 7) 2.35 ->
// 2.29; 64 pairs up to 300 x 480 in the wide form 137 -> 79 us.  kLeanWide (scores
// of 960 to 2,016) takes 2 % more cycles: a call of 100,000 pairs of 101-319 bases
// at 5, -4, -12, -2 with 5 % re-run 2.88 -> 2.51 ms.
// No step is masked: cells left of column 1 keep H = 0; cells right of a
// pair's last column and rows below its query never match (padding
// selectors, bit 7 of a padding row's table), so they score strictly below
// the pair's best cell.  (A packed padding cell's diagonal loses 255, which
// leaves its key 4 past a multiple of 8: half a score, which stays among padding
// cells, as none leads back into the matrix.)
// ---------------------------------------------------------------------------
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

template <bool PK> __device__ __forceinline__ uint32_t vmax3(uint32_t a, uint32_t b, uint32_t c) {
    if constexpr (PK) {
        const v2h x = __builtin_bit_cast(v2h, a), y = __builtin_bit_cast(v2h, b),
                  z = __builtin_bit_cast(v2h, c);
        return __builtin_bit_cast(
            uint32_t, __builtin_elementwise_maximum(__builtin_elementwise_maximum(x, y), z));
    } else {
        return max(max(a, b), c);
    }
}
template <bool PK> __device__ __forceinline__ uint32_t vsub_sat(uint32_t a, uint32_t b) {
    if constexpr (PK) return as_u(__builtin_elementwise_sub_sat(as_us(a), as_us(b)));
    else return __builtin_elementwise_sub_sat(a, b);
}

// 32-bit lanes compare bytes in dual-rail code: bits 14..21 the byte, bits
// 22..29 its complement on the query side, swapped on the reference side, so
// q & r is zero exactly where the bytes are equal; N has neither (the
// wildcard).  Bit 30: set in every query row and in padding columns; bit 31:
// set in padding rows and in every column.  A non-zero q & r is >= 2^14,
// above every mismatch penalty.
__device__ __forceinline__ uint32_t rail_query(uint32_t c, bool pad_row) {
    const uint32_t rails = c == 'N' ? 0u : c | (~c & 0xFFu) << 8;
    return (rails << 14) | (1u << 30) | (pad_row ? 1u << 31 : 0u);
}
__device__ __forceinline__ uint32_t rail_ref(uint32_t c, bool pad_col) {
    const uint32_t u = (uint32_t)upper_byte((int)c) & 0xFFu;
    const uint32_t rails = u == 'N' ? 0u : (~u & 0xFFu) | u << 8;
    return (rails << 14) | (1u << 31) | (pad_col ? 1u << 30 : 0u);
}
// Packed lanes: a row's match table (a byte per class A C G T: 0 where the
// query byte matches, else the mismatch penalty; 0xFF throughout in padding
// rows) and a column's selector, low byte: its class; N the sign of table
// byte 1, 0xFF in padding rows and 0 else; padding and other bytes 0xFF.  The
// high byte selects 0.
__device__ __forceinline__ uint32_t lean_table(uint32_t c, bool pad_row, uint32_t pm) {
    if (pad_row) return 0xFFFFFFFFu;
    return ~query_table(query_mask_bf((unsigned char)c)) & (pm * 0x01010101u);
}
__device__ __forceinline__ uint32_t lean_selector(uint32_t cls, int half) {
    const uint32_t s = cls < 4 ? cls + 4u * (uint32_t)half : cls == 4 ? 8u + 2u * (uint32_t)half : 13u;
    return s | 0x0C00u;
}

template <int G, int R, bool PK, int FORM = kLean>
struct Lean {
    static constexpr int KPW = PK ? 8 : 16;          // rows per trace word
    static constexpr int W = (R + KPW - 1) / KPW;     // trace words per step
    static constexpr uint32_t CMASK = PK ? 0x00030003u : 3u;
    static constexpr int CTRL = G == 16 ? kRowShr1 : kWaveShr1;
    // row r = block * B + k, coded so that smaller rows are larger: NB blocks,
    // below the key's H; B - 1 - k, KB bits
    static constexpr int NB = PK ? 8 : 4, KB = PK ? 2 : 3;
    static constexpr int B = (R + NB - 1) / NB;
    static_assert(B <= 1 << KB, "row codes");

    uint32_t q[R];             // PK: match tables of half 0; else dual-rail bytes
    uint32_t q2[PK ? R : 1];   // PK: match tables of half 1
    uint32_t x[R];             // u(H + match) + 3 of (row, j-1); u = 8 packed, else 4
    uint32_t el[R];            // left exit of (row, j-1)
    uint32_t x_top, eu_last;
    uint32_t best, tbest;      // best key and the step of its first cell
    uint32_t c_x, c_sign, tab_u, tab_l, pm, c_add, c_four;

    __device__ __forceinline__ void init(const KeyConsts &k) {
        c_x = splat<PK>(PK ? k.px : k.x);
        c_sign = splat<PK>(k.sign);
        tab_u = PK ? k.ptab_u : k.tab_u;
        tab_l = PK ? k.ptab_l : k.tab_l;
        pm = (uint32_t)k.pm;
        if constexpr (PK) {
            c_add = c_x - splat<true>(7);
            c_four = opaque(splat<true>(4));  // kept a multiplier: one v_pk_mad per key
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            x[r] = c_x;  // column 0: H = 0, start
            el[r] = 0;
        }
        x_top = c_x;
        eu_last = 0;
        best = first_key() + splat<PK>(31);  // H = 0 at any row
        tbest = 0;
    }

    // the key of H = 0 at the last row code
    __device__ __forceinline__ uint32_t first_key() const {
        return PK ? 4u * (c_x - splat<PK>(3)) : 8u * (c_x - 3u);
    }

    // One step on the reference code(s) rr of column t - g; tcode: t in every
    // element.
    __device__ __forceinline__ void step(uint32_t rr, uint32_t tcode, uint32_t *acc) {
        // from the lane above; a group's first lane sees matrix row 0 (H = 0: x =
        // c_x, no up exit).  (No maximum with c_x: a padding cell's x may be less,
        // and would take the other half's with it.)
        const uint32_t eu_in =
            (uint32_t)__builtin_amdgcn_update_dpp(0, (int)eu_last, CTRL, 0xF, 0xF, true);
        const uint32_t x_in =
            PK ? (uint32_t)__builtin_amdgcn_update_dpp((int)c_x, (int)x[R - 1], CTRL, 0xF, 0xF, false)
               : max((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x[R - 1], CTRL, 0xF, 0xF, true),
                     c_x);
        uint32_t diag[R];
#pragma unroll
        for (int r = R - 1; r >= 0; --r) {
            const uint32_t pen = PK ? __builtin_amdgcn_perm(q2[PK ? r : 0], q[r], rr)
                                    : min(q[r] & rr, pm);
            diag[r] = vsub_sat<PK>(r ? x[r - 1] : x_top, pen);
        }
        x_top = x_in;
        uint32_t eu = eu_in;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t K = vmax3<PK>(diag[r], el[r], eu);
            if constexpr (PK) {
                const uint32_t c = (~K & CMASK) | c_four;  // 4 + (3 - direction)
                acc[r / KPW] += c << (2 * (r % KPW));
                eu = vsub_sat<true>(K, __builtin_amdgcn_perm(tab_u, 0u, c));
                el[r] = vsub_sat<true>(K, __builtin_amdgcn_perm(tab_l, 0u, c));
                x[r] = (K ^ c) + c_add;  // 8H + 7 + (8*match - 4)
            } else {
                const uint32_t c = K & CMASK;
                acc[r / KPW] |= c << (2 * (r % KPW));
                eu = vsub_sat<PK>(K, __builtin_amdgcn_perm(tab_u, tab_u, c));
                el[r] = vsub_sat<PK>(K, __builtin_amdgcn_perm(tab_l, tab_l, c));
                x[r] = (K & ~CMASK) + c_x;
            }
        }
        if constexpr (PK) {
            // the codes: what the rows' sums of 7 - direction fall short by
#pragma unroll
            for (int w = 0; w < W; ++w) {
                uint32_t sevens = 0;
#pragma unroll
                for (int k = 0; k < KPW && w * KPW + k < R; ++k) sevens += splat<true>(7) << (2 * k);
                acc[w] = sevens - acc[w];
            }
        }
        eu_last = eu;
        // the step's best key: rows of one k by block, then over k
        uint32_t kb[B];
#pragma unroll
        for (int k = 0; k < B; ++k) {
            uint32_t v[NB];
            int n = 0;
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (b * B + k < R) v[n++] = x[b * B + k] - splat<PK>(b);
            uint32_t m = v[0];  // below 0x7C00 in either form
            int i = 1;
#pragma unroll
            for (; i + 1 < n; i += 2) m = vmax3<PK>(m, v[i], v[i + 1]);
            if (i < n) m = vmax<PK>(m, v[i]);
            if constexpr (PK)
                kb[k] = vmad<true>(m, c_four, splat<true>(16 + B - 1 - k));
            else kb[k] = (m << 3) + (uint32_t)(B - 1 - k);
        }
        uint32_t m = kb[0];
        if constexpr (PK && FORM == kLeanWide) {
#pragma unroll
            for (int k = 1; k < B; ++k)
                m = as_u(__builtin_elementwise_max(as_us(m), as_us(kb[k])));
            // all-ones where m > best: the saturated difference is not 0
            const uint32_t d = as_u(__builtin_elementwise_sub_sat(as_us(m), as_us(best)));
            const uint32_t up = vsub<true>(0u, vmin1<true>(d));
            tbest = (up & tcode) | (~up & tbest);
            best = as_u(__builtin_elementwise_max(as_us(best), as_us(m)));
        } else {
#pragma unroll
            for (int k = 1; k + 1 < B; k += 2) m = vmax3<PK>(m, kb[k], kb[k + 1]);
            if constexpr (B % 2 == 0) m = vmax<PK>(m, kb[B - 1]);
            if constexpr (PK) {
                const uint32_t up = as_u(as_s(vsub<true>(best, m)) >> as_s(c_sign));
                tbest = (up & tcode) | (~up & tbest);
                best = vmax<true>(best, m);
            } else {
                tbest = m > best ? tcode : tbest;
                best = max(best, m);
            }
        }
    }

    // best cell of the lane: H, its row within the lane (0-based), its step
    __device__ __forceinline__ void result(int half, uint32_t &h, int &r, int &t) const {
        const uint32_t s = 16u * (uint32_t)half, m = PK ? 0xFFFFu : ~0u;
        const uint32_t k = ((best >> s) & m) - ((first_key() >> s) & m);
        h = k >> 5;
        r = (int)(NB - 1 - ((k >> KB) & (NB - 1))) * B + B - 1 - (int)(k & ((1 << KB) - 1));
        t = (int)((tbest >> s) & m);
    }
};

// T steps of a lean sweep, rounded up to whole granules of 4 (the columns past
// the last are padding): a granule's columns, at col[t], are read during the
// granule before (4 words past the end are read), its trace words stored 16
// bytes a lane and word.  (Global stores: a 16-byte buffer store with its
// offset in a scalar register was seen to lose data to a 2-cycle instruction
// overwriting its source right after it; the compiler keeps only the other
// forms of wide stores apart from such writes.)
template <class S, bool PK>
__device__ __forceinline__ void lean_sweep(S &sw, const uint32_t *col, int T, uint32_t *trace) {
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63;
    v4u *tr = reinterpret_cast<v4u *>(trace);
    uint32_t nx[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) nx[u] = col[u];
    for (int t = 0; t < T; t += 4) {
        uint32_t cur[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            cur[u] = nx[u];
            nx[u] = col[t + 4 + u];
        }
        uint32_t acc[4][S::W];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int w = 0; w < S::W; ++w) acc[u][w] = 0;
            sw.step(cur[u], splat<PK>(t + u), acc[u]);
        }
#pragma unroll
        for (int w = 0; w < S::W; ++w)
            tr[w * 64 + lane] = (v4u){acc[0][w], acc[1][w], acc[2][w], acc[3][w]};
        tr += S::W * 64;
    }
}

// ---------------------------------------------------------------------------
// Result of a lane group: per lane, best (H, row, col) over its valid rows,
// then a group-wide max of (H desc, row asc) -- the reference's first strict
// maximum in row-major order.  Every lane of the group receives the result.
// ---------------------------------------------------------------------------
struct GroupResult {
    int32_t score, row, col, flag;
};

template <int G>
__device__ __forceinline__ GroupResult group_best(uint32_t lane_h, uint32_t lane_row,
                                                  uint32_t lane_col, int R, bool flag_overflow,
                                                  uint32_t h_limit, uint32_t force_flag) {
    uint64_t key = lane_h ? (((uint64_t)lane_h << 32) | (0xFFFFFFFFu - lane_row)) : 0;
    uint64_t m = key;
#pragma unroll
    for (int s = G / 2; s >= 1; s >>= 1) {
        uint64_t o = __shfl_xor(m, s, G);
        m = o > m ? o : m;
    }
    GroupResult gr;
    gr.score = (int32_t)(m >> 32);
    gr.row = m ? (int32_t)(0xFFFFFFFFu - (uint32_t)m) : 0;
    // the column lives in the lane that owns the best row
    const int base = (int)(threadIdx.x & 63) & ~(G - 1);
    const int src = base + (gr.row > 0 ? (gr.row - 1) / R : 0);
    gr.col = m ? __shfl((int)lane_col, src, 64) : 0;
    gr.flag = ((flag_overflow && (uint32_t)gr.score * 4 >= h_limit) || force_flag) ? 1 : 0;
    return gr;
}

// Output of one consensus string, four bytes per store when its start is
// 4-byte aligned.
struct ConsWriter {
    char *base;
    uint32_t word = 0;
    int n = 0;
    bool aligned;
    __device__ explicit ConsWriter(char *b) : base(b), aligned(((uintptr_t)b & 3) == 0) {}
    __device__ __forceinline__ void put(char c) {
        if (aligned) {
            word |= (uint32_t)(unsigned char)c << (8 * (n & 3));
            if ((n & 3) == 3) {
                *(uint32_t *)(base + (n & ~3)) = word;
                word = 0;
            }
        } else {
            base[n] = c;
        }
        ++n;
    }
    __device__ __forceinline__ void finish() {  // NUL terminator
        put('\0');
        if (aligned && (n & 3)) *(uint32_t *)(base + (n & ~3)) = word;
    }
};

// Trace layout: granules of 4 steps, [t/4][w][lane][t%4] (16 bytes per lane
// and word index), so a walk that stays on one lane for a few columns reads
// one granule instead of one cache line per step.
struct TraceReader {
    const uint4 *tr;
    PairTrace pt;
    uint32_t inv;  // ceil(2^16 / R): x / R == (x * inv) >> 16 for R <= 20, x < 2048
    int64_t cached = -1;
    uint4 gran;
    __device__ TraceReader(const uint4 *t, const PairTrace &p)
        : tr(t), pt(p), inv((65536u + (uint32_t)p.rows - 1) / (uint32_t)p.rows) {}
    __device__ __forceinline__ int code(int i, int j) {
        const int R = pt.rows;
        const int kpw = (pt.half & 2) ? 8 : 16;
        const int g = (int)(((uint32_t)(i - 1) * inv) >> 16), k = (i - 1) - g * R;
        const int lane = pt.lane0 + g, t = (j - 1) + g;
        const int w = k / kpw;
        const int bit = (pt.half & 1) * 16 + 2 * (k - w * kpw);
        const int64_t gi = pt.base / 4 + ((int64_t)(t >> 2) * pt.words + w) * 64 + lane;
        if (gi != cached) {
            gran = tr[gi];
            cached = gi;
        }
        const int u = t & 3;
        uint32_t word = u == 0 ? gran.x : u == 1 ? gran.y : u == 2 ? gran.z : gran.w;
        return (word >> bit) & 3;
    }
};

// TraceReader for the deferred walk kernel, which issues in the gaps the
// sweeps leave: per step only 32-bit arithmetic on (i, j), the pair's first
// granule resolved once, rows per word a shift, and the step's word picked
// by selects, not branches (80 instructions per step against 125).  The
// fused walk inside the sweep kernels keeps TraceReader: this one's extra
// live values spill there.
struct TraceReaderLean {
    const uint4 *tr;  // the pair's lane group at step 0, word 0
    int R, W, kl, bitb;
    uint32_t inv;
    int cached = -1;
    uint4 gran;
    __device__ TraceReaderLean(const uint4 *t, const PairTrace &p)
        : tr(t + p.base / 4 + p.lane0), R(p.rows), W(p.words), kl((p.half & 2) ? 3 : 4),
          bitb((p.half & 1) * 16), inv((65536u + (uint32_t)p.rows - 1) / (uint32_t)p.rows) {}
    __device__ __forceinline__ int code(int i, int j) {
        const int g = (int)(((uint32_t)(i - 1) * inv) >> 16), k = (i - 1) - g * R;
        const int t = (j - 1) + g;
        const int w = k >> kl;  // rows per word: 8 (packed halves) or 16
        const int bit = bitb + 2 * (k & ((1 << kl) - 1));
        // 32-bit granule index (a 24-bit multiply: t < 2^12, W <= 3); the
        // byte offset is formed once, in 64 bits, at the load
        const uint32_t gi = ((__umul24((uint32_t)(t >> 2), (uint32_t)W) + w) << 6) + g;
        if ((int)gi != cached) {
            gran = *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(tr) +
                                                     ((size_t)gi << 4));
            cached = (int)gi;
        }
        const uint32_t lo = (t & 1) ? gran.y : gran.x, hi = (t & 1) ? gran.w : gran.z;
        const uint32_t word = (t & 2) ? hi : lo;
        return (word >> bit) & 3;
    }
};

// Word offset of step t, trace word w, lane `lane` in the granule layout.
template <int W>
__device__ __forceinline__ int64_t trace_word(int t, int w, int lane) {
    return (((int64_t)(t >> 2) * W + w) * 64 + lane) * 4 + (t & 3);
}

// Runs steps [0, T): masked before lo and from hi on, unmasked between.
template <class Run>
__device__ __forceinline__ void sweep_steps(int T, int lo, int hi, Run &run) {
    int t = 0;
    for (; t < lo; ++t) run(std::true_type{}, t);
    for (; t < hi; ++t) run(std::false_type{}, t);
    for (; t < T; ++t) run(std::true_type{}, t);
}

struct WalkOut {
    int start, end, len;
};

// backtrack_cpu (src/smithWaterman.cu:263-335) over the packed direction
// codes: emit the current cell while its pointer leads elsewhere; a pointer
// into row 0 or column 0 emits the current cell and stops; a start pointer
// stops without emitting.  Each emitted cell is handed to `emit(k, op, i, j)`
// in walk order (the reference stores the strings reversed, i.e. in this
// order) with op 0 = diagonal (both bases), 1 = up (reference gap), 2 = left
// (query gap).
template <class Reader = TraceReader, class Emit>
__device__ __forceinline__ WalkOut walk_cells(const uint32_t *trace, int score, int row, int col,
                                              const PairTrace &pt, int qlen, int rlen, Emit &emit) {
    int start = 0, nrb = -1, tick = 0;
    if (score > 0 && row >= 1 && row <= qlen && col >= 1 && col <= rlen) {
        int ci = row, cj = col, ni, nj;
        Reader rd(reinterpret_cast<const uint4 *>(trace), pt);
        auto back = [&](int i, int j, int &oi, int &oj) {
            int c = rd.code(i, j);
            oi = (c & 2) ? i - 1 : i;            // diag (3) and up (2) move up
            oj = (c == 3 || c == 1) ? j - 1 : j;  // diag (3) and left (1) move left
        };
        back(ci, cj, ni, nj);
        for (;;) {
            if (ci == ni && cj == nj) break;
            const int op = nj == cj ? 1 : ni == ci ? 2 : 0;
            if (op != 1) ++nrb;
            emit(tick, op, ci, cj);
            start = cj;
            ++tick;
            if (ni == 0 || nj == 0) break;  // the target is in row/column 0
            ci = ni;
            cj = nj;
            back(ci, cj, ni, nj);
        }
    }
    return WalkOut{start, start + nrb, tick};
}

// Walk emitting the consensus strings directly (fused mode), NUL terminated.
__device__ WalkOut walk_pair(const uint32_t *trace, int score, int row, int col,
                             const PairTrace &pt, const char *qs, const char *rs, int qlen,
                             int rlen, char *qcons, char *rcons) {
    ConsWriter qc(qcons), rc(rcons);
    auto emit = [&](int, int op, int i, int j) {
        rc.put(op == 1 ? '-' : rs[j - 1]);
        qc.put(op == 2 ? '-' : qs[i - 1]);
    };
    WalkOut wo = walk_cells(trace, score, row, col, pt, qlen, rlen, emit);
    qc.finish();
    rc.finish();
    return wo;
}

// Makes this wave's earlier global stores (trace words) visible to its own
// later loads from other lanes.
__device__ __forceinline__ void wave_store_fence() {
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
}

// Orders one wave's LDS stores before its later LDS loads from other lanes
// (each wave of sw_expand_kernel works alone on its own LDS region, so no
// workgroup barrier is involved).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Deferred walk of one pair by a whole wave, for calls too small to fill
// the chip (a lane per pair leaves each wave waiting on one dependent
// granule load after another, and every lane's wait is the wave's).  The
// walk's state is wave-uniform; the trace around it is loaded as a window
// of granules, one per lane -- lane groups (g0 - NG, g0], every trace word,
// step blocks (tb0 - NT, tb0].  Lane l reads the code of the cell l steps
// down the diagonal from the window lane holding its granule (ds_bpermute);
// a ballot gives the length of the leading diagonal run, which the walk
// takes at once, then the move off it.  The walk only moves up and left, so
// it stays in a window until its lane group or step block passes the
// window's lower edge; a new window is then loaded at the current cell, one
// load per lane.  Same path, moves and results as walk_cells.  tr: the
// pair's lane group at step 0, word 0.
//
// The moves go to `mv`, a word (16 moves) at a time; RegMoves keeps them in
// registers, word m * 64 + lane in r[m], and stores them at the end (a store
// to global memory inside the walk would be waited for with the next window
// load).
template <int NMV> struct RegMoves {
    uint32_t *out;
    uint32_t r[NMV];
    __device__ explicit RegMoves(uint32_t *o) : out(o) {
#pragma unroll
        for (int m = 0; m < NMV; ++m) r[m] = 0;
    }
    __device__ __forceinline__ void put(int word, uint32_t value) {
#pragma unroll
        for (int m = 0; m < NMV; ++m)
            if (word == m * 64 + (int)(threadIdx.x & 63)) r[m] = value;
    }
    __device__ __forceinline__ void finish(int nwords) {
#pragma unroll
        for (int m = 0; m < NMV; ++m) {
            const int i = m * 64 + (int)(threadIdx.x & 63);
            if (i < nwords) out[i] = r[m];
        }
    }
};
// moves straight into LDS (the expansion follows in the same wave)
struct LdsMoves {
    uint32_t *out;
    __device__ __forceinline__ void put(int word, uint32_t value) {
        if ((threadIdx.x & 63) == 0) out[word] = value;
    }
    __device__ __forceinline__ void finish(int) {}
};
template <class Moves>
__device__ __forceinline__ WalkOut walk_wave(const uint4 *tr, int R, int W, int kl, int bitb,
                                             int score, int row, int col, int qlen, int rlen,
                                             Moves &mv) {
    const int lane = threadIdx.x & 63;
    int start = 0, nrb = -1, tick = 0;
    if (!(score > 0 && row >= 1 && row <= qlen && col >= 1 && col <= rlen))
        return WalkOut{start, start + nrb, tick};
    const uint32_t inv = (65536u + (uint32_t)R - 1) / (uint32_t)R;  // x / R for x < 2048
    // window shape: about 24 rows of lane groups, the rest of the 64 lanes
    // in step blocks; lanes past NG x W x NT load a copy of a window granule
    const int NG = min(8, (24 + R - 1) / R + 1);
    const int WT = 64 / NG, NT = WT / W;
    const int dg = min(lane / WT, NG - 1), r0 = lane - (lane / WT) * WT;
    const int lw = min(r0 / NT, W - 1), dtb = r0 - (r0 / NT) * NT;
    const int kmask = (1 << kl) - 1;
    int g0 = -1, tb0 = 0;
    uint4 v = make_uint4(0, 0, 0, 0);
    uint32_t mword = 0;
    int ci = row, cj = col;
    for (;;) {
        const int g = (int)(((uint32_t)(ci - 1) * inv) >> 16);
        const int tb = ((cj - 1) + g) >> 2;
        if (g0 < 0 || g0 - g >= NG || tb0 - tb >= NT) {
            g0 = g;
            tb0 = tb;
            v = tr[(max(tb0 - dtb, 0) * W + lw) * 64 + max(g0 - dg, 0)];
        }
        // Lane l reads the code of cell (ci - l, cj - l), l steps down the
        // diagonal, from the window lane holding its granule; the walk then
        // takes every leading diagonal move at once.
        const int il = ci - lane, jl = cj - lane;
        const int gl = (int)(__umul24((uint32_t)max(il - 1, 0), inv) >> 16);
        const int kl_ = (il - 1) - gl * R, tl = (jl - 1) + gl;
        const bool in_win = il >= 1 && jl >= 1 && g0 - gl < NG && tb0 - (tl >> 2) < NT;
        const int L = in_win ? (g0 - gl) * WT + (kl_ >> kl) * NT + (tb0 - (tl >> 2)) : 0;
        const uint32_t x = (uint32_t)__builtin_amdgcn_ds_bpermute(L << 2, (int)v.x);
        const uint32_t y = (uint32_t)__builtin_amdgcn_ds_bpermute(L << 2, (int)v.y);
        const uint32_t z = (uint32_t)__builtin_amdgcn_ds_bpermute(L << 2, (int)v.z);
        const uint32_t u = (uint32_t)__builtin_amdgcn_ds_bpermute(L << 2, (int)v.w);
        const uint32_t word = (tl & 2) ? ((tl & 1) ? u : z) : ((tl & 1) ? y : x);
        const int cl = in_win ? (int)((word >> (bitb + 2 * (kl_ & kmask))) & 3u) : -1;
        const uint64_t stop = __ballot(cl != 3);
        // the first cell off the diagonal run (or outside the window)
        const int first = stop ? (int)__builtin_ctzll(stop) : 64;
        if (first > 0) {
            // `first` diagonal moves (op 0: no bits to set); the move words
            // they complete are flushed as the count passes them
            nrb += first;
            start = cj - first + 1;
            ci -= first;
            cj -= first;
            int rest = first;
            while ((tick & 15) + rest >= 16) {
                const int adv = 16 - (tick & 15);
                mv.put(tick >> 4, mword);
                mword = 0;
                tick += adv;
                rest -= adv;
            }
            tick += rest;
            if (ci == 0 || cj == 0) break;  // the target is in row/column 0
        }
        if (first >= 64) continue;
        // that cell is now the current one; outside the window, a window is
        // loaded around it first
        if (!__builtin_amdgcn_readlane((int)in_win, first)) continue;
        const int c = __builtin_amdgcn_readlane(cl, first);
        if (c == 0) break;  // a start pointer: stop without emitting
        // up (2) or left (1)
        const int di = c >> 1, dj = c & 1;
        const int op = dj == 0 ? 1 : 2;
        nrb += dj;
        mword |= (uint32_t)op << (2 * (tick & 15));
        if ((tick & 15) == 15) {
            mv.put(tick >> 4, mword);
            mword = 0;
        }
        start = cj;
        ++tick;
        ci -= di;
        cj -= dj;
        if (ci == 0 || cj == 0) break;  // the target is in row/column 0
    }
    if (tick & 15) mv.put(tick >> 4, mword);
    mv.finish((tick + 15) >> 4);
    return WalkOut{start, start + nrb, tick};
}

// A flag in mapped host memory, read by the host after it has waited for the
// kernel.
__device__ __forceinline__ void host_flag(int32_t *f) {
    __hip_atomic_store(f, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// One pair's consensus expansion, by one row of L lanes of a wave (lane sl of
// the row; L = 16: four pairs per wave).  A pair's moves are taken in chunks
// of 16 per lane; a prefix sum of the row and column steps over the row's lanes gives each
// lane the cell its 16 moves start from, and the lane builds its 16 bytes of
// each string in registers from the pair's bases staged in LDS, then stores
// them as dwords where the strings are dword aligned (bytes at the string's
// end, then the NUL).  live = false: the row only takes part in the wave's
// LDS ordering.
struct ExpandPair {
    bool live = false;
    int len = 0, row = 0, col = 0;   // moves, best cell (1-based)
    int nq = 0, nr = 0;              // bases the path can reach
    const unsigned char *qsrc = nullptr, *rsrc = nullptr;
    char *qc = nullptr, *rc = nullptr;
    const uint32_t *mv = nullptr;    // 2-bit moves, 16 per word, walk order
};

template <int L>
__device__ __forceinline__ void expand_row(const ExpandPair &e, uint32_t *lq4, uint32_t *lr4,
                                           int sl) {
    // the bases into LDS, from the aligned dwords holding them (an aligned
    // dword holding a sequence byte lies within that byte's page)
    const int qm = (int)((uintptr_t)e.qsrc & 3), rm = (int)((uintptr_t)e.rsrc & 3);
    const int nqw = e.nq > 0 ? (qm + e.nq + 3) >> 2 : 0;
    const int nrw = e.nr > 0 ? (rm + e.nr + 3) >> 2 : 0;
    for (int u = sl; u < nqw; u += L)
        lq4[u] = reinterpret_cast<const uint32_t *>(e.qsrc - qm)[u];
    for (int u = sl; u < nrw; u += L)
        lr4[u] = reinterpret_cast<const uint32_t *>(e.rsrc - rm)[u];
    wave_lds_sync();
    const unsigned char *lq = (const unsigned char *)lq4 + qm;
    const unsigned char *lr = (const unsigned char *)lr4 + rm;
    char *qc = e.qc, *rc = e.rc;
    const bool aligned = (((uintptr_t)qc | (uintptr_t)rc) & 3) == 0;
    const int len = e.len;
    int ci = e.row, cj = e.col;
    constexpr int CH = 16 * L;  // moves a chunk
    const int nchunk = (len + CH - 1) / CH;
    for (int c = 0; c < nchunk; ++c) {
        const int k0 = c * CH + sl * 16;
        const int cnt = max(0, min(16, len - k0));
        const uint32_t w = cnt > 0 ? e.mv[k0 >> 4] : 0u;
        // row steps: every move but left (2); column steps: every move but
        // up (1); ops are 0, 1 or 2
        const uint32_t lo2 = cnt == 16 ? 0x55555555u : ((1u << (2 * cnt)) - 1u) & 0x55555555u;
        const uint32_t hib = (w >> 1) & lo2, lob = w & lo2;
        const int di = cnt - __builtin_popcount(hib & ~lob);
        const int dj = cnt - __builtin_popcount(lob & ~hib);
        int ei = di, ej = dj;  // inclusive scans over the row's lanes
#pragma unroll
        for (int d = 1; d < L; d <<= 1) {
            const int oi = __shfl_up(ei, d, L), oj = __shfl_up(ej, d, L);
            if (sl >= d) {
                ei += oi;
                ej += oj;
            }
        }
        int xi = ci - (ei - di), xj = cj - (ej - dj);
        uint32_t oq[4] = {0u, 0u, 0u, 0u}, orr[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            if (k < cnt) {
                const int op = (w >> (2 * k)) & 3;
                const uint32_t qb = op == 2 ? (uint32_t)'-' : (uint32_t)lq[xi - 1];
                const uint32_t rb = op == 1 ? (uint32_t)'-' : (uint32_t)lr[xj - 1];
                oq[k >> 2] |= qb << (8 * (k & 3));
                orr[k >> 2] |= rb << (8 * (k & 3));
                xi -= op != 2;
                xj -= op != 1;
            }
        }
        if (cnt == 16 && aligned) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                reinterpret_cast<uint32_t *>(qc + k0)[d] = oq[d];
                reinterpret_cast<uint32_t *>(rc + k0)[d] = orr[d];
            }
        } else {
            for (int k = 0; k < cnt; ++k) {
                qc[k0 + k] = (char)(oq[k >> 2] >> (8 * (k & 3)));
                rc[k0 + k] = (char)(orr[k >> 2] >> (8 * (k & 3)));
            }
        }
        ci -= __shfl(ei, L - 1, L);
        cj -= __shfl(ej, L - 1, L);
    }
    if (e.live && sl == 0) {
        qc[len] = 0;
        rc[len] = 0;
    }
    wave_lds_sync();  // before the next pairs overwrite this row's buffers
}

}  // namespace swift
