// Semi-local queries on a seaweed permutation: the quadrant -> dominance map
// shared by host validation and the device kernels, and the wavelet-matrix
// index layout.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lcs_hip.h"

namespace lcsq {

// Query q = (q0, q1) of `kind` on P(a, b) (m rows of a, n columns of b) as
//     result = sign * (base - D(r0, c0)) + (1 - sign) * D(r0, c0),
//     D(r0, c0) = #{ r >= r0 : P[r] < c0 }.
// The four quadrants are H(i, j) = (j - i) - D(m + i, j) at
//   string-substring  (i, j) = (q0, q1)               H
//   substring-string  (i, j) = (-q0, n + m - q1)      H - q0 - (m - q1) = n - D
//   prefix-suffix     (i, j) = (q1, n + m - q0)       H - (m - q0)       = (n - q1) - D
//   suffix-prefix     (i, j) = (-q0, q1)              H - q0             = q1 - D
// Returns false when the query lies outside its quadrant.
struct Window {
    int64_t r0, c0;
    int32_t base;
    bool score;   // false: the raw dominance count
};

__host__ __device__ inline bool query_window(int kind, int32_t m, int32_t n, int32_t q0, int32_t q1, Window &w)
{
    const int64_t M = m, N = n;
    switch (kind) {
    case LCS_SEMI_STRING_SUBSTRING:
        if (q0 < 0 || q0 > q1 || q1 > n) return false;
        w = {M + q0, q1, q1 - q0, true};
        return true;
    case LCS_SEMI_SUBSTRING_STRING:
        if (q0 < 0 || q0 > q1 || q1 > m) return false;
        w = {M - q0, N + M - q1, n, true};
        return true;
    case LCS_SEMI_PREFIX_SUFFIX:
        if (q0 < 0 || q0 > m || q1 < 0 || q1 > n) return false;
        w = {M + q1, N + M - q0, n - q1, true};
        return true;
    case LCS_SEMI_SUFFIX_PREFIX:
        if (q0 < 0 || q0 > m || q1 < 0 || q1 > n) return false;
        w = {M - q0, q1, q1, true};
        return true;
    case LCS_SEMI_DOMINANCE:
        w = {q0 < 0 ? 0 : q0, q1, 0, false};
        return true;
    }
    return false;
}

// The index: a wavelet matrix with two bits (a digit, 0..3) per level, and for
// an odd number of bits a last level of one bit.  16 bytes per record, so a
// rank is one gathered load, and half as many levels as with one bit each.

// 32 rows of a two-bit level: the digits' bits, and in `counts` the rows
// before these, back to the last multiple of kSuperRows, whose digit is below
// 1, 2 and 3 (kCountBits each).
struct Rank4 {
    uint32_t hi, lo;
    unsigned long long counts;
};
constexpr int kSuperLog = 20, kCountBits = 21;   // a count is at most kSuperRows
constexpr uint32_t kCountMask = (1u << kCountBits) - 1;

// 64 rows of the one-bit level.
struct Rank2 {
    unsigned long long bits;
    uint32_t zeros_before;
    uint32_t pad;
};

// The counts below 1, 2 and 3 (x, y, z) before each multiple of 2^kSuperLog
// rows of a two-bit level (`super`), and of the whole level (`totals`; of the
// one-bit level, x is the number of zeros).
struct IndexView {
    Rank4 *rec;
    Rank2 *last;
    uint4 *super, *totals;
    int32_t size;
    int bits, quads, supers;      // value bits, two-bit levels, entries of `super` per level
    int64_t w4, w2;               // records per level; both cover row `size`
};

inline IndexView index_view(void *mem, int32_t size, int bits)
{
    IndexView v{};
    v.size = size;
    v.bits = bits;
    v.quads = bits / 2;
    v.supers = (size >> kSuperLog) + 1;
    v.w4 = ((int64_t)size >> 5) + 1;
    v.w2 = bits % 2 ? ((int64_t)size >> 6) + 1 : 0;
    v.rec = (Rank4 *)mem;
    v.last = (Rank2 *)(v.rec + v.quads * v.w4);
    v.super = (uint4 *)(v.last + v.w2);
    v.totals = v.super + v.quads * v.supers;
    return v;
}

inline size_t index_bytes(int32_t size, int bits)
{
    const IndexView v = index_view(nullptr, size, bits);
    return (size_t)(v.totals + v.quads + bits % 2);
}

// Rows per workgroup of a build kernel: at least kTileRows, as many as keep
// the workgroups at kMaxBuildBlocks (each adds up the counts of all others).
constexpr int kTileRowsLog = 11, kMaxBuildBlocks = 2048;
inline int build_rows_log(int32_t size)
{
    int l = kTileRowsLog;
    while ((((int64_t)size >> l) + 1) > kMaxBuildBlocks) ++l;
    return l;   // at most kSuperLog
}
inline int build_blocks(int32_t size) { return (int)(((int64_t)size >> build_rows_log(size)) + 1); }   // covers row `size`
inline size_t build_scratch_words(int32_t size) { return 2 * (((size_t)size + 3) & ~(size_t)3) + 13 * (size_t)build_blocks(size) + 1; }

}  // namespace lcsq

// Launchers (query_kernels.hip); 0 or a negative LCS_E* status.
int lcsq_launch_scan(const int32_t *perm, int32_t size, int kind, int32_t m, int32_t n, const int32_t *q0,
                     const int32_t *q1, int32_t nq, int32_t *out, hipStream_t s);
// Builds the index of `perm` (size rows).  `scratch` holds
// build_scratch_words(size) words, 16-byte aligned; its last word becomes 1 if
// a value lies outside [-1, size), else 0.
int lcsq_launch_index_build(const int32_t *perm, const lcsq::IndexView &index, int32_t *scratch, hipStream_t s);
int lcsq_launch_index_query(const lcsq::IndexView &index, int kind, int32_t m, int32_t n, const int32_t *q0,
                            const int32_t *q1, int32_t nq, int32_t *out, hipStream_t s);
