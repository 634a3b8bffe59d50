// Semi-local score queries read from a seaweed permutation.
//
// For the permutation P of a (m) against b (n) in row_to_col form (row =
// strand id: 0..m-1 enter the rows, m..m+n-1 the columns; column = exit:
// 0..n-1 the bottom, n..n+m-1 the right side), every semi-local score is
//     H(i, j) = (j - i) - D(m + i, j),   D(r0, c0) = #{ r >= r0 : P[r] < c0 },
// read at a fixed offset per quadrant (query_kernels.h).  Two ways to count D:
//
//  * scan: one wave per query, each lane counts a strided share of the rows
//    (HBM/L2-bound, size*4 bytes per query; no set-up);
//  * wavelet matrix over the values P + 1 (so unset rows, -1, become 0) with
//    two bits per level: level k holds digit k from the top of the values in
//    that level's order; the next level is a stable sort by the digit.
//    D(r0, c) walks the levels with two ranks each (dependent 16-byte loads).
//    One launch per level builds it (index_level_kernel).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "query_kernels.h"

namespace lcsq {

constexpr int kBuildThreads = 512;            // 8 waves
constexpr int kTileWords = 4;                 // 64-row words of a wave in a tile
static_assert(1 << kTileRowsLog == 64 * kTileWords * (kBuildThreads / 64), "rows of a tile");

__global__ void scan_kernel(const int32_t *perm, int32_t size, int kind, int32_t m, int32_t n, const int32_t *q0,
                            const int32_t *q1, int32_t nq, int32_t *out)
{
    const int wave = (int)((blockIdx.x * (unsigned)blockDim.x + threadIdx.x) >> 6);
    const int lane = threadIdx.x & 63;
    if (wave >= nq) return;
    Window w;
    if (!query_window(kind, m, n, q0[wave], q1[wave], w)) {
        if (lane == 0) out[wave] = -1;
        return;
    }
    int cnt = 0;
    if (w.r0 < size)
        for (int32_t r = (int32_t)w.r0 + lane; r < size; r += 64) cnt += (int64_t)perm[r] < w.c0;
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off);
    if (lane == 0) out[wave] = w.score ? w.base - cnt : cnt;
}

struct LevelArgs {
    const int32_t *A;      // the level's values in its order, less `add`
    int32_t *next;         // the next level's order; null at the last
    const uint32_t *hist;  // rows per digit (4) of each workgroup's rows
    uint32_t *hist_next;   // the same of the next level, zero on entry
    uint4 *hist_after;     // cleared here: the level after next counts there
    Rank4 *rec;
    Rank2 *last;           // instead of rec at the one-bit level
    uint4 *super, *totals;
    const uint32_t *bad;   // at the last level: workgroups that saw a bad value
    int32_t *bad_out;
    int64_t words;         // records of the level
    int32_t size, add;
    uint32_t value_mask, digit_mask, next_digit_mask;
    int shift, next_shift, rows_log, blocks;
};

__device__ inline uint32_t digit_of(int32_t x, uint32_t value_mask, int shift, uint32_t digit_mask)
{
    // of a bad value (the build then fails), the same digits in every kernel
    return (((uint32_t)x & value_mask) >> shift) & digit_mask;
}

// hist of the first level; flags workgroups with a value outside [-1, size)
__global__ __launch_bounds__(kBuildThreads) void index_prep_kernel(const int32_t *perm, int32_t size, int rows_log,
                                                                   uint32_t value_mask, int shift,
                                                                   uint32_t digit_mask, uint4 *hist, uint4 *hist_next,
                                                                   uint32_t *bad)
{
    __shared__ uint32_t sum[5];
    const int t = threadIdx.x;
    if (t < 5) sum[t] = 0;
    __syncthreads();
    const int64_t row0 = (int64_t)blockIdx.x << rows_log;
    const int64_t row1 = min(row0 + ((int64_t)1 << rows_log), (int64_t)size);
    uint32_t c[4] = {0, 0, 0, 0}, wrong = 0;
    for (int64_t r = row0 + t; r < row1; r += kBuildThreads) {
        const int32_t x = perm[r];
        wrong |= x < -1 || x >= size;
        const uint32_t d = digit_of((int32_t)((uint32_t)x + 1), value_mask, shift, digit_mask);
#pragma unroll
        for (int k = 0; k < 4; ++k) c[k] += d == (uint32_t)k;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        for (int off = 32; off > 0; off >>= 1) c[k] += __shfl_xor(c[k], off);
        if ((t & 63) == 0) atomicAdd(&sum[k], c[k]);
    }
    if (wrong) atomicOr(&sum[4], 1u);
    __syncthreads();
    if (t == 0) {
        hist[blockIdx.x] = make_uint4(sum[0], sum[1], sum[2], sum[3]);
        hist_next[blockIdx.x] = make_uint4(0, 0, 0, 0);
        bad[blockIdx.x] = sum[4];
    }
}

// One level: its records, its values in the next level's order, and the next
// level's digit counts per workgroup.
//
// A workgroup's rows keep their order within each digit, so they land in (up
// to) four runs of the next order, each no longer than a workgroup's rows and
// hence within two workgroups of the next level: 4 x 2 x 4 counters in LDS
// take the place of a pass that counts.  Where the runs start, every
// workgroup adds up from the counts of all (at most kMaxBuildBlocks) itself:
// the launch and the dependent pass of a scan kernel cost more.
//
// Launches and the latency of their dependent loads bound the build at 2^19
// rows: 10 levels take 82 us of kernels, where 20 levels of one bit, each
// counted, scanned and placed by a launch of its own, took 301.  8 waves with
// 4 words each rather than 4 with 8 halve a wave's serial part (128 -> 82 us,
// with the rows loaded before the counts are).  A query reads one 16-byte
// record per rank and level: 2^20 queries take 28 us.
__global__ __launch_bounds__(kBuildThreads) void index_level_kernel(LevelArgs G)
{
    constexpr int kWaves = kBuildThreads / 64;
    __shared__ uint32_t part[kWaves][12], sum[12], next_count[32], wrong;
    __shared__ uint4 wave_count[kWaves];
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const int blk = (int)blockIdx.x;
    const int per_super_log = kSuperLog - G.rows_log;
    const int super0 = blk >> per_super_log << per_super_log;

    const int64_t rows0 = (int64_t)blk << G.rows_log, cover = (int64_t)G.size + 1;   // the records cover row `size`
    int32_t x[kTileWords];
    const auto load_tile = [&](int64_t w0) {
#pragma unroll
        for (int j = 0; j < kTileWords; ++j) {
            const int64_t r = w0 + j * 64 + lane;
            x[j] = r < G.size ? (int32_t)((uint32_t)G.A[r] + (uint32_t)G.add) : 0;
        }
    };
    load_tile(rows0 + wave * (64 * kTileWords));

    // rows per digit (one per thread, t & 3): of all workgroups, of those
    // before this one, and of those before the superblock
    uint32_t all = 0, pre = 0, sup = 0;
    for (int i = t; i < G.blocks * 4; i += kBuildThreads) {
        const uint32_t h = G.hist[i];
        all += h;
        pre += (i >> 2) < blk ? h : 0;
        sup += (i >> 2) < super0 ? h : 0;
    }
#pragma unroll
    for (int off = 4; off < 64; off <<= 1) {
        all += __shfl_xor(all, off);
        pre += __shfl_xor(pre, off);
        sup += __shfl_xor(sup, off);
    }
    if (lane < 4) {
        part[wave][lane] = all;
        part[wave][4 + lane] = pre;
        part[wave][8 + lane] = sup;
    }
    if (t < 32) next_count[t] = 0;
    if (t == 0) wrong = 0;
    __syncthreads();
    if (t < 12) {
        uint32_t v = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) v += part[w][t];
        sum[t] = v;
    }
    __syncthreads();
    uint32_t at[4], rel[4];   // where the next row of each digit goes; such rows since the superblock's start
    uint32_t before[4], base = 0, start[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        before[d] = sum[4 + d];
        at[d] = base + before[d];
        rel[d] = before[d] - sum[8 + d];
        start[d] = base;
        base += sum[d];
    }
    if (t == 0) {
        if (blk == 0) *G.totals = make_uint4(start[1], start[2], start[3], 0);
        if (blk == super0 && G.rec)
            G.super[blk >> per_super_log] =
                make_uint4(before[0], before[0] + before[1], before[0] + before[1] + before[2], 0);
        if (G.hist_after) G.hist_after[blk] = make_uint4(0, 0, 0, 0);
    }
    uint32_t first[4];   // the workgroup of the next level where the run of a digit starts
#pragma unroll
    for (int d = 0; d < 4; ++d) first[d] = at[d] >> G.rows_log;

    const int tiles = 1 << (G.rows_log - kTileRowsLog);
    for (int tile = 0; tile < tiles; ++tile) {
        const int64_t r0 = rows0 + ((int64_t)tile << kTileRowsLog);
        if (r0 >= cover) break;
        const int64_t w0 = r0 + wave * (64 * kTileWords);
        if (tile) load_tile(w0);
        unsigned long long hi[kTileWords], lo[kTileWords];
        uint32_t count[4] = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < kTileWords; ++j) {
            const int64_t r = w0 + j * 64 + lane;
            const bool valid = r < G.size;
            const uint32_t d = digit_of(x[j], G.value_mask, G.shift, G.digit_mask);
            hi[j] = __ballot(valid && (d & 2));
            lo[j] = __ballot(valid && (d & 1));
            const unsigned long long live = __ballot(valid);
            count[0] += (uint32_t)__popcll(live & ~hi[j] & ~lo[j]);
            count[1] += (uint32_t)__popcll(~hi[j] & lo[j]);
            count[2] += (uint32_t)__popcll(hi[j] & ~lo[j]);
            count[3] += (uint32_t)__popcll(hi[j] & lo[j]);
        }
        if (lane == 0) wave_count[wave] = make_uint4(count[0], count[1], count[2], count[3]);
        __syncthreads();
        uint32_t tile_count[4], run[4];   // run: rows of the digit earlier in the tile
#pragma unroll
        for (int d = 0; d < 4; ++d) tile_count[d] = run[d] = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const uint4 v = wave_count[w];
            const uint32_t c[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                tile_count[d] += c[d];
                run[d] += w < wave ? c[d] : 0;
            }
        }
        __syncthreads();   // wave_count is free for the next tile
#pragma unroll
        for (int j = 0; j < kTileWords; ++j) {
            const int64_t row = w0 + j * 64, r = row + lane;
            const bool valid = r < G.size;
            const unsigned long long h = hi[j], l = lo[j], live = __ballot(valid);
            const unsigned long long mask[4] = {live & ~h & ~l, ~h & l, h & ~l, h & l};
            // records: lane 0 the word's first half, lane 1 the second
            if (G.rec) {
                const int64_t w = (row >> 5) + lane;
                if (lane < 2 && w < G.words) {
                    uint32_t c[3], total = 0;
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        total += rel[d] + run[d] + (lane ? (uint32_t)__popc((uint32_t)mask[d]) : 0u);
                        c[d] = total;
                    }
                    Rank4 rec;
                    rec.hi = (uint32_t)(h >> (32 * lane));
                    rec.lo = (uint32_t)(l >> (32 * lane));
                    rec.counts = (unsigned long long)c[0] | ((unsigned long long)c[1] << kCountBits) |
                                 ((unsigned long long)c[2] << (2 * kCountBits));
                    G.rec[w] = rec;
                }
            } else if (lane == 0 && (row >> 6) < G.words) {
                Rank2 rec;
                rec.bits = l;
                rec.zeros_before = before[0] + run[0];
                rec.pad = 0;
                G.last[row >> 6] = rec;
            }
            if (G.next && valid) {
                const unsigned long long earlier = (1ull << lane) - 1;
                const bool dh = (h >> lane) & 1, dl = (l >> lane) & 1;
                const unsigned long long mine = dh ? (dl ? mask[3] : mask[2]) : (dl ? mask[1] : mask[0]);
                const uint32_t to = dh ? (dl ? at[3] + run[3] : at[2] + run[2]) : (dl ? at[1] + run[1] : at[0] + run[0]);
                const uint32_t from = dh ? (dl ? first[3] : first[2]) : (dl ? first[1] : first[0]);
                const uint32_t dest = to + (uint32_t)__popcll(mine & earlier);
                G.next[dest] = x[j];
                const uint32_t nd = digit_of(x[j], G.value_mask, G.next_shift, G.next_digit_mask);
                const uint32_t d = (dh ? 2u : 0u) + (dl ? 1u : 0u), second = (dest >> G.rows_log) != from;
                atomicAdd(&next_count[d * 8 + second * 4 + nd], 1u);
            }
#pragma unroll
            for (int d = 0; d < 4; ++d) run[d] += (uint32_t)__popcll(mask[d]);
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            at[d] += tile_count[d];
            rel[d] += tile_count[d];
            before[d] += tile_count[d];
        }
    }
    if (G.next) {
        __syncthreads();
        if (t < 32) {
            const uint32_t c = next_count[t];
            const int d = t >> 3;
            const uint32_t from = d == 0 ? first[0] : d == 1 ? first[1] : d == 2 ? first[2] : first[3];
            if (c) atomicAdd(&G.hist_next[(from + ((t >> 2) & 1)) * 4 + (t & 3)], c);
        }
    } else if (blk == 0) {
        uint32_t any = 0;
        for (int i = t; i < G.blocks; i += kBuildThreads) any |= G.bad[i];
        if (any) atomicOr(&wrong, 1u);
        __syncthreads();
        if (t == 0) *G.bad_out = wrong ? 1 : 0;
    }
}

// rows before i of a two-bit level whose digit is below d, and d
struct Counts {
    uint32_t below, equal;
};
__device__ inline Counts rank4(const Rank4 *rec, const uint4 *super, uint32_t i, uint32_t d)
{
    const Rank4 r = rec[i >> 5];
    const uint32_t lt = (1u << (i & 31)) - 1;
    const uint32_t b1 = (uint32_t)r.counts & kCountMask, b2 = (uint32_t)(r.counts >> kCountBits) & kCountMask,
                   b3 = (uint32_t)(r.counts >> (2 * kCountBits));
    uint32_t s1 = 0, s2 = 0, s3 = 0;
    if (super) {
        const uint4 s = super[i >> kSuperLog];
        s1 = s.x, s2 = s.y, s3 = s.z;
    }
    // rows before i with a digit below 1, 2, 3
    const uint32_t c1 = s1 + b1 + __popc(~(r.hi | r.lo) & lt), c2 = s2 + b2 + __popc(~r.hi & lt),
                   c3 = s3 + b3 + __popc(~(r.hi & r.lo) & lt);
    const uint32_t below = d == 0 ? 0 : d == 1 ? c1 : d == 2 ? c2 : c3;
    const uint32_t upto = d == 0 ? c1 : d == 1 ? c2 : d == 2 ? c3 : i;
    return {below, upto - below};
}

__device__ inline uint32_t rank0(const Rank2 *wk, uint32_t i)
{
    const Rank2 r = wk[i >> 6];
    return r.zeros_before + (uint32_t)__popcll(~r.bits & ((1ull << (i & 63)) - 1));
}

__global__ void index_query_kernel(IndexView I, int kind, int32_t m, int32_t n, const int32_t *q0, const int32_t *q1,
                                   int32_t nq, int32_t *out)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nq) return;
    Window w;
    if (!query_window(kind, m, n, q0[q], q1[q], w)) {
        out[q] = -1;
        return;
    }
    uint32_t s = (uint32_t)(w.r0 < I.size ? w.r0 : I.size), e = (uint32_t)I.size;
    const int64_t c = w.c0 + 1;   // values are stored shifted by one
    uint32_t cnt = 0;
    if (s >= e || c <= 0) {
        cnt = 0;
    } else if (c >= ((int64_t)1 << I.bits)) {
        cnt = e - s;
    } else {
        for (int k = 0; k < I.quads && s < e; ++k) {
            const Rank4 *rec = I.rec + k * I.w4;
            const uint4 *super = I.supers > 1 ? I.super + k * I.supers : nullptr;
            const uint32_t d = (uint32_t)(c >> (I.bits - 2 - 2 * k)) & 3;
            const Counts cs = rank4(rec, super, s, d), ce = rank4(rec, super, e, d);
            const uint4 total = I.totals[k];
            const uint32_t base = d == 0 ? 0 : d == 1 ? total.x : d == 2 ? total.y : total.z;
            cnt += ce.below - cs.below;
            s = base + cs.equal;
            e = base + ce.equal;
        }
        if (I.bits % 2 && s < e && (c & 1)) cnt += rank0(I.last, e) - rank0(I.last, s);
    }
    out[q] = w.score ? w.base - (int32_t)cnt : (int32_t)cnt;
}

}  // namespace lcsq

using namespace lcsq;

static int launch_status() { return hipGetLastError() == hipSuccess ? 0 : LCS_EIO; }

int lcsq_launch_scan(const int32_t *perm, int32_t size, int kind, int32_t m, int32_t n, const int32_t *q0,
                     const int32_t *q1, int32_t nq, int32_t *out, hipStream_t s)
{
    if (nq <= 0) return 0;
    const int blocks = (int)(((int64_t)nq * 64 + 255) / 256);
    hipLaunchKernelGGL(scan_kernel, dim3(blocks), dim3(256), 0, s, perm, size, kind, m, n, q0, q1, nq, out);
    return launch_status();
}

int lcsq_launch_index_build(const int32_t *perm, const IndexView &I, int32_t *scratch, hipStream_t s)
{
    if (I.size <= 0) return 0;
    const int nb = build_blocks(I.size);
    const size_t padded = ((size_t)I.size + 3) & ~(size_t)3;
    int32_t *buf[2] = {scratch, scratch + padded};
    uint4 *hist = (uint4 *)(scratch + 2 * padded);   // of this level, the next and the one after, in turn
    uint32_t *bad = (uint32_t *)(hist + 3 * (size_t)nb);
    LevelArgs G{};
    G.size = I.size;
    G.rows_log = build_rows_log(I.size);
    G.blocks = nb;
    G.value_mask = (uint32_t)(((uint64_t)1 << I.bits) - 1);
    G.bad = bad;
    G.bad_out = (int32_t *)(bad + nb);
    const int levels = I.quads + I.bits % 2;
    const auto shift_of = [&](int k) { return k < I.quads ? I.bits - 2 - 2 * k : 0; };
    const auto mask_of = [&](int k) { return k < I.quads ? 3u : 1u; };
    hipLaunchKernelGGL(index_prep_kernel, dim3(nb), dim3(kBuildThreads), 0, s, perm, I.size, G.rows_log, G.value_mask,
                       shift_of(0), mask_of(0), hist, hist + nb, bad);
    for (int k = 0; k < levels; ++k) {
        G.A = k ? buf[(k - 1) & 1] : perm;
        G.add = k ? 0 : 1;
        G.next = k + 1 < levels ? buf[k & 1] : nullptr;
        G.hist = (const uint32_t *)(hist + (k % 3) * (size_t)nb);
        G.hist_next = (uint32_t *)(hist + ((k + 1) % 3) * (size_t)nb);
        G.hist_after = k + 2 < levels ? hist + ((k + 2) % 3) * (size_t)nb : nullptr;
        G.rec = k < I.quads ? I.rec + k * I.w4 : nullptr;
        G.last = I.last;
        G.super = I.super + (k < I.quads ? k * I.supers : 0);
        G.totals = I.totals + k;
        G.words = k < I.quads ? I.w4 : I.w2;
        G.shift = shift_of(k);
        G.digit_mask = mask_of(k);
        G.next_shift = shift_of(k + 1);
        G.next_digit_mask = mask_of(k + 1);
        hipLaunchKernelGGL(index_level_kernel, dim3(nb), dim3(kBuildThreads), 0, s, G);
    }
    return launch_status();
}

int lcsq_launch_index_query(const IndexView &I, int kind, int32_t m, int32_t n, const int32_t *q0, const int32_t *q1,
                            int32_t nq, int32_t *out, hipStream_t s)
{
    if (nq <= 0) return 0;
    hipLaunchKernelGGL(index_query_kernel, dim3((unsigned)(((int64_t)nq + 255) / 256)), dim3(256), 0, s, I, kind, m, n,
                       q0, q1, nq, out);
    return launch_status();
}
