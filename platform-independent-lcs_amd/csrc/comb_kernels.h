// Launch interface of the combing kernels (internal to the library).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// One comb problem: a (m symbols, row r holds a[r]) against b (n symbols),
// cut into bands of 64*tile_m rows.  Band g reads its top-edge strands from
// ring slot g&1 of E and writes its bottom edge to slot (g+1)&1; the prep
// kernel seeds slot 0, the extract kernel copies the last slot to v_out.
struct PairDesc {
    const int32_t *a;            // m symbols, original order
    const int32_t *b;            // n symbols
    const int32_t *h_in;         // nullable: initial h strands (reference order), else i
    const int32_t *v_in;         // nullable: initial v strands, else m + j
    int32_t *h_out;              // m strands, reference order (index m-1-r)
    int32_t *v_out;              // n strands
    unsigned long long *E;       // 2*n ring words (tag << 32 | strand) + 64 spare words
    int32_t m, n, nbands, tile_m;
    // Nullable: b as byte symbols (lcsk_launch_sym8), read instead of b by
    // the band chains unless *sym8_flags has kSym8Bad.
    const uint32_t *sym8;
    const int32_t *sym8_flags;
    int32_t sym8_stride, pad;
    // Nullable, as are h_out and v_out: the pair's permutation (row_to_col,
    // m + n entries).
    int32_t *perm;
};

// One pair cut into GR x GC tiles of H rows and W columns (the last ones may
// be smaller), each combed from its own identity; described by value in the
// launch arguments, so that a single-pair call uploads nothing.  Tile (i, j)
// combs a[iH ..) against b[jW ..) with ring slot iGC + j of `pair.E` and the
// byte copies of strip j of `pair.sym8`.  With one tile the pair's own
// h_in, v_in, h_out, v_out and perm are used; with more, each tile writes only
// its permutation, at `perm` + perm_off(i, j).
struct TileGrid {
    PairDesc pair;
    int32_t H, W, GR, GC;
    int32_t *perm;
    int32_t *sym8_flags;   // pair.sym8_flags, cleared by the extract kernel for the next launch
    int32_t *status;       // nullable: receives the launch's abort flag
    __host__ __device__ int32_t rows(int32_t i) const { return pair.m - i * H < H ? pair.m - i * H : H; }
    __host__ __device__ int32_t cols(int32_t j) const { return pair.n - j * W < W ? pair.n - j * W : W; }
    __host__ __device__ int64_t perm_off(int32_t i, int32_t j) const
    {
        return (int64_t)i * ((int64_t)GC * H + pair.n) + (int64_t)j * (rows(i) + W);
    }
};

// Byte symbols of a string b of n symbols: four copies (stride words each,
// lcsk_sym8_stride(n)), copy j holding at byte x the symbol of column
// x + j - kSym8Pad as a byte (255 outside [0, n)).  A lane whose C-step
// window starts at byte x0 reads copy x0 % 4 from a word boundary.
constexpr int32_t kSym8Pad = 128;
// flags of a staged string: a symbol outside [0, 255]; a symbol 255, the
// padding of the copies; bit 8 + i: the symbol -1 - i (i < 24), so that a
// 32-bit chain can pad its rows with one of them that is absent
constexpr int32_t kSym8Bad = 1, kSym8Has255 = 2, kSym8RowPads = 24;
inline int32_t lcsk_sym8_stride(int32_t n) { return (int32_t)((((int64_t)n + 2 * kSym8Pad + 15) / 16) * 4); }
// Writes the four copies of b into `out` (4 * stride words) and b's flags.
int lcsk_launch_sym8(const int32_t *b, int32_t n, uint32_t *out, int32_t stride, int32_t *flags, hipStream_t stream);

// Whether a byte chain's bands keep one chunk more than they need between
// themselves and the band above (band_pass).  It costs 32 steps a band and
// spares up to half of every step, so it is for bands that are long beside
// their number, and long enough to fall out of step at all.  Median times
// without and with it: 8 bands of 6000 columns 103 and 108 us, of 8192 139 and
// 134, of 12000 209 and 181; 16 of 8192 176 and 159; 32 of 16384 477 and 306;
// 64 of 16384 404 and 395; 256 of 50000 1184 and 1367.
constexpr int kSlackMinColumns = 8192, kSlackColumnsPerBand = 384;
__host__ __device__ inline bool band_slack(int tile_m, int32_t nbands, int32_t n)
{
    return tile_m == 1 && n >= kSlackMinColumns && n / kSlackColumnsPerBand > nbands;
}

// Two pairs combed together by the 16-bit packed chain
// (LCS_VARIANT_PACKED16): pair q (0 = X, low halves; 1 = Y, high halves)
// reads a[q], b[q] (m_[q], n_[q] int32 symbols in [0, 0xfffd]) and writes
// h_out[q], v_out[q]; each has m_[q] + n_[q] <= 65535 and m_[q], n_[q] >= 1.
// m, n are the larger extents; the shorter pair is padded with rows and
// columns that never match and never swap.
struct CoupleDesc {
    const int32_t *a[2];
    const int32_t *b[2];
    int32_t *h_out[2];
    int32_t *v_out[2];
    int32_t m_[2], n_[2];
    unsigned long long *E;       // 2*n ring words (tag << 32 | Y strand << 16 | X strand) + 64 spare words
    int32_t m, n, nbands, tile_m;
    int32_t onehot;              // both pairs' symbols in [0, 15]: one-hot cells (1 << symbol per half)
};

// Words of ring a pair of n columns needs.
inline size_t lcsk_ring_words(int32_t n) { return 2 * (size_t)n + 64; }

// One persistent chain launch: waves take tickets in order; ticket t runs
// band tasks[t].y of pair tasks[t].x (group_w == 1), or bands
// group_w*tasks[t].y .. +group_w-1 in one workgroup (group_w > 1).  Tasks must list every band after the
// band above it (same pair), which makes every wait one on a resident wave.
struct ChainArgs {
    const PairDesc *pairs;       // the register chain and linked groups; null: the tiles of `grid`, task t being
                                 // band (or group) t / (GR GC) of tile t % (GR GC)
    const CoupleDesc *couples;   // the packed chain (tasks[t].x indexes couples)
    const int2 *tasks;
    int32_t ntasks;
    int32_t group_w;             // 1: one wave per task (register chain); W > 1: LDS groups of W bands
    unsigned *ticket;            // zeroed by the prep kernel
    unsigned *abort_flag;        // zeroed by the prep kernel
    unsigned long long timeout_ticks;  // 100 MHz realtime ticks per wait
    unsigned long long *trace;   // nullable: [2t] start, [2t+1] end of task t (realtime ticks)
    int32_t trace_cap;           // tasks the trace buffer holds
    int32_t poll_sleep;          // 1: a wave waiting for its inputs sleeps between polls (launches that
                                 // share SIMDs with other launches' waves)
    unsigned *sticky;            // nullable: the prep kernel ORs the abort flag into it before clearing it
    TileGrid grid;               // when pairs is null
};

// The same for the tiles of args.grid, with the byte copies of b (when
// grid.pair.sym8 is set) staged by the seeding kernel.
int lcsk_launch_grid(const ChainArgs &args, int grid_blocks, int block_threads, hipStream_t stream);
// Seeds the rings of pairs[0..npairs) and clears ticket/abort; then runs the
// chain for tile height tile_m; then extracts v_out.  All on `stream`.
int lcsk_launch_chain(const ChainArgs &args, const PairDesc *d_pairs, int npairs, int max_n, int tile_m,
                      int grid_blocks, int block_threads, hipStream_t stream);
// Strands (and, when perm is given, the permutation) of an empty grid (m == 0
// or n == 0).
int lcsk_launch_identity(int32_t *h_out, int32_t m, int32_t *v_out, int32_t n, hipStream_t stream,
                         int32_t *perm = nullptr);
// A string whose symbols the packed chain needs in [0, 0xfffd]: bit 0 of
// bad[item] is set when one is outside, bit 1 when one is above 15 (the
// one-hot cells then cannot take the pair).
struct SymbolRange {
    const int32_t *x;
    int32_t len, item;
};
int lcsk_launch_check16(const SymbolRange *d_ranges, int32_t nranges, int32_t *d_bad, int32_t nitems,
                        hipStream_t stream);
// The same sequence (seed, chain, extract) for couples of pairs combed by
// the 16-bit packed chain.
int lcsk_launch_chain16(const ChainArgs &args, const CoupleDesc *d_couples, int ncouples, int max_n, int tile_m,
                        int grid_blocks, int block_threads, hipStream_t stream);
// row_to_col of the permutation of each pair from its strands (m+n entries
// each, written at perm + perm_off[p]).
int lcsk_launch_from_strands(const PairDesc *d_pairs, int npairs, int max_len, int32_t *perm,
                             const int64_t *d_perm_off, hipStream_t stream);
// dst[0..count) = src[0..count) (a kernel, so it can sit in a captured graph).
int lcsk_launch_copy(int32_t *dst, const int32_t *src, long long count, hipStream_t stream);
// Strands from a permutation (row_to_col, size m+n): h_out[l] = row of col
// n+l, v_out[j] = row of col j.
// copy (nullable) receives r2c itself.
int lcsk_launch_strands_from_perm(const int32_t *r2c, int32_t m, int32_t n, int32_t *h_out, int32_t *v_out,
                                  int32_t *copy, hipStream_t stream);
