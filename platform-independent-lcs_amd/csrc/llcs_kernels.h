// Launch interface of the score-only bit-parallel LCS kernels (internal).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lcsl {

constexpr int kWave = 64;
constexpr int kWordRows = 32;                    // rows of the row string per lane
constexpr int kBandRows = kWave * kWordRows;     // 2048 rows per band (one wave)
constexpr int kChunk = 32;                       // columns per carry word
constexpr int kMaxBlock = 4;                     // columns a lane takes per turn: 4 or 2
constexpr int kMaxSigma = 200;                   // one table row per symbol, 51 KB of LDS
// Up to this alphabet a table row can serve two columns: (sigma + 1)^2 rows of
// 512 bytes, lanes 0 .. 31 in one half of the table and 32 .. 63 in the other,
// 128 rows of 256 bytes on (58 KB at 9).  A column then takes 15.0 ns instead
// of 17.3, but above 4 symbols a CU's LDS holds fewer than four such tables.
constexpr int kMaxPairSigma = 9;

// One LCS-length problem: `rows` (nrows symbols) is cut into bands of 2048
// rows, one 32-bit word per lane; `cols` (ncols symbols) streams through the
// band as codes.  Band g reads the carry words of band g-1 from ring slot g&1
// (tag g) and writes its own to slot (g+1)&1; the seeding kernel fills slot 0
// with empty words of tag 0 for band 0.  A slot has a word per 32 columns and
// two that the last prefetches read.
struct LlcsDesc {
    const int32_t *rows;
    const int32_t *cols;
    int32_t nrows, ncols;
    unsigned long long *ring;    // 2 * llcs_slot_words(ncols) words (tag << 32 | 32 carry bits)
    uint8_t *codes;              // llcs_code_bytes(ncols, pairs), 16-byte aligned; null in a launch without codes
    int32_t *out;                // LCS length (zeroed by the prep kernel); -1 on a symbol outside [0, sigma)
    int32_t *err;                // zero before the launch; set on a symbol outside [0, sigma)
};

inline int32_t llcs_nbands(int32_t nrows) { return (int32_t)(((int64_t)nrows + kBandRows - 1) / kBandRows); }
__host__ __device__ inline int32_t llcs_nwords(int32_t ncols) { return ncols > 0 ? (ncols - 1) / kChunk + 1 : 0; }
__host__ __device__ inline int64_t llcs_slot_words(int32_t ncols) { return ncols > 0 ? (int64_t)llcs_nwords(ncols) + 2 : 0; }
// Chunks between the column word q of a band and the one in which it is whole:
// with blocks of B columns a chunk has 32 / B turns and lane 63 takes block b
// in turn b + 63, so word q is whole after the last turn but one of chunk q +
// word_lag(B).
__host__ __device__ constexpr int word_lag(int B) { return kWave * B / kChunk; }
// Codes: 64 blocks of padding (lane 63 starts 63 blocks back), the string, and
// padding up to the last prefetch (three chunks past the last, in steps of
// six); a byte per column, or per two.
constexpr int kFrontPad = kWave * kMaxBlock;   // columns
__host__ __device__ inline int64_t llcs_code_columns(int32_t nwords)
{
    return kFrontPad + (int64_t)kChunk * (nwords + word_lag(kMaxBlock) + 10);
}
inline size_t llcs_code_bytes(int32_t ncols, bool pairs)
{
    return ((size_t)llcs_code_columns(llcs_nwords(ncols)) / (pairs ? 2 : 1) + 31) & ~(size_t)15;
}

struct LlcsArgs {
    const LlcsDesc *descs;
    const int2 *tasks;           // (pair, band), every band after the band below it
    int32_t ntasks;
    int32_t sigma;               // symbols in [0, sigma), sigma <= kMaxSigma
    unsigned *ticket;            // zeroed by the prep kernel
    unsigned *abort_flag;        // zeroed by the prep kernel
    unsigned long long timeout_ticks;
    unsigned long long *trace;   // nullable: [2t] start, [2t+1] end of task t (realtime ticks)
    int32_t trace_cap;
    int32_t block;               // columns per turn, 4 or 2
    int32_t pairs;               // table rows and code bytes serve two columns (sigma <= kMaxPairSigma)
    int32_t codes;               // 0: no descriptor has codes, the bands read `cols`
    unsigned *sticky;            // nullable: the prep kernel ORs the abort flag into it before clearing it
};

// LDS of one band: the match-mask table, a zero row for the padding included
inline size_t llcs_lds_bytes(int sigma, bool pairs)
{
    return pairs ? (size_t)32768 + (size_t)(sigma + 1) * (sigma + 1) * 256 : (size_t)(sigma + 1) * 256;
}

}  // namespace lcsl

// Clears outputs, ticket and abort flag, invalidates every ring word and
// writes the codes; runs the band chain (lds_bytes >= llcs_lds_bytes(sigma, pairs)
// per workgroup); marks pairs with a bad symbol (-1).
int lcsl_launch(const lcsl::LlcsArgs &args, const lcsl::LlcsDesc *d_descs, int npairs, int max_words,
                int grid_blocks, int lds_bytes, hipStream_t stream);
