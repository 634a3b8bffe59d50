// Launch interface of the steady-ant kernels (internal to the library).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// Largest padded core (2^L): cores up to 2^10 run in one workgroup's LDS,
// larger ones over the whole GPU (their grid of boxes is sized for nodes of
// at most 2^22 points).  With in_lds a core of 2^11 runs in LDS as well, with
// a workspace that is 65 KB smaller (k = 2048: 71 us over the GPU, 86 in LDS).
constexpr int kMaxCoreL = 22;
constexpr int kMaxCoreK = 1 << kMaxCoreL;

size_t lcsb_core_scratch_words(int32_t k, bool in_lds);
// One-time kernel attribute setup (called by the launches; call it before
// capturing a launch sequence in a graph).
int lcsb_init(void);
int lcsb_core_L(int32_t k);
size_t lcsb_multiply_ws_words(int32_t p_size, int32_t q_size, int32_t k, bool in_lds = false);
// staggered_multiply<row_glue>(p, q, k) on device pointers.
int lcsb_multiply_device(const int32_t *p, int32_t p_size, const int32_t *q, int32_t q_size, int32_t k,
                         int32_t row_glue, int32_t *out, int32_t *ws, hipStream_t stream, bool in_lds = false);
// Several independent products; their cores share one launch.  ws of each
// holds lcsb_multiply_ws_words(p_size, q_size, k) words.
struct MulSpec {
    const int32_t *p;
    int32_t p_size;
    const int32_t *q;
    int32_t q_size, k, row_glue;
    int32_t *out, *ws;
};
int lcsb_multiply_many_device(const MulSpec *specs, int count, hipStream_t stream, bool in_lds = false);
