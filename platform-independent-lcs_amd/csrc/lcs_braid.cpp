// lcs_braid_multiply: staggered_multiply<RowGlue> of the reference
// (src/braid_multiplication.hpp:273-406) on the GPU, host pointers.
#include <hip/hip_runtime.h>

#include <cstring>
#include <vector>

#include "braid_kernels.h"
#include "lcs_hip.h"
#include "lcs_internal.h"

using namespace lcs;

namespace {
// From kBranchMin entries the byte table misses every cache, and a branch on
// what an earlier value stored lets the loads run ahead of the stores (2^24
// entries 7.9 ms each with it, 8.8 without; 2^26 314 and 365); below, the loop
// without it is the faster one (65000 entries 46 and 59 us).
constexpr int32_t kBranchMin = 1 << 24;
bool is_permutation(const int32_t *x, int32_t n)
{
    std::vector<unsigned char> seen((size_t)n, 0);
    if (n >= kBranchMin) {
        for (int32_t i = 0; i < n; ++i) {
            if (x[i] < 0 || x[i] >= n || seen[(size_t)x[i]]) return false;
            seen[(size_t)x[i]] = 1;
        }
        return true;
    }
    unsigned twice = 0;
    for (int32_t i = 0; i < n; ++i) {
        const uint32_t v = (uint32_t)x[i];
        if (v >= (uint32_t)n) return false;
        twice |= seen[v];
        seen[v] = 1;
    }
    return twice == 0;
}
}  // namespace

extern "C" int lcs_braid_multiply(lcs_ctx *ctx, const int32_t *p_row_to_col, int32_t p_size,
                                  const int32_t *q_row_to_col, int32_t q_size, int32_t k, int32_t row_glue,
                                  int32_t *out_row_to_col)
{
    if (!ctx || p_size < 0 || q_size < 0 || k < 0 || k > p_size || k > q_size) return LCS_EINVAL;
    if ((p_size && !p_row_to_col) || (q_size && !q_row_to_col)) return LCS_EINVAL;
    const int32_t out_size = p_size + q_size - k;
    if (out_size && !out_row_to_col) return LCS_EINVAL;
    if (!is_permutation(p_row_to_col, p_size) || !is_permutation(q_row_to_col, q_size)) return LCS_EINVAL;
    if (k > kMaxCoreK) return LCS_ERANGE;
    if (out_size == 0) return LCS_OK;
    if (hipSetDevice(ctx->device) != hipSuccess) return LCS_EIO;
    const size_t io_words = (size_t)p_size + q_size + out_size;
    size_t words = io_words + lcsb_multiply_ws_words(p_size, q_size, k) + 16;
    // kept between calls: with it, the staged copies and the results returned
    // uncopied, a product with k = 65000 fell from 430 to 320 us
    DevBuf buf = ctx->scratch.take(words * 4, kKeptMax);
    int rc = buf.reserve(ctx, words * 4);
    const bool in_lds = rc == LCS_ENOMEM;   // a workspace that may still fit
    if (in_lds) {
        words = io_words + lcsb_multiply_ws_words(p_size, q_size, k, true);
        rc = buf.reserve(ctx, words * 4);
    }
    if (rc) return rc;
    int32_t *dp = (int32_t *)buf.ptr, *dq = dp + p_size, *dout = dq + q_size, *dws = dout + out_size;
    hipStream_t s = ctx->stream;
    // dp, dq and dout lie side by side: one copy in and one out, through pinned memory up to kPinnedMax bytes
    const size_t in_words = (size_t)p_size + q_size, io_bytes = (in_words + out_size) * 4;
    int32_t *pin = io_bytes <= kPinnedMax ? (int32_t *)pinned_staging(ctx, io_bytes) : nullptr;
    bool ok;
    if (pin) {
        if (p_size) std::memcpy(pin, p_row_to_col, (size_t)p_size * 4);
        if (q_size) std::memcpy(pin + p_size, q_row_to_col, (size_t)q_size * 4);
        ok = hipMemcpyAsync(dp, pin, in_words * 4, hipMemcpyHostToDevice, s) == hipSuccess;
    } else {
        ok = (!p_size || hipMemcpyAsync(dp, p_row_to_col, (size_t)p_size * 4, hipMemcpyHostToDevice, s) == hipSuccess) &&
             (!q_size || hipMemcpyAsync(dq, q_row_to_col, (size_t)q_size * 4, hipMemcpyHostToDevice, s) == hipSuccess);
    }
    ctx->pending_timing = false;   // its events are recorded anew
    if (!ok || hipEventRecord(ctx->ev0, s) != hipSuccess) { buf.release(ctx); return LCS_EIO; }
    rc = lcsb_multiply_device(dp, p_size, dq, q_size, k, row_glue ? 1 : 0, dout, dws, s, in_lds);
    if (!rc) {
        (void)hipEventRecord(ctx->ev1, s);
        ok = hipMemcpyAsync(pin ? pin + in_words : out_row_to_col, dout, (size_t)out_size * 4, hipMemcpyDeviceToHost, s) == hipSuccess &&
             hipStreamSynchronize(s) == hipSuccess;
        rc = ok ? LCS_OK : LCS_EIO;
        float ms = 0.f;
        if (ok && pin) std::memcpy(out_row_to_col, pin + in_words, (size_t)out_size * 4);
        if (ok && hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess) ctx->last_kernel_ms = ms;
    }
    if (rc) buf.release(ctx);   // waits for what was enqueued
    ctx->scratch.give(ctx, buf);
    return rc;
}
