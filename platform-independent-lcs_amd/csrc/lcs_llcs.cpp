// Score-only LCS length (bit-parallel kernel) behind the C ABI; declarations
// in include/lcs_hip.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "lcs_hip.h"
#include "lcs_internal.h"
#include "llcs_kernels.h"

using namespace lcs;

namespace {

struct LlcsPair {
    const int32_t *a, *b;   // device
    int32_t m, n;
    int32_t *out;           // device int32
};

// Microseconds from the first band's start to the last band's end with blocks
// of 4 and of 2 columns: a band lags the one below by 64 blocks of skew, the
// chunk that a carry word fills, two chunks of prefetch and the word's trip
// (measured 390 columns at 4, 260 at 2), and bands beyond the resident ones run
// in later rounds.  A column takes 15.0 ns at 4 and 17.0 at 2.
struct PipelineUs {
    double of4, of2;
    double best() const { return std::min(of4, of2); }
};
PipelineUs pipeline_us(int32_t rows, int32_t cols, int64_t resident)
{
    const int64_t bands = lcsl::llcs_nbands(rows);
    const double rounds = bands <= resident ? 1.0 : (double)((bands + resident - 1) / resident);
    return {(rounds * ((double)cols + lcsl::kWave * 4) + (double)bands * 390.0) * 0.0150,
            (rounds * ((double)cols + lcsl::kWave * 2) + (double)bands * 260.0) * 0.0170};
}

// LDS of a CU, and the bands it holds at once: one per SIMD, fewer when the
// match-mask tables fill the LDS
constexpr int kCuLdsBytes = 160 * 1024;
int bands_per_cu(int sigma, bool pairs)
{
    return (int)std::min<size_t>(4, kCuLdsBytes / lcsl::llcs_lds_bytes(sigma, pairs));
}

// Enqueues one launch over `pairs` on `s`: the longer-pipelined orientation
// is chosen per pair (LCS is symmetric).  Rings and descriptors live in the
// context's buffers, error words after the descriptors.
static int enqueue_llcs_ws(lcs_ctx *ctx, const std::vector<LlcsPair> &pairs, int32_t sigma, hipStream_t s);

int enqueue_llcs(lcs_ctx *ctx, const std::vector<LlcsPair> &pairs, int32_t sigma, hipStream_t s)
{
    int rc = ws_acquire(ctx, s);
    if (rc) return rc;
    rc = enqueue_llcs_ws(ctx, pairs, sigma, s);
    const int rc2 = ws_release(ctx, s);
    ctx->ws_reserved = 0;
    return rc ? rc : rc2;
}

static int enqueue_llcs_ws(lcs_ctx *ctx, const std::vector<LlcsPair> &pairs, int32_t sigma, hipStream_t s)
{
    const int np = (int)pairs.size();
    if (np == 0) return LCS_OK;
    // tables of column pairs while every band still has its SIMD, or the tables
    // are small enough for four to a CU: of 5 to 9 symbols, 20 pairs of 100000
    // take 3.87 ms with them and 2.34 without
    bool two_columns = sigma <= lcsl::kMaxPairSigma;
    int64_t bands_a = 0, bands_b = 0;
    for (const LlcsPair &P : pairs) {
        bands_a += lcsl::llcs_nbands(P.m);
        bands_b += lcsl::llcs_nbands(P.n);
    }
    const int tables = two_columns ? bands_per_cu(sigma, true) : 0;
    if (tables < 4 && std::min(bands_a, bands_b) > (int64_t)ctx->num_cus * tables) two_columns = false;
    const int64_t resident = (int64_t)ctx->num_cus * bands_per_cu(sigma, two_columns);
    std::vector<lcsl::LlcsDesc> descs((size_t)np);
    size_t ring_words = 0, code_bytes = 0;
    int max_words = 0;
    double us[2] = {0.0, 0.0};   // blocks of 4, of 2: the slowest pair
    int64_t all_bands = 0;
    for (int p = 0; p < np; ++p) {
        const LlcsPair &P = pairs[(size_t)p];
        const PipelineUs as_given = pipeline_us(P.m, P.n, resident), swapped = pipeline_us(P.n, P.m, resident);
        const bool swap = swapped.best() < as_given.best();
        lcsl::LlcsDesc &D = descs[(size_t)p];
        D = lcsl::LlcsDesc{};
        D.rows = swap ? P.b : P.a;
        D.cols = swap ? P.a : P.b;
        D.nrows = swap ? P.n : P.m;
        D.ncols = swap ? P.m : P.n;
        // the widest b of the ABI; the band loop itself counts chunks
        if (D.ncols > 0x7fffffff - 4096) return LCS_ERANGE;
        us[0] = std::max(us[0], swap ? swapped.of4 : as_given.of4);
        us[1] = std::max(us[1], swap ? swapped.of2 : as_given.of2);
        all_bands += lcsl::llcs_nbands(D.nrows);
        D.out = P.out;
        ring_words += 2 * (size_t)lcsl::llcs_slot_words(D.ncols);
        code_bytes += lcsl::llcs_code_bytes(D.ncols, two_columns);
        max_words = std::max(max_words, lcsl::llcs_nwords(D.ncols));
    }
    ctx->ws_reserved = 0;
    int rc = reserve_ws(ctx, kWsRing, ring_words * sizeof(unsigned long long));
    if (rc) return rc;
    std::vector<int2> tasks;
    for (int p = 0; p < np; ++p)
        for (int32_t g = 0; g < lcsl::llcs_nbands(descs[(size_t)p].nrows); ++g) tasks.push_back(make_int2(p, g));
    const size_t desc_bytes = sizeof(lcsl::LlcsDesc) * (size_t)np, task_bytes = sizeof(int2) * tasks.size();
    // the error words travel with the descriptors, as zeros
    const size_t err_off = (desc_bytes + task_bytes + 255) / 256 * 256;
    if ((rc = ctx->descs.reserve(ctx, err_off + 4 * (size_t)np + 256))) return rc;
    // a budget that does not hold the codes: the bands read the symbols themselves
    const bool coded = reserve_ws(ctx, kWsSym8, code_bytes) == LCS_OK;
    uint8_t *codes = coded ? (uint8_t *)ctx->sym8.ptr : nullptr;
    unsigned long long *ring = (unsigned long long *)ctx->ring.ptr;
    int32_t *err = (int32_t *)((unsigned char *)ctx->descs.ptr + err_off);
    for (int p = 0; p < np; ++p) {
        descs[(size_t)p].ring = ring;
        ring += 2 * (size_t)lcsl::llcs_slot_words(descs[(size_t)p].ncols);
        descs[(size_t)p].codes = codes;
        if (coded) codes += lcsl::llcs_code_bytes(descs[(size_t)p].ncols, two_columns);
        descs[(size_t)p].err = err + p;
    }
    std::vector<unsigned char> blob(err_off + 4 * (size_t)np, 0);
    std::memcpy(blob.data(), descs.data(), desc_bytes);
    if (task_bytes) std::memcpy(blob.data() + desc_bytes, tasks.data(), task_bytes);
    if ((rc = upload(ctx, ctx->descs.ptr, blob.data(), blob.size(), s))) return rc;
    lcsl::LlcsArgs A{};
    A.descs = (const lcsl::LlcsDesc *)ctx->descs.ptr;
    A.tasks = (const int2 *)((unsigned char *)ctx->descs.ptr + desc_bytes);
    A.ntasks = (int32_t)tasks.size();
    A.sigma = sigma;
    A.ticket = ctx->ctrl;
    A.abort_flag = ctx->ctrl + 1;
    A.sticky = ctx->ctrl + kStickyWord;
    A.timeout_ticks = ctx->timeout_ticks;
    A.trace = ctx->band_trace;
    A.trace_cap = ctx->band_trace_cap;
    A.pairs = two_columns;
    A.codes = coded;
    // more bands than SIMDs over several pairs: the time per column counts
    A.block = us[1] < us[0] && (np == 1 || all_bands <= resident) ? 2 : 4;
    const int blocks = (int)std::min<int64_t>((int64_t)tasks.size(), resident);
    // as much LDS per band as leaves each CU its share of them: the dispatcher
    // then spreads the bands over the CUs, and a band has its SIMD to itself
    const int share = std::max(1, (blocks + ctx->num_cus - 1) / ctx->num_cus);
    const int lds = std::max((int)lcsl::llcs_lds_bytes(sigma, two_columns), kCuLdsBytes / share / 512 * 512);
    return lcsl_launch(A, A.descs, np, max_words, blocks, lds, s) == 0 ? LCS_OK : LCS_EIO;
}

bool valid_sigma(int32_t sigma) { return sigma >= 1 && sigma <= lcsl::kMaxSigma; }

// Runs host pairs: copies the strings in, launches, copies the lengths out.
int run_host(lcs_ctx *ctx, int32_t npairs, const int32_t *a_all, const int64_t *a_off, const int32_t *m,
             const int32_t *b_all, const int64_t *b_off, const int32_t *n, int32_t sigma, int32_t *out)
{
    if (hipSetDevice(ctx->device) != hipSuccess) return LCS_EIO;
    int64_t a_len = 0, b_len = 0;
    for (int32_t p = 0; p < npairs; ++p) {
        a_len = std::max<int64_t>(a_len, a_off[p] + m[p]);
        b_len = std::max<int64_t>(b_len, b_off[p] + n[p]);
    }
    int rc = ctx->strings.reserve(ctx, (size_t)std::max<int64_t>(a_len + b_len, 1) * 4);
    if (!rc) rc = ctx->results.reserve(ctx, (size_t)std::max(npairs, 1) * 4);
    if (rc) return rc;
    hipStream_t s = ctx->stream;
    int32_t *da = (int32_t *)ctx->strings.ptr, *db = da + a_len, *dout = (int32_t *)ctx->results.ptr;
    if (a_len && hipMemcpyAsync(da, a_all, (size_t)a_len * 4, hipMemcpyHostToDevice, s) != hipSuccess) return LCS_EIO;
    if (b_len && hipMemcpyAsync(db, b_all, (size_t)b_len * 4, hipMemcpyHostToDevice, s) != hipSuccess) return LCS_EIO;
    std::vector<LlcsPair> pairs((size_t)npairs);
    for (int32_t p = 0; p < npairs; ++p)
        pairs[(size_t)p] = LlcsPair{da + a_off[p], db + b_off[p], m[p], n[p], dout + p};
    if (hipEventRecord(ctx->ev0, s) != hipSuccess) return LCS_EIO;
    if ((rc = enqueue_llcs(ctx, pairs, sigma, s))) return rc;
    if (hipEventRecord(ctx->ev1, s) != hipSuccess) return LCS_EIO;
    ctx->time_from = ctx->ev0;
    ctx->time_to = ctx->ev1;
    ctx->pending_timing = true;
    if (hipMemcpyAsync(out, dout, (size_t)npairs * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return LCS_EIO;
    if ((rc = check_abort(ctx))) return rc;
    for (int32_t p = 0; p < npairs; ++p)
        if (out[p] < 0) return LCS_ERANGE;
    return LCS_OK;
}

}  // namespace

extern "C" int lcs_llcs(lcs_ctx *ctx, const int32_t *a, int32_t m, const int32_t *b, int32_t n, int32_t sigma,
                        int32_t *llcs)
{
    if (!ctx || !llcs || m < 0 || n < 0 || (m && !a) || (n && !b) || !valid_sigma(sigma)) return LCS_EINVAL;
    const int64_t zero = 0;
    return run_host(ctx, 1, a, &zero, &m, b, &zero, &n, sigma, llcs);
}

extern "C" int lcs_llcs_device(lcs_ctx *ctx, const int32_t *d_a, int32_t m, const int32_t *d_b, int32_t n,
                               int32_t sigma, int32_t *d_llcs)
{
    if (!ctx || !d_llcs || m < 0 || n < 0 || (m && !d_a) || (n && !d_b) || !valid_sigma(sigma)) return LCS_EINVAL;
    if (hipSetDevice(ctx->device) != hipSuccess) return LCS_EIO;
    hipStream_t s = ctx->stream;
    std::vector<LlcsPair> pairs{LlcsPair{d_a, d_b, m, n, d_llcs}};
    if (hipEventRecord(ctx->ev0, s) != hipSuccess) return LCS_EIO;
    int rc = enqueue_llcs(ctx, pairs, sigma, s);
    if (rc) return rc;
    if (hipEventRecord(ctx->ev1, s) != hipSuccess) return LCS_EIO;
    ctx->time_from = ctx->ev0;
    ctx->time_to = ctx->ev1;
    ctx->pending_timing = true;
    return LCS_OK;
}

extern "C" int lcs_llcs_batch(lcs_ctx *ctx, int32_t npairs, const int32_t *a_all, const int64_t *a_off,
                              const int32_t *m, const int32_t *b_all, const int64_t *b_off, const int32_t *n,
                              int32_t sigma, int32_t *out)
{
    if (!ctx || npairs < 0 || !valid_sigma(sigma)) return LCS_EINVAL;
    if (npairs == 0) return LCS_OK;
    if (!a_off || !m || !b_off || !n || !out) return LCS_EINVAL;
    for (int32_t p = 0; p < npairs; ++p)
        if (m[p] < 0 || n[p] < 0 || a_off[p] < 0 || b_off[p] < 0 || (m[p] && !a_all) || (n[p] && !b_all))
            return LCS_EINVAL;
    return run_host(ctx, npairs, a_all, a_off, m, b_all, b_off, n, sigma, out);
}
