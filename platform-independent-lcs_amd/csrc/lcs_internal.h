// Internal state of a context (shared by the C ABI translation units).
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "comb_kernels.h"
#include "lcs_hip.h"

namespace lcs {

// A grow-only device buffer whose bytes count against the context's budget.
struct DevBuf {
    void *ptr = nullptr;
    size_t bytes = 0;
    int reserve(lcs_ctx *ctx, size_t want);
    void release(lcs_ctx *ctx);
};

// Device memory kept between calls that each need some for their own time.  A
// caller takes it, reserves what it needs, and gives it back once the device
// is done with it; what is kept is at most kKeptMax bytes and is freed when
// another buffer needs its share of the budget or of the device's memory.
// A thread other than the context's may give back, under ContextLife.
constexpr size_t kKeptMax = (size_t)256 << 20;
struct KeptBuf {
    std::mutex mu;
    DevBuf buf;
    DevBuf take(size_t at_least, size_t at_most);   // empty when what is kept does not fit
    void give(lcs_ctx *ctx, DevBuf &b);
    void trim(lcs_ctx *ctx);
};

// Whether a context is there still, for what may be dropped after it and on
// another thread (an index, by whoever collects it).  The lock is held for a
// whole give-back, and by lcs_ctx_destroy to mark the context gone.
struct ContextLife {
    std::mutex mu;
    bool alive = true;
};

struct Extras;  // batch / server resources, created on first use

// Pinned host staging for descriptor uploads.  `done` is recorded after the
// last copy out of `pinned`; the next upload through the same staging waits
// for it before rewriting the buffer.
struct Staging {
    void *pinned = nullptr;
    size_t bytes = 0;
    hipEvent_t done = nullptr;
    int init();
    void destroy();
};

// A chain launch whose descriptors are already on the device.  Between
// build_launch and rebase_launch, args.pairs and args.tasks hold byte
// offsets into the host descriptor blob instead of device addresses.
struct PreparedLaunch {
    ChainArgs args{};
    int blocks = 0, threads = 0, npairs = 0, max_n = 0, tile_m = 0;
    bool packed = false;   // args.couples (the 16-bit packed chain), npairs couples
};

// Schedule selection state of one mode (LCS_TUNE_SINGLE / LCS_TUNE_BATCH):
// the autotune table, the attached cost model and the autotune-on-miss
// candidates.  Model and on-miss choices are memoised per shape.
struct TunedShape {
    int32_t m, n;
    lcs_schedule s;
};
struct Selector {
    std::vector<TunedShape> table;
    lcs_mlp *model = nullptr;                 // not owned; same context
    std::vector<lcs_schedule> model_cands;
    std::vector<lcs_schedule> miss_cands;     // empty: no autotune on a miss
    int32_t miss_reps = 1;
    std::map<std::tuple<int32_t, int32_t, int32_t>, std::pair<lcs_schedule, int>> memo;
};

}  // namespace lcs

namespace lcs {
// ctrl word that collects the abort flags of finished launches (folded in by
// each launch's prep kernel); lcs_ctx_status reads and clears it
constexpr int kStickyWord = 63;
// ctrl word of the byte-symbol flags of single-pair launches; zero between
// launches (each one's extract kernel clears it)
constexpr int kSym8FlagWord = 62;
constexpr int kZeroWord = 61;   // always zero
}  // namespace lcs

struct lcs_ctx {
    int device = 0;
    int num_cus = 0;
    std::string name, arch;
    size_t budget = 0;
    std::atomic<size_t> held{0};         // device bytes; freed on any thread, reserved on the context's
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // around the band-chain launch (seed, chain, extract) of the last
    // single-pair call: its time alone, without merges or conversions
    hipEvent_t evc0 = nullptr, evc1 = nullptr;
    bool chain_timed = false;
    unsigned *ctrl = nullptr;            // [0] ticket, [1] abort flag, rest spare
    unsigned long long timeout_ticks = 500000000ull;  // 5 s at 100 MHz
    double last_kernel_ms = 0.0;
    bool pending_timing = false;
    // events around the last timed call's kernels (of ev0, ev1, evc0, evc1)
    hipEvent_t time_from = nullptr, time_to = nullptr;
    lcs::DevBuf ring, strings, results, descs, strip_ws;   // strings, results: of the host calls
    void *pinned = nullptr;              // host staging of strings and results, at most lcs::kPinnedMax bytes
    size_t pinned_bytes = 0;
    lcs::KeptBuf scratch;                // braid products and index builds
    lcs::KeptBuf index_mem;              // the memory of a destroyed index
    std::shared_ptr<lcs::ContextLife> life = std::make_shared<lcs::ContextLife>();
    lcs::DevBuf sym8;                    // byte copies of b and their range flag (single-pair chains)
    unsigned ws_reserved = 0;            // bit per lcs::PairWs: reserved by the single-pair call being enqueued
    // The shared workspace (ring, descriptors, ctrl words) is used by one
    // launch at a time: a call on another stream first waits for ws_done,
    // recorded after the last call's kernels on ws_stream.
    hipEvent_t ws_done = nullptr;
    hipStream_t ws_stream = nullptr;
    lcs::Staging staging;                // descriptor uploads of the context's own calls
    lcs::Extras *extras = nullptr;
    lcs::Selector select[2];             // schedule selection per mode (single pair, batch)
    unsigned long long *band_trace = nullptr;  // device buffer set by lcs_debug_band_trace
    int32_t band_trace_cap = 0;
};

namespace lcs {
// Reserves one of the single-pair workspaces for the call being enqueued; those
// that it has not reserved are freed where the budget or the device runs short.
enum PairWs { kWsRing, kWsStrips, kWsSym8 };
int reserve_ws(lcs_ctx *ctx, PairWs which, size_t bytes);
int enqueue_chain(lcs_ctx *ctx, const int32_t *d_a, int32_t m, const int32_t *d_b, int32_t n,
                  const lcs_schedule *sched, int32_t *d_h, int32_t *d_v, hipStream_t stream,
                  const int32_t *d_h_in = nullptr, const int32_t *d_v_in = nullptr, int32_t *d_r2c = nullptr,
                  int32_t *d_status = nullptr);
int check_abort(lcs_ctx *ctx);
void settle_timing(lcs_ctx *ctx);
// The register chain's time per step and the steps from one band's start to
// the next one's (lcs_capi.cpp).
struct ChainPace {
    double step_ns, lag;
};
ChainPace chain_pace(int tm, double waves, double bands, double columns);
// Host staging of host single-pair calls up to this size; larger ones are
// copied straight from and to the caller's memory.
constexpr size_t kPinnedMax = (size_t)4 << 20;
void *pinned_staging(lcs_ctx *ctx, size_t bytes);
// order a call on `s` after the previous user of the shared workspace, and
// mark `s` as its latest user once the call's kernels are enqueued
int ws_acquire(lcs_ctx *ctx, hipStream_t s);
int ws_release(lcs_ctx *ctx, hipStream_t s);
int upload(lcs_ctx *ctx, void *dst, const void *src, size_t bytes, hipStream_t stream);
int upload_via(Staging &st, void *dst, const void *src, size_t bytes, hipStream_t stream);
size_t pairs_ring_words(const std::vector<PairDesc> &pairs);
// Appends one chain launch over `pairs` (descriptors and task list) to
// `blob` and fills `L` with offsets into it; several launches share one
// blob, so they go to the device in one upload.  rebase_launch turns the
// offsets into addresses once the blob lies at `device_blob`.
int build_launch(lcs_ctx *ctx, std::vector<PairDesc> &pairs, int tm, int wps, unsigned long long *ring,
                 unsigned *ctrl, int group_w, std::vector<unsigned char> &blob, PreparedLaunch &L);
void rebase_launch(PreparedLaunch &L, const void *device_blob);
// The same for couples of pairs combed by the 16-bit packed chain.
int build_launch16(lcs_ctx *ctx, std::vector<CoupleDesc> &couples, int tm, int wps, unsigned long long *ring,
                   unsigned *ctrl, std::vector<unsigned char> &blob, PreparedLaunch &L);
size_t couples_ring_words(const std::vector<CoupleDesc> &couples);
// group_w: 1 = register chain (one wave per band), 4 = LDS groups of 4 bands
int prepare_pairs(lcs_ctx *ctx, std::vector<PairDesc> &pairs, int tm, int wps, unsigned long long *ring,
                  DevBuf &descs, unsigned *ctrl, PreparedLaunch &L, hipStream_t stream, int group_w = 1);
// group width of a schedule variant (LCS_VARIANT_*), 0 if unknown
int group_width(int variant);
int launch_prepared(const PreparedLaunch &L, hipStream_t stream);
// whether a single pair's register chain stages its b as byte symbols
// (lcsk_launch_sym8): pairs of 2^22 cells or more, or LCS_VARIANT_CHAIN_BYTES
bool use_sym8(int variant, int32_t m, int32_t n);
int default_batch_tile_m(int32_t m);
bool valid_tile_m(int tm);
int32_t bands_of(int32_t m, int32_t n, int tm);
void destroy_extras(lcs_ctx *ctx);
// layer sizes of a cost model
int mlp_shape(const lcs_mlp *M, int *n_in, int *hidden, int *n_out);
const lcs_ctx *mlp_ctx(const lcs_mlp *M);
// Schedule of a pair whose schedule leaves tile_m at 0: the context's
// autotune table, then its cost model, then the autotune on a miss, then
// the built-in default (all fields 0).  Non-zero fields of `given` are
// kept.  `source` (nullable) receives LCS_SCHED_FROM_*.
int choose_schedule(lcs_ctx *ctx, int mode, int32_t m, int32_t n, int32_t alphabet, float rate,
                    const lcs_schedule *given, lcs_schedule *out, int32_t *source);
// The same for npairs pairs at once (one model evaluation for all misses).
int choose_schedules(lcs_ctx *ctx, int mode, int32_t npairs, const int32_t *m, const int32_t *n,
                     const int32_t *alphabet, const lcs_schedule *given, std::vector<lcs_schedule> &out);
// 1 + the largest symbol of a host string, at least 2 (the cost model's
// alphabet input); 4 when unknown
int32_t alphabet_of(const int32_t *x, int32_t len);
void detach_model(lcs_ctx *ctx, const lcs_mlp *M);
}  // namespace lcs
