// C ABI of the engine: contexts, single-pair combing, permutation helpers.
// Declarations and the reference interfaces each entry replaces are in
// include/lcs_hip.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "lcs_hip.h"
#include "braid_kernels.h"
#include "comb_kernels.h"
#include "lcs_internal.h"

namespace lcs {

static int hip_status(hipError_t e) { return e == hipSuccess ? LCS_OK : LCS_EIO; }

DevBuf KeptBuf::take(size_t at_least, size_t at_most)
{
    std::lock_guard<std::mutex> lock(mu);
    DevBuf out;
    if (buf.bytes >= at_least && buf.bytes <= at_most) std::swap(out, buf);
    return out;
}

void KeptBuf::give(lcs_ctx *ctx, DevBuf &b)
{
    {
        std::lock_guard<std::mutex> lock(mu);
        if (b.bytes <= kKeptMax && b.bytes > buf.bytes) std::swap(b, buf);
    }
    b.release(ctx);
}

void KeptBuf::trim(lcs_ctx *ctx)
{
    std::lock_guard<std::mutex> lock(mu);
    buf.release(ctx);
}

// Frees what the context keeps for later calls and no call is using: products'
// and index builds' memory, and the single-pair workspaces that the call under
// way has not reserved.  (hipFree waits for the kernels that still use them.)
static void trim_kept(lcs_ctx *ctx, const DevBuf *reserving)
{
    ctx->scratch.trim(ctx);
    ctx->index_mem.trim(ctx);
    DevBuf *const bufs[] = {&ctx->ring, &ctx->strip_ws, &ctx->sym8};
    for (int i = 0; i < 3; ++i)
        if (!(ctx->ws_reserved >> i & 1) && bufs[i] != reserving) bufs[i]->release(ctx);
}

int reserve_ws(lcs_ctx *ctx, PairWs which, size_t bytes)
{
    DevBuf &buf = which == kWsRing ? ctx->ring : which == kWsStrips ? ctx->strip_ws : ctx->sym8;
    const int rc = buf.reserve(ctx, bytes);
    if (!rc) ctx->ws_reserved |= 1u << which;
    return rc;
}

int DevBuf::reserve(lcs_ctx *ctx, size_t want)
{
    if (want <= bytes) return LCS_OK;
    size_t grow = std::max(want, bytes + bytes / 2);
    if (ctx->held + grow - bytes > ctx->budget) grow = want;
    if (ctx->held + grow - bytes > ctx->budget) trim_kept(ctx, this);
    if (ctx->held + grow - bytes > ctx->budget) return LCS_ENOMEM;
    if (ptr) {
        (void)hipFree(ptr);
        ctx->held -= bytes;
        ptr = nullptr;
        bytes = 0;
    }
    void *p = nullptr;
    if (hipMalloc(&p, grow) != hipSuccess) {
        (void)hipGetLastError();
        trim_kept(ctx, this);
        if (hipMalloc(&p, grow) != hipSuccess) {
            (void)hipGetLastError();
            return LCS_ENOMEM;
        }
    }
    ptr = p;
    bytes = grow;
    ctx->held += grow;
    return LCS_OK;
}

void DevBuf::release(lcs_ctx *ctx)
{
    if (ptr) {
        (void)hipFree(ptr);
        ctx->held -= bytes;
    }
    ptr = nullptr;
    bytes = 0;
}

bool valid_tile_m(int tm) { return tm == 1 || tm == 2 || tm == 4 || tm == 8 || tm == 16 || tm == 32; }

int32_t bands_of(int32_t m, int32_t n, int tm)
{
    if (m <= 0 || n <= 0) return 0;
    return (int32_t)(((long long)m + 64LL * tm - 1) / (64LL * tm));
}

int Staging::init()
{
    return hipEventCreateWithFlags(&done, hipEventDisableTiming) == hipSuccess ? LCS_OK : LCS_EIO;
}

void Staging::destroy()
{
    if (done) (void)hipEventSynchronize(done);
    if (pinned) (void)hipHostFree(pinned);
    if (done) (void)hipEventDestroy(done);
    pinned = nullptr;
    bytes = 0;
    done = nullptr;
}

// Stages host bytes into a pinned buffer and copies them to `dst` on
// `stream`.  The previous upload through the same staging is waited for
// first, so the buffer is never rewritten while a copy from it is pending.
int upload_via(Staging &st, void *dst, const void *src, size_t bytes, hipStream_t stream)
{
    if (bytes == 0) return LCS_OK;
    if (hipEventSynchronize(st.done) != hipSuccess) return LCS_EIO;
    if (bytes > st.bytes) {
        if (st.pinned) (void)hipHostFree(st.pinned);
        st.pinned = nullptr;
        st.bytes = 0;
        void *p = nullptr;
        if (hipHostMalloc(&p, bytes * 2, hipHostMallocDefault) != hipSuccess) return LCS_ENOMEM;
        st.pinned = p;
        st.bytes = bytes * 2;
    }
    std::memcpy(st.pinned, src, bytes);
    if (hipMemcpyAsync(dst, st.pinned, bytes, hipMemcpyHostToDevice, stream) != hipSuccess) return LCS_EIO;
    if (hipEventRecord(st.done, stream) != hipSuccess) return LCS_EIO;
    return LCS_OK;
}

int upload(lcs_ctx *ctx, void *dst, const void *src, size_t bytes, hipStream_t stream)
{
    return upload_via(ctx->staging, dst, src, bytes, stream);
}

// Ring words of a launch over `pairs` (one ring of lcsk_ring_words(n) each).
size_t pairs_ring_words(const std::vector<PairDesc> &pairs)
{
    size_t w = 0;
    for (const auto &P : pairs) w += lcsk_ring_words(P.n);
    return w;
}

int group_width(int variant)
{
    switch (variant) {
    case LCS_VARIANT_AUTO:
    case LCS_VARIANT_CHAIN:
    case LCS_VARIANT_CHAIN_BYTES: return 1;
    case LCS_VARIANT_CHAIN_LDS: return 4;
    case LCS_VARIANT_PACKED16: return 1;   // one pair per wave outside batches
    default: return 0;
    }
}

constexpr int32_t kMaxChainN = 0x7fffffff - 4096;   // widest b a band chain combs

// One chain launch over `pairs` (one tile height): assigns each pair its
// ring inside `ring` (which must hold pairs_ring_words(pairs) words; NULL
// when every pair carries its own) and lists the tasks band-major (all pairs
// start at once, and every band comes after the band above it).
int build_launch(lcs_ctx *ctx, std::vector<PairDesc> &pairs, int tm, int wps, unsigned long long *ring,
                 unsigned *ctrl, int group_w, std::vector<unsigned char> &blob, PreparedLaunch &L)
{
    if (!valid_tile_m(tm) || wps < 1 || wps > 8 || (group_w != 1 && group_w != 4)) return LCS_EINVAL;
    const int np = (int)pairs.size();
    L = PreparedLaunch{};
    if (np == 0) return LCS_OK;
    int32_t max_bands = 0, max_n = 0;
    unsigned long long *E = ring;
    for (auto &P : pairs) {
        // the band loop counts steps up to n + 64 + 2 chunks in int
        if (P.n > kMaxChainN) return LCS_ERANGE;
        P.tile_m = tm;
        P.nbands = bands_of(P.m, P.n, tm);
        if (ring) {  // else every pair already carries its own ring
            P.E = E;
            E += lcsk_ring_words(P.n);
        }
        max_bands = std::max(max_bands, P.nbands);
        max_n = std::max(max_n, std::max(P.n, P.m));
    }
    // tasks: bands (or groups of group_w bands), band-major over the pairs
    std::vector<int2> tasks;
    const int32_t max_units = (max_bands + group_w - 1) / group_w;
    for (int32_t g = 0; g < max_units; ++g)
        for (int p = 0; p < np; ++p)
            if (g < (pairs[(size_t)p].nbands + group_w - 1) / group_w) tasks.push_back(make_int2(p, g));
    const size_t pair_bytes = sizeof(PairDesc) * (size_t)np, task_bytes = sizeof(int2) * tasks.size();
    const size_t base = (blob.size() + 15) & ~(size_t)15;
    blob.resize(base + pair_bytes + task_bytes);
    std::memcpy(blob.data() + base, pairs.data(), pair_bytes);
    if (task_bytes) std::memcpy(blob.data() + base + pair_bytes, tasks.data(), task_bytes);
    ChainArgs &A = L.args;
    A.pairs = (const PairDesc *)(uintptr_t)base;
    A.tasks = (const int2 *)(uintptr_t)(base + pair_bytes);
    A.ntasks = (int32_t)tasks.size();
    A.ticket = ctrl;
    A.abort_flag = ctrl + 1;
    A.sticky = ctx->ctrl + kStickyWord;
    A.timeout_ticks = ctx->timeout_ticks;
    A.trace = ctx->band_trace;
    A.trace_cap = ctx->band_trace_cap;
    A.group_w = group_w;
    const int waves_per_block = 4;
    if (group_w == 1) {
        const long long waves = std::min<long long>((long long)tasks.size(), 4LL * ctx->num_cus * wps);
        L.blocks = (int)std::max<long long>(1, (waves + waves_per_block - 1) / waves_per_block);
    } else {
        // one group per workgroup, wps groups per CU
        L.blocks = (int)std::max<long long>(1, std::min<long long>((long long)tasks.size(), (long long)ctx->num_cus * wps));
    }
    L.threads = 64 * waves_per_block;
    L.npairs = np;
    L.max_n = max_n;
    L.tile_m = tm;
    return LCS_OK;
}

void rebase_launch(PreparedLaunch &L, const void *device_blob)
{
    const uintptr_t b = (uintptr_t)device_blob;
    if (L.packed) L.args.couples = (const CoupleDesc *)(b + (uintptr_t)L.args.couples);
    else L.args.pairs = (const PairDesc *)(b + (uintptr_t)L.args.pairs);
    L.args.tasks = (const int2 *)(b + (uintptr_t)L.args.tasks);
}

// Ring words of a packed launch: one ring of lcsk_ring_words(max n) per
// couple, from the pairs' own extents (D.n is only set by build_launch16).
size_t couples_ring_words(const std::vector<CoupleDesc> &couples)
{
    size_t w = 0;
    for (const auto &D : couples) w += lcsk_ring_words(std::max(D.n_[0], D.n_[1]));
    return w;
}

// One packed-chain launch over `couples` (one tile height): rings carved
// from `ring`, tasks band-major over the couples.
int build_launch16(lcs_ctx *ctx, std::vector<CoupleDesc> &couples, int tm, int wps, unsigned long long *ring,
                   unsigned *ctrl, std::vector<unsigned char> &blob, PreparedLaunch &L)
{
    if (!valid_tile_m(tm) || wps < 1 || wps > 8) return LCS_EINVAL;
    const int nc = (int)couples.size();
    L = PreparedLaunch{};
    L.packed = true;
    if (nc == 0) return LCS_OK;
    int32_t max_bands = 0, max_n = 0;
    unsigned long long *E = ring;
    for (auto &D : couples) {
        D.tile_m = tm;
        D.m = std::max(D.m_[0], D.m_[1]);
        D.n = std::max(D.n_[0], D.n_[1]);
        D.nbands = bands_of(D.m, D.n, tm);
        D.E = E;
        E += lcsk_ring_words(D.n);
        max_bands = std::max(max_bands, D.nbands);
        max_n = std::max(max_n, std::max(D.n, D.m));
    }
    std::vector<int2> tasks;
    for (int32_t g = 0; g < max_bands; ++g)
        for (int c = 0; c < nc; ++c)
            if (g < couples[(size_t)c].nbands) tasks.push_back(make_int2(c, g));
    const size_t cbytes = sizeof(CoupleDesc) * (size_t)nc, task_bytes = sizeof(int2) * tasks.size();
    const size_t base = (blob.size() + 15) & ~(size_t)15;
    blob.resize(base + cbytes + task_bytes);
    std::memcpy(blob.data() + base, couples.data(), cbytes);
    if (task_bytes) std::memcpy(blob.data() + base + cbytes, tasks.data(), task_bytes);
    ChainArgs &A = L.args;
    A.couples = (const CoupleDesc *)(uintptr_t)base;
    A.tasks = (const int2 *)(uintptr_t)(base + cbytes);
    A.ntasks = (int32_t)tasks.size();
    A.ticket = ctrl;
    A.abort_flag = ctrl + 1;
    A.sticky = ctx->ctrl + kStickyWord;
    A.timeout_ticks = ctx->timeout_ticks;
    A.trace = ctx->band_trace;
    A.trace_cap = ctx->band_trace_cap;
    A.group_w = 1;
    const long long waves = std::min<long long>((long long)tasks.size(), 4LL * ctx->num_cus * wps);
    L.blocks = (int)std::max<long long>(1, (waves + 3) / 4);
    L.threads = 256;
    L.npairs = nc;
    L.max_n = max_n;
    L.tile_m = tm;
    return LCS_OK;
}

// Prepares one chain launch over `pairs` (one tile height): assigns each
// pair its ring inside `ring`, lists the tasks and uploads descriptors and
// tasks to `descs` through the context's staging.
int prepare_pairs(lcs_ctx *ctx, std::vector<PairDesc> &pairs, int tm, int wps, unsigned long long *ring,
                  DevBuf &descs, unsigned *ctrl, PreparedLaunch &L, hipStream_t stream, int group_w)
{
    std::vector<unsigned char> blob;
    int rc = build_launch(ctx, pairs, tm, wps, ring, ctrl, group_w, blob, L);
    if (rc || pairs.empty()) return rc;
    if ((rc = descs.reserve(ctx, blob.size() + 256))) return rc;
    if ((rc = upload(ctx, descs.ptr, blob.data(), blob.size(), stream))) return rc;
    rebase_launch(L, descs.ptr);
    return LCS_OK;
}

// Prep, chain and extract kernels of a prepared launch (no copies or
// memsets: capturable in a hipGraph).
int launch_prepared(const PreparedLaunch &L, hipStream_t stream)
{
    if (L.npairs == 0) return LCS_OK;
    if (L.packed)
        return lcsk_launch_chain16(L.args, L.args.couples, L.npairs, L.max_n, L.tile_m, L.blocks, L.threads, stream);
    return lcsk_launch_chain(L.args, L.args.pairs, L.npairs, L.max_n, L.tile_m, L.blocks, L.threads, stream);
}

// Byte symbols: a chain band takes each lane's column symbols from byte copies
// of b when every symbol of b lies in [0, 255] (which the staging finds out on
// the device), and pads the rows of a partial band with a symbol that b does
// not hold.  A single pair's copies are written by the launch's seeding
// kernel, whatever its size; a b longer than kSym8MaxN, or a context whose
// budget cannot hold them, keeps the 32-bit symbols.  The server stages them
// in two launches of their own (about 8 us of device time at n = 16384), which
// pays from kSym8MinCells cells.
constexpr int32_t kSym8MaxN = 1 << 30;
constexpr double kSym8MinCells = 4194304.0;   // 2^22
bool use_sym8(int variant, int32_t m, int32_t n)
{
    if (n <= 0 || n > kSym8MaxN) return false;
    return variant == LCS_VARIANT_CHAIN_BYTES || (double)m * (double)n >= kSym8MinCells;
}

// How one pair is cut and combed: GR x GC tiles of tm rows per lane.
struct GridPlan {
    int32_t tm, wps, group_w, GR, GC;
};

// The merge tree over a grid of tiles: every level joins neighbours along the
// shorter side of the current tiles (two tiles side by side glue on their
// common rows, one above the other on their common columns).
// level(products, k, p_size) sees each level with its largest product.
template <typename Level>
static void merge_levels(int32_t m, int32_t n, int32_t GR, int32_t GC, Level level)
{
    int32_t gr = GR, gc = GC, h = (m + GR - 1) / GR, w = (n + GC - 1) / GC;
    while (gr * gc > 1) {
        const bool side = gc > 1 && (gr == 1 || h <= w);
        level(side ? gr * (gc / 2) : gc * (gr / 2), side ? h : w, h + w);
        if (side) {
            gc = (gc + 1) / 2;
            w = std::min(n, 2 * w);
        } else {
            gr = (gr + 1) / 2;
            h = std::min(m, 2 * h);
        }
    }
}

// Words of the merge workspaces (the level that needs most).
static size_t grid_merge_words(int32_t m, int32_t n, const GridPlan &G)
{
    size_t most = 0;
    merge_levels(m, n, G.GR, G.GC, [&](int32_t products, int32_t k, int32_t size) {
        most = std::max(most, (size_t)products * lcsb_multiply_ws_words(size, size, k));
    });
    return most;
}

// Words of the tiles' permutations: every tile row holds its rows once per
// tile column and the columns once.
static size_t grid_perm_words(int32_t m, int32_t n, const GridPlan &G)
{
    return (size_t)G.GC * m + (size_t)G.GR * n;
}

// The pace of a byte chain: nanoseconds a step, and steps from one band's
// start to the next one's (64 of lane skew, a chunk of 32 published, a chunk
// prefetched, and with band_slack a chunk more).  `bands` of one pair with
// `columns` each, `waves` bands in the whole launch.  Measured on MI355X, one
// strip, n = 65536, 1 / 8 / 64 bands: 12.6 / 12.6 / 13.7 ns at 1 row per lane,
// 19.3 / 19.5 / 20.1 at 2, 32.3 / 32.3 / 32.8 at 4, 59.3 / 59.4 / 60.0 at 8 and
// 112.7 / 112.8 / 113.6 at 16; from 4 rows on 2 % more with every SIMD busy.
// Without the slack one row takes about 17.4 once
// a launch's bands lie on several XCDs (n = 4096 .. 50000, from 16 bands), two
// 20 to 24 in chains of 8 to 64 bands.
ChainPace chain_pace(int tm, double waves, double bands, double columns)
{
    const bool slack = band_slack(tm, (int32_t)bands, (int32_t)columns);
    const double lag = slack ? 162.0 : 130.0;
    if (tm == 1) return {slack ? 13.3 : waves < 16 ? 12.9 : 17.4, lag};
    return {tm == 2 ? 21.4 : tm == 4 ? 33.3 : tm == 8 ? 61.4 : 114.4 / 16 * tm, lag};
}

// Predicted microseconds of a plan.  The chain: one wave per band and SIMD, at
// chain_pace; bands beyond the SIMDs run in further rounds.  The merges: a
// level's products share its launches, about 60 us for a core of 2^11 points
// plus 8 per doubling, and about 0.6 ns per point (k = 2^16 155 us, 2^18 285,
// eight of 2^16 390).  Checked against the whole grid of plans at 2^14,
// 50021 x 70207, 2^16, 200000 and 2^18: the chain within 8 %, the plan it
// picks within 3 % of the best one measured (200000^2: 20 tiles of 16 rows
// 7.1 ms, one 10.6).  Small cores merge faster than that (k = 64 about 15 us a
// level), so a short a is cut into fewer strips than would be best (64 x
// 100000: 8 strips 223 us, 32 136, one 1254).
static double plan_us(const lcs_ctx *ctx, int32_t m, int32_t n, const GridPlan &G)
{
    const int32_t H = (m + G.GR - 1) / G.GR, W = (n + G.GC - 1) / G.GC, tiles = G.GR * G.GC;
    const double bands = bands_of(H, W, G.tm), waves = bands * tiles, simds = 4.0 * ctx->num_cus * G.wps;
    const ChainPace pace = chain_pace(G.tm, waves, bands, W);
    const double rounds = std::ceil(waves / simds), last = std::fmod(waves - 1, simds) / tiles;
    const double steps = std::max(rounds * (W + 64.0) + last * pace.lag, W + 64.0 + (bands - 1) * pace.lag);
    double us = steps * pace.step_ns * 1e-3;
    merge_levels(m, n, G.GR, G.GC, [&](int32_t products, int32_t k, int32_t) {
        const int L = std::max(6, lcsb_core_L(k));
        us += 60.0 + 8.0 * std::max(0, L - 11) + 0.6e-3 * products * (double)(1LL << L);
    });
    return us + (tiles > 1 ? 10.0 : 0.0);
}

// The plan of a pair: the cheapest predicted one with the fields that the
// schedule fixes (tm, strips; 0 = open).  A pair with explicit strands is one
// tile.  Below kGridMinCells cells a pair is cut only into columns, and from
// kWideMinN of them: m is then so small that its merges are short beside the
// columns (64 x 16384 216 us as one tile, 103 as four; 512 x 100000 1268 and
// 261; 4000 x 16400 446 and 371), while a square one gains nothing (8192^2
// 0.36 ms as one tile).
constexpr double kGridMinCells = 67108864.0;   // 2^26
constexpr int32_t kWideMinN = 16384;
static GridPlan choose_grid(const lcs_ctx *ctx, int32_t m, int32_t n, int tm, int strips, bool whole, GridPlan G)
{
    static const int32_t kCols[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64}, kRows[] = {1, 2, 3, 4, 6, 8};
    const bool open_rows = !whole && !strips && (double)m * n >= kGridMinCells;
    const bool open_cols = open_rows || (!whole && !strips && n >= kWideMinN);
    double best = 0.0;
    GridPlan B = G;
    B.tm = 0;
    for (int32_t t = 1; t <= 16; t *= 2) {
        if (tm && t != (tm < 16 ? tm : 16)) continue;
        for (const int32_t r : kRows) {
            if (r > 1 && (!open_rows || m / r < 2048 || n > kMaxCoreK)) break;
            for (int32_t c : kCols) {
                if (c > 1 && (!open_cols || n / c < 2048 || m > kMaxCoreK)) break;
                GridPlan T = G;
                T.tm = tm ? tm : t;
                T.GR = r;
                T.GC = strips ? strips : c;
                const double us = plan_us(ctx, m, n, T);
                if (!B.tm || us < best) {
                    best = us;
                    B = T;
                }
            }
        }
    }
    return B;
}

// Merges the tiles' permutations to the whole pair's and writes its strands,
// all products of a level (merge_levels) in one launch sequence.
static int merge_tiles(const TileGrid &T, int32_t *permA, int32_t *permB, int32_t *ws, const PairDesc &out,
                       hipStream_t stream)
{
    const int32_t m = T.pair.m, n = T.pair.n;
    struct Tile {
        int32_t *p;
        int32_t m, n;
    };
    int32_t gr = T.GR, gc = T.GC;
    std::vector<Tile> cur((size_t)gr * gc);
    for (int32_t i = 0; i < gr; ++i)
        for (int32_t j = 0; j < gc; ++j) cur[(size_t)i * gc + j] = Tile{permA + T.perm_off(i, j), T.rows(i), T.cols(j)};
    int32_t *dst_base = permB;
    while (gr * gc > 1) {
        const bool side = gc > 1 && (gr == 1 || cur[0].m <= cur[0].n);
        int32_t *next_ws = ws;
        const int32_t nr = side ? gr : (gr + 1) / 2, nc = side ? (gc + 1) / 2 : gc;
        std::vector<Tile> nxt((size_t)nr * nc);
        std::vector<MulSpec> specs;
        int32_t *dst = dst_base;
        for (int32_t i = 0; i < nr; ++i)
            for (int32_t j = 0; j < nc; ++j) {
                const Tile &p = cur[(size_t)(side ? i : 2 * i) * gc + (side ? 2 * j : j)];
                Tile &o = nxt[(size_t)i * nc + j];
                o = Tile{dst, p.m, p.n};
                if (side ? 2 * j + 1 < gc : 2 * i + 1 < gr) {
                    const Tile &q = side ? cur[(size_t)i * gc + 2 * j + 1] : cur[(size_t)(2 * i + 1) * gc + j];
                    const int32_t k = side ? p.m : p.n;
                    specs.push_back(MulSpec{p.p, p.m + p.n, q.p, q.m + q.n, k, side ? 0 : 1, dst, next_ws});
                    next_ws += lcsb_multiply_ws_words(p.m + p.n, q.m + q.n, k);
                    if (side) o.n += q.n;
                    else o.m += q.m;
                } else if (lcsk_launch_copy(dst, p.p, (long long)p.m + p.n, stream)) {
                    return LCS_EIO;   // an odd tile moves on unchanged
                }
                dst += o.m + o.n;
            }
        const int rc = lcsb_multiply_many_device(specs.data(), (int)specs.size(), stream);
        if (rc) return rc;
        cur.swap(nxt);
        gr = nr;
        gc = nc;
        dst_base = dst_base == permB ? permA : permB;
    }
    return lcsk_launch_strands_from_perm(cur[0].p, m, n, out.h_out, out.v_out, out.perm, stream);
}

// Combs one pair as the tiles of `G` in one chain launch and merges them.
// The launch is described by its arguments alone: nothing is uploaded.
static int enqueue_grid(lcs_ctx *ctx, const PairDesc &pair, GridPlan G, int32_t *status, hipStream_t stream)
{
    const int32_t m = pair.m, n = pair.n;
    TileGrid T{};
    T.pair = pair;
    T.status = status;
    T.H = (m + G.GR - 1) / G.GR;
    T.W = (n + G.GC - 1) / G.GC;
    T.GR = G.GR = (m + T.H - 1) / T.H;   // no empty tile
    T.GC = G.GC = (n + T.W - 1) / T.W;
    const int32_t tiles = T.GR * T.GC;
    T.pair.tile_m = G.tm;
    T.pair.nbands = bands_of(T.H, T.W, G.tm);
    // what the call cannot do without first; the byte copies take what is left
    ctx->ws_reserved = 0;
    int rc = reserve_ws(ctx, kWsRing, (size_t)tiles * lcsk_ring_words(T.W) * sizeof(unsigned long long));
    if (rc) return rc;
    size_t perm_words = 0;
    if (tiles > 1) {
        perm_words = grid_perm_words(m, n, G);
        if ((rc = reserve_ws(ctx, kWsStrips, (2 * perm_words + grid_merge_words(m, n, G)) * 4))) return rc;
        T.perm = (int32_t *)ctx->strip_ws.ptr;
    }
    T.pair.E = (unsigned long long *)ctx->ring.ptr;
    if (n <= kSym8MaxN) {
        const int32_t stride = lcsk_sym8_stride(T.W);
        if (reserve_ws(ctx, kWsSym8, (size_t)T.GC * 16 * (size_t)stride) == LCS_OK) {
            T.pair.sym8 = (const uint32_t *)ctx->sym8.ptr;
            T.pair.sym8_stride = stride;
            T.sym8_flags = (int32_t *)ctx->ctrl + kSym8FlagWord;
            T.pair.sym8_flags = T.sym8_flags;
        }
    }
    ChainArgs A{};
    const long long units = (T.pair.nbands + G.group_w - 1) / G.group_w * (long long)tiles;
    if (units > 0x7fffffffLL) return LCS_ERANGE;
    A.grid = T;
    A.ntasks = (int32_t)units;
    A.group_w = G.group_w;
    A.ticket = ctx->ctrl;
    A.abort_flag = ctx->ctrl + 1;
    A.sticky = ctx->ctrl + kStickyWord;
    A.timeout_ticks = ctx->timeout_ticks;
    A.trace = ctx->band_trace;
    A.trace_cap = ctx->band_trace_cap;
    const long long per_cu = G.group_w == 1 ? 4LL : 1LL, resident = per_cu * ctx->num_cus * G.wps;
    const long long blocks = (std::min(units, resident) + per_cu - 1) / per_cu;
    ctx->pending_timing = false;   // its events are recorded anew
    if (hipEventRecord(ctx->evc0, stream) != hipSuccess) return LCS_EIO;
    if ((rc = lcsk_launch_grid(A, (int)blocks, 256, stream))) return rc;
    if (hipEventRecord(ctx->evc1, stream) != hipSuccess) return LCS_EIO;
    ctx->chain_timed = true;
    ctx->time_from = ctx->evc0;
    ctx->time_to = ctx->evc1;
    if (tiles == 1) return LCS_OK;
    if ((rc = merge_tiles(T, T.perm, T.perm + perm_words, T.perm + 2 * perm_words, pair, stream))) return rc;
    ctx->time_to = ctx->ev1;
    return hipEventRecord(ctx->ev1, stream) == hipSuccess ? LCS_OK : LCS_EIO;
}

int ws_acquire(lcs_ctx *ctx, hipStream_t s)
{
    if (ctx->ws_stream && ctx->ws_stream != s && hipStreamWaitEvent(s, ctx->ws_done, 0) != hipSuccess) return LCS_EIO;
    return LCS_OK;
}

int ws_release(lcs_ctx *ctx, hipStream_t s)
{
    if (hipEventRecord(ctx->ws_done, s) != hipSuccess) return LCS_EIO;
    ctx->ws_stream = s;
    return LCS_OK;
}

static int enqueue_chain_ws(lcs_ctx *ctx, const int32_t *d_a, int32_t m, const int32_t *d_b, int32_t n,
                            const lcs_schedule *sched, int32_t *d_h, int32_t *d_v, hipStream_t stream,
                            const int32_t *d_h_in, const int32_t *d_v_in, int32_t *d_r2c, int32_t *d_status);

// Enqueue one pair on `stream` with device pointers, following `sched`,
// after the previous user of the context's workspace.
int enqueue_chain(lcs_ctx *ctx, const int32_t *d_a, int32_t m, const int32_t *d_b, int32_t n,
                  const lcs_schedule *sched, int32_t *d_h, int32_t *d_v, hipStream_t stream,
                  const int32_t *d_h_in, const int32_t *d_v_in, int32_t *d_r2c, int32_t *d_status)
{
    int rc = ws_acquire(ctx, stream);
    if (rc) return rc;
    rc = enqueue_chain_ws(ctx, d_a, m, d_b, n, sched, d_h, d_v, stream, d_h_in, d_v_in, d_r2c, d_status);
    const int rc2 = ws_release(ctx, stream);
    ctx->ws_reserved = 0;
    return rc ? rc : rc2;
}

static int enqueue_chain_ws(lcs_ctx *ctx, const int32_t *d_a, int32_t m, const int32_t *d_b, int32_t n,
                            const lcs_schedule *sched, int32_t *d_h, int32_t *d_v, hipStream_t stream,
                            const int32_t *d_h_in, const int32_t *d_v_in, int32_t *d_r2c, int32_t *d_status)
{
    if (m == 0 || n == 0) {
        ctx->pending_timing = false;   // its events are recorded anew
        ctx->time_from = ctx->ev0;
        ctx->time_to = ctx->ev1;
        bool ok = hipEventRecord(ctx->ev0, stream) == hipSuccess;
        if (ok && d_status)
            ok = hipMemcpyAsync(d_status, ctx->ctrl + kZeroWord, 4, hipMemcpyDeviceToDevice, stream) == hipSuccess;
        if (d_h_in || d_v_in) {
            if (ok && m) ok = hipMemcpyAsync(d_h, d_h_in, (size_t)m * 4, hipMemcpyDeviceToDevice, stream) == hipSuccess;
            if (ok && n) ok = hipMemcpyAsync(d_v, d_v_in, (size_t)n * 4, hipMemcpyDeviceToDevice, stream) == hipSuccess;
        } else if (ok) {
            const int rc = lcsk_launch_identity(d_h, m, d_v, n, stream, d_r2c);
            if (rc) return rc;
        }
        return ok && hipEventRecord(ctx->ev1, stream) == hipSuccess ? LCS_OK : LCS_EIO;
    }
    if (n > kMaxChainN) return LCS_ERANGE;   // before any buffer is reserved
    const int strips_req = sched ? sched->strips : 0;
    int tm = (sched && sched->tile_m) ? sched->tile_m : 0;
    if (tm && !valid_tile_m(tm)) return LCS_EINVAL;
    const int wps = (sched && sched->waves_per_simd) ? sched->waves_per_simd : 1;
    if (wps < 1 || wps > 8) return LCS_EINVAL;
    if (strips_req < 0) return LCS_EINVAL;
    const int group_w = group_width(sched ? sched->variant : LCS_VARIANT_AUTO);
    if (!group_w) return LCS_EINVAL;
    const bool whole = d_h_in || d_v_in;   // fixups use explicit strands: one tile
    if (strips_req > 1 && whole) return LCS_EINVAL;
    if (strips_req > 1 && m > kMaxCoreK) return LCS_ERANGE;
    const GridPlan G = choose_grid(ctx, m, n, tm, std::min(strips_req, n), whole, GridPlan{0, wps, group_w, 1, 1});
    PairDesc P{};
    P.a = d_a;
    P.b = d_b;
    P.h_in = d_h_in;
    P.v_in = d_v_in;
    P.h_out = d_h;
    P.v_out = d_v;
    P.perm = d_r2c;
    P.m = m;
    P.n = n;
    const int rc = enqueue_grid(ctx, P, G, d_status, stream);
    if (rc != LCS_ENOMEM || strips_req || G.GR * G.GC == 1) return rc;
    // the budget cannot hold the library's own cut (its workspaces are reserved
    // before anything is launched): one tile
    return enqueue_grid(ctx, P, choose_grid(ctx, m, n, tm, 1, whole, G), d_status, stream);
}

void *pinned_staging(lcs_ctx *ctx, size_t bytes)
{
    if (bytes <= ctx->pinned_bytes) return ctx->pinned;
    if (ctx->pinned) (void)hipHostFree(ctx->pinned);   // its last user has waited for its copies
    ctx->pinned = nullptr;
    ctx->pinned_bytes = 0;
    void *p = nullptr;
    const size_t want = std::min(kPinnedMax, bytes * 2);
    if (hipHostMalloc(&p, want, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    ctx->pinned = p;
    ctx->pinned_bytes = want;
    return p;
}

// Reads the time of an asynchronous call off its events (waiting for them),
// before a call that times nothing itself records into the same ones.
void settle_timing(lcs_ctx *ctx)
{
    float ms = 0.f;
    if (ctx->pending_timing && hipEventSynchronize(ctx->time_to) == hipSuccess &&
        hipEventElapsedTime(&ms, ctx->time_from, ctx->time_to) == hipSuccess)
        ctx->last_kernel_ms = ms;
    ctx->pending_timing = false;
}

// The abort flag of the last launch on the context's own ctrl words (the
// caller has synchronised).  A raised flag is cleared once reported, so the
// next launch's prep kernel does not fold it into the status word again.
int check_abort(lcs_ctx *ctx)
{
    unsigned flag = 0;
    if (hipMemcpy(&flag, ctx->ctrl + 1, sizeof(flag), hipMemcpyDeviceToHost) != hipSuccess) return LCS_EIO;
    if (!flag) return LCS_OK;
    const unsigned zero = 0;
    if (hipMemcpy(ctx->ctrl + 1, &zero, sizeof(zero), hipMemcpyHostToDevice) != hipSuccess) return LCS_EIO;
    return LCS_ETIMEDOUT;
}

// The schedule a single-pair call runs with (host strings give the cost
// model the alphabet; device strings are taken as alphabet 4).
static int single_schedule(lcs_ctx *ctx, const int32_t *a_host, int32_t m, const int32_t *b_host, int32_t n,
                           const lcs_schedule *sched, lcs_schedule &out)
{
    if (sched && sched->tile_m) {
        out = *sched;
        return LCS_OK;
    }
    const Selector &S = ctx->select[LCS_TUNE_SINGLE];
    int32_t alphabet = 4;
    if ((S.model || !S.miss_cands.empty()) && (a_host || b_host))
        alphabet = std::max(alphabet_of(a_host, a_host ? m : 0), alphabet_of(b_host, b_host ? n : 0));
    return choose_schedule(ctx, LCS_TUNE_SINGLE, m, n, alphabet, 0.1f, sched, &out, nullptr);
}

}  // namespace lcs

using namespace lcs;

extern "C" {

int lcs_ctx_create(int device, size_t hbm_budget, lcs_ctx **out)
{
    if (!out) return LCS_EINVAL;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
        (void)hipGetLastError();
        return LCS_EIO;
    }
    if (device < 0 || device >= ndev) return LCS_EINVAL;
    if (hipSetDevice(device) != hipSuccess) return LCS_EIO;
    lcs_ctx *ctx = new (std::nothrow) lcs_ctx();
    if (!ctx) return LCS_ENOMEM;
    ctx->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) { delete ctx; return LCS_EIO; }
    ctx->num_cus = prop.multiProcessorCount;
    ctx->name = prop.name;
    ctx->arch = prop.gcnArchName;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) { delete ctx; return LCS_EIO; }
    ctx->budget = hbm_budget ? hbm_budget : free_b / 4 * 3;
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) { delete ctx; return LCS_EIO; }
    if (hipEventCreate(&ctx->ev0) != hipSuccess || hipEventCreate(&ctx->ev1) != hipSuccess ||
        hipEventCreate(&ctx->evc0) != hipSuccess || hipEventCreate(&ctx->evc1) != hipSuccess ||
        ctx->staging.init() != LCS_OK ||
        hipEventCreateWithFlags(&ctx->ws_done, hipEventDisableTiming) != hipSuccess) {
        lcs_ctx_destroy(ctx);
        return LCS_EIO;
    }
    void *p = nullptr;
    if (hipMalloc(&p, 256) != hipSuccess) { lcs_ctx_destroy(ctx); return LCS_ENOMEM; }
    ctx->ctrl = (unsigned *)p;
    if (hipMemset(ctx->ctrl, 0, 256) != hipSuccess) { lcs_ctx_destroy(ctx); return LCS_EIO; }
    *out = ctx;
    return LCS_OK;
}

int lcs_ctx_destroy(lcs_ctx *ctx)
{
    if (!ctx) return LCS_EINVAL;
    {
        const std::lock_guard<std::mutex> lock(ctx->life->mu);   // of an index being dropped: after it
        ctx->life->alive = false;
    }
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    destroy_extras(ctx);
    ctx->ring.release(ctx);
    ctx->descs.release(ctx);
    ctx->strip_ws.release(ctx);
    ctx->sym8.release(ctx);
    ctx->staging.destroy();
    if (ctx->ws_done) (void)hipEventDestroy(ctx->ws_done);
    ctx->strings.release(ctx);
    ctx->results.release(ctx);
    trim_kept(ctx, nullptr);
    if (ctx->pinned) (void)hipHostFree(ctx->pinned);
    if (ctx->ctrl) (void)hipFree(ctx->ctrl);
    if (ctx->band_trace) (void)hipFree(ctx->band_trace);
    if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
    if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
    if (ctx->evc0) (void)hipEventDestroy(ctx->evc0);
    if (ctx->evc1) (void)hipEventDestroy(ctx->evc1);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return LCS_OK;
}

int lcs_ctx_device_name(lcs_ctx *ctx, char *buf, size_t len)
{
    if (!ctx || !buf || len == 0) return LCS_EINVAL;
    std::snprintf(buf, len, "%s (%s)", ctx->name.c_str(), ctx->arch.c_str());
    return LCS_OK;
}

int lcs_ctx_status(lcs_ctx *ctx)
{
    if (!ctx) return LCS_EINVAL;
    if (hipSetDevice(ctx->device) != hipSuccess) return LCS_EIO;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return LCS_EIO;
    if (ctx->ws_stream && hipEventSynchronize(ctx->ws_done) != hipSuccess) return LCS_EIO;
    unsigned words[64];
    if (hipMemcpy(words, ctx->ctrl, sizeof(words), hipMemcpyDeviceToHost) != hipSuccess) return LCS_EIO;
    const bool aborted = words[1] || words[kStickyWord];
    if (aborted) {
        const unsigned zero = 0;
        if (hipMemcpy(ctx->ctrl + 1, &zero, 4, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(ctx->ctrl + kStickyWord, &zero, 4, hipMemcpyHostToDevice) != hipSuccess)
            return LCS_EIO;
    }
    return aborted ? LCS_ETIMEDOUT : LCS_OK;
}

int lcs_ctx_memory(lcs_ctx *ctx, size_t *held, size_t *budget)
{
    if (!ctx) return LCS_EINVAL;
    if (held) *held = ctx->held;
    if (budget) *budget = ctx->budget;
    return LCS_OK;
}

int lcs_ctx_set_timeout(lcs_ctx *ctx, uint64_t ticks)
{
    if (!ctx) return LCS_EINVAL;
    ctx->timeout_ticks = ticks;
    return LCS_OK;
}

int lcs_ctx_info(lcs_ctx *ctx, int32_t *num_cus, double *last_kernel_ms)
{
    if (!ctx) return LCS_EINVAL;
    if (ctx->pending_timing && hipEventQuery(ctx->time_to) == hipSuccess) settle_timing(ctx);
    if (num_cus) *num_cus = ctx->num_cus;
    if (last_kernel_ms) *last_kernel_ms = ctx->last_kernel_ms;
    return LCS_OK;
}

int lcs_ctx_chain_ms(lcs_ctx *ctx, double *chain_ms)
{
    if (!ctx || !chain_ms) return LCS_EINVAL;
    if (!ctx->chain_timed) return LCS_ENOENT;
    if (hipSetDevice(ctx->device) != hipSuccess) return LCS_EIO;
    if (hipEventSynchronize(ctx->evc1) != hipSuccess) return LCS_EIO;
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, ctx->evc0, ctx->evc1) != hipSuccess) return LCS_EIO;
    *chain_ms = ms;
    return LCS_OK;
}

// The host single-pair calls.  Strings and results each lie in one device
// buffer, so that a call makes one copy in and one out, through pinned host
// memory up to kPinnedMax bytes: a small call's time is its copies, launches
// and waits, and a copy from or to pageable memory costs a wait of its own.
// 300 x 500 took 127 us with 2 copies in, 2 out, one of the abort flag and
// 5 events, and takes 66 us.  The limit bounds the pinned memory a context
// holds; past it the two waits are small beside the call.
// Results on the device: kStatusWords words (the launch's abort flag in the
// first), row_to_col (if asked for), v, h -- col_to_row is v then h.
static int comb_host(lcs_ctx *ctx, const int32_t *a, int32_t m, const int32_t *b, int32_t n, const lcs_schedule *sched,
                     int32_t *r2c, int32_t *v_out, int32_t *h_out, int32_t *llcs_out)
{
    constexpr size_t kStatusWords = 16;
    if (hipSetDevice(ctx->device) != hipSuccess) return LCS_EIO;
    int rc;
    lcs_schedule chosen{};
    if ((rc = single_schedule(ctx, a, m, b, n, sched, chosen))) return rc;
    const size_t mm = (size_t)m, nn = (size_t)n, a_words = (mm + 15) & ~(size_t)15;   // b 64-byte aligned
    const size_t in_bytes = (a_words + nn) * 4, perm_words = r2c ? mm + nn : 0;
    const size_t out_bytes = (kStatusWords + perm_words + mm + nn) * 4;
    if ((rc = ctx->strings.reserve(ctx, std::max<size_t>(in_bytes, 4)))) return rc;
    if ((rc = ctx->results.reserve(ctx, out_bytes))) return rc;
    int32_t *da = (int32_t *)ctx->strings.ptr, *db = da + a_words;
    int32_t *dstatus = (int32_t *)ctx->results.ptr, *dr2c = dstatus + kStatusWords, *dv = dr2c + perm_words, *dh = dv + n;
    hipStream_t s = ctx->stream;
    // an error leaves no copy of the staging or the caller's memory queued
    const auto drained = [s](int rc) {
        (void)hipStreamSynchronize(s);
        return rc;
    };
    int32_t *pin = in_bytes + out_bytes <= kPinnedMax ? (int32_t *)pinned_staging(ctx, in_bytes + out_bytes) : nullptr;
    if (pin) {
        if (m) std::memcpy(pin, a, mm * 4);
        if (n) std::memcpy(pin + a_words, b, nn * 4);
        if (in_bytes && hipMemcpyAsync(da, pin, in_bytes, hipMemcpyHostToDevice, s) != hipSuccess) return drained(LCS_EIO);
    } else {
        if (m && hipMemcpyAsync(da, a, mm * 4, hipMemcpyHostToDevice, s) != hipSuccess) return drained(LCS_EIO);
        if (n && hipMemcpyAsync(db, b, nn * 4, hipMemcpyHostToDevice, s) != hipSuccess) return drained(LCS_EIO);
    }
    if ((rc = enqueue_chain(ctx, da, m, db, n, &chosen, dh, dv, s, nullptr, nullptr, r2c ? dr2c : nullptr, dstatus)))
        return drained(rc);
    int32_t status = 0;
    if (pin) {
        int32_t *res = pin + in_bytes / 4;
        if (hipMemcpyAsync(res, dstatus, out_bytes, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return drained(LCS_EIO);
        status = res[0];
        if (!status) {
            res += kStatusWords;
            if (perm_words) std::memcpy(r2c, res, perm_words * 4);
            if (n) std::memcpy(v_out, res + perm_words, nn * 4);
            if (m) std::memcpy(h_out, res + perm_words + nn, mm * 4);
        }
    } else {
        if (perm_words && hipMemcpyAsync(r2c, dr2c, perm_words * 4, hipMemcpyDeviceToHost, s) != hipSuccess) return drained(LCS_EIO);
        if (n && hipMemcpyAsync(v_out, dv, nn * 4, hipMemcpyDeviceToHost, s) != hipSuccess) return drained(LCS_EIO);
        if (m && hipMemcpyAsync(h_out, dh, mm * 4, hipMemcpyDeviceToHost, s) != hipSuccess) return drained(LCS_EIO);
        if (hipMemcpyAsync(&status, dstatus, 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return drained(LCS_EIO);
    }
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, ctx->time_from, ctx->time_to) == hipSuccess) ctx->last_kernel_ms = ms;
    ctx->pending_timing = false;
    if (status) return (rc = check_abort(ctx)) ? rc : LCS_ETIMEDOUT;   // clears the flag
    if (llcs_out) {
        int32_t c = 0;
        for (int32_t j = 0; j < n; ++j) c += v_out[j] < m;
        *llcs_out = c;
    }
    return LCS_OK;
}

int lcs_comb(lcs_ctx *ctx, const int32_t *a, int32_t m, const int32_t *b, int32_t n,
             const lcs_schedule *sched, int32_t *h_out, int32_t *v_out, int32_t *llcs_out)
{
    if (!ctx || m < 0 || n < 0) return LCS_EINVAL;
    if ((m > 0 && (!a || !h_out)) || (n > 0 && (!b || !v_out))) return LCS_EINVAL;
    if ((long long)m + n > 0x7fffffffLL) return LCS_ERANGE;
    return comb_host(ctx, a, m, b, n, sched, nullptr, v_out, h_out, llcs_out);
}

int lcs_comb_permutation(lcs_ctx *ctx, const int32_t *a, int32_t m, const int32_t *b, int32_t n,
                         const lcs_schedule *sched, int32_t *row_to_col, int32_t *col_to_row, int32_t *llcs_out)
{
    if (!ctx || m < 0 || n < 0) return LCS_EINVAL;
    if ((m > 0 && !a) || (n > 0 && !b) || (m + n > 0 && (!row_to_col || !col_to_row))) return LCS_EINVAL;
    if ((long long)m + n > 0x7fffffffLL) return LCS_ERANGE;
    // col_to_row is v then h (FromStrands: col j <- v[j], col n+l <- h[l])
    return comb_host(ctx, a, m, b, n, sched, row_to_col, col_to_row, col_to_row ? col_to_row + n : nullptr, llcs_out);
}

int lcs_comb_device(lcs_ctx *ctx, const int32_t *d_a, int32_t m, const int32_t *d_b, int32_t n,
                    const lcs_schedule *sched, int32_t *d_h_out, int32_t *d_v_out, void *stream)
{
    if (!ctx || m < 0 || n < 0) return LCS_EINVAL;
    if ((m > 0 && (!d_a || !d_h_out)) || (n > 0 && (!d_b || !d_v_out))) return LCS_EINVAL;
    if ((long long)m + n > 0x7fffffffLL) return LCS_ERANGE;
    if (hipSetDevice(ctx->device) != hipSuccess) return LCS_EIO;
    hipStream_t s = stream ? (hipStream_t)stream : ctx->stream;
    lcs_schedule chosen{};
    int rc = single_schedule(ctx, nullptr, m, nullptr, n, sched, chosen);
    if (rc) return rc;
    rc = enqueue_chain(ctx, d_a, m, d_b, n, &chosen, d_h_out, d_v_out, s);
    if (rc) return rc;
    ctx->pending_timing = true;
    return LCS_OK;
}

int lcs_debug_band_trace(lcs_ctx *ctx, int32_t max_bands, uint64_t *host_out)
{
    // max_bands > 0: (re)arm tracing of up to max_bands bands; 0: disarm;
    // host_out != NULL: copy the last trace (2 words per band) out.
    if (!ctx || max_bands < 0) return LCS_EINVAL;
    if (hipSetDevice(ctx->device) != hipSuccess) return LCS_EIO;
    if (host_out) {
        if (!ctx->band_trace || max_bands > ctx->band_trace_cap) return LCS_EINVAL;
        if (hipMemcpy(host_out, ctx->band_trace, (size_t)max_bands * 16, hipMemcpyDeviceToHost) != hipSuccess)
            return LCS_EIO;
        return LCS_OK;
    }
    if (ctx->band_trace) {
        (void)hipFree(ctx->band_trace);
        ctx->band_trace = nullptr;
        ctx->band_trace_cap = 0;
    }
    if (max_bands == 0) return LCS_OK;
    void *p = nullptr;
    if (hipMalloc(&p, (size_t)max_bands * 16) != hipSuccess) return LCS_ENOMEM;
    ctx->band_trace = (unsigned long long *)p;
    ctx->band_trace_cap = max_bands;
    return LCS_OK;
}

int lcs_permutation_from_strands(const int32_t *h, int32_t m, const int32_t *v, int32_t n,
                                 int32_t *row_to_col, int32_t *col_to_row)
{
    if (m < 0 || n < 0 || (m && !h) || (n && !v)) return LCS_EINVAL;
    const int32_t size = m + n;
    if (size && (!row_to_col || !col_to_row)) return LCS_EINVAL;
    for (int32_t i = 0; i < size; ++i) row_to_col[i] = col_to_row[i] = -1;
    for (int32_t l = 0; l < m; ++l)
        if (h[l] >= 0 && h[l] < size) { row_to_col[h[l]] = n + l; col_to_row[n + l] = h[l]; }
    for (int32_t j = 0; j < n; ++j)
        if (v[j] >= 0 && v[j] < size) { row_to_col[v[j]] = j; col_to_row[j] = v[j]; }
    return LCS_OK;
}

int64_t lcs_permutation_hash(const int32_t *col_to_row, int32_t size)
{
    // result = (R * result + row) % M in 64-bit two's complement, the wrap made
    // explicit with unsigned arithmetic.
    const uint64_t R = 4294967279ull;
    const int64_t M = 4294967291ll;
    int64_t res = 0;
    for (int32_t c = 0; c < size; ++c) {
        const uint64_t t = R * (uint64_t)res + (uint64_t)(int64_t)col_to_row[c];
        res = (int64_t)t % M;
    }
    return res;
}

}  // extern "C"
