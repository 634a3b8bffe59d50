// Steady-ant braid multiplication on the GPU (gfx950).
//
// Computes staggered_multiply<RowGlue>(p, q, k) of the reference
// (src/braid_multiplication.hpp:273-406): the sticky-braid (distance) product
// of two seaweed permutations glued on k strands.  The k x k core product is
// the steady ant of src/braid_multiplication.hpp:204-270, organised for a
// workgroup instead of a recursion:
//
//  * the core is padded to K = 2^L with fixed points (strands that never meet
//    another strand do not change the product), so every node of the
//    recursion at depth d is an aligned segment of K >> d positions;
//  * top-down, one stable partition per depth orders the points of P by
//    (node, row) and those of Q by (node, column) -- the reference's
//    get_vert_slice / get_horz_slice (:5-36) for all nodes of a depth at
//    once -- and remembers where each point came from;
//  * bottom-up, each depth lifts the children's products into the node's
//    coordinates (the reference's inverse_mapping, :191-202) and runs the ant
//    passage (:123-189) for all nodes at once.  The dominance-sum difference
//        delta(r, c) = #{hi points: row < r, col < c} - #{lo points: row >= r, col >= c}
//    is non-decreasing in r and c, so the ant leaves row r at the first
//    column T(r) where delta >= 0, and the product's point of row r follows
//    from T(r) and the row's own point alone: it is T(r) - 1 when T(r) > 0
//    and the point is counted at T(r) (lo ? col >= T : col < T), else the
//    point itself.  So nothing is walked: waves find T at every 64th row line
//    and the row where the path crosses every 64th column line, and one wave
//    per box finds T for its 64 rows, a lane each, from bit masks of the
//    box's columns.
// The last six depths (nodes of 64 points) run in one wave's registers.  The
// union of the children's points, the per-column view and the parents of the
// depths above live in LDS (16-bit entries, the lo/hi flag in bit 15) for
// cores up to K = 2048.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "braid_kernels.h"

namespace lcsb {

constexpr int kThreads = 1024;
constexpr uint16_t kLoFlag = 0x8000u;
constexpr uint16_t kIdx = 0x7fffu;
// cores up to this size keep keys, products and parents in LDS
// (braid_core_lds_kernel and the leaves of larger cores)
constexpr int kLdsCoreL = 11;
constexpr int kLdsCoreK = 1 << kLdsCoreL;
constexpr int kBox = 64;   // side of a box: one wave, a lane per row
constexpr int kMaxLeafLines = kLdsCoreK / kBox;   // grid lines of the largest node in LDS
// dynamic LDS of a core of 2^L points: keys / U, CI, R, Rn (4K uint16), the
// K/64+1 group counts of P and of Q, then the parents of P and of Q at each
// depth above the 64-point nodes (2 (L - 6) K uint16)
constexpr size_t lds_core_bytes(int L)
{
    return (size_t)4 * (1 << L) * sizeof(uint16_t) + 2 * ((size_t)(1 << L) / 64 + 1) * 4 +
           (size_t)2 * (L - 6) * (1 << L) * sizeof(uint16_t);
}

// Inclusive prefix sum over the 64 lanes of a wave with DPP: four row_shr
// steps scan each row of 16 lanes, then row_bcast:15 and row_bcast:31 carry
// the row totals forward (lanes without a source add the old value, 0).
__device__ __forceinline__ int wave_incl_scan(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);   // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);   // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);   // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1, 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2, 3
    return x;
}

// An entry of U or CI counts at line r: lo ? idx >= r : idx < r.  With the
// lo flag in bit F of the entry and idx, r below 2^F this is bit F of e - r.
template <int F>
__device__ __forceinline__ uint32_t counted(uint32_t e, int r)
{
    return ((e - (uint32_t)r) >> F) & 1u;
}

// Position of the k-th set bit of w, of 2H bits (1 <= k <= popcount(w)).
template <int H>
__device__ __forceinline__ int select_bit(uint32_t w, int k)
{
    int pos = 0;
#pragma unroll
    for (int h = H; h >= 1; h >>= 1) {
        const int c = __popc(w & ((1u << h) - 1));
        const bool up = k > c;
        k -= up ? c : 0;
        w = up ? w >> h : w;
        pos += up ? h : 0;
    }
    return pos;
}
__device__ __forceinline__ int select64(uint32_t lo, uint32_t hi, int k)
{
    const int c = __popc(lo);
    const bool up = k > c;
    return (up ? 32 : 0) + select_bit<16>(up ? hi : lo, up ? k - c : k);
}

// Bit c (of 16) = entry c counts at this lane's line, for 16 entries held by
// the 16 lanes of each DPP row (lane l of the row: entry l), every entry and
// line shifted so that the counted bit of their difference is bit 31.  Each of
// the 16 rotations of the row subtracts and shifts one bit in (a v_sub with a
// DPP operand and a v_alignbit); after them bit b is the entry of lane
// (b + l + 1) mod 16.
__device__ __forceinline__ uint32_t counted_row16(uint32_t up, uint32_t rr, int lane)
{
    uint32_t w = (up - rr) >> 31, t;
    // in one block, as the compiler does not fold the rotation into the
    // subtract; the s_nop covers a DPP read of an `up` written just before
#define LCSB_ROR(I)                                                                     \
    "v_sub_u32_dpp %[t], %[e], %[r] row_ror:" #I " row_mask:0xf bank_mask:0xf\n\t"      \
    "v_alignbit_b32 %[w], %[w], %[t], 31\n\t"
    asm("s_nop 1\n\t" LCSB_ROR(1) LCSB_ROR(2) LCSB_ROR(3) LCSB_ROR(4) LCSB_ROR(5) LCSB_ROR(6) LCSB_ROR(7) LCSB_ROR(8)
            LCSB_ROR(9) LCSB_ROR(10) LCSB_ROR(11) LCSB_ROR(12) LCSB_ROR(13) LCSB_ROR(14) LCSB_ROR(15)
        : [w] "+v"(w), [t] "=&v"(t)
        : [e] "v"(up), [r] "v"(rr));
#undef LCSB_ROR
    return ((w | w << 16) >> (~lane & 15)) & 0xffffu;
}

__device__ __forceinline__ int lane_push(int dst, int x) { return __builtin_amdgcn_ds_permute(dst << 2, x); }
__device__ __forceinline__ int lane_pull(int src, int x) { return __builtin_amdgcn_ds_bpermute(src << 2, x); }

// The sticky product of 64 points in one wave: lane x holds row x's shared
// column kp and column x's shared row kq; returns row x's column.  All six
// depths stay in registers: the partitions and lifts move between lanes by
// ds_permute, and a node's T(r) comes from one mask of its columns per lane
// (each node is a single box entered at T(s) = 0).  Bound by VALU issue:
// about 1000 instructions per 64 points, 12 us of a 2048-point core's 75.
__device__ __forceinline__ int wave_product64(int kp, int kq, int lane)
{
    const unsigned long long lt = (1ull << lane) - 1;
    int pp[6], pq[6];
    auto split = [&](int &key, int s, int bit) {
        const int b = (key >> bit) & 1, seg = lane & ~(s - 1);
        const unsigned long long in = s == 64 ? ~0ull : ((1ull << (s & 63)) - 1) << seg, m = __ballot(b) & in;
        const int before = __popcll(m & lt), ones = __popcll(m);
        const int pos = b ? seg + s - ones + before : lane - before;
        const int v = lane_push(pos, key << 6 | lane);
        key = v >> 6;
        return v & 63;
    };
#pragma unroll
    for (int d = 0; d < 6; ++d) {
        pp[d] = split(kp, 64 >> d, 5 - d);
        pq[d] = split(kq, 64 >> d, 5 - d);
    }
    int R = 0;   // 1 x 1 nodes
#pragma unroll
    for (int d = 5; d >= 0; --d) {
        const int s = 64 >> d, h = s >> 1;
        const int p_pos = pp[d], q_pos = lane_pull((lane & ~(h - 1)) + R, pq[d]);
        const int p0 = p_pos & ~(s - 1);
        const uint32_t flag = (lane & h) ? 0u : 0x80u;
        const uint32_t u = (uint32_t)lane_push(p_pos, (int)((uint32_t)(q_pos - p0) | flag));
        const uint32_t ci = (uint32_t)lane_push(q_pos, (int)((uint32_t)(p_pos - p0) | flag));
        const int v0 = lane & ~(s - 1), r = lane - v0;
        const unsigned long long in = s == 64 ? ~0ull : ((1ull << (s & 63)) - 1) << v0;
        const int need = __popcll(__ballot((u & 0x80u) != 0) & in & ~lt);   // lo rows >= r
        // the node's columns 16 at a time: the lane's own DPP row and, in
        // larger nodes, the rows that lane_pull brings alongside
        const uint32_t up = ci << 24, rr = (uint32_t)r << 24;
        int T = 0;
        if (s <= 16) {
            const uint32_t w = (counted_row16(up, rr, lane) >> (v0 & 15)) & ((1u << (s & 31)) - 1);
            T = 1 + (s == 16 ? select_bit<8>(w, need) : s == 8 ? select_bit<4>(w, need) : s == 4 ? select_bit<2>(w, need)
                                                                                     : select_bit<1>(w, need));
        } else {
            uint32_t q[4] = {};
#pragma unroll
            for (int i = 0; i < s / 16; ++i)
                q[i] = counted_row16((uint32_t)lane_pull(v0 + 16 * i + (lane & 15), (int)up), rr, lane);
            const uint32_t lo = q[0] | q[1] << 16;
            T = 1 + (s == 32 ? select_bit<16>(lo, need) : select64(lo, q[2] | q[3] << 16, need));
        }
        T = need ? T : 0;
        const int lc = (int)(u & 0x7fu);
        R = T > 0 && counted<7>(u, T) ? T - 1 : lc;
        R &= s - 1;   // in range whatever an aborted comb fed in
    }
    return R;
}

// One wave's box of kBox rows r_lo .. r_lo + 63 of a node (lane l: row r_lo +
// l, entry u): the rows that the ant's path crosses with T in (cs, ce] (or T =
// cs, from a row line), ce - cs <= 64.  From a row line (COL false) every row
// is open and delta(r_lo + 64, cs) = 0; from a column line cs the rows up to
// rho are, and delta(rho, cs) = -1.  -delta(r, cs) adds the rows from r down
// to the line that count at cs; T(r) is the position after that many counted
// columns.  entry(c) reads column c's entry, c < ce; the caller may lower ce
// to T(r_lo), which no open row exceeds.  Returns the row's new column or -1.
template <int F, bool COL, typename Entry>
__device__ __forceinline__ int box_rows(uint32_t u, Entry entry, int r_lo, int rho, int cs, int ce, int lane)
{
    const int r = r_lo + lane;
    const bool uc = counted<F>(u, cs);
    const unsigned long long m = __ballot(COL ? uc && r < rho : uc);
    const int need = (COL ? 1 : 0) + (int)__popcll(m >> lane);
    const uint32_t rr = (uint32_t)r << (31 - F);
    uint32_t q[4] = {};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = cs + 16 * i + (lane & 15);
        if (cs + 16 * i < ce)   // uniform; past ce an entry that counts at no line
            q[i] = counted_row16(c < ce ? (uint32_t)entry(c) << (31 - F) : 0x7fffffffu, rr, lane);
    }
    const uint32_t lo = q[0] | q[1] << 16, hi = q[2] | q[3] << 16;
    const bool open = (!COL || r <= rho) && need <= __popc(lo) + __popc(hi);
    const int T = need ? cs + 1 + select64(lo, hi, need) : cs;
    return open && T > 0 && counted<F>(u, T) ? T - 1 : -1;
}

// One bottom-up depth (node size s >= 128) of a core in LDS: lift the
// children's products into node coordinates (the reference's
// inverse_mapping, :191-202), then the ant passage (:123-189) for every node:
// counts per 64-entry block and line, the crossing of each line, the boxes.
struct LeafLines {
    uint16_t T[2][kMaxLeafLines];                      // [0] row lines, [1] column lines (T = rho + 1), per node nb
    uint16_t lo[2][kMaxLeafLines];                     // lo entries per block of CI, of U
    uint8_t cnt[2][kMaxLeafLines][kMaxLeafLines];      // [dir][block][j]: z_j entries of the block
};
__device__ __forceinline__ void bottom_up_depth(uint16_t *U, uint16_t *CI, const uint16_t *R, uint16_t *Rn,
                                                const uint16_t *pp, const uint16_t *pq, int K, int s, LeafLines &B)
{
    const int h = s >> 1;
    // lift the children's products into node coordinates
#pragma unroll 2
    for (int x = threadIdx.x; x < K; x += kThreads) {
        const int p_pos = pp[x];
        const int cseg = x & ~(h - 1);
        const int q_pos = pq[cseg + (int)R[x]];
        const int v0 = p_pos & ~(s - 1);
        const uint16_t lo = (x & h) ? 0 : kLoFlag;
        const int lr = p_pos - v0, lc = q_pos - v0;
        U[p_pos] = (uint16_t)lc | lo;
        CI[v0 + lc] = (uint16_t)lr | lo;
        Rn[p_pos] = (uint16_t)lc;
    }
    __syncthreads();
    // Line j of a node (row line Dr = s - 64 j over the columns' entries CI,
    // column line c = s - 64 j over the rows' entries U): with bucket b =
    // (s-1-idx) / 64 of an entry, z_j = lo ? b < j : b >= j, Y_j = #{lo
    // entries with b < j} and T_j = the first position with Y_j z_j entries
    // before it.
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    constexpr int kWaves = kThreads / 64;
    const int nb = s >> 6, blocks = K >> 6, nodes = K / s;
    const unsigned long long lt = (1ull << lane) - 1;
    for (int t = wave; t < 2 * blocks; t += kWaves) {
        const int dir = t >= blocks, g = dir ? t - blocks : t;
        const uint32_t e = (dir ? U : CI)[g * 64 + lane];
        const unsigned long long los = __ballot((e & kLoFlag) != 0);
        const int bk = (s - 1 - (int)(e & kIdx)) >> 6;
        // lane j: the entries with bucket < j, from the buckets' bit planes
        unsigned long long lt_j = 0, eq = ~0ull;
        for (int p = nb >> 1; p; p >>= 1) {
            const unsigned long long plane = __ballot((bk & p) != 0), mine = (lane & p) ? ~0ull : 0ull;
            lt_j |= eq & ~plane & mine;
            eq &= ~(plane ^ mine);
        }
        if (lane < nb) B.cnt[dir][g][lane] = (uint8_t)(__popcll(los & lt_j) + __popcll(~los & ~lt_j));
        if (lane == 0) B.lo[dir][g] = (uint16_t)__popcll(los);
    }
    __syncthreads();
    // lines, up to kLineBatch per wave at once so that their LDS reads overlap
    constexpr int kLineBatch = 2 * kMaxLeafLines / kWaves;
    int lY[kLineBatch], lc[kLineBatch];
    uint32_t le[kLineBatch];
#pragma unroll
    for (int i = 0; i < kLineBatch; ++i) {
        const int t = wave + i * kWaves, dir = t >= blocks, q = dir ? t - blocks : t, j = q & (nb - 1), b0 = q - j;
        const bool on = t < 2 * blocks;
        // Y_j: the lo entries of the other array's last j blocks (their idx is
        // the position there)
        lY[i] = on && lane >= nb - j && lane < nb ? B.lo[dir ^ 1][b0 + lane] : 0;
        lc[i] = on && lane < nb ? B.cnt[dir][b0 + lane][j] : 0;
    }
#pragma unroll
    for (int i = 0; i < kLineBatch; ++i) {
        const int t = wave + i * kWaves, dir = t >= blocks, q = dir ? t - blocks : t;
        const int Y = __builtin_amdgcn_readlane(wave_incl_scan(lY[i]), 63), incl = wave_incl_scan(lc[i]);
        const unsigned long long reach = __ballot(lane < nb && incl >= Y);
        const int g = reach ? __ffsll((long long)reach) - 1 : 0;
        lY[i] = reach ? Y - __builtin_amdgcn_readlane(incl - lc[i], g) : 0;   // still needed in block g
        lc[i] = g;
        le[i] = t < 2 * blocks ? (dir ? U : CI)[(q & ~(nb - 1)) * 64 + g * 64 + lane] : 0;
    }
#pragma unroll
    for (int i = 0; i < kLineBatch; ++i) {
        const int t = wave + i * kWaves, dir = t >= blocks, q = dir ? t - blocks : t, j = q & (nb - 1);
        const int bk = (s - 1 - (int)(le[i] & kIdx)) >> 6;
        const bool z = (le[i] & kLoFlag) ? bk < j : bk >= j;
        const unsigned long long zm = __ballot(z);
        const unsigned long long hit = __ballot(z && (int)__popcll(zm & lt) == lY[i] - 1);
        if (lane == 0 && t < 2 * blocks && j) B.T[dir][q] = (uint16_t)(hit ? lc[i] * 64 + __ffsll((long long)hit) : 0);
    }
    __syncthreads();
    // boxes: piece q < nb of a node starts at row line j = q (q = 0: at T(s) =
    // 0), q >= nb at column line i = q - nb + 1
    const int per_node = 2 * nb - 1;
    for (int t = wave; t < nodes * per_node; t += kWaves) {
        const int node = t / per_node, q = t - node * per_node, v0 = node * s;
        int r_lo, cs, ce, rho;
        if (q < nb) {
            r_lo = s - (q + 1) * 64;
            rho = r_lo + 63;
            cs = q == 0 ? 0 : min((int)B.T[0][node * nb + q], s);
            ce = cs == 0 ? 64 : (((cs - 1) >> 6) + 1) << 6;
        } else {
            const int i = q - nb + 1, Tc = min((int)B.T[1][node * nb + nb - i], s);
            if (Tc == 0) continue;   // the ant never reaches this column line
            rho = Tc - 1;
            r_lo = rho & ~63;
            cs = i * 64;
            ce = cs + 64;
        }
        if (r_lo) ce = min(ce, (int)B.T[0][node * nb + nb - (r_lo >> 6)]);   // T(r_lo): open rows stay below it
        const uint32_t u = U[v0 + r_lo + lane];
        auto entry = [&](int c) { return CI[v0 + c]; };
        const int c = q < nb ? box_rows<15, false>(u, entry, r_lo, rho, cs, ce, lane)
                             : box_rows<15, true>(u, entry, r_lo, rho, cs, ce, lane);
        if (c >= 0) Rn[v0 + r_lo + lane] = (uint16_t)c;
    }
    __syncthreads();
}

// One depth of the top-down split with the keys in LDS, for P (waves
// 0 .. kSideW-1) and Q (the other half) at once: a stable partition of every
// aligned segment of size s by bit `bit` (zeros first), the ranks from wave
// ballots; par[pos] = old position.  Each wave counts the ones of its 64-key
// groups (gc, one word per group); after one barrier every wave scans all
// of its side's group counts itself (K <= 4096: at most 64 groups, one DPP
// scan), so a depth costs two barriers.  A wave takes the groups w, w +
// kSideW, ..., U at a time, with every load of the U groups issued before
// the first ballot, so their LDS latencies overlap (the compiler does not
// unroll a loop around a ballot by itself).  K >= 64.
constexpr int kSideW = kThreads / 128;
static_assert(kLdsCoreK <= 64 * 64, "one DPP scan covers a side's group counts");
template <int U>
__device__ __forceinline__ void split_count_groups(const uint16_t *key, int bit, int32_t *gc, int g0, int lane)
{
    uint16_t kv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) kv[u] = key[(g0 + u * kSideW) * 64 + lane];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const unsigned long long m = __ballot((kv[u] >> bit) & 1);
        if (lane == 0) gc[g0 + u * kSideW] = __popcll(m);
    }
}

// excl = exclusive prefix of the group counts at lane g, total = all ones
template <int U>
__device__ __forceinline__ void split_place_groups(const uint16_t *key, uint16_t *key_new, uint16_t *par, int s,
                                                   int bit, int excl, int total, int ngroups, int g0, int lane)
{
    const unsigned long long lt = (1ull << lane) - 1;
    uint16_t kv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) kv[u] = key[(g0 + u * kSideW) * 64 + lane];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int g = g0 + u * kSideW, x = g * 64 + lane;
        const int b = (kv[u] >> bit) & 1;
        const unsigned long long m = __ballot(b);
        const int seg = x & ~(s - 1);
        int before, ones;
        if (s >= 64) {
            // the segment's groups are gs .. ge-1; prefixes read from the scan
            const int gs = seg >> 6, ge = gs + (s >> 6);
            const int p_g = __builtin_amdgcn_readlane(excl, g), p_s = __builtin_amdgcn_readlane(excl, gs);
            const int p_e = ge < ngroups ? __builtin_amdgcn_readlane(excl, ge) : total;
            before = p_g - p_s + __popcll(m & lt);
            ones = p_e - p_s;
        } else {
            const unsigned long long segmask = ((1ull << s) - 1) << (lane & ~(s - 1));
            before = __popcll(m & lt & segmask);
            ones = __popcll(m & segmask);
        }
        const int pos = b ? seg + (s - ones) + before : seg + (x - seg - before);
        key_new[pos] = kv[u];
        par[pos] = (uint16_t)x;
    }
}

__device__ __forceinline__ void split_depth_pq(const uint16_t *keyP, uint16_t *keyP_new, uint16_t *parP,
                                               const uint16_t *keyQ, uint16_t *keyQ_new, uint16_t *parQ,
                                               int32_t *gcP, int32_t *gcQ, int K, int s, int bit)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool q_side = wave >= kSideW;
    const int w = q_side ? wave - kSideW : wave;
    const uint16_t *key = q_side ? keyQ : keyP;
    uint16_t *key_new = q_side ? keyQ_new : keyP_new, *par = q_side ? parQ : parP;
    int32_t *gc = q_side ? gcQ : gcP;
    const int ngroups = K >> 6;
    int g = w;
    for (; g + 3 * kSideW < ngroups; g += 4 * kSideW) split_count_groups<4>(key, bit, gc, g, lane);
    for (; g < ngroups; g += kSideW) split_count_groups<1>(key, bit, gc, g, lane);
    __syncthreads();
    const int c = lane < ngroups ? gc[lane] : 0;
    const int incl = wave_incl_scan(c);
    const int excl = incl - c, total = __builtin_amdgcn_readlane(incl, 63);
    g = w;
    for (; g + 3 * kSideW < ngroups; g += 4 * kSideW)
        split_place_groups<4>(key, key_new, par, s, bit, excl, total, ngroups, g, lane);
    for (; g < ngroups; g += kSideW) split_place_groups<1>(key, key_new, par, s, bit, excl, total, ngroups, g, lane);
    __syncthreads();
}

// The sticky product with keys, both products, the parents of every depth
// and the chunk entries in LDS for cores up to K = kLdsCoreK, one workgroup
// per core; the dynamic LDS is laid out as lds_core_bytes(L) says.  P holds
// row -> shared column; Q holds shared row -> column, or (QKEY) column ->
// shared row, the keys themselves.  Values are read modulo K (a leaf of a
// big core reads its slice of the big core's keys).
template <bool QKEY>
__device__ __forceinline__ void core_lds_body(const int32_t *P, const int32_t *Q, int32_t *Rout, int k, int L,
                                              uint16_t *lds, LeafLines &B)
{
    const int K = 1 << L, mask = K - 1;
    uint16_t *keyP = lds, *keyP2 = lds + K;                       // top-down
    uint16_t *keyQ = lds + 2 * (size_t)K, *keyQ2 = lds + 3 * (size_t)K;
    uint16_t *U = lds, *CI = lds + K;                             // bottom-up (reuses the key space)
    uint16_t *R = lds + 2 * (size_t)K, *Rn = lds + 3 * (size_t)K;
    int32_t *gcP = (int32_t *)(lds + 4 * (size_t)K), *gcQ = gcP + (K / 64 + 1);
    uint16_t *parP = lds + 4 * (size_t)K + 4 * ((size_t)K / 64 + 1);   // (L - 6) * K
    uint16_t *parQ = parP + (size_t)(L - 6) * K;                        // (L - 6) * K

    // P ordered by row (key = shared column), Q ordered by column (key = shared row)
    for (int x = threadIdx.x; x < K; x += kThreads) keyP[x] = (uint16_t)(x < k ? (P[x] & mask) : x);
    if (QKEY) {
        for (int x = threadIdx.x; x < K; x += kThreads) keyQ[x] = (uint16_t)(Q[x] & mask);
    } else {
        for (int x = threadIdx.x; x < K; x += kThreads)
            if (x >= k) keyQ[x] = (uint16_t)x;
        for (int r = threadIdx.x; r < k; r += kThreads)
            if ((uint32_t)Q[r] < (uint32_t)k) keyQ[Q[r]] = (uint16_t)r;
    }
    __syncthreads();
    const int D = L - 6;   // depths above the 64-point nodes
    for (int d = 0; d < D; ++d) {
        split_depth_pq(keyP, keyP2, parP + (size_t)d * K, keyQ, keyQ2, parQ + (size_t)d * K, gcP, gcQ, K, K >> d,
                       L - d - 1);
        uint16_t *t = keyP; keyP = keyP2; keyP2 = t;
        t = keyQ; keyQ = keyQ2; keyQ2 = t;
    }
    // the 64-point nodes, a wave each; R takes the place of Q's spare keys
    // only once every wave has read its keys
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    constexpr int kWaves = kThreads / 64, kPerWave = kLdsCoreK / 64 / kWaves;
    int prod[kPerWave];
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
        const int node = wave + i * kWaves;
        prod[i] = node < K / 64 ? wave_product64(keyP[node * 64 + lane] & 63, keyQ[node * 64 + lane] & 63, lane) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
        const int node = wave + i * kWaves;
        if (node < K / 64) R[node * 64 + lane] = (uint16_t)prod[i];
    }
    __syncthreads();
    for (int d = D - 1; d >= 0; --d) {
        bottom_up_depth(U, CI, R, Rn, parP + (size_t)d * K, parQ + (size_t)d * K, K, K >> d, B);
        uint16_t *tmp = R; R = Rn; Rn = tmp;
    }
    for (int x = threadIdx.x; x < k; x += kThreads) Rout[x] = R[x];
}

__global__ __launch_bounds__(kThreads) void braid_core_lds_kernel(CoreBatch batch)
{
    const BraidCoreDesc D = batch.d[blockIdx.x];
    extern __shared__ uint16_t lds[];
    __shared__ LeafLines lines;
    core_lds_body<false>(D.P, D.Q, D.R, D.k, D.L, lds, lines);
}

// ---------------------------------------------------------------- big cores
// Cores above kLdsCoreK run the same recursion spread over the whole GPU
// (the one-workgroup core finishes its top depths in the same boxes):
//  * the top d0 = L - L0 depths of the top-down split are device-wide
//    stable partitions (count, scan, scatter per depth);
//  * the 2^d0 nodes of depth d0 are independent sticky products of 2^L0
//    points each, one workgroup per node (core_lds_body on their keys);
//  * bottom-up, each top depth lifts the children's products into node
//    coordinates (inverse_mapping, src/braid_multiplication.hpp:191-202)
//    and runs the ant passage (:123-189) cut into boxes that a wave each
//    finishes.  The ant leaves row r at T(r) = min{c : delta(r, c) >= 0}
//    (delta non-decreasing in r and c), so its path is fixed by where it
//    crosses a grid of lines every g rows and every g columns of a node:
//      - row line Dr (= s - j g): enters row Dr-1 at column T(Dr), with
//        delta(Dr, T) = 0;
//      - column line c = i g: the ant steps right from (rho, c) to
//        (rho, c+1) at rho + 1 = min{r : delta(r, c) >= 0}, with
//        delta(rho, c) = -1.
//    Both are "first position where a running count reaches a target" over
//    the node's columns (row lines) or rows (column lines): with bucket
//    b(e) = (s-1-idx(e)) >> log2 g of an entry and boundary j,
//        z_j(e) = lo(e) ? b(e) < j : b(e) >= j,  Y_j = #{lo entries: b < j},
//        T_j = min{x : #{x' < x : z_j(e_x')} >= Y_j},
//    the column line c = i g being boundary j = s/g - i over the rows
//    (T_j = rho + 1).  Block histograms (big_hist_kernel), a search over
//    the blocks per boundary and a sweep of the one block where the count
//    crosses (big_sweep_kernel) find every T_j.  A piece starts at a
//    crossing and ends at the next one, so it stays inside one g x g box,
//    whose rows' T follow from its columns' entries (big_box_kernel).
// Entries of U (row -> column) and CI (column -> row) are node-local
// indices with the lo flag in bit 31.
constexpr int kBigBatch = 32;          // products per big-core launch
constexpr int kSplitTile = 2048;       // elements per block of a device-wide partition
constexpr int kMaxLines = 8192;        // grid lines per node and direction
// Box side of a node's grid: one wave per box takes 64 rows and 64 columns
// at a time, so 64 up to nodes of kMaxLines * 64 points, s / kMaxLines above.
constexpr uint32_t kLo31 = 0x80000000u;

struct BigCore {
    const int32_t *P, *Q;   // k: row -> shared column, shared row -> column
    int32_t *R;             // k: row -> column of the product
    int32_t *ws;            // lcsb_big_ws_words(k, L0) words
    int32_t k;
};
// grid of one top depth (node size s): lines every g = s / nb
struct BigDepth {
    int32_t s, nb, glog, w, nsegs;   // w entries per histogram block, nsegs per node
};

// Histogram blocks of w entries: every open boundary sweeps (on average)
// half a block, nb w / 2 entries per node and direction, while the
// blocks' prefixes cost about 2 (s / w)(nb + 1) words written and read;
// w = 2 sqrt(s) balances the two (clamped to [2^LCS_BIG_MIN_W_LOG, 8192],
// at most s = 2^e).
#ifndef LCS_BIG_MIN_W_LOG
#define LCS_BIG_MIN_W_LOG 9
#endif
static_assert(LCS_BIG_MIN_W_LOG >= 7 && LCS_BIG_MIN_W_LOG <= 11, "histogram block width");
__host__ __device__ constexpr int big_w_log(int e)
{
    const int wl = 1 + (e + 1) / 2;
    return wl < LCS_BIG_MIN_W_LOG ? LCS_BIG_MIN_W_LOG : (wl > 13 ? 13 : wl);
}
constexpr bool big_blocks_fit(int max_blocks)
{
    for (int e = 11; e <= kMaxCoreL; ++e)
        if ((1 << (e - (big_w_log(e) < e ? big_w_log(e) : e))) > max_blocks) return false;
    return true;
}

__host__ __device__ inline BigDepth big_depth(int L, int d)
{
    BigDepth D;
    D.s = 1 << (L - d);
    D.nb = D.s / kBox < kMaxLines ? D.s / kBox : kMaxLines;
    D.glog = __builtin_ctz((unsigned)(D.s / D.nb));
    D.w = 1 << big_w_log(L - d);
    if (D.w > D.s) D.w = D.s;
    D.nsegs = D.s / D.w;
    return D;
}

// word offsets inside one product's workspace
struct BigLayout {
    size_t keyP, keyQ, keyP2, keyQ2, parP, parQ, R, Rn, U, CI, cnt, hist, T, total;
};

__host__ __device__ inline BigLayout big_layout(int L, int L0)
{
    const size_t K = (size_t)1 << L;
    const int d0 = L - L0;
    BigLayout B;
    size_t o = 0;
    B.keyP = o; o += K;
    B.keyQ = o; o += K;
    B.keyP2 = o; o += K;
    B.keyQ2 = o; o += K;
    B.parP = o; o += (size_t)d0 * K;
    B.parQ = o; o += (size_t)d0 * K;
    B.R = o; o += K;
    B.Rn = o; o += K;
    B.U = o; o += K;
    B.CI = o; o += K;
    B.cnt = o; o += 3 * 2 * (K / kSplitTile);   // tile counts of P and Q, three depths in rotation
    size_t hist = 0, lines = 0;
    for (int d = 0; d < d0; ++d) {
        const BigDepth D = big_depth(L, d);
        const size_t nodes = K / (size_t)D.s;
        const size_t h = 2 * nodes * (size_t)D.nsegs * (size_t)(D.nb + 1);
        hist = h > hist ? h : hist;
        lines = nodes * (size_t)D.nb > lines ? nodes * (size_t)D.nb : lines;
    }
    B.hist = o; o += hist;
    B.T = o; o += 2 * lines;
    B.total = o;
    return B;
}

// The launch arguments of the big-core kernels: the products, and the
// workspace layout and the grid of every top depth, computed once on the
// host (per wave they were a loop of 64-bit divisions on the scalar unit).
struct BigBatch {
    BigCore c[kBigBatch];
    int32_t L, L0;
    BigLayout Y;
    BigDepth D[kMaxCoreL];
};

__global__ void big_init_kernel(BigBatch B)
{
    const BigCore &C = B.c[blockIdx.z];
    const BigLayout &Y = B.Y;
    const int K = 1 << B.L, x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= K) return;
    int32_t *keyP = C.ws + Y.keyP, *keyQ = C.ws + Y.keyQ;
    keyP[x] = x < C.k ? C.P[x] : x;
    if (x >= C.k) keyQ[x] = x;
    else if ((uint32_t)C.Q[x] < (uint32_t)C.k) keyQ[C.Q[x]] = x;
    // the tile counts of depths 1 and 2 are accumulated by the scatters
    // before them and start at zero
    const int ntiles = K / kSplitTile;
    if (x < 2 * 2 * ntiles) C.ws[Y.cnt + 2 * (size_t)ntiles + x] = 0;
}

// Depth-0 ones of the top bit per tile of kSplitTile keys (y = 0: P keys,
// 1: Q keys), into count buffer 0; every later depth's counts are
// accumulated by the scatter of the depth before.
__global__ __launch_bounds__(256) void big_split_count_kernel(BigBatch B, int d)
{
    const BigCore &C = B.c[blockIdx.z];
    const BigLayout &Y = B.Y;
    const int K = 1 << B.L, bit = B.L - d - 1, y = blockIdx.y;
    const int32_t *key = C.ws + (y ? ((d & 1) ? Y.keyQ2 : Y.keyQ) : ((d & 1) ? Y.keyP2 : Y.keyP));
    const int base = blockIdx.x * kSplitTile + threadIdx.x * 8;
    int c = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) c += (key[base + q] >> bit) & 1;
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    __shared__ int red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0)
        C.ws[Y.cnt + ((size_t)(d % 3) * 2 + y) * (K / kSplitTile) + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// Stable partition of every segment of size s by bit `bit` (zeros first);
// par[pos] = old position.  The block's own tile count prefix and its
// segment's total ones come from the tile counts of this depth (count
// buffer d % 3), summed by the block itself.  When another device-wide
// depth follows (NEXT), the block also counts the next bit's ones of the
// keys it places per destination tile -- its zeros and its ones each land
// in a run of at most kSplitTile positions, so at most two tiles each --
// and adds them to buffer (d + 1) % 3, and clears its own tile in buffer
// (d + 2) % 3 for the depth after that.
template <bool NEXT>
__global__ __launch_bounds__(256) void big_split_scatter_kernel(BigBatch B, int d)
{
    const BigCore &C = B.c[blockIdx.z];
    const BigLayout &Y = B.Y;
    const int K = 1 << B.L, s = K >> d, bit = B.L - d - 1, y = blockIdx.y;
    const int ntiles = K / kSplitTile;
    const int32_t *key = C.ws + (y ? ((d & 1) ? Y.keyQ2 : Y.keyQ) : ((d & 1) ? Y.keyP2 : Y.keyP));
    int32_t *key_new = C.ws + (y ? ((d & 1) ? Y.keyQ : Y.keyQ2) : ((d & 1) ? Y.keyP : Y.keyP2));
    int32_t *par = C.ws + (y ? Y.parQ : Y.parP) + (size_t)d * K;
    const int32_t *cnt = C.ws + Y.cnt + ((size_t)(d % 3) * 2 + y) * ntiles;
    const int base = blockIdx.x * kSplitTile + threadIdx.x * 8;
    int32_t kv[8];
    int c = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        kv[q] = key[base + q];
        c += (kv[q] >> bit) & 1;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // the segment's tiles t0 .. t0+nt-1; ones in the tiles before this one and in all of them
    const int seg = (blockIdx.x * kSplitTile) & ~(s - 1);
    const int t0 = seg / kSplitTile, nt = s / kSplitTile, mine = blockIdx.x - t0;
    int pre = 0, all = 0;
    for (int i = threadIdx.x; i < nt; i += 256) {
        const int v = cnt[t0 + i];
        all += v;
        pre += i < mine ? v : 0;
    }
    // exclusive prefix of the thread counts over the block, and the block sums
    const int incl = wave_incl_scan(c);
    for (int off = 32; off > 0; off >>= 1) {
        pre += __shfl_xor(pre, off);
        all += __shfl_xor(all, off);
    }
    __shared__ int wsum[4], wpre[4], wall[4];
    __shared__ int nz[2], no[2];
    if (lane == 63) wsum[wave] = incl;
    if (lane == 0) {
        wpre[wave] = pre;
        wall[wave] = all;
    }
    if (NEXT && threadIdx.x < 2) {
        nz[threadIdx.x] = 0;
        no[threadIdx.x] = 0;
    }
    __syncthreads();
    int before = incl - c;
    for (int w2 = 0; w2 < wave; ++w2) before += wsum[w2];
    const int before_tiles = wpre[0] + wpre[1] + wpre[2] + wpre[3];
    const int ones_total = wall[0] + wall[1] + wall[2] + wall[3];
    before += before_tiles;
    const int zeros_total = s - ones_total;
    // first destinations of the block's zeros and ones (their runs' first tiles)
    const int z0 = blockIdx.x * kSplitTile - before_tiles, o0 = seg + zeros_total + before_tiles;
    const int zt = z0 / kSplitTile, ot = o0 / kSplitTile;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int x = base + q;
        const int b = (kv[q] >> bit) & 1;
        const int pos = b ? seg + zeros_total + before : seg + (x - seg - before);
        before += b;
        key_new[pos] = kv[q];
        par[pos] = x;
        if (NEXT && ((kv[q] >> (bit - 1)) & 1))
            atomicAdd(b ? &no[pos / kSplitTile - ot] : &nz[pos / kSplitTile - zt], 1);
    }
    if (NEXT) {
        int32_t *next = C.ws + Y.cnt + ((size_t)((d + 1) % 3) * 2 + y) * ntiles;
        __syncthreads();
        if (threadIdx.x < 4) {
            const int v = threadIdx.x < 2 ? nz[threadIdx.x] : no[threadIdx.x - 2];
            const int tile = (threadIdx.x < 2 ? zt : ot) + (threadIdx.x & 1);
            if (v) atomicAdd(&next[tile], v);
        }
        if (threadIdx.x == 0) C.ws[Y.cnt + ((size_t)((d + 2) % 3) * 2 + y) * ntiles + blockIdx.x] = 0;
    }
}

// the 2^d0 independent nodes of depth d0, one workgroup each
__global__ __launch_bounds__(kThreads) void big_leaf_kernel(BigBatch B)
{
    const BigCore &C = B.c[blockIdx.z];
    const BigLayout &Y = B.Y;
    const int d0 = B.L - B.L0, s0 = 1 << B.L0;
    const size_t v0 = (size_t)blockIdx.x * s0;
    const int32_t *keyP = C.ws + ((d0 & 1) ? Y.keyP2 : Y.keyP) + v0;
    const int32_t *keyQ = C.ws + ((d0 & 1) ? Y.keyQ2 : Y.keyQ) + v0;
    extern __shared__ uint16_t lds[];
    __shared__ LeafLines lines;
    // depth d0 of the big core's own recursion: the products go to R
    core_lds_body<true>(keyP, keyQ, C.ws + Y.R + v0, s0, B.L0, lds, lines);
}

// lift the children's products into node coordinates (node size s).  The
// children's products are in R (flip = 0) or Rn (flip = 1), the node's go
// to the other one.
__global__ void big_lift_kernel(BigBatch B, int d, int flip)
{
    const BigCore &C = B.c[blockIdx.z];
    const BigLayout &Y = B.Y;
    const int K = 1 << B.L, s = K >> d, h = s >> 1;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= K) return;
    const int32_t *pp = C.ws + Y.parP + (size_t)d * K, *pq = C.ws + Y.parQ + (size_t)d * K;
    const int32_t *R = C.ws + (flip ? Y.Rn : Y.R);
    int32_t *Rn = C.ws + (flip ? Y.R : Y.Rn);
    uint32_t *U = (uint32_t *)(C.ws + Y.U), *CI = (uint32_t *)(C.ws + Y.CI);
    const int p_pos = pp[x];
    const int cseg = x & ~(h - 1);
    const int q_pos = pq[cseg + R[x]];
    const int v0 = p_pos & ~(s - 1);
    const uint32_t lo = (x & h) ? 0u : kLo31;
    const int lr = p_pos - v0, lc = q_pos - v0;
    U[p_pos] = (uint32_t)lc | lo;
    CI[v0 + lc] = (uint32_t)lr | lo;
    Rn[p_pos] = lc;
}

// Per histogram block (w entries of CI for y = 0, of U for y = 1): packed
// exclusive prefix over the buckets of (lo count | hi count << 16) for each
// boundary j < nb, and the packed totals at [nb].
__global__ __launch_bounds__(256) void big_hist_kernel(BigBatch B, int d)
{
    const BigCore &C = B.c[blockIdx.z];
    const BigLayout &Y = B.Y;
    const BigDepth &D = B.D[d];
    const int K = 1 << B.L, y = blockIdx.y;
    const uint32_t *E = (const uint32_t *)(C.ws + (y ? Y.U : Y.CI));
    __shared__ uint32_t h[kMaxLines];
    __shared__ uint32_t sums[4];
    for (int j = threadIdx.x; j < D.nb; j += 256) h[j] = 0;
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * D.w;
    for (int i = threadIdx.x; i < D.w; i += 256) {
        const uint32_t e = E[base + i];
        const int bk = (D.s - 1 - (int)(e & ~kLo31)) >> D.glog;
        atomicAdd(&h[bk], (e & kLo31) ? 1u : 0x10000u);
    }
    __syncthreads();
    // exclusive prefix in place: each of nw waves scans its nb / nw
    // consecutive buckets 64 at a time (DPP scan plus a carry; the packed
    // halves stay below 2^16, so they add without carrying into each
    // other), then the prefix leaves with consecutive threads on
    // consecutive buckets plus the totals of the waves before
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nw = D.nb >= 256 ? 4 : 1, chunk = D.nb / nw;   // nb is a power of two
    if (wave < nw) {
        uint32_t carry = 0;
        const int jb = wave * chunk, je = jb + chunk;
        for (int j0 = jb; j0 < je; j0 += 64) {
            const int j = j0 + lane;
            const uint32_t c = j < je ? h[j] : 0u;
            const uint32_t incl = (uint32_t)wave_incl_scan((int)c);
            if (j < je) h[j] = carry + incl - c;
            carry += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        }
        if (lane == 0) sums[wave] = carry;
    }
    __syncthreads();
    // per (y, node): the nsegs blocks' prefix rows of nb words (each block
    // writes its own row, coalesced), then the nsegs block totals in a row
    // of their own (read coalesced by the search)
    const int node = blockIdx.x / D.nsegs, g = blockIdx.x % D.nsegs, nodes = K / D.s;
    uint32_t *rows = (uint32_t *)(C.ws + Y.hist) + ((size_t)y * nodes + node) * D.nsegs * (size_t)(D.nb + 1);
    uint32_t *out = rows + (size_t)g * D.nb;
    const uint32_t w1 = sums[0], w2 = w1 + (nw > 1 ? sums[1] : 0u), w3 = w2 + (nw > 2 ? sums[2] : 0u);
    for (int j = threadIdx.x; j < D.nb; j += 256) {
        const int wj = j / chunk;
        out[j] = h[j] + (wj == 0 ? 0u : wj == 1 ? w1 : wj == 2 ? w2 : w3);
    }
    if (threadIdx.x == 0) rows[(size_t)D.nsegs * D.nb + g] = nw > 1 ? w3 + sums[3] : w1;
}

// The block of a node where the running count of z_j entries reaches Y_j.
// Hj[g * nb] = block g's prefix at j (lo | hi << 16 entries with bucket <
// j), Ht[g] = its totals: Y_j sums the lo parts; the block holds lo(P) +
// hi(total) - hi(P) z_j entries.  Lane l holds blocks l, l + 64, ... (R
// rounds, 64 R >= nsegs), all loaded in one batch from clamped (valid)
// blocks and masked afterwards; the rounds' wave scans find the first block
// where Z (z_j entries before it) plus its own count reaches Y_j.
template <int R>
__device__ __forceinline__ void block_search(const uint32_t *Hj, const uint32_t *Ht, int nb, int nsegs, int lane,
                                             int &Yj, int &Z, int &seg)
{
    uint32_t Pv[R], Tv[R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const int g = min(64 * u + lane, nsegs - 1);
        Pv[u] = Hj[(size_t)g * nb];
        Tv[u] = Ht[g];
    }
    int lo_sum = 0;
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const bool mine = 64 * u + lane < nsegs;
        Pv[u] = mine ? Pv[u] : 0u;
        Tv[u] = mine ? Tv[u] : 0u;
        lo_sum += (int)(Pv[u] & 0xffffu);
    }
    Yj = lo_sum;
    for (int off = 32; off > 0; off >>= 1) Yj += __shfl_xor(Yj, off);
    Z = 0;
    seg = nsegs - 1;
    bool found = false;   // uniform
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const int c = (int)(Pv[u] & 0xffffu) + (int)(Tv[u] >> 16) - (int)(Pv[u] >> 16);
        const int incl = wave_incl_scan(c);
        const unsigned long long reach = found ? 0ull : __ballot(Z + incl >= Yj);
        if (reach) {
            const int l = __ffsll((long long)reach) - 1;
            seg = min(64 * u + l, nsegs - 1);
            Z += __shfl(incl - c, l);
            found = true;
        } else if (!found) {
            Z += __builtin_amdgcn_readlane(incl, 63);
        }
    }
}

// The entry of a block of w entries (w >= 64 RS, a multiple of it) where
// the count of z_j entries reaches `need`: the block is read RS x 64
// entries at a time, all loads issued before the first ballot, so one
// memory latency covers that much of it.  Returns the entry's position
// + 1 in the block (0 if the count never gets there).
template <int RS>
__device__ __forceinline__ int sweep_block(const uint32_t *E, int w, int s, int glog, int j, int need, int lane)
{
    const unsigned long long lt = (1ull << lane) - 1;
    for (int r0 = 0; r0 < w; r0 += 64 * RS) {
        uint32_t ev[RS];
#pragma unroll
        for (int u = 0; u < RS; ++u) ev[u] = E[r0 + 64 * u + lane];
#pragma unroll
        for (int u = 0; u < RS; ++u) {
            const uint32_t e = ev[u];
            const int bk = (s - 1 - (int)(e & ~kLo31)) >> glog;
            const bool z = (e & kLo31) ? bk < j : bk >= j;
            const unsigned long long ball = __ballot(z);
            const int cnt = __popcll(ball);
            if (need <= cnt) {
                const bool hit = z && __popcll(ball & lt) == need - 1;
                return r0 + 64 * u + __ffsll((long long)__ballot(hit));
            }
            need -= cnt;
        }
    }
    return 0;
}

// One wave per (y, node, boundary j): Y_j and the block where the running
// count reaches it (block_search, at most kSegRounds x 64 blocks per node),
// then a sweep of that block (sweep_block) for the entry where the count
// reaches the rank still needed; T = that entry's position + 1.
// Boundaries with j = 0 or Y_j = 0 get T = 0.
constexpr int kSegRounds = 16;
static_assert(big_blocks_fit(64 * kSegRounds), "histogram blocks per node");
#ifndef LCS_SWEEP_WAVES
#define LCS_SWEEP_WAVES 4
#endif
constexpr int kSweepWaves = LCS_SWEEP_WAVES;   // waves (boundaries) per workgroup
__global__ __launch_bounds__(64 * kSweepWaves) void big_sweep_kernel(BigBatch B, int d)
{
    const BigCore &C = B.c[blockIdx.z];
    const BigLayout &Y = B.Y;
    const BigDepth &D = B.D[d];
    const int K = 1 << B.L, nodes = K / D.s, y = blockIdx.y;
    // the wave's boundary, made scalar so that its addresses stay in SGPRs
    const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * kSweepWaves + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (t >= nodes * D.nb) return;
    const int node = t / D.nb, j = t % D.nb;
    int32_t *T = C.ws + Y.T + (size_t)y * nodes * D.nb + t;
    if (j == 0) {
        if (lane == 0) *T = 0;
        return;
    }
    const uint32_t *H = (const uint32_t *)(C.ws + Y.hist) + ((size_t)y * nodes + node) * D.nsegs * (size_t)(D.nb + 1);
    const uint32_t *Hj = H + j, *Ht = H + (size_t)D.nsegs * D.nb;
    int Yj, Z, seg;
    if (D.nsegs <= 64) block_search<1>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    else if (D.nsegs <= 128) block_search<2>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    else if (D.nsegs <= 256) block_search<4>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    else if (D.nsegs <= 512) block_search<8>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    else block_search<kSegRounds>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    if (Yj == 0) {
        if (lane == 0) *T = 0;
        return;
    }
    const uint32_t *E = (const uint32_t *)(C.ws + (y ? Y.U : Y.CI)) + (size_t)node * D.s + (size_t)seg * D.w;
    // w is a power of two >= 128: the whole block in one batch up to 1024 entries
    const int need = Yj - Z;
    const int pos = D.w <= 128   ? sweep_block<2>(E, D.w, D.s, D.glog, j, need, lane)
                    : D.w <= 256 ? sweep_block<4>(E, D.w, D.s, D.glog, j, need, lane)
                    : D.w <= 512 ? sweep_block<8>(E, D.w, D.s, D.glog, j, need, lane)
                                 : sweep_block<16>(E, D.w, D.s, D.glog, j, need, lane);
    if (lane == 0 && pos) *T = seg * D.w + pos;
}

// One wave per piece of the ant's path.  Piece q < nb of a node starts at
// row line j = q (q = 0: the start of the passage at T(s) = 0), q >= nb at
// column line i = q - nb + 1; it stays in one g x g box (box_rows above says
// how its rows find T).  With g above 64 the rows go 64 at a time from the
// line upwards, carrying the rows counted so far, and the columns 64 at a
// time.  About 200 VALU and a few coalesced loads per wave; walking the boxes
// one lane each took 21 us per depth of a k = 2^16 product, this 3.  Whole
// products (random, kernel time, before and after boxes and wave_product64
// took the walks' place): k = 2^11 142 and 100 us, 2^16 344 and 215, 2^20
// 1419 and 1178.
constexpr int kBoxWaves = 4;   // pieces per workgroup
__global__ __launch_bounds__(64 * kBoxWaves) void big_box_kernel(BigBatch B, int d, int flip)
{
    const BigCore &C = B.c[blockIdx.z];
    const BigLayout &Y = B.Y;
    const BigDepth &D = B.D[d];
    const int K = 1 << B.L, s = D.s, nodes = K / s, g = 1 << D.glog, nb = D.nb;
    const int pieces = 2 * nb - 1, lane = threadIdx.x & 63;
    const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * kBoxWaves + (threadIdx.x >> 6));
    if (t >= nodes * pieces) return;
    const int node = t / pieces, q = t - node * pieces;
    const size_t v0 = (size_t)node * s;
    const uint32_t *U = (const uint32_t *)(C.ws + Y.U) + v0, *CI = (const uint32_t *)(C.ws + Y.CI) + v0;
    int32_t *Rn = C.ws + (flip ? Y.R : Y.Rn) + v0;
    // T lies in [0, s]; the clamps only keep every access inside the node
    // after an aborted comb fed undefined input
    int r_lo, rho, cs, ce;
    const bool col = q >= nb;
    if (!col) {
        r_lo = s - (q + 1) * g;
        rho = r_lo + g - 1;
        cs = q == 0 ? 0 : min(max(C.ws[Y.T + (size_t)node * nb + q], 0), s);
        ce = cs == 0 ? g : (((cs - 1) >> D.glog) + 1) << D.glog;
    } else {
        const int i = q - nb + 1;
        const int Tc = min(max(C.ws[Y.T + (size_t)nodes * nb + (size_t)node * nb + nb - i], 0), s);
        if (Tc == 0) return;   // the ant never reaches this column line
        rho = Tc - 1;
        r_lo = rho & ~(g - 1);
        cs = i * g;
        ce = cs + g;
    }
    auto entry = [&](int c) { return CI[c]; };
    if (g == kBox) {
        if (r_lo) ce = min(ce, min(max(C.ws[Y.T + (size_t)node * nb + nb - (r_lo >> D.glog)], 0), s));
        const uint32_t u = U[r_lo + lane];
        const int c = col ? box_rows<31, true>(u, entry, r_lo, rho, cs, ce, lane)
                          : box_rows<31, false>(u, entry, r_lo, rho, cs, ce, lane);
        if (c >= 0) Rn[r_lo + lane] = c;
        return;
    }
    int below = col ? 1 : 0;   // -delta(r, cs) just below the rows in hand
    for (int rb = (rho & ~63); rb >= r_lo; rb -= 64) {
        const int r = rb + lane;
        const uint32_t u = U[r];
        const bool uc = counted<31>(u, cs);
        const unsigned long long m = __ballot(col ? uc && r < rho : uc);
        int need = below + (int)__popcll(m >> lane);
        below += (int)__popcll(m);
        int T = need ? -1 : cs;
        for (int c0 = cs; c0 < ce; c0 += 64) {
            uint32_t q[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = c0 + 16 * i + (lane & 15);
                q[i] = counted_row16(c < ce ? entry(c) : ~kLo31, (uint32_t)r, lane);
            }
            const uint32_t lo = q[0] | q[1] << 16, hi = q[2] | q[3] << 16;
            const int cnt = __popc(lo) + __popc(hi);
            if (T < 0 && need <= cnt) T = c0 + 1 + select64(lo, hi, need);
            need -= cnt;
        }
        if ((!col || r <= rho) && T > 0 && counted<31>(u, T)) Rn[r] = T - 1;
    }
}

// the product of the last depth is in R (flip = 0) or Rn (flip = 1)
__global__ void big_out_kernel(BigBatch B, int flip)
{
    const BigCore &C = B.c[blockIdx.z];
    const BigLayout &Y = B.Y;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x < C.k) C.R[x] = C.ws[(flip ? Y.Rn : Y.R) + x];
}

// ---------------------------------------------------------------- slicing
// Device-wide stable compaction in three kernels: per-block counts, a scan
// of the counts in one block, per-block scatter.  The products of one merge
// level go through each kernel in one launch: blockIdx.y picks the slice
// (two per product, p's rows at even y and q's columns at odd y).
constexpr int kScanBlock = 256, kScanPer = 8, kScanTile = kScanBlock * kScanPer;
constexpr int kMulBatch = 32;   // products per slicing / assembly launch

struct SliceSpec {
    // selects element i of `src` (size n) when lo <= src[i] < hi; per-block
    // counts (then their exclusive scan) in `counts`; records, for slice j of
    // the selected elements (j < cap):
    //   even slice (vertical slice of p, rows in order):   map[j] = i, val[j] = src[i] - lo
    //   odd slice (horizontal slice of q, cols in order):  map[j] = i (a column), val[src[i] - lo] = j
    const int32_t *src;
    int32_t *counts, *map, *val;
    int32_t n, lo, hi, cap;
};
struct SliceBatch {
    SliceSpec s[2 * kMulBatch];
};

__device__ __forceinline__ bool sel(const SliceSpec &S, int i) { const int v = S.src[i]; return v >= S.lo && v < S.hi; }

__global__ void slice_count_kernel(SliceBatch B)
{
    const SliceSpec &S = B.s[blockIdx.y];
    if ((int64_t)blockIdx.x * kScanTile >= S.n) return;   // past this slice's blocks (whole block)
    __shared__ int32_t red[kScanBlock];
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanPer;
    int c = 0;
    for (int q = 0; q < kScanPer; ++q) c += (base + q < S.n) && sel(S, base + q);
    red[threadIdx.x] = c;
    __syncthreads();
    for (int off = kScanBlock / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) S.counts[blockIdx.x] = red[0];
}

__global__ void scan_counts_kernel(SliceBatch B)
{
    // exclusive scan of slice blockIdx.x's block counts in place, one block of 1024
    const SliceSpec &S = B.s[blockIdx.x];
    int32_t *counts = S.counts;
    const int nblocks = (S.n + kScanTile - 1) / kScanTile;
    __shared__ int32_t s[1024];
    const int t = threadIdx.x;
    const int per = (nblocks + 1023) / 1024;
    const int lo = min(t * per, nblocks), hi = min(lo + per, nblocks);
    int run = 0;
    for (int i = lo; i < hi; ++i) run += counts[i];
    s[t] = run;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        int v = t >= off ? s[t - off] : 0;
        __syncthreads();
        s[t] += v;
        __syncthreads();
    }
    int acc = s[t] - run;
    for (int i = lo; i < hi; ++i) { const int c = counts[i]; counts[i] = acc; acc += c; }
}

__global__ void slice_scatter_kernel(SliceBatch B)
{
    const SliceSpec &S = B.s[blockIdx.y];
    if ((int64_t)blockIdx.x * kScanTile >= S.n) return;   // past this slice's blocks (whole block)
    const bool rows = (blockIdx.y & 1) == 0;
    __shared__ int32_t s[kScanBlock];
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanPer;
    int c = 0;
    for (int q = 0; q < kScanPer; ++q) c += (base + q < S.n) && sel(S, base + q);
    s[threadIdx.x] = c;
    __syncthreads();
    for (int off = 1; off < kScanBlock; off <<= 1) {
        int v = (int)threadIdx.x >= off ? s[threadIdx.x - off] : 0;
        __syncthreads();
        s[threadIdx.x] += v;
        __syncthreads();
    }
    int j = S.counts[blockIdx.x] + s[threadIdx.x] - c;
    for (int q = 0; q < kScanPer; ++q) {
        const int i = base + q;
        if (i < S.n && sel(S, i) && j < S.cap) {
            S.map[j] = i;
            if (rows) S.val[j] = S.src[i] - S.lo;
            else S.val[S.src[i] - S.lo] = j;
            ++j;
        }
    }
}

struct InvertBatch {
    struct {
        const int32_t *r2c;
        int32_t *c2r;
        int32_t n;
    } s[kMulBatch];
};

__global__ void invert_kernel(InvertBatch B)
{
    const auto &S = B.s[blockIdx.y];
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;   // no wrap near 2^31
    if (i < S.n && (uint32_t)S.r2c[i] < (uint32_t)S.n) S.c2r[S.r2c[i]] = (int32_t)i;
}

struct AssembleBatch {
    AssembleArgs a[kMulBatch];
};

// Writes the product (row -> col) from the core result and the untouched
// points of p and q (braid_multiplication.hpp:353-401).
__global__ void assemble_kernel(AssembleBatch B)
{
    const AssembleArgs &A = B.a[blockIdx.y];
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;   // no wrap near 2^31
    const int k = A.k, ps = A.p_size, qs = A.q_size;
    // the range tests only matter after an aborted comb fed undefined input
    if (i < k && (uint32_t)A.core[i] < (uint32_t)k) {
        const int row = A.map_row[i], col = A.map_col[A.core[i]];
        if ((uint32_t)row < (uint32_t)ps) {
            if (A.row_glue) A.out[qs - k + row] = col;
            else A.out[row] = col + ps - k;
        }
    }
    if (i < ps) {
        const int c = A.p[i];
        if (A.row_glue) { if (c >= k) A.out[i + qs - k] = c + qs - k; }
        else { if (c < ps - k) A.out[i] = c; }
    }
    if (i < qs) {
        const int c = A.q[i];
        if (A.row_glue) { if (i < qs - k) A.out[i] = c; }
        else { if (i >= k) A.out[i - k + ps] = c - k + ps; }
    }
}

}  // namespace lcsb

using namespace lcsb;

// Cores of 2^L points with L >= kBigMinL run over the whole GPU, with
// leaves of at most 2^kBigLeafMaxL points (at least 2^10: the device-wide
// partitions work on tiles of 2048 keys inside nodes of 2^(leaf+1); at most
// 2^kLdsCoreL: a leaf is one workgroup's LDS core).
// Measured on the Zipf pair's five merge levels (k = 2^14, 16 .. 1 products
// per level): one workgroup per core 15.6 ms for the whole pair; whole-GPU
// cores with leaves of 2^10 / 2^11 / 2^12 points 12.5 / 12.3 / 12.5 ms.
#ifndef LCS_BIG_MIN_L
#define LCS_BIG_MIN_L 12
#endif
#ifndef LCS_BIG_LEAF_L
#define LCS_BIG_LEAF_L 11
#endif
// cores of 2^16 points and more take leaves of up to 2^LCS_BIG_LEAF_L_LARGE
#ifndef LCS_BIG_LEAF_L_LARGE
#define LCS_BIG_LEAF_L_LARGE 11
#endif
constexpr int kBigMinL = LCS_BIG_MIN_L;
constexpr int kBigLeafMaxL = LCS_BIG_LEAF_L;
constexpr int kBigLeafLargeL = LCS_BIG_LEAF_L_LARGE;
static_assert(kBigMinL >= 11 && kBigMinL <= kLdsCoreL + 1 && kBigLeafMaxL >= 10 && kBigLeafMaxL <= kLdsCoreL &&
                  kBigLeafLargeL >= 10 && kBigLeafLargeL <= kLdsCoreL,
              "big-core leaf sizes");
static int big_leaf_L(int L)
{
    const int lim = L >= 16 ? kBigLeafLargeL : kBigLeafMaxL;
    return L - 1 < lim ? L - 1 : lim;
}
static bool is_big(int L) { return L >= kBigMinL; }

size_t lcsb_core_scratch_words(int32_t k)
{
    const int L = lcsb_core_L(k);
    if (!is_big(L)) return 0;   // the one-workgroup core keeps everything in LDS
    return big_layout(L, big_leaf_L(L)).total;
}

// Padded core size 2^L: at least 64 (the LDS kernel ranks keys by wave
// ballots over groups of 64); padding adds fixed points only.
int lcsb_core_L(int32_t k)
{
    int L = 6;
    while ((1 << L) < k) ++L;
    return L;
}

// The big-core sequence for up to kBigBatch products of one padded size.
static int launch_big(const BigBatch &B, int cnt, hipStream_t stream)
{
    const int L = B.L, L0 = B.L0, d0 = L - L0, K = 1 << L;
    const dim3 lin((unsigned)(K / 256), 1, (unsigned)cnt), tiles((unsigned)(K / kSplitTile), 2, (unsigned)cnt);
    hipLaunchKernelGGL(big_init_kernel, lin, dim3(256), 0, stream, B);
    hipLaunchKernelGGL(big_split_count_kernel, tiles, dim3(256), 0, stream, B, 0);
    for (int d = 0; d < d0; ++d) {
        if (d + 1 < d0) hipLaunchKernelGGL(big_split_scatter_kernel<true>, tiles, dim3(256), 0, stream, B, d);
        else hipLaunchKernelGGL(big_split_scatter_kernel<false>, tiles, dim3(256), 0, stream, B, d);
    }
    hipLaunchKernelGGL(big_leaf_kernel, dim3(1u << d0, 1, (unsigned)cnt), dim3(kThreads), lds_core_bytes(L0),
                       stream, B);
    int flip = 0;
    for (int d = d0 - 1; d >= 0; --d) {
        const BigDepth D = big_depth(L, d);
        const int lines = (K / D.s) * D.nb, pieces = (K / D.s) * (2 * D.nb - 1);
        hipLaunchKernelGGL(big_lift_kernel, lin, dim3(256), 0, stream, B, d, flip);
        hipLaunchKernelGGL(big_hist_kernel, dim3((unsigned)(K / D.w), 2, (unsigned)cnt), dim3(256), 0, stream, B, d);
        hipLaunchKernelGGL(big_sweep_kernel, dim3((unsigned)((lines + kSweepWaves - 1) / kSweepWaves), 2, (unsigned)cnt),
                           dim3(64 * kSweepWaves), 0, stream,
                           B, d);
        hipLaunchKernelGGL(big_box_kernel, dim3((unsigned)((pieces + kBoxWaves - 1) / kBoxWaves), 1, (unsigned)cnt),
                           dim3(64 * kBoxWaves), 0, stream, B, d, flip);
        flip ^= 1;
    }
    hipLaunchKernelGGL(big_out_kernel, lin, dim3(256), 0, stream, B, flip);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

// The dynamic LDS limit of the core kernels, set once per process (before
// any capture: it is not a stream operation).
int lcsb_init(void)
{
    static std::once_flag once;
    static int rc = 0;
    std::call_once(once, [] {
        if (hipFuncSetAttribute((const void *)braid_core_lds_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds_core_bytes(kLdsCoreL)) != hipSuccess ||
            hipFuncSetAttribute((const void *)big_leaf_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds_core_bytes(kLdsCoreL)) != hipSuccess)
            rc = -5;
    });
    return rc;
}

int lcsb_launch_core(const BraidCoreDesc *descs, int count, hipStream_t stream)
{
    if (lcsb_init()) return -5;
    // small cores: one workgroup each, descriptors by value in the arguments
    std::vector<BraidCoreDesc> small;
    std::vector<BraidCoreDesc> big;
    for (int i = 0; i < count; ++i) {
        if (descs[i].L > kMaxCoreL) return -34;
        (is_big(descs[i].L) ? big : small).push_back(descs[i]);
    }
    for (size_t base = 0; base < small.size(); base += kCoreBatch) {
        CoreBatch batch{};
        const int cnt = (int)std::min<size_t>(small.size() - base, kCoreBatch);
        int max_L = 0;
        for (int i = 0; i < cnt; ++i) {
            batch.d[i] = small[base + (size_t)i];
            max_L = std::max(max_L, (int)batch.d[i].L);
        }
        if (max_L > kLdsCoreL) return -34;
        hipLaunchKernelGGL(braid_core_lds_kernel, dim3(cnt), dim3(kThreads), lds_core_bytes(max_L), stream, batch);
    }
    // big cores: products of one padded size share each launch of the sequence
    std::sort(big.begin(), big.end(), [](const BraidCoreDesc &x, const BraidCoreDesc &y) { return x.L < y.L; });
    for (size_t i = 0; i < big.size();) {
        BigBatch B{};
        B.L = big[i].L;
        B.L0 = big_leaf_L(B.L);
        B.Y = big_layout(B.L, B.L0);
        for (int d = 0; d < B.L - B.L0; ++d) B.D[d] = big_depth(B.L, d);
        int cnt = 0;
        while (i < big.size() && big[i].L == B.L && cnt < kBigBatch) {
            B.c[cnt++] = BigCore{big[i].P, big[i].Q, big[i].R, big[i].scratch, big[i].k};
            ++i;
        }
        const int rc = launch_big(B, cnt, stream);
        if (rc) return rc;
    }
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

// staggered_multiply for `count` independent products on device pointers.
// Their slicing, cores and assembly each go to one launch per kind (in
// groups of kMulBatch products for the slicing and assembly), so the
// products of a merge-tree level run side by side.  specs[i].ws holds
// lcsb_multiply_ws_words(p_size, q_size, k) words.
int lcsb_multiply_many_device(const MulSpec *specs, int count, hipStream_t stream)
{
    std::vector<BraidCoreDesc> cores;
    cores.reserve((size_t)count);
    auto nblocks = [](int32_t n) { return (n + kScanTile - 1) / kScanTile; };
    for (int base = 0; base < count; base += kMulBatch) {
        const int cnt = count - base < kMulBatch ? count - base : kMulBatch;
        InvertBatch ib{};
        SliceBatch sb{};
        int ni = 0, inv_blocks = 0, slice_blocks = 0;
        for (int i = 0; i < cnt; ++i) {
            const MulSpec &M = specs[base + i];
            const int32_t p_size = M.p_size, q_size = M.q_size, k = M.k;
            if (k == 0) continue;
            const int nmax = p_size > q_size ? p_size : q_size;
            const int nblocks_max = nblocks(nmax) + 1;
            int32_t *q_c2r = M.ws;                // q_size
            int32_t *map_row = q_c2r + q_size;    // k
            int32_t *map_col = map_row + k;       // k
            int32_t *Pred = map_col + k;          // k
            int32_t *Qred = Pred + k;             // k
            int32_t *core = Qred + k;             // k
            int32_t *counts_p = core + k;         // nblocks_max
            int32_t *counts_q = counts_p + nblocks_max;
            int32_t *core_ws = counts_q + nblocks_max;
            ib.s[ni].r2c = M.q;
            ib.s[ni].c2r = q_c2r;
            ib.s[ni].n = q_size;
            // vertical slice of p: rows whose column lies in the glued range
            sb.s[2 * ni] = SliceSpec{M.p, counts_p, map_row, Pred, p_size, M.row_glue ? 0 : p_size - k,
                                     M.row_glue ? k : p_size, k};
            // horizontal slice of q: columns whose row lies in the glued range
            sb.s[2 * ni + 1] = SliceSpec{q_c2r, counts_q, map_col, Qred, q_size, M.row_glue ? q_size - k : 0,
                                         M.row_glue ? q_size : k, k};
            ++ni;
            inv_blocks = std::max(inv_blocks, (q_size + 255) / 256);
            slice_blocks = std::max(slice_blocks, std::max(nblocks(p_size), nblocks(q_size)));
            BraidCoreDesc h{};
            h.P = Pred;
            h.Q = Qred;
            h.R = core;
            h.k = k;
            h.L = lcsb_core_L(k);
            h.scratch = core_ws;
            cores.push_back(h);
        }
        if (ni == 0) continue;
        hipLaunchKernelGGL(invert_kernel, dim3(inv_blocks, ni), dim3(256), 0, stream, ib);
        hipLaunchKernelGGL(slice_count_kernel, dim3(slice_blocks, 2 * ni), dim3(kScanBlock), 0, stream, sb);
        hipLaunchKernelGGL(scan_counts_kernel, dim3(2 * ni), dim3(1024), 0, stream, sb);
        hipLaunchKernelGGL(slice_scatter_kernel, dim3(slice_blocks, 2 * ni), dim3(kScanBlock), 0, stream, sb);
    }
    if (!cores.empty()) {
        const int rc = lcsb_launch_core(cores.data(), (int)cores.size(), stream);
        if (rc) return rc;
    }
    for (int base = 0; base < count; base += kMulBatch) {
        const int cnt = count - base < kMulBatch ? count - base : kMulBatch;
        AssembleBatch ab{};
        int blocks = 1;
        for (int i = 0; i < cnt; ++i) {
            const MulSpec &M = specs[base + i];
            int32_t *map_row = M.ws + M.q_size, *map_col = map_row + M.k, *core = map_col + 3 * (size_t)M.k;
            ab.a[i] = AssembleArgs{M.p, M.q, M.out, map_row, map_col, core, M.p_size, M.q_size, M.k, M.row_glue};
            const int n = std::max(std::max(M.p_size, M.q_size), M.k);
            blocks = std::max(blocks, (n + 255) / 256);
        }
        hipLaunchKernelGGL(assemble_kernel, dim3(blocks, cnt), dim3(256), 0, stream, ab);
    }
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

// staggered_multiply on device pointers; ws must hold lcsb_multiply_ws_words(...)
int lcsb_multiply_device(const int32_t *p, int32_t p_size, const int32_t *q, int32_t q_size, int32_t k,
                         int32_t row_glue, int32_t *out, int32_t *ws, hipStream_t stream)
{
    const MulSpec M{p, p_size, q, q_size, k, row_glue, out, ws};
    return lcsb_multiply_many_device(&M, 1, stream);
}

size_t lcsb_multiply_ws_words(int32_t p_size, int32_t q_size, int32_t k)
{
    const int nmax = p_size > q_size ? p_size : q_size;
    const size_t nblocks_max = (size_t)(nmax + kScanTile - 1) / kScanTile + 1;
    return (size_t)q_size + 5 * (size_t)k + 2 * nblocks_max + lcsb_core_scratch_words(k > 0 ? k : 1);
}
