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
#include <vector>

#include "braid_kernels.h"
#include "per_device.h"

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
// to T(r_lo), which no open row exceeds.  Returns the row's column in the
// product, or -1 for a row of another piece.
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
    const int c = T > 0 && counted<F>(u, T) ? T - 1 : (int)(u & ~(1u << F));
    return open ? c : -1;
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

// One product p (.) q glued on k strands, as every kernel of the sequence
// takes it (by value in the launch arguments).  The workspace holds q's
// inverse, the rows of p and the columns of q that the core's strands stand
// for, the block counts of the two slices, and the core's own words, which
// begin with the keys: keyP[x] = shared strand of the core's row x, keyQ[x] =
// shared strand of its column x.
constexpr int kScanBlock = 256, kScanPer = 8, kScanTile = kScanBlock * kScanPer;
// Every workgroup of a slice adds up the counts of those before it, so their
// number is bounded (2^26 points a side, k = 64: 2.47 ms with a workgroup per
// tile, 2.36 with at most 4096, 2.18 with whole lines stored as well).
constexpr int kMaxSliceBlocks = 4096;
constexpr int kLinesMin = 1 << 18;   // points from which a slice stores whole lines (slice_scatter_kernel)
static_assert(kLinesMin / kScanTile < kMaxSliceBlocks, "one tile a workgroup below");
constexpr int kMulBatch = 32;   // products per launch
struct MulArgs {
    const int32_t *p, *q;
    int32_t *out, *ws;
    int32_t p_size, q_size, k, row_glue, L;
    int32_t run, blocks;   // tiles of kScanTile points that a workgroup of a slice takes, and the workgroups
    int32_t big;           // the core runs over the whole GPU
    __host__ __device__ int32_t *q_c2r() const { return ws; }
    __host__ __device__ int32_t *map_row() const { return ws + q_size; }
    __host__ __device__ int32_t *map_col() const { return map_row() + k; }
    // (on the host: a division in every kernel of a product took 6 of 155 us)
    void set_blocks()
    {
        const int32_t tiles = (p_size > q_size ? p_size : q_size) / kScanTile + 1;
        run = (tiles + kMaxSliceBlocks - 1) / kMaxSliceBlocks;
        blocks = (tiles + run - 1) / run;
    }
    __host__ __device__ int32_t *counts(int side) const { return map_col() + k + side * blocks; }
    __host__ __device__ int32_t *core() const { return counts(2); }
    // row i of the core goes to column c: the product's point
    // (braid_multiplication.hpp:353-401); the range tests only matter after an
    // aborted comb fed undefined input
    __device__ __forceinline__ void put(int i, int c) const
    {
        if (i >= k || (uint32_t)c >= (uint32_t)k) return;
        const int row = map_row()[i], col = map_col()[c];
        if ((uint32_t)row >= (uint32_t)p_size) return;
        if (row_glue) out[q_size - k + row] = col;
        else out[row] = col + p_size - k;
    }
};
struct MulBatch {
    MulArgs m[kMulBatch];
};

// The sticky product with keys, both products, the parents of the depths
// above the 64-point nodes and the line tables in LDS for cores up to K =
// kLdsCoreK, one workgroup per core; the dynamic LDS is laid out as
// lds_core_bytes(L) says.  P holds row -> shared strand, Q column -> shared
// strand, for the first k of K (the rest are fixed points); values are read
// modulo K (a leaf of a big core reads its slice of the big core's keys).
// done(x, c) receives row x's column.
template <typename Done>
__device__ __forceinline__ void core_lds_body(const int32_t *P, const int32_t *Q, int k, int L, uint16_t *lds,
                                              LeafLines &B, Done done)
{
    const int K = 1 << L, mask = K - 1;
    uint16_t *keyP = lds, *keyP2 = lds + K;                       // top-down
    uint16_t *keyQ = lds + 2 * (size_t)K, *keyQ2 = lds + 3 * (size_t)K;
    uint16_t *U = lds, *CI = lds + K;                             // bottom-up (reuses the key space)
    uint16_t *R = lds + 2 * (size_t)K, *Rn = lds + 3 * (size_t)K;
    int32_t *gcP = (int32_t *)(lds + 4 * (size_t)K), *gcQ = gcP + (K / 64 + 1);
    uint16_t *parP = lds + 4 * (size_t)K + 4 * ((size_t)K / 64 + 1);   // (L - 6) * K
    uint16_t *parQ = parP + (size_t)(L - 6) * K;                        // (L - 6) * K

    for (int x = threadIdx.x; x < K; x += kThreads) {
        const int kp = x < k ? P[x] : x, kq = x < k ? Q[x] : x;
        keyP[x] = (uint16_t)(kp & mask);
        keyQ[x] = (uint16_t)(kq & mask);
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
    for (int x = threadIdx.x; x < K; x += kThreads) done(x, (int)R[x]);
}

__global__ __launch_bounds__(kThreads) void braid_core_lds_kernel(MulBatch B)
{
    const MulArgs &M = B.m[blockIdx.x];
    extern __shared__ uint16_t lds[];
    __shared__ LeafLines lines;
    const int32_t *key = M.core();
    core_lds_body(key, key + (1 << M.L), M.k, M.L, lds, lines, [&](int x, int c) { M.put(x, c); });
}

// ---------------------------------------------------------------- big cores
// Cores from 2^kBigMinL on run the same recursion spread over the whole GPU
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
constexpr int kSplitTile = 2048;       // elements per block of a device-wide partition
constexpr int kMaxLines = 8192;        // grid lines per node and direction
// Box side of a node's grid: one wave per box takes 64 rows and 64 columns
// at a time, so 64 up to nodes of kMaxLines * 64 points, s / kMaxLines above.
constexpr uint32_t kLo31 = 0x80000000u;

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

// word offsets inside one core's words; U and CI (64-bit pairs would not
// coalesce with the row and column reads) alternate between two sets, as a
// depth's boxes read one while they lift into the next depth's
struct BigLayout {
    size_t keyP, keyQ, keyP2, keyQ2, parP, parQ, U[2], CI[2], cnt, hist, total;
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
    for (int i = 0; i < 2; ++i) {
        B.U[i] = o; o += K;
        B.CI[i] = o; o += K;
    }
    B.cnt = o; o += 3 * 2 * (K / kSplitTile);   // tile counts of P and Q, three depths in rotation
    size_t hist = 0;
    for (int d = 0; d < d0; ++d) {
        const BigDepth D = big_depth(L, d);
        const size_t h = 2 * (K / (size_t)D.s) * (size_t)D.nsegs * (size_t)(D.nb + 1);
        hist = h > hist ? h : hist;
    }
    B.hist = o; o += hist;
    B.total = o;
    return B;
}

// Leaves of a core of 2^L points: one workgroup's LDS core each, of 2^10 points
// up to 2^18 (the leaf is VALU-bound on its CU, and few leaves leave most CUs
// idle), of 2^11 above (one device-wide depth less).  Kernel time with leaves
// of 2^10 and 2^11: k = 2^12 106 and 127 us, 2^16 197 and 215, 2^18 355 and
// 361, 2^20 1249 and 1178.
constexpr int kBigMinL = 11;
__host__ __device__ constexpr int big_leaf_L(int L) { return L > 18 ? 11 : 10; }
static_assert(kLdsCoreL >= 11, "leaves fit the LDS core");
// the tile counts' offset, for kernels without a BigBatch
__host__ __device__ inline size_t big_layout_cnt(int L)
{
    return ((size_t)8 + 2 * (size_t)(L - big_leaf_L(L))) << L;
}

// The launch arguments of the big-core kernels: the products, and the
// workspace layout and the grid of every top depth, computed once on the
// host (per wave they were a loop of 64-bit divisions on the scalar unit).
struct BigBatch {
    MulArgs c[kMulBatch];
    int32_t L, L0;
    BigLayout Y;
    BigDepth D[kMaxCoreL];
};

// Row x of a node of depth d + 1 goes to its local column c (node at v0, size
// h): its point in the parent, node size 2 h at depth d, written to that
// depth's U (row -> column) and CI (column -> row).
__device__ __forceinline__ void big_lift(const BigBatch &B, int32_t *w, int d, int v0, int h, int x, int c)
{
    const size_t K = (size_t)1 << B.L;
    const int p_pos = w[B.Y.parP + (size_t)d * K + x], q_pos = w[B.Y.parQ + (size_t)d * K + v0 + (c & (h - 1))];
    const int p0 = p_pos & ~(2 * h - 1);
    const uint32_t lo = (x & h) ? 0u : kLo31;
    ((uint32_t *)w)[B.Y.U[d & 1] + p_pos] = (uint32_t)(q_pos - p0) | lo;
    ((uint32_t *)w)[B.Y.CI[d & 1] + q_pos] = (uint32_t)(p_pos - p0) | lo;
}

// Depth-0 ones of the top bit per tile of kSplitTile keys (y = 0: P keys,
// 1: Q keys), into count buffer 0; every later depth's counts are
// accumulated by the scatter of the depth before.
__global__ __launch_bounds__(256) void big_split_count_kernel(BigBatch B, int d)
{
    int32_t *const w = B.c[blockIdx.z].core();
    const BigLayout &Y = B.Y;
    const int K = 1 << B.L, bit = B.L - d - 1, y = blockIdx.y;
    const int32_t *key = w + (y ? ((d & 1) ? Y.keyQ2 : Y.keyQ) : ((d & 1) ? Y.keyP2 : Y.keyP));
    const int base = blockIdx.x * kSplitTile + threadIdx.x * 8;
    int c = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) c += (key[base + q] >> bit) & 1;
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    __shared__ int red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0)
        w[Y.cnt + ((size_t)(d % 3) * 2 + y) * (K / kSplitTile) + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
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
    int32_t *const w = B.c[blockIdx.z].core();
    const BigLayout &Y = B.Y;
    const int K = 1 << B.L, s = K >> d, bit = B.L - d - 1, y = blockIdx.y;
    const int ntiles = K / kSplitTile;
    const int32_t *key = w + (y ? ((d & 1) ? Y.keyQ2 : Y.keyQ) : ((d & 1) ? Y.keyP2 : Y.keyP));
    int32_t *key_new = w + (y ? ((d & 1) ? Y.keyQ : Y.keyQ2) : ((d & 1) ? Y.keyP : Y.keyP2));
    int32_t *par = w + (y ? Y.parQ : Y.parP) + (size_t)d * K;
    const int32_t *cnt = w + Y.cnt + ((size_t)(d % 3) * 2 + y) * ntiles;
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
        int32_t *next = w + Y.cnt + ((size_t)((d + 1) % 3) * 2 + y) * ntiles;
        __syncthreads();
        if (threadIdx.x < 4) {
            const int v = threadIdx.x < 2 ? nz[threadIdx.x] : no[threadIdx.x - 2];
            const int tile = (threadIdx.x < 2 ? zt : ot) + (threadIdx.x & 1);
            if (v) atomicAdd(&next[tile], v);
        }
        if (threadIdx.x == 0) w[Y.cnt + ((size_t)((d + 2) % 3) * 2 + y) * ntiles + blockIdx.x] = 0;
    }
}

// the 2^d0 independent nodes of depth d0, one workgroup each, lifted into
// depth d0 - 1
__global__ __launch_bounds__(kThreads) void big_leaf_kernel(BigBatch B)
{
    int32_t *const w = B.c[blockIdx.z].core();
    const BigLayout &Y = B.Y;
    const int d0 = B.L - B.L0, s0 = 1 << B.L0, v0 = (int)blockIdx.x * s0;
    const int32_t *keyP = w + ((d0 & 1) ? Y.keyP2 : Y.keyP) + v0;
    const int32_t *keyQ = w + ((d0 & 1) ? Y.keyQ2 : Y.keyQ) + v0;
    extern __shared__ uint16_t lds[];
    __shared__ LeafLines lines;
    core_lds_body(keyP, keyQ, s0, B.L0, lds, lines,
                  [&](int x, int c) { big_lift(B, w, d0 - 1, v0, s0, v0 + x, c); });
}

// Per histogram block (w entries of CI for y = 0, of U for y = 1): packed
// exclusive prefix over the buckets of (lo count | hi count << 16) for each
// boundary j < nb, and the packed totals at [nb].
__global__ __launch_bounds__(256) void big_hist_kernel(BigBatch B, int d)
{
    int32_t *const w = B.c[blockIdx.z].core();
    const BigLayout &Y = B.Y;
    const BigDepth &D = B.D[d];
    const int K = 1 << B.L, y = blockIdx.y;
    const uint32_t *E = (const uint32_t *)w + (y ? Y.U[d & 1] : Y.CI[d & 1]);
    __shared__ uint32_t h[kMaxLines];
    __shared__ uint32_t sums[4];
    for (int j = threadIdx.x; j < D.nb; j += 256) h[j] = 0;
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * D.w;
    for (int i = threadIdx.x; i < D.w; i += 256) {
        const uint32_t e = E[base + i];
        // an aborted comb can leave entries unwritten: keep the bucket in range
        const int bk = (D.s - 1 - (int)(e & (uint32_t)(D.s - 1))) >> D.glog;
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
    uint32_t *rows = (uint32_t *)(w + Y.hist) + ((size_t)y * nodes + node) * D.nsegs * (size_t)(D.nb + 1);
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

constexpr int kSegRounds = 16;
static_assert(big_blocks_fit(64 * kSegRounds), "histogram blocks per node");

// T of boundary j > 0 over the entries E of a node: Y_j and the block where
// the running count reaches it (block_search, at most kSegRounds x 64 blocks
// per node), then a sweep of that block for the entry where the count reaches
// the rank still needed; T is that entry's position + 1, 0 when Y_j = 0.
__device__ __forceinline__ int big_line(const BigDepth &D, const uint32_t *H, const uint32_t *E, int j, int lane)
{
    const uint32_t *Hj = H + j, *Ht = H + (size_t)D.nsegs * D.nb;
    int Yj, Z, seg;
    if (D.nsegs <= 64) block_search<1>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    else if (D.nsegs <= 128) block_search<2>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    else if (D.nsegs <= 256) block_search<4>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    else if (D.nsegs <= 512) block_search<8>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    else block_search<kSegRounds>(Hj, Ht, D.nb, D.nsegs, lane, Yj, Z, seg);
    if (Yj == 0) return 0;
    E += (size_t)seg * D.w;
    // w is a power of two >= 128: the whole block in one batch up to 1024 entries
    const int need = Yj - Z;
    const int pos = D.w <= 128   ? sweep_block<2>(E, D.w, D.s, D.glog, j, need, lane)
                    : D.w <= 256 ? sweep_block<4>(E, D.w, D.s, D.glog, j, need, lane)
                    : D.w <= 512 ? sweep_block<8>(E, D.w, D.s, D.glog, j, need, lane)
                                 : sweep_block<16>(E, D.w, D.s, D.glog, j, need, lane);
    return pos ? min(seg * D.w + pos, D.s) : 0;
}

// One wave per piece of the ant's path: (y = 0) from row line j = 0 .. nb - 1
// (j = 0: the start of the passage at T(s) = 0), (y = 1) from column line i =
// nb - j.  The wave finds its own crossing (big_line), then its box's rows
// (box_rows), and hands every row it decides straight to the parent node
// (big_lift), or from the top depth to the product: each row lies in exactly
// one piece's box.  A wave's chain of dependent loads (histogram, block, box,
// parents) is what bounds it.  Sweep, boxes, lift and output were kernels of
// their own, each a launch (about 4 us with its gap) and a pass over U and CI;
// with them in one and the slicing in three, a k = 2^16 product takes 24
// launches instead of 38: 197 -> 155 us, 2^11 86 -> 71, 2^20 1178 -> 991.  With g above 64 the rows go
// 64 at a time from the line upwards, carrying the rows counted so far, and
// the columns 64 at a time.
constexpr int kBoxWaves = 4;   // pieces per workgroup
__global__ __launch_bounds__(64 * kBoxWaves) void big_box_kernel(BigBatch B, int d)
{
    const MulArgs &M = B.c[blockIdx.z];
    int32_t *const w = M.core();
    const BigLayout &Y = B.Y;
    const BigDepth &D = B.D[d];
    const int K = 1 << B.L, s = D.s, nodes = K / s, g = 1 << D.glog, nb = D.nb, lane = threadIdx.x & 63;
    const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * kBoxWaves + (threadIdx.x >> 6));
    if (t >= 2 * nodes * nb) return;
    const bool col = t >= nodes * nb;
    const int q = col ? t - nodes * nb : t, node = q / nb, j = q - node * nb;
    if (col && j == 0) return;
    const int v0 = node * s;
    const uint32_t *U = (const uint32_t *)w + Y.U[d & 1] + v0, *CI = (const uint32_t *)w + Y.CI[d & 1] + v0;
    int T0 = 0;
    if (j) {
        const uint32_t *H = (const uint32_t *)w + Y.hist + ((size_t)(col ? 1 : 0) * nodes + node) * D.nsegs * (size_t)(D.nb + 1);
        T0 = big_line(D, H, col ? U : CI, j, lane);
    }
    int r_lo, rho, cs, ce;
    if (!col) {
        r_lo = s - (j + 1) * g;
        rho = r_lo + g - 1;
        cs = T0;
        ce = cs == 0 ? g : (((cs - 1) >> D.glog) + 1) << D.glog;
    } else {
        if (T0 == 0) return;   // the ant never reaches this column line
        rho = T0 - 1;
        r_lo = rho & ~(g - 1);
        cs = (nb - j) * g;
        ce = cs + g;
    }
    auto finish = [&](int r, int c) {
        if (d) big_lift(B, w, d - 1, v0, s, v0 + r, c);
        else M.put(r, c);
    };
    auto entry = [&](int c) { return CI[c]; };
    if (g == kBox) {
        const uint32_t u = U[r_lo + lane];
        const int c = col ? box_rows<31, true>(u, entry, r_lo, rho, cs, ce, lane)
                          : box_rows<31, false>(u, entry, r_lo, rho, cs, ce, lane);
        if (c >= 0) finish(r_lo + lane, c);
        return;
    }
    int below = col ? 1 : 0;   // -delta(r, cs) just below the rows in hand
    for (int rb = rho & ~63; rb >= r_lo; rb -= 64) {
        const int r = rb + lane;
        const uint32_t u = U[r];
        const bool uc = counted<31>(u, cs);
        const unsigned long long m = __ballot(col ? uc && r < rho : uc);
        int need = below + (int)__popcll(m >> lane);
        below += (int)__popcll(m);
        int T = need ? -1 : cs;
        for (int c0 = cs; c0 < ce; c0 += 64) {
            uint32_t qm[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = c0 + 16 * i + (lane & 15);
                qm[i] = counted_row16(c < ce ? entry(c) : ~kLo31, (uint32_t)r, lane);
            }
            const uint32_t lo = qm[0] | qm[1] << 16, hi = qm[2] | qm[3] << 16;
            const int cnt = __popc(lo) + __popc(hi);
            if (T < 0 && need <= cnt) T = c0 + 1 + select64(lo, hi, need);
            need -= cnt;
        }
        if ((!col || r <= rho) && T >= 0) finish(r, T > 0 && counted<31>(u, T) ? T - 1 : (int)(u & ~kLo31));
    }
}

// ---------------------------------------------------------------- slicing
// The points of p in the glued columns (p's rows in order) and those of q in
// the glued rows (q's columns in order) become the core's keys; every other
// point goes to the product unchanged (braid_multiplication.hpp:353-401).
// Device-wide stable compaction: per-block counts, then a scatter whose
// blocks sum the counts before them themselves.  The products of one merge
// level go through each kernel in one launch: blockIdx.y / 2 picks the
// product, blockIdx.y & 1 its side (0: p by rows, 1: q by columns).
struct SliceSide {
    const int32_t *src;
    int32_t n, lo, hi;
    __device__ bool sel(int i) const { return src[i] >= lo && src[i] < hi; }
};
__device__ __forceinline__ SliceSide slice_side(const MulArgs &M, int side)
{
    if (side == 0) return {M.p, M.p_size, M.row_glue ? 0 : M.p_size - M.k, M.row_glue ? M.k : M.p_size};
    return {M.q_c2r(), M.q_size, M.row_glue ? M.q_size - M.k : 0, M.row_glue ? M.q_size : M.k};
}

__device__ __forceinline__ int block_sum256(int x, int *red)
{
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

template <bool LINES>
__global__ __launch_bounds__(kScanBlock) void slice_count_kernel(MulBatch B)
{
    const MulArgs &M = B.m[blockIdx.y >> 1];
    const int side = blockIdx.y & 1, run = LINES ? M.run : 1;
    const SliceSide S = slice_side(M, side);
    const int64_t first = (int64_t)blockIdx.x * run * kScanTile;
    if (first >= S.n) return;   // past this slice's blocks (whole block)
    __shared__ int red[kScanBlock / 64];
    int c = 0;
    for (int t = 0; t < run; ++t) {
        constexpr int kStep = LINES ? kScanBlock : 1;
        const int64_t base = first + (int64_t)t * kScanTile + threadIdx.x * (LINES ? 1 : kScanPer);
#pragma unroll
        for (int q = 0; q < kScanPer; ++q) c += base + q * kStep < S.n && S.sel((int)(base + q * kStep));
    }
    c = block_sum256(c, red);
    if (threadIdx.x == 0) M.counts(side)[blockIdx.x] = c;
}

// LINES: consecutive threads take consecutive points, so that those passed on
// unchanged leave in whole lines, and a workgroup takes as many tiles as keep
// their number bounded; else each thread takes kScanPer consecutive points,
// whose ranks are one scan.  Kernel time of a product, else / LINES: 5000
// points, k = 64 19 / 22 us; 100000, 65000 153 / 156; 2^20, 1 49 / 45; 2^22,
// 64 159 / 142; 2^26, 64 2470 / 2180.
// Also pads the keys of a core smaller than 2^L with fixed points, and zeroes
// the tile counts of a big core's depths 1 and 2, which the partitions before
// them accumulate
template <bool LINES>
__global__ __launch_bounds__(kScanBlock) void slice_scatter_kernel(MulBatch B)
{
    const MulArgs &M = B.m[blockIdx.y >> 1];
    const int side = blockIdx.y & 1;
    const SliceSide S = slice_side(M, side);
    const int K = 1 << M.L, k = M.k, ps = M.p_size, qs = M.q_size;
    int32_t *const key = M.core() + (side ? K : 0), *const map = side ? M.map_col() : M.map_row();
    for (int64_t x = k + (int64_t)blockIdx.x * kScanBlock + threadIdx.x; x < K; x += (int64_t)gridDim.x * kScanBlock)
        key[x] = (int32_t)x;
    if (M.big) {
        const int ntiles = K / kSplitTile;
        const size_t cnt = big_layout_cnt(M.L) + (size_t)ntiles * 2;
        for (int x = blockIdx.x * kScanBlock + threadIdx.x; x < 2 * ntiles; x += gridDim.x * kScanBlock)
            M.core()[cnt + (size_t)side * 2 * ntiles + x] = 0;
    }
    const int run = LINES ? M.run : 1;
    const int64_t first = (int64_t)blockIdx.x * run * kScanTile;
    if (first >= S.n) return;   // past this slice's blocks (whole block)
    constexpr int kWaves = kScanBlock / 64, kGroups = kScanPer * kWaves;   // groups of 64 points, in order
    static_assert(kGroups <= 64, "one wave scans the groups' counts");
    __shared__ int red[kWaves], group[LINES ? kGroups : kWaves];
    const int32_t *counts = M.counts(side);
    int before = 0;
    for (int i = threadIdx.x; i < (int)blockIdx.x; i += kScanBlock) before += counts[i];
    before = block_sum256(before, red);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // point i (value v) goes to place j of the core's, or on unchanged
    auto place = [&](int i, int32_t v, bool selected, int j) {
        if (selected) {
            if (j < k) {
                map[j] = i;
                key[j] = v - S.lo;
            }
            return;
        }
        // an untouched point (row, col) of p or q; the range test only matters
        // after an aborted comb fed undefined input
        int row = side ? v : i, col = side ? i : v;
        if (side == 0 && M.row_glue) { row += qs - k; col += qs - k; }
        if (side == 1 && !M.row_glue) { row += ps - k; col += ps - k; }
        if ((uint32_t)row < (uint32_t)(ps + qs - k)) M.out[row] = col;
    };
    int32_t v[kScanPer];
    if constexpr (!LINES) {
        const int64_t base = first + threadIdx.x * kScanPer;
        int c = 0;
#pragma unroll
        for (int q = 0; q < kScanPer; ++q) {
            v[q] = base + q < S.n ? S.src[base + q] : -1;
            c += v[q] >= S.lo && v[q] < S.hi;
        }
        const int incl = wave_incl_scan(c);
        if (lane == 63) group[wave] = incl;
        __syncthreads();
        int j = before + incl - c;
        for (int q = 0; q < wave; ++q) j += group[q];
#pragma unroll
        for (int q = 0; q < kScanPer; ++q) {
            if (base + q >= S.n) break;
            const bool selected = v[q] >= S.lo && v[q] < S.hi;
            place((int)(base + q), v[q], selected, j);
            j += selected;
        }
    } else {
        for (int t = 0; t < run; ++t) {
            const int64_t base = first + (int64_t)t * kScanTile + threadIdx.x;
            unsigned long long mask[kScanPer];
#pragma unroll
            for (int q = 0; q < kScanPer; ++q) v[q] = base + q * kScanBlock < S.n ? S.src[base + q * kScanBlock] : -1;
#pragma unroll
            for (int q = 0; q < kScanPer; ++q) {
                mask[q] = __ballot(v[q] >= S.lo && v[q] < S.hi);
                if (lane == 0) group[q * kWaves + wave] = __popcll(mask[q]);
            }
            __syncthreads();
            const int c = lane < kGroups ? group[lane] : 0, incl = wave_incl_scan(c);
            if (t + 1 < run) __syncthreads();   // before the next tile's counts
            int start[kScanPer];   // read here, where every lane is there to be read
#pragma unroll
            for (int q = 0; q < kScanPer; ++q)
                start[q] = before + __builtin_amdgcn_readlane(incl - c, q * kWaves + wave);
            before += __builtin_amdgcn_readlane(incl, 63);
#pragma unroll
            for (int q = 0; q < kScanPer; ++q) {
                if (base + q * kScanBlock >= S.n) break;
                place((int)(base + q * kScanBlock), v[q], mask[q] >> lane & 1,
                      start[q] + __popcll(mask[q] & ((1ull << lane) - 1)));
            }
        }
    }
}

__global__ void invert_kernel(MulBatch B)
{
    const MulArgs &M = B.m[blockIdx.y];
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;   // no wrap near 2^31
    if (i < M.q_size && (uint32_t)M.q[i] < (uint32_t)M.q_size) M.q_c2r()[M.q[i]] = (int32_t)i;
}

// A product with no glued strands: p's points, then q's.
__global__ void juxtapose_kernel(MulBatch B)
{
    const MulArgs &M = B.m[blockIdx.y];
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int ps = M.p_size, qs = M.q_size;
    if (i < ps) M.out[M.row_glue ? i + qs : i] = M.p[i] + (M.row_glue ? qs : 0);
    if (i < qs) M.out[M.row_glue ? i : i + ps] = M.q[i] + (M.row_glue ? 0 : ps);
}

}  // namespace lcsb

using namespace lcsb;

static bool core_is_big(int L, bool in_lds) { return L >= kBigMinL && !(in_lds && L <= kLdsCoreL); }

size_t lcsb_core_scratch_words(int32_t k, bool in_lds)
{
    const int L = lcsb_core_L(k);
    return core_is_big(L, in_lds) ? big_layout(L, big_leaf_L(L)).total : (size_t)2 << L;   // small cores: the keys
}

// Padded core size 2^L: at least 64 (the LDS kernel ranks keys by wave
// ballots over groups of 64); padding adds fixed points only.
int lcsb_core_L(int32_t k)
{
    int L = 6;
    while ((1 << L) < k) ++L;
    return L;
}

// The big-core sequence for up to kMulBatch products of one padded size.
static int launch_big(const BigBatch &B, int cnt, hipStream_t stream)
{
    const int L = B.L, L0 = B.L0, d0 = L - L0, K = 1 << L;
    const dim3 tiles((unsigned)(K / kSplitTile), 2, (unsigned)cnt);
    hipLaunchKernelGGL(big_split_count_kernel, tiles, dim3(256), 0, stream, B, 0);
    for (int d = 0; d < d0; ++d) {
        if (d + 1 < d0) hipLaunchKernelGGL(big_split_scatter_kernel<true>, tiles, dim3(256), 0, stream, B, d);
        else hipLaunchKernelGGL(big_split_scatter_kernel<false>, tiles, dim3(256), 0, stream, B, d);
    }
    hipLaunchKernelGGL(big_leaf_kernel, dim3(1u << d0, 1, (unsigned)cnt), dim3(kThreads), lds_core_bytes(L0),
                       stream, B);
    for (int d = d0 - 1; d >= 0; --d) {
        const BigDepth D = big_depth(L, d);
        const int pieces = 2 * (K / D.s) * D.nb;
        hipLaunchKernelGGL(big_hist_kernel, dim3((unsigned)(K / D.w), 2, (unsigned)cnt), dim3(256), 0, stream, B, d);
        hipLaunchKernelGGL(big_box_kernel, dim3((unsigned)((pieces + kBoxWaves - 1) / kBoxWaves), 1, (unsigned)cnt),
                           dim3(64 * kBoxWaves), 0, stream, B, d);
    }
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

// The dynamic LDS limit of the core kernels, set once per device (before any
// capture: it is not a stream operation).
int lcsb_init(void)
{
    static PerDevice lds;
    return lds.once([] {
        for (const void *k : {(const void *)braid_core_lds_kernel, (const void *)big_leaf_kernel})
            if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_core_bytes(kLdsCoreL)) !=
                hipSuccess)
                return -5;
        return 0;
    });
}

// staggered_multiply for `count` independent products on device pointers.
// The products of one padded core size go through each kernel of the
// sequence side by side (in groups of kMulBatch), so the products of a
// merge-tree level share their launches.  specs[i].ws holds
// lcsb_multiply_ws_words(p_size, q_size, k) words.
int lcsb_multiply_many_device(const MulSpec *specs, int count, hipStream_t stream, bool in_lds)
{
    if (lcsb_init()) return -5;
    std::vector<MulArgs> mul((size_t)count);
    for (int i = 0; i < count; ++i) {
        const MulSpec &M = specs[i];
        mul[(size_t)i] = MulArgs{M.p, M.q, M.out, M.ws, M.p_size, M.q_size, M.k, M.row_glue ? 1 : 0,
                                 M.k ? lcsb_core_L(M.k) : 0, 0, 0, 0};
        mul[(size_t)i].big = core_is_big(mul[(size_t)i].L, in_lds);
        mul[(size_t)i].set_blocks();
        if (mul[(size_t)i].L > kMaxCoreL) return -34;
    }
    std::stable_sort(mul.begin(), mul.end(), [](const MulArgs &x, const MulArgs &y) { return x.L < y.L; });
    for (size_t i = 0; i < mul.size();) {
        MulBatch B{};
        const int L = mul[i].L;
        int cnt = 0, q_max = 0, n_max = 0;
        while (i < mul.size() && mul[i].L == L && cnt < kMulBatch) {
            q_max = std::max(q_max, mul[i].q_size);
            n_max = std::max(n_max, std::max(mul[i].p_size, mul[i].q_size));
            B.m[cnt++] = mul[i++];
        }
        const dim3 by_point((unsigned)((n_max + 255) / 256), (unsigned)cnt);
        if (L == 0) {
            if (n_max) hipLaunchKernelGGL(juxtapose_kernel, by_point, dim3(256), 0, stream, B);
            continue;
        }
        int slice_blocks = 0;
        for (int c = 0; c < cnt; ++c) slice_blocks = std::max(slice_blocks, B.m[c].blocks);
        const dim3 slices((unsigned)slice_blocks, 2 * (unsigned)cnt);
        hipLaunchKernelGGL(invert_kernel, dim3((unsigned)((q_max + 255) / 256), (unsigned)cnt), dim3(256), 0, stream, B);
        if (n_max >= kLinesMin) {
            hipLaunchKernelGGL(slice_count_kernel<true>, slices, dim3(kScanBlock), 0, stream, B);
            hipLaunchKernelGGL(slice_scatter_kernel<true>, slices, dim3(kScanBlock), 0, stream, B);
        } else {
            hipLaunchKernelGGL(slice_count_kernel<false>, slices, dim3(kScanBlock), 0, stream, B);
            hipLaunchKernelGGL(slice_scatter_kernel<false>, slices, dim3(kScanBlock), 0, stream, B);
        }
        if (!B.m[0].big) {
            hipLaunchKernelGGL(braid_core_lds_kernel, dim3((unsigned)cnt), dim3(kThreads), lds_core_bytes(L), stream, B);
            continue;
        }
        BigBatch G{};
        for (int c = 0; c < cnt; ++c) G.c[c] = B.m[c];
        G.L = L;
        G.L0 = big_leaf_L(L);
        G.Y = big_layout(L, G.L0);
        for (int d = 0; d < L - G.L0; ++d) G.D[d] = big_depth(L, d);
        const int rc = launch_big(G, cnt, stream);
        if (rc) return rc;
    }
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

// staggered_multiply on device pointers; ws must hold lcsb_multiply_ws_words(...)
int lcsb_multiply_device(const int32_t *p, int32_t p_size, const int32_t *q, int32_t q_size, int32_t k,
                         int32_t row_glue, int32_t *out, int32_t *ws, hipStream_t stream, bool in_lds)
{
    const MulSpec M{p, p_size, q, q_size, k, row_glue, out, ws};
    return lcsb_multiply_many_device(&M, 1, stream, in_lds);
}

size_t lcsb_multiply_ws_words(int32_t p_size, int32_t q_size, int32_t k, bool in_lds)
{
    // at least MulArgs::blocks counts a side, and no fewer for a larger product:
    // merges reserve for the largest of a level
    const int32_t tiles = std::max(p_size, q_size) / kScanTile + 1;
    return (size_t)q_size + 2 * (size_t)k + 2 * (size_t)std::min(tiles, kMaxSliceBlocks) + lcsb_core_scratch_words(k > 0 ? k : 1, in_lds);
}
