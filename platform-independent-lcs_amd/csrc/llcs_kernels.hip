// Score-only LCS length by bit-parallel combing on gfx950.
//
// The reference's binary bit-parallel LLCS (src/lcs_reference.hpp:135-211,
// disabled by #if 0) packs strands into machine words.  This kernel uses the
// word-parallel LCS recurrence over the row string a (Allison-Dix; Hyyro's
// form): with V an m-bit vector, initially all ones, and M[c] the bits i with
// a[i] == c, every symbol c of the column string does
//     U = V & M[c];   V = (V + U) | (V & ~M[c])
// and LCS = number of zero bits of V at the end.  The addition carries from
// row i to row i+1, which is the only coupling between rows.
//
// MI355X mapping: one wave64 per band of 2048 rows, one 32-bit word of V per
// lane.  Lane l takes the columns in blocks of B = 4, block k - l in turn k, so
// what it needs from lane l-1 -- the four carries of that block -- was
// finished the turn before and moves as one register by one DPP per turn.
// Inside a turn everything is VALU and lane-private: per column
//     cin:  shift the carry word left, its top bit to an SGPR pair (v_add_co)
//     U, sum with carry in and out (v_and, v_addc_co), V (v_bitop3)
//     cout: shift the carry out into the outgoing word (v_addc_co),
// five VALU for 2048 cells.  The columns of one band are a serial chain, so
// the kernel's time is columns x time per column plus the bands' fill.  By the
// counters a lone wave's six instructions a column take 5.8 cycles each, about
// 30 % of them stall in the turn's chain of carries (a comb wave, without such
// a chain, issues every four): their count and that chain are what matters.
// With one column per step, carries in lane-skewed SGPR masks and a second wave
// fetching through LDS a column took 30.5 ns and m = n = 2^20 38.0 ms; now 15.0
// and 19.9.  A band follows the one
// below by 64 blocks, so blocks of two (15 instead of 12 issues a turn for two
// columns, 17 ns a column) halve the skew where bands, not columns, make the
// time: the caller picks by that.
//
//  * Match masks: a table in LDS, built once per band: one row of 64 words per
//    symbol, or (alphabets of at most 9, the caller's choice) one row of 64 pairs of words per two
//    consecutive symbols, so that one address (a v_perm of the code byte and
//    the lane) and one ds_read_b64 serve two columns.  A zero row serves the
//    padding before and after the column string.
//  * Column symbols: the seeding kernel writes them as code bytes; a lane
//    loads its own 32 columns of codes per chunk (32 / B turns), two chunks
//    before their masks are read, and those are read a chunk before use.
//  * Band hand-off: after the last turn but one of chunk q + 2 B lane 63's
//    outgoing word holds exactly the 32 carries of columns 32q ..; it goes to the band above as
//    one tagged 64-bit word (tag << 32 | bits), stored with an agent-scope
//    relaxed atomic.  The band above loads each word two chunks ahead and
//    polls, bounded in time, when it comes too early.
//  * Bands are handed out by an atomic ticket in order, so every wait is on a
//    band that a resident wave already holds.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "llcs_kernels.h"
#include "per_device.h"

namespace lcsl {

#define LCSL_GLOBAL __attribute__((address_space(1)))
typedef LCSL_GLOBAL unsigned long long gword;
typedef LCSL_GLOBAL const unsigned long long gcword;
typedef LCSL_GLOBAL const int32_t gsym;
typedef LCSL_GLOBAL const uint8_t gbyte;
typedef uint32_t unaligned_u32 __attribute__((aligned(1)));
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;

constexpr unsigned kNoTag = 0xffffffffu;
constexpr int kMaxLdsBytes = 160 * 1024;

__device__ __forceinline__ unsigned long long ld_relaxed(gcword *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_relaxed(gword *p, unsigned long long x)
{
    __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned ld_flag(const unsigned *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One turn: the B columns of a lane's block, their match masks in M.
// First the carries move: lane l-1's cout of the turn before (its low B
// bits), left-aligned, becomes cin; lane 0, which the DPP leaves alone, keeps
// shifting the band's own input word out of its cin.  Column k: N(k) u = V &
// m, A(k) cin <<= 1 with its top bit to sA[k % 2], S(k) sum = V + u + sA with
// the carry to sB[k % 2], B(k) V = sum | (V & ~m), O(k) cout = cout << 1 | sB.
// A VALU-written SGPR mask, and a VGPR that a DPP reads, want two issues in
// between, so A runs a column ahead and O a column behind, and the two table
// addresses of the caller's next reads (bytes sel0, sel1 of w over the lane's
// place in a row) fill the turn's head: no s_nop, 24 issues for four columns
// (14 for two).
#define LCSL_N(K) "v_and_b32 %[u], %[v], %[m" #K "]\n\t"
#define LCSL_A(X) "v_add_co_u32_e64 %[ci], %[a" #X "], %[ci], %[ci]\n\t"
#define LCSL_S(X) "v_addc_co_u32_e64 %[s], %[b" #X "], %[v], %[u], %[a" #X "]\n\t"
#define LCSL_B(K) "v_bitop3_b32 %[v], %[s], %[v], %[m" #K "] bitop3:0xf4\n\t"
#define LCSL_O(X) "v_addc_co_u32_e64 %[co], %[d], %[co], %[co], %[b" #X "]\n\t"
__device__ __forceinline__ void turn(uint32_t &V, uint32_t &cout, uint32_t &cin, const uint32_t (&M)[4], uint32_t w,
                                     uint32_t lane_off, uint32_t sel0, uint32_t sel1, uint32_t &p0, uint32_t &p1)
{
    uint32_t t, u, sum;
    uint64_t a0, a1, b0, b1, d;
    asm volatile("v_lshlrev_b32 %[t], 28, %[co]\n\t"
                 LCSL_N(0)
                 "v_perm_b32 %[p0], %[w], %[l], %[s0]\n\t"
                 "v_mov_b32_dpp %[ci], %[t] wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                 LCSL_A(0) LCSL_A(1)
                 "v_perm_b32 %[p1], %[w], %[l], %[s1]\n\t"
                 LCSL_S(0) LCSL_B(0)
                 LCSL_N(1) LCSL_A(0) LCSL_S(1) LCSL_B(1) LCSL_O(0)
                 LCSL_N(2) LCSL_A(1) LCSL_S(0) LCSL_B(2) LCSL_O(1)
                 LCSL_N(3) LCSL_S(1) LCSL_B(3) LCSL_O(0) LCSL_O(1)
                 : [v] "+v"(V), [co] "+v"(cout), [ci] "+v"(cin), [t] "=&v"(t), [u] "=&v"(u), [s] "=&v"(sum),
                   [a0] "=&s"(a0), [a1] "=&s"(a1), [b0] "=&s"(b0), [b1] "=&s"(b1), [d] "=&s"(d), [p0] "=&v"(p0),
                   [p1] "=&v"(p1)
                 : [w] "v"(w), [l] "v"(lane_off), [s0] "s"(sel0), [s1] "s"(sel1), [m0] "v"(M[0]), [m1] "v"(M[1]),
                   [m2] "v"(M[2]), [m3] "v"(M[3]));
}

__device__ __forceinline__ void turn(uint32_t &V, uint32_t &cout, uint32_t &cin, const uint32_t (&M)[2], uint32_t w,
                                     uint32_t lane_off, uint32_t sel0, uint32_t sel1, uint32_t &p0, uint32_t &p1)
{
    uint32_t t, u, sum;
    uint64_t a0, a1, b0, b1, d;
    asm volatile("v_lshlrev_b32 %[t], 30, %[co]\n\t"
                 LCSL_N(0)
                 "v_perm_b32 %[p0], %[w], %[l], %[s0]\n\t"
                 "v_mov_b32_dpp %[ci], %[t] wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                 LCSL_A(0) LCSL_A(1)
                 "v_perm_b32 %[p1], %[w], %[l], %[s1]\n\t"
                 LCSL_S(0) LCSL_B(0)
                 LCSL_N(1) LCSL_S(1) LCSL_B(1) LCSL_O(0) LCSL_O(1)
                 : [v] "+v"(V), [co] "+v"(cout), [ci] "+v"(cin), [t] "=&v"(t), [u] "=&v"(u), [s] "=&v"(sum),
                   [a0] "=&s"(a0), [a1] "=&s"(a1), [b0] "=&s"(b0), [b1] "=&s"(b1), [d] "=&s"(d), [p0] "=&v"(p0),
                   [p1] "=&v"(p1)
                 : [w] "v"(w), [l] "v"(lane_off), [s0] "s"(sel0), [s1] "s"(sel1), [m0] "v"(M[0]), [m1] "v"(M[1]));
}

// One band.  PAIRS: a code byte stands for two columns; B: columns per turn.
// RAW: no codes (a budget that does not hold them): a lane turns the 32
// symbols of its chunk into codes itself (m = n = 2^20: 57.8 ms against 20.1).
template <bool PAIRS, int B, bool RAW = false>
__device__ bool band(const LlcsArgs &A, const LlcsDesc &D, int g, int lane, lds_u32 *tab)
{
    constexpr int kBlock = B, kTurns = kChunk / B, kWordLag = word_lag(B);
    static_assert(!(PAIRS && RAW), "raw symbols have a code each");
    constexpr int kCodeWords = PAIRS ? kChunk / 8 : kChunk / 4;   // code words of a lane's chunk
    const int sigma = A.sigma;
    bool bad = false;
    // the masks of this lane's 32 rows; row `sigma` stays zero (padding)
    {
        // the single-symbol rows: the table itself, or in its first words until
        // the lane holds them in registers, before the first pair row is written
        const int rows1 = sigma + 1;
        for (int c = 0; c < rows1; ++c) tab[c * kWave + lane] = 0u;
        const int64_t r0 = ((int64_t)g * kWave + lane) * kWordRows;
        for (int i = 0; i < kWordRows; ++i) {
            const int64_t r = r0 + i;
            if (r < D.nrows) {
                const int32_t s = ((gsym *)D.rows)[r];
                if ((uint32_t)s < (uint32_t)sigma) tab[s * kWave + lane] |= 1u << i;
                else bad = true;
            }
        }
        if constexpr (PAIRS) {
            uint32_t one[kMaxPairSigma + 1];
#pragma unroll
            for (int c = 0; c <= kMaxPairSigma; ++c) one[c] = c < rows1 ? tab[c * kWave + lane] : 0u;
            __syncthreads();   // one wave: only keeps the reads before the writes
            for (int c = 0; c < rows1; ++c) {
                uint32_t mc = 0;
#pragma unroll
                for (int x = 0; x <= kMaxPairSigma; ++x) mc = x == c ? one[x] : mc;
#pragma unroll
                for (int x = 0; x <= kMaxPairSigma; ++x)
                    if (x < rows1)
                        *((lds_u32x2 *)tab + (c * rows1 + x + (lane & 32) * 4) * 32 + (lane & 31)) = u32x2{mc, one[x]};
            }
        }
        __syncthreads();
    }
    // (readfirstlane: with the word count's range known to it the compiler
    // computes every chunk's addresses anew, 1 % of the time)
    const int32_t nwords = __builtin_amdgcn_readfirstlane(llcs_nwords(D.ncols));
    const int32_t nchunks = nwords > 0 ? nwords + kWordLag : 0;
    gcword *rin = (gcword *)(D.ring + (g & 1) * llcs_slot_words(D.ncols));
    gword *rout = (gword *)(D.ring + ((g + 1) & 1) * llcs_slot_words(D.ncols));
    const uint32_t tag_in = (uint32_t)g;
    const unsigned long long tag_out = (unsigned long long)(g + 1) << 32;
    // lane l's codes of chunk q start at column kFrontPad + 32 q - B l
    gbyte *codes = (gbyte *)D.codes + (size_t)(kFrontPad - B * lane) / (PAIRS ? 2 : 1);
    auto load_codes = [&](int q, uint32_t (&c)[kCodeWords]) {
        if constexpr (RAW) {
            // all loads, from clamped addresses, before the first symbol is used
            const int32_t c0 = q * kChunk - B * lane;
            uint32_t x[kChunk];
#pragma unroll
            for (int k = 0; k < kChunk; ++k) x[k] = (uint32_t)((gsym *)D.cols)[min(max(c0 + k, 0), D.ncols - 1)];
#pragma unroll
            for (int i = 0; i < kCodeWords; ++i) {
                c[i] = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int32_t col = c0 + 4 * i + k;
                    const uint32_t s = col >= 0 && col < D.ncols ? x[4 * i + k] : (uint32_t)sigma;
                    c[i] |= min(s, (uint32_t)sigma) << (8 * k);
                }
            }
        } else {
            typedef LCSL_GLOBAL const unaligned_u32 gcode;
#pragma unroll
            for (int i = 0; i < kCodeWords; ++i) c[i] = ((gcode *)(codes + (size_t)q * kCodeWords * 4))[i];
        }
    };
    // The masks of turn i of a chunk from its codes: per code byte the LDS
    // address byte * 256 + the lane's place in a row (the table is the
    // kernel's only LDS and starts at address 0), put together by v_perm, the
    // first two of a turn inside turn().
    const uint32_t lane_off = PAIRS ? (uint32_t)(lane & 31) * 8u : (uint32_t)lane * 4u;
    const uint32_t half = PAIRS && lane >= 32 ? 0x80808080u : 0u;
    constexpr int kPerTurn = PAIRS ? B / 2 : B;   // code bytes
    auto code_word = [&](const uint32_t (&c)[kCodeWords], int i) {
        return PAIRS ? c[i * kPerTurn / 4] | half : c[i * kPerTurn / 4];
    };
    auto sel = [](int i, int k) { return 0x0c0c0000u | (uint32_t)(4 + i * kPerTurn % 4 + k) << 8; };
    auto read_masks = [&](uint32_t w, int i, uint32_t p0, uint32_t p1, uint32_t (&M)[B]) {
        if constexpr (PAIRS) {
            const u32x2 x = *(const lds_u32x2 *)(uintptr_t)p0;
            M[0] = x.x;
            M[1] = x.y;
            if constexpr (B == 4) {
                const u32x2 y = *(const lds_u32x2 *)(uintptr_t)p1;
                M[2] = y.x;
                M[3] = y.y;
            }
        } else {
            M[0] = *(const lds_u32 *)(uintptr_t)p0;
            M[1] = *(const lds_u32 *)(uintptr_t)p1;
#pragma unroll
            for (int k = 2; k < B; ++k) M[k] = *(const lds_u32 *)(uintptr_t)__builtin_amdgcn_perm(w, lane_off, sel(i, k));
        }
    };
    auto sel1 = [&](int i) { return PAIRS && B == 2 ? sel(i, 0) : sel(i, 1); };   // (a turn of one pair has no second byte)
    int dead = 0;   // set when a wait gave up: nothing is waited for after that
    // the word of chunk q as loaded ahead (all lanes load the same one), once
    // it carries this band's tag
    auto take_word = [&](int q, unsigned long long e) -> uint32_t {
        if (__builtin_expect(__builtin_amdgcn_readfirstlane((uint32_t)(e >> 32)) != tag_in, 0)) {
            unsigned long long t0 = 0;
#pragma nounroll
            for (int polls = 0; !dead; ++polls) {
                e = ld_relaxed(rin + q);
                if (__builtin_amdgcn_readfirstlane((uint32_t)(e >> 32)) == tag_in) break;
                if (polls % 8 == 0) {
                    const unsigned long long now = __builtin_amdgcn_s_memrealtime();
                    if (polls == 0) t0 = now;
                    const bool late = A.timeout_ticks == 0 || now - t0 > A.timeout_ticks;
                    if (late) __hip_atomic_store(A.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    dead = late || __builtin_amdgcn_readfirstlane(ld_flag(A.abort_flag)) != 0;
                }
            }
        }
        return __builtin_amdgcn_readfirstlane((uint32_t)e);
    };

    uint32_t V = 0xffffffffu, cout = 0;
    uint32_t cA[kCodeWords], cB[kCodeWords], cC[kCodeWords];
    uint32_t MA[kTurns][kBlock], MB[kTurns][kBlock];
    unsigned long long wA = 0, wB = 0;
    if (nchunks > 0) {
        load_codes(0, cA);
        load_codes(1, cB);
        load_codes(2, cC);
        wA = ld_relaxed(rin);
        wB = ld_relaxed(rin + 1);
#pragma unroll
        for (int i = 0; i < kTurns; ++i) {
            const uint32_t w = code_word(cA, i);
            read_masks(w, i, __builtin_amdgcn_perm(w, lane_off, sel(i, 0)), __builtin_amdgcn_perm(w, lane_off, sel1(i)),
                       MA[i]);
        }
    }
    // Chunk q: its masks are in M; the next chunk's are read between the turns
    // from cN into N; the codes of chunk q + 3 and the word of chunk q + 2 take
    // the place of this chunk's.  Chunks before kWordLag publish nothing and
    // those from nwords on have no input (EDGE); the others run without a test
    // on q, six per iteration, so that no register that a load is still to fill
    // is copied.
    auto chunk = [&](auto edge, int q, uint32_t (&cur)[kCodeWords], unsigned long long &word,
                     const uint32_t (&cN)[kCodeWords], uint32_t (&M)[kTurns][kBlock], uint32_t (&N)[kTurns][kBlock]) {
        constexpr bool EDGE = decltype(edge)::value;
        uint32_t cin = 0;   // lane 0's; the others take theirs from the lane below each turn
        if (!EDGE || q < nwords) cin = take_word(q, word);
        load_codes(q + 3, cur);
        word = ld_relaxed(rin + (EDGE ? min(q + 2, nwords + 1) : q + 2));
#pragma unroll
        for (int i = 0; i < kTurns; ++i) {
            const uint32_t w = code_word(cN, i);
            uint32_t p0, p1;
            turn(V, cout, cin, M[i], w, lane_off, sel(i, 0), sel1(i), p0, p1);
            if (i == kTurns - 2 && (!EDGE || q >= kWordLag)) {
                // lane 63: the carries of columns 32 (q - kWordLag) ..; all
                // lanes store the same word, so no lane mask puts a branch
                // between the loads and their waits
                uint32_t bits;   // (a v_readlane wants an issue between it and the VALU write)
                asm volatile("s_nop 0\n\tv_readlane_b32 %0, %1, 63" : "=s"(bits) : "v"(cout));
                st_relaxed(rout + (q - kWordLag), tag_out | bits);
            }
            read_masks(w, i, p0, p1, N[i]);
        }
    };
    using Edge = std::integral_constant<bool, true>;
    using Inner = std::integral_constant<bool, false>;
    auto edges = [&](int q, int end) {   // q a multiple of six, where the sets' roles start over
        for (; q < end; q += 6) {
            chunk(Edge{}, q, cA, wA, cB, MA, MB);
            if (q + 1 < end) chunk(Edge{}, q + 1, cB, wB, cC, MB, MA);
            if (q + 2 < end) chunk(Edge{}, q + 2, cC, wA, cA, MA, MB);
            if (q + 3 < end) chunk(Edge{}, q + 3, cA, wB, cB, MB, MA);
            if (q + 4 < end) chunk(Edge{}, q + 4, cB, wA, cC, MA, MB);
            if (q + 5 < end) chunk(Edge{}, q + 5, cC, wB, cA, MB, MA);
        }
    };
    constexpr int kRampChunks = (kWordLag + 5) / 6 * 6;
    int q = min(kRampChunks, nchunks);
    edges(0, q);
    for (; q + 6 <= nwords; q += 6) {
        chunk(Inner{}, q, cA, wA, cB, MA, MB);
        chunk(Inner{}, q + 1, cB, wB, cC, MB, MA);
        chunk(Inner{}, q + 2, cC, wA, cA, MA, MB);
        chunk(Inner{}, q + 3, cA, wB, cB, MB, MA);
        chunk(Inner{}, q + 4, cB, wA, cC, MA, MB);
        chunk(Inner{}, q + 5, cC, wB, cA, MB, MA);
    }
    edges(q, nchunks);

    if (__any(bad) && lane == 0) *D.err = 1;
    const int64_t live = (int64_t)D.nrows - ((int64_t)g * kWave + lane) * kWordRows;
    const uint32_t valid = live >= kWordRows ? 0xffffffffu : live <= 0 ? 0u : ((1u << live) - 1u);
    int zeros = __popc(~V & valid);
    for (int off = 32; off > 0; off >>= 1) zeros += __shfl_xor(zeros, off);
    if (lane == 0) atomicAdd(D.out, zeros);
    return !dead;
}

template <bool PAIRS, int B, bool RAW = false>
__global__ __launch_bounds__(kWave) void llcs_chain_kernel(LlcsArgs A)
{
    extern __shared__ uint32_t lds_dyn[];
    const int lane = threadIdx.x;
    for (;;) {
        unsigned t = 0;
        if (lane == 0) t = atomicAdd(A.ticket, 1u);
        t = __builtin_amdgcn_readfirstlane(t);
        if ((int)t >= A.ntasks) break;
        if (__builtin_amdgcn_readfirstlane(ld_flag(A.abort_flag))) break;
        const int2 task = A.tasks[t];
        const LlcsDesc D = A.descs[task.x];
        const bool traced = A.trace && (int)t < A.trace_cap && lane == 0;
        if (traced) A.trace[2 * (size_t)t] = __builtin_amdgcn_s_memrealtime();
        if (!band<PAIRS, B, RAW>(A, D, task.y, lane, (lds_u32 *)lds_dyn)) break;
        if (traced) A.trace[2 * (size_t)t + 1] = __builtin_amdgcn_s_memrealtime();
        __syncthreads();   // the table is rebuilt
    }
}

// grid (x: columns / 4, y: pair): ring words (band 0's empty input, and no tag any
// band waits for), the column string as codes (one thread per four columns); block (0,0) clears
// the ticket and abort words, after folding the previous launch's abort flag
// into `sticky`
__global__ void llcs_prep_kernel(const LlcsDesc *descs, int sigma, bool pairs, unsigned *ticket, unsigned *abort_flag,
                                 unsigned *sticky)
{
    const LlcsDesc D = descs[blockIdx.y];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x, i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t slot = llcs_slot_words(D.ncols);
    for (int64_t i = i0; i < 2 * slot; i += stride) D.ring[i] = i < slot ? 0ull : (unsigned long long)kNoTag << 32;
    bool bad = false;
    auto code = [&](int64_t c) -> uint32_t {
        if (c < 0 || c >= D.ncols) return (uint32_t)sigma;
        const uint32_t s = (uint32_t)D.cols[c];
        bad = bad || s >= (uint32_t)sigma;
        return s < (uint32_t)sigma ? s : (uint32_t)sigma;
    };
    if (D.ncols > 0) {
        const int64_t quads = llcs_code_columns(llcs_nwords(D.ncols)) / 4;
        for (int64_t b = i0; b < quads; b += stride) {
            const int64_t c0 = 4 * b - kFrontPad;
            const uint32_t x = code(c0), y = code(c0 + 1), z = code(c0 + 2), w = code(c0 + 3), row = (uint32_t)sigma + 1;
            if (!D.codes) continue;   // only checked
            if (pairs) ((uint16_t *)D.codes)[b] = (uint16_t)((x * row + y) | (z * row + w) << 8);
            else ((uint32_t *)D.codes)[b] = x | y << 8 | z << 16 | w << 24;
        }
    }
    if (bad) *D.err = 1;
    if (i0 == 0) *D.out = 0;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        if (sticky && *abort_flag) *sticky = 1u;
        *ticket = 0u;
        *abort_flag = 0u;
    }
}

__global__ void llcs_finish_kernel(const LlcsDesc *descs, int npairs)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npairs) return;
    const LlcsDesc D = descs[p];
    if (*D.err) *D.out = -1;
}

}  // namespace lcsl

int lcsl_launch(const lcsl::LlcsArgs &args, const lcsl::LlcsDesc *d_descs, int npairs, int max_words,
                int grid_blocks, int lds_bytes, hipStream_t stream)
{
    using namespace lcsl;
    if (npairs <= 0) return 0;
    if (args.sigma < 1 || args.sigma > kMaxSigma || (args.pairs && args.sigma > kMaxPairSigma) ||
        lds_bytes < (int)llcs_lds_bytes(args.sigma, args.pairs))
        return -22;
    const bool pairs = args.pairs && args.codes;
    static PerDevice lds;   // no stream operation
    const int rc = lds.once([] {
        for (const void *k : {(const void *)llcs_chain_kernel<true, 4>, (const void *)llcs_chain_kernel<false, 4>,
                              (const void *)llcs_chain_kernel<true, 2>, (const void *)llcs_chain_kernel<false, 2>,
                              (const void *)llcs_chain_kernel<false, 4, true>})
            if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLdsBytes) != hipSuccess) return -5;
        return 0;
    });
    if (rc) return rc;
    // one thread per four columns, the padding among them
    const unsigned px = (unsigned)std::min<int64_t>(4096, (llcs_code_columns(max_words) / 4 + 255) / 256);
    for (int base = 0; base < npairs; base += 65535) {   // grid y is at most 65535
        const int cnt = std::min(65535, npairs - base);
        hipLaunchKernelGGL(llcs_prep_kernel, dim3(px, (unsigned)cnt), dim3(256), 0, stream, d_descs + base, args.sigma,
                           pairs, args.ticket, args.abort_flag, base ? nullptr : args.sticky);
    }
    if (args.ntasks > 0 && grid_blocks > 0) {
        const dim3 grid(grid_blocks), block(kWave);
        if (!args.codes) llcs_chain_kernel<false, 4, true><<<grid, block, lds_bytes, stream>>>(args);
        else if (pairs && args.block == 4) llcs_chain_kernel<true, 4><<<grid, block, lds_bytes, stream>>>(args);
        else if (pairs) llcs_chain_kernel<true, 2><<<grid, block, lds_bytes, stream>>>(args);
        else if (args.block == 4) llcs_chain_kernel<false, 4><<<grid, block, lds_bytes, stream>>>(args);
        else llcs_chain_kernel<false, 2><<<grid, block, lds_bytes, stream>>>(args);
    }
    hipLaunchKernelGGL(llcs_finish_kernel, dim3((npairs + 255) / 256), dim3(256), 0, stream, d_descs, npairs);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}
