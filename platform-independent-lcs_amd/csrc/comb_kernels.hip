// Seaweed (strand) combing kernels for CDNA4 / gfx950.
//
// Grid orientation used on the device: row r = 0..m-1 holds a[r] (the
// reference's reversed row i = m-1-r, src/lcs_reference.hpp:13-20), column c
// holds b[c].  Horizontal strands travel left to right along a row, vertical
// strands travel top to bottom (from row r-1 into row r, the reference's "from
// high i to low i", src/lcs_common.hpp:76-88).  Cell rule
// (src/lcs_common.hpp:7-24): swap iff a[r] == b[c] || h > v.  Strand ids are
// non-negative, so the signed compare equals the unsigned one and the swap is
//     h' = min(match ? ~0u : h, v),   v' = h ^ v ^ h'
// i.e. v_cmp_eq + v_min_u32 + v_cndmask + v_bitop3 (xor3): 4 VALU, no SALU.
//
// Band chain.  One wave64 owns a band of 64*TM consecutive rows; lane L keeps
// TM rows (symbols and h strands) in VGPRs.  At step t lane L combs column
// t-L, so the wave sweeps the band along anti-diagonals.  The v strand and the
// b symbol move one lane down per step by DPP wave_shr:1; lane 0 receives the
// band's inputs from two "conveyor" registers shifted by wave_shl:1, and the
// strand conveyor also catches the v strand leaving lane 63: a chunk's C
// inputs drain out at lane 0 while its C outputs fill lanes 64-C .. 63.
// Nothing touches LDS.
// Every C = 32 steps (a chunk) the wave publishes the C newest bottom-edge
// strands of its band to a ring in global memory as 64-bit (tag, strand) words stored with
// device-scope relaxed atomics; the band below polls for words carrying its
// tag, so no fence, flag or cache flush is needed.  Bands are handed out by an
// atomic ticket in launch order, so a wave only ever waits for a band that a
// resident wave already owns: any grid size makes progress.  Every wait is
// bounded in time; on expiry the kernel raises an abort flag that every wave
// checks, and all waves exit.
//
// Residuals (the reference's CPU fixup, src/lcs_grid.hpp:451-493) are handled
// in the kernel: lanes whose column is outside [0, n) hold a symbol no row
// matches and the largest strand (or, where no such symbol is known, skip the
// cells), rows beyond m in the last band never match and hold the smallest
// strand id; both pass every v strand through unchanged.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "cell_asm.h"
#include "comb_kernels.h"

namespace lcsk {

constexpr int kWave = 64;
constexpr int kDppWaveShl1 = 0x130;  // lane L reads lane L+1
constexpr int kDppWaveShr1 = 0x138;  // lane L reads lane L-1

__device__ __forceinline__ int32_t shl1_zero_i(int32_t x)
{
    return __builtin_amdgcn_mov_dpp(x, kDppWaveShl1, 0xf, 0xf, true);
}
// lane L <- x[L-1]; lane 0 keeps `old`
__device__ __forceinline__ uint32_t shr1_keep(uint32_t old_, uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old_, (int)x, kDppWaveShr1, 0xf, 0xf, false);
}
__device__ __forceinline__ int32_t shr1_keep_i(int32_t old_, int32_t x)
{
    return __builtin_amdgcn_update_dpp(old_, x, kDppWaveShr1, 0xf, 0xf, false);
}
// lane L <- x[L+1]; lane 63 keeps `old`
__device__ __forceinline__ uint32_t shl1_keep(uint32_t old_, uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old_, (int)x, kDppWaveShl1, 0xf, 0xf, false);
}

// Pointers read from a pair descriptor are generic; the band loop casts them
// to the global address space so its loads and stores are global_* rather
// than flat_* instructions.  A flat access may hit LDS, whose results return
// out of order, and that forces a full vmcnt(0) wait (on the in-flight ring
// store too) where a global access needs only vmcnt(1).
#define LCSK_GLOBAL __attribute__((address_space(1)))
typedef LCSK_GLOBAL unsigned long long gword;
typedef LCSK_GLOBAL const unsigned long long gcword;
typedef LCSK_GLOBAL const int32_t gsym;
typedef LCSK_GLOBAL const uint32_t gsym8;   // a word of four byte symbols
typedef LCSK_GLOBAL int32_t gout;
// LDS words polled through a pointer: the explicit address space keeps the
// reads ds_read (a volatile generic pointer would be a flat access, and a
// flat access waits for every outstanding global store).
typedef __attribute__((address_space(3))) volatile unsigned lds_flag;

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
__device__ __forceinline__ void raise_abort(unsigned *p)
{
    __hip_atomic_store(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One cell.  `sb` is the column symbol; `valid` is false for padding rows.
template <bool ROWMASK>
__device__ __forceinline__ void cell(int32_t sa, int32_t sb, bool valid, uint32_t &h, uint32_t &v)
{
    bool match = (sa == sb);
    if (ROWMASK) match = match && valid;
    uint32_t hx = match ? 0xffffffffu : h;
    uint32_t hn = min(hx, v);
    v = __builtin_amdgcn_bitop3_b32(h, v, hn, 0x96);
    h = hn;
}

// All TM rows of one column for one lane.
template <int TM, bool ROWMASK>
__device__ __forceinline__ void column_cells(const int32_t (&a)[TM], uint32_t (&h)[TM], const bool (&valid)[TM],
                                             int32_t sb, uint32_t &v)
{
    // Rows go through hand-scheduled blocks of up to 16 (cell_asm.h); one
    // block per column keeps the whole chain free of hazard nops.
    if constexpr (!ROWMASK && TM >= 4) {
        constexpr int R = TM >= 16 ? 16 : TM;
#pragma unroll
        for (int k = 0; k < TM; k += R) {
            uint32_t hn[R];
            if constexpr (R == 16) cell_block16(&a[k], &h[k], hn, sb, v);
            else if constexpr (R == 8) cell_block8(&a[k], &h[k], hn, sb, v);
            else cell_block4(&a[k], &h[k], hn, sb, v);
#pragma unroll
            for (int q = 0; q < R; ++q) h[k + q] = hn[q];
        }
    } else {
#pragma unroll
        for (int k = 0; k < TM; ++k) cell<ROWMASK>(a[k], sb, valid[k], h[k], v);
    }
}

// Two cells at once, pair X in the low and pair Y in the high 16 bits of
// every register (the packed chain): per half, swap iff sa == sb || h > v,
// as the 32-bit cell.  With e = sa ^ sb, sat(1 - e) is 1 on a match, and
// sat(h + 1 * 0xffff) = 0xffff replaces h there, so
//     hx = mad_sat(sat_sub(1, e), 0xffff, h),  hn = min(hx, v),  v' = h ^ v ^ hn
// is v_xor + v_pk_sub_u16 clamp + v_pk_mad_u16 clamp + v_pk_min_u16 +
// v_bitop3: 5 VALU for 2 cells (4 per cell in 32 bits).  Strand ids stay
// below 0xffff, the value a padded column carries.
typedef unsigned short lcsk_u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void cell16(uint32_t sa, uint32_t sb, uint32_t &h, uint32_t &v)
{
    const lcsk_u16x2 one = {1, 1};
    const lcsk_u16x2 mk = __builtin_elementwise_sub_sat(one, __builtin_bit_cast(lcsk_u16x2, sa ^ sb));
    uint32_t hx;
    asm("v_pk_mad_u16 %0, %1, -1, %2 clamp" : "=v"(hx) : "v"(__builtin_bit_cast(uint32_t, mk)), "v"(h));
    const uint32_t hn = __builtin_bit_cast(
        uint32_t, __builtin_elementwise_min(__builtin_bit_cast(lcsk_u16x2, hx), __builtin_bit_cast(lcsk_u16x2, v)));
    v = __builtin_amdgcn_bitop3_b32(h, v, hn, 0x96);
    h = hn;
}

// The packed cell with one-hot symbols (each half holds 1 << symbol, 0 for
// padding; alphabets of at most 16): sa & sb is nonzero exactly on a match,
// and sat(mk * 0xffff + h) is 0xffff there, so the match mask costs one
// v_and instead of v_xor + v_pk_sub_u16: 4 VALU for 2 cells.
__device__ __forceinline__ void cell16_oh(uint32_t sa, uint32_t sb, uint32_t &h, uint32_t &v)
{
    uint32_t hx;
    asm("v_pk_mad_u16 %0, %1, -1, %2 clamp" : "=v"(hx) : "v"(sa & sb), "v"(h));
    const uint32_t hn = __builtin_bit_cast(
        uint32_t, __builtin_elementwise_min(__builtin_bit_cast(lcsk_u16x2, hx), __builtin_bit_cast(lcsk_u16x2, v)));
    v = __builtin_amdgcn_bitop3_b32(h, v, hn, 0x96);
    h = hn;
}

// Steps t0 .. t0+C-1 of a band.  COLMASK: some lane's column leaves [0, n).
// Q (strands) and IB (symbols) are the conveyors.  On entry Q's lanes
// 0 .. C-1 hold the chunk's inputs (the input of step t0+s in lane s); each
// step hands Q's lane 0 to the band and shifts Q down one lane while lane
// 63's strand enters at the top, so on return Q's lanes 64-C .. 63 hold the
// chunk's outputs (columns t0-64 .. t0-64+C-1).  One shift serves both
// directions: C <= 64, so the inputs and outputs never meet.
template <int TM, int C, bool ROWMASK, bool COLMASK, bool PK = false, bool OH = false>
__device__ __forceinline__ void band_steps(const int32_t (&a)[TM], uint32_t (&h)[TM], const bool (&valid)[TM],
                                           uint32_t &v, int32_t &bq, uint32_t &Q, int32_t &IB, int t0, int lane, int n)
{
    if constexpr (PK && !COLMASK && C == 32 && TM >= 4 && TM <= 16) {
        // the packed chain's 32 steps, hand-offs included, in one asm block
        // (cell_asm.h): no step waits out a hazard with an s_nop
        uint32_t ua[TM];
#pragma unroll
        for (int q = 0; q < TM; ++q) ua[q] = (uint32_t)a[q];
        if constexpr (OH) cell16oh_chunk<TM>(ua, h, v, Q, IB, bq);
        else cell16_chunk<TM>(ua, h, v, Q, IB, bq);
        return;
    }
#pragma unroll
    for (int s = 0; s < C; ++s) {
        const int32_t bin = IB;
        IB = shl1_zero_i(IB);
        const uint32_t vn = shr1_keep(Q, v);   // lane 0 takes the band input Q[0]
        Q = shl1_keep(v, Q);                   // inputs move toward lane 0; lane 63's output enters at the top
        v = vn;
        bq = shr1_keep_i(bin, bq);
        bool active = true;
        if (COLMASK) {
            const int j = t0 + s - lane;
            active = (j >= 0) && (j < n);
        }
        if (active) {
            if constexpr (PK && OH) {
#pragma unroll
                for (int k = 0; k < TM; ++k) cell16_oh((uint32_t)a[k], (uint32_t)bq, h[k], v);
            } else if constexpr (PK && !COLMASK && TM >= 4) {
                // software-pipelined rows (cell_asm.h): no packed result is
                // read by the next issue, so no s_nop between the rows
                constexpr int R = TM >= 16 ? 16 : TM;
#pragma unroll
                for (int k = 0; k < TM; k += R) {
                    uint32_t ua[R], hn[R];
#pragma unroll
                    for (int q = 0; q < R; ++q) ua[q] = (uint32_t)a[k + q];
                    cell16_block<R>(ua, &h[k], hn, (uint32_t)bq, v);
#pragma unroll
                    for (int q = 0; q < R; ++q) h[k + q] = hn[q];
                }
            } else if constexpr (PK) {
#pragma unroll
                for (int k = 0; k < TM; ++k) cell16((uint32_t)a[k], (uint32_t)bq, h[k], v);
            } else {
                column_cells<TM, ROWMASK>(a, h, valid, bq, v);
            }
        }
    }
}

// All TM rows of one column for one lane when the column symbol is byte SEL
// of `word` (byte symbols; a row symbol matches it zero-extended, so row
// symbols outside [0, 255] never match, as no column symbol is).
template <int TM, bool ROWMASK, int SEL>
__device__ __forceinline__ void column_cells8(const int32_t (&a)[TM], uint32_t (&h)[TM], const bool (&valid)[TM],
                                              uint32_t word, uint32_t &v)
{
    if constexpr (!ROWMASK && TM >= 4) {
        constexpr int R = TM >= 16 ? 16 : TM;
#pragma unroll
        for (int k = 0; k < TM; k += R) {
            uint32_t hn[R];
            cell_block_byte<R, SEL>(&a[k], &h[k], hn, (int32_t)word, v);
#pragma unroll
            for (int q = 0; q < R; ++q) h[k + q] = hn[q];
        }
    } else {
        const int32_t sb = (int32_t)((word >> (8 * SEL)) & 0xffu);
#pragma unroll
        for (int k = 0; k < TM; ++k) cell<ROWMASK>(a[k], sb, valid[k], h[k], v);
    }
}

// Step t of a band with byte symbols: the strand moves as in band_steps;
// the column symbol is byte SEL of `word`, which the lane holds itself.
// An unmasked step of four or more rows runs as one asm block (cell_asm.h:
// the strand hand-off sits behind the step's first two compares, so the DPP
// read of v needs no s_nop after the previous step's last cell wrote it);
// band_steps8 uses this for 32-row tiles.
template <int TM, bool ROWMASK, bool COLMASK, int SEL>
__device__ __forceinline__ void band_step8(const int32_t (&a)[TM], uint32_t (&h)[TM], const bool (&valid)[TM],
                                           uint32_t &v, uint32_t &Q, uint32_t word, int t, int lane, int n)
{
    if constexpr (!ROWMASK && !COLMASK && TM >= 4) {
        constexpr int R = TM >= 16 ? 16 : TM;
        uint32_t w = v, vt;
        {
            uint32_t hn[R];
            cell_step_byte<R, SEL>(&a[0], &h[0], hn, (int32_t)word, Q, w, vt);
#pragma unroll
            for (int q = 0; q < R; ++q) h[q] = hn[q];
        }
#pragma unroll
        for (int k = R; k < TM; k += R) {
            uint32_t hn[R];
            cell_block_byte<R, SEL>(&a[k], &h[k], hn, (int32_t)word, vt);
#pragma unroll
            for (int q = 0; q < R; ++q) h[k + q] = hn[q];
        }
        Q = w;    // moved down one lane, lane 63 holding the strand that left the band
        v = vt;
        return;
    }
    const uint32_t vn = shr1_keep(Q, v);
    Q = shl1_keep(v, Q);
    v = vn;
    bool active = true;
    if (COLMASK) {
        const int j = t - lane;
        active = (j >= 0) && (j < n);
    }
    if (active) column_cells8<TM, ROWMASK, SEL>(a, h, valid, word, v);
}

// Steps t0 .. t0+C-1 of a band whose column symbols are bytes: sym[s / 4]
// byte s % 4 is the symbol of the column this lane combs at step t0 + s
// (every lane holds its own C symbols), so only the strand conveyor Q
// moves between lanes.
template <int TM, int C, bool ROWMASK, bool COLMASK>
__device__ __forceinline__ void band_steps8(const int32_t (&a)[TM], uint32_t (&h)[TM], const bool (&valid)[TM],
                                            uint32_t &v, uint32_t &Q, const uint32_t (&sym)[C / 4], int t0, int lane,
                                            int n)
{
// The compiler puts an s_nop 0 before every asm block that reads the strand,
// so larger blocks pay it less often (m = n = 2^20: 131.5 ms per comb with
// chunk blocks, 132.0 with a block per symbol word on the same box; 133.6 with
// a block per step against 132.1 for words on another).
    if constexpr (C == 32 && !ROWMASK && !COLMASK && TM <= 16) {
        // the whole chunk in one asm block (cell_asm.h)
        uint32_t qn;
        cell_chunk32<TM>(a, h, sym, Q, v, qn);
        Q = qn;
        return;
    }
    if constexpr (C == 16 && !ROWMASK && !COLMASK && TM <= 16) {
        // half a chunk of a linked band (cell_asm.h)
        uint32_t qn;
        cell_chunk16<TM>(a, h, sym, Q, v, qn);
        Q = qn;
        return;
    }
#pragma unroll
    for (int w = 0; w < C / 4; ++w) {
        const int t = t0 + 4 * w;
        band_step8<TM, ROWMASK, COLMASK, 0>(a, h, valid, v, Q, sym[w], t, lane, n);
        band_step8<TM, ROWMASK, COLMASK, 1>(a, h, valid, v, Q, sym[w], t + 1, lane, n);
        band_step8<TM, ROWMASK, COLMASK, 2>(a, h, valid, v, Q, sym[w], t + 2, lane, n);
        band_step8<TM, ROWMASK, COLMASK, 3>(a, h, valid, v, Q, sym[w], t + 3, lane, n);
    }
}

constexpr int kRingPolls = 8;    // ring polls per look at the abort flag and the clock

// Linked bands (comb_group_kernel): the four bands of a workgroup hand
// strands to each other through LDS.  Link w carries the strands leaving
// wave w's band to wave w+1's as a ring of kLinkSlots column chunks guarded
// by two progress words: the producer's last published chunk and the
// consumer's last consumed one.
constexpr int kGroupW = 4;       // bands (waves) per workgroup, one per SIMD
constexpr int kLinkSlots = 16;   // column chunks in flight on one link
struct GroupLds {
    volatile int prog[kGroupW];   // prog[w]: last column chunk wave w published (-1: none)
    volatile int cons[kGroupW];   // cons[w]: last chunk wave w took from wave w-1
    volatile unsigned stop;       // set by a wave whose wait expired
};
typedef __attribute__((address_space(3))) GroupLds lds_group;
typedef __attribute__((address_space(3))) volatile uint32_t lds_word;

// A linked wave's ends: its position in the group and the rings on both
// sides (in: from wave w-1, out: to wave w+1).
struct BandLink {
    lds_group *G;
    lds_word *in, *out;
    int w;
    bool first, last;   // wave-uniform: reads the global ring / has no consumer in the group
};

// Spins until *word >= target (LDS).  When the stop word is set or the time
// runs out (then both abort words are raised) `dead` is set instead; a dead
// wave waits for nothing any more and runs its band to the end on whatever
// it holds, so no wait has an exit that the band loop would have to carry.
// A wave in step with the one above it comes here every chunk, so most polls
// read nothing else: the clock is a memory round trip away.
constexpr int kFastPolls = 64;
__device__ __forceinline__ void lds_wait_ge(__attribute__((address_space(3))) volatile int *word, int target,
                                            lds_group *G, const ChainArgs &A, int &dead)
{
    unsigned long long t_start = 0;
#pragma nounroll
    for (int i = 1; !dead; ++i) {
        if (__builtin_amdgcn_readfirstlane(*word) >= target) return;
        if (A.poll_sleep) __builtin_amdgcn_s_sleep(1);
        if (i % kFastPolls == 0) {
            const unsigned long long now = __builtin_amdgcn_s_memrealtime();
            if (t_start == 0) t_start = now;
            const bool late = A.timeout_ticks == 0 || now - t_start > A.timeout_ticks;
            if (late) raise_abort(A.abort_flag);
            if (late) G->stop = 1u;
            dead = __builtin_amdgcn_readfirstlane(G->stop) != 0;
        }
    }
}

// Every band runs the same sequence of memory operations: it reads its top
// edge from ring slot g&1 (tag g) and writes its bottom edge to slot (g+1)&1
// (tag g+1).  The prep kernel seeds slot 0 with the grid's top edge (tag 0)
// and the extract kernel reads v_out from the last band's slot, so no
// branch on the band's position sits between a load and its wait.
// PK: the packed chain over a CoupleDesc -- every symbol and strand
// register holds pair X in its low and pair Y in its high 16 bits.  Rows
// past a pair's m hold symbol kPadRow16 and strand 0 and columns past its n
// carry symbol kPadCol16 and strand 0xffff: they never match and never
// swap, so they pass every strand through unchanged and ROWMASK is not
// needed.
constexpr uint32_t kPadRow16 = 0xffffu, kPadCol16 = 0xfffeu;

// What a band's column symbols are: 32-bit words, bytes, or bytes whose
// padding (255) no symbol of b equals.
constexpr int kSymWords = 0, kSymBytes = 1, kSymBytesPadded = 2;

// S8: the column symbols come from the byte copies of b (P.sym8) instead of
// b; every lane loads its own C symbols of the next chunk (C/4 words from
// the copy that starts its window on a word boundary) and no symbol
// conveyor runs.
//
// LK: a band of a linked group.  Its first wave reads the global ring and the
// others the LDS link of the wave above; every wave also stores to the global
// ring as an unlinked band does (only the last wave's words are read from
// there, by the next group or the extract kernel), so that no path skips the
// store and no wait for a load ever covers a store in flight.  A chunk's
// outputs go to the link as soon as its steps are done, and the next chunk's
// inputs are read from the link halfway through the chunk: a lag of 64 + 32 +
// 16 steps against the global hand-off's 64 + 32 + 32 (its load is issued a
// chunk ahead, which hides the trip through memory).  The link's reads,
// progress words and branches cost more than those 16 steps: m = n = 16384
// at 4 rows per lane 0.94 ms against the chain's 0.85 (1.24 and 1.09 before
// the groups shared band_pass), so only LCS_VARIANT_CHAIN_LDS comes here.
//
// The first and last chunks of a band (some lane's column outside [0, n))
// run the same unmasked steps as the others where a symbol exists that no
// row of the band can match (PAD): lanes outside [0, n) then carry that
// symbol and the strand ~0, which every row lets pass unchanged
// (hn = min(h, ~0) = h, v' = ~0).  The packed chain has its pad symbols, the
// byte copies are padded with 255 (kSym8Has255 in the flag word keeps the
// masked steps for a b that holds it), and the 32-bit path looks for a value
// that none of the band's rows holds.  A masked step takes several times an
// unmasked one's time, and the first 96 steps of a band lie between its first
// input and its first output, so masked ramps set the band-to-band lag of the
// whole chain: m = n = 16384 at 4 rows per lane, one strip, took 1.09 ms with
// masked ramps and 0.91 without; with the wait loops and the publish below
// as they are now, 0.85 (2 rows per lane: 1.18, 0.93, 0.73).
template <int TM, int C, bool ROWMASK, bool PK, typename Desc, int S8 = kSymWords, bool OH = false, bool LK = false>
__device__ __forceinline__ bool band_pass(const ChainArgs &A, const Desc &P, int g, int lane, int t_id,
                                          const BandLink &K = BandLink{}, int32_t row_pad = 0)
{
    static_assert(!LK || (!PK && C == 32), "linked bands");
    constexpr bool PAD = PK || S8 == kSymBytesPadded || (!S8 && !ROWMASK);
    const int m = P.m, n = P.n;
    const int r0 = g * (kWave * TM) + lane * TM;
    if (A.trace && t_id < A.trace_cap && lane == 0) A.trace[2 * (size_t)t_id] = __builtin_amdgcn_s_memrealtime();
    int32_t a[TM];
    uint32_t h[TM];
    bool valid[TM];
#pragma unroll
    for (int k = 0; k < TM; ++k) {
        const int r = r0 + k;
        if constexpr (PK) {
            uint32_t sa = 0, hh = 0;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const bool in = r < P.m_[q];
                uint32_t sym;
                if constexpr (OH) sym = in ? 1u << ((uint32_t)P.a[q][r] & 15u) : 0u;
                else sym = in ? ((uint32_t)P.a[q][r] & 0xffffu) : kPadRow16;
                const uint32_t id = in ? (uint32_t)(P.m_[q] - 1 - r) : 0u;
                sa |= sym << (16 * q);
                hh |= id << (16 * q);
            }
            valid[k] = true;
            a[k] = (int32_t)sa;
            h[k] = hh;
        } else if constexpr (S8) {
            // rows past m hold a symbol no byte equals and strand 0: they
            // never match and never swap (min(0, v) = 0), so every strand
            // passes them unchanged and the band needs no row mask
            valid[k] = r < m;
            a[k] = valid[k] ? P.a[r] : -1;
            if (S8 == kSymBytesPadded && a[k] == 255) a[k] = -1;   // b holds no 255
            h[k] = valid[k] ? (P.h_in ? (uint32_t)P.h_in[m - 1 - r] : (uint32_t)(m - 1 - r)) : 0u;
        } else {
            // rows past m: masked, or (row_pad) a symbol that b does not hold and
            // strand 0, as in the byte chain
            valid[k] = r < m;
            a[k] = valid[k] ? P.a[r] : row_pad;
            h[k] = valid[k] ? (P.h_in ? (uint32_t)P.h_in[m - 1 - r] : (uint32_t)(m - 1 - r)) : 0u;
        }
    }
    // the symbol of a column outside [0, n) (PAD): one that no row holds; the
    // search ends within 64 TM + 1 values and nearly always at once
    [[maybe_unused]] int32_t pad = OH ? 0 : (int32_t)(kPadCol16 << 16 | kPadCol16);
    if constexpr (PAD && !PK && !S8) {
        for (pad = -1;; --pad) {
            bool hit = false;
#pragma unroll
            for (int k = 0; k < TM; ++k) hit = hit || a[k] == pad;
            if (__builtin_amdgcn_ballot_w64(hit) == 0) break;
        }
    }
    const uint32_t tag_in = (uint32_t)g;
    const unsigned long long tag_out = (unsigned long long)(g + 1) << 32;
    gcword *Ein = (gcword *)(P.E + (size_t)(g & 1) * (size_t)n);
    gword *Eout = (gword *)(P.E + (size_t)((g + 1) & 1) * (size_t)n);
    const int nchunks = (n + kWave + C - 1) / C;
    // the column symbol of column c >= 0 (any from n on, or for the packed chain
    // the pad symbol), always loaded from an in-bounds address; INSIDE: c < n
    // is known
    auto load_b = [&](auto c, auto inside) -> int32_t {
        if constexpr (PK) {
            uint32_t x = 0;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const uint32_t raw = (uint32_t)((gsym *)P.b[q])[min((int)c, P.n_[q] - 1)];
                if constexpr (OH) x |= ((int)c < P.n_[q] ? 1u << (raw & 15u) : 0u) << (16 * q);
                else x |= ((int)c < P.n_[q] ? raw & 0xffffu : kPadCol16) << (16 * q);
            }
            return (int32_t)x;
        } else if constexpr (decltype(inside)::value) {
            return ((gsym *)P.b)[c];
        } else {
            return ((gsym *)P.b)[min((int)c, n - 1)];
        }
    };
    // the pad symbol in place of a 32-bit symbol loaded for column c >= n: done
    // where the chunk's steps take the symbols over, as anything computed from
    // a prefetched symbol before them waits for its load (one row per lane, one
    // band of 100000 columns: 20.0 ns a step with the select at the load, 18.7
    // here)
    auto pad_past_n = [&](int32_t x, int c) -> int32_t { return PAD && !PK && c >= n ? pad : x; };

    // Byte symbols: lane L combs column t - L at step t, the byte at
    // x0 + t of the padded symbol string (x0 = kSym8Pad - L >= 65);
    // copy j = x0 % 4 holds it at byte x0 - j + t, a word boundary for
    // every chunk (t0 is a multiple of C).  The copies extend kSym8Pad
    // bytes past column n, beyond the last prefetch (t0 <= n + 64 + C).
    static_assert(!S8 || (C % 4 == 0 && kWave + 2 * C - 2 < kSym8Pad), "byte-symbol window");
    [[maybe_unused]] uint32_t sym[C / 4], psym[C / 4];
    [[maybe_unused]] gsym8 *sym_base = nullptr;
    if constexpr (S8) {
        const int x0 = kSym8Pad - lane;
        const int j = x0 & 3;
        sym_base = (gsym8 *)P.sym8 + (size_t)j * (size_t)P.sym8_stride + ((x0 - j) >> 2);
    }
    auto load_sym = [&](uint32_t (&d)[C / 4], int t) {
        gsym8 *p = sym_base + (t >> 2);
#pragma unroll
        for (int q = 0; q < C / 4; ++q) d[q] = p[q];
    };
    // prefetch chunk 0.  Every lane loads from a clamped in-bounds address
    // (no exec masking, no select), so the waits before each chunk cover
    // exactly these loads.
    const int nm1 = n - 1;
    // Only lanes < C use their words (the conveyors start at lane 0 and
    // shift C times); lanes >= C load the same addresses, so each chunk
    // fetches C words, not 64.
    int32_t pB = 0;
    if constexpr (S8) load_sym(sym, 0);
    else pB = pad_past_n(load_b(lane & (C - 1), std::false_type{}), lane & (C - 1));
    unsigned long long pE = 0;
    if (!LK || K.first) pE = ld_relaxed(Ein + min(lane & (C - 1), nm1));
    // Publishes the C bottom-edge strands caught in O during the chunk that
    // started at step t: lanes 64-C .. 63 hold columns t-64 .. t-64+C-1.
    // Inside the grid every lane stores (lane L the word of lane 64-C + L%C,
    // which v_permlane32_swap brings down for C = 32): a lane mask would put
    // a branch round the store, and the waits for the prefetch loads could
    // then not leave it in flight.  The first and last chunks of a band leave
    // columns outside [0, n) out.  A chunk's words are published at the start
    // of the next chunk, behind that chunk's loads.
    static_assert(C == kWave / 2, "publish moves the upper half of the wave to both halves");
    auto both_halves = [](uint32_t x) {
        return (uint32_t)__builtin_amdgcn_permlane32_swap((int)x, (int)x, false, false)[1];
    };
    // INSIDE: every column is known to be in [0, n) (the interior chunks below)
    auto publish = [&](uint32_t Ox, int t, auto inside) {
        const int col = t - kWave + (lane & (C - 1));
        const uint32_t x = both_halves(Ox);
        if (decltype(inside)::value || (col >= 0 && col < n))
            st_relaxed(Eout + (uint32_t)col, tag_out | (unsigned long long)x);
    };
    // Turns the prefetched ring words of the chunk starting at t into lane 0's
    // conveyor I (waiting, bounded in time, until they carry this band's tag).
    // INSIDE: the chunk's columns are known to be < n.
    // Set when a wait gave up: nothing is waited for after that, and the band
    // runs to its end on whatever it holds.  An early return from each wait
    // made the compiler carry the band's registers over every exit (about 20
    // copies and several branches a chunk).
    int dead = 0;
    // Byte chains of one row per lane: a chunk of 32 steps is shorter
    // than the trips through memory, and a band that is just in time prefetches
    // the words of a chunk before the band above has stored them.  The lines it
    // then holds make that band's stores slow, and a store two chunks back is
    // what its next loads queue behind (vmcnt counts both in order), so the
    // whole chain falls to the pace of its stores and stays there: one row, 16
    // bands, 100000 columns 1.75 to 2.5 ms, some runs 1.3.  So a band that had
    // to wait waits for one chunk more (band_slack, comb_kernels.h): 1.33 ms
    // (50000 columns and 32 bands 1.25 -> 0.73).  Two rows fall to 24 ns a step
    // from 20 at worst, but the longer poll loop costs them 1 % where it does
    // not help (50021 x 70207 as a grid 1540 -> 1551 us), so they have none.
    const int slack = TM == 1 && S8 != kSymWords && band_slack(TM, P.nbands, n) ? C : 0;
    auto take_inputs = [&](int t, uint32_t &I, auto inside) {
        const int c = t + (lane & (C - 1));   // lanes >= C repeat lanes < C
        const bool need = decltype(inside)::value || c < n;
        unsigned long long e = pE;
        // keeps the tag test (and so the wait for the prefetched word) after
        // the chunk's last step: I still holds the conveyor the chunk left,
        // which that step wrote, so the compare cannot be hoisted next to
        // the load to wait there for the whole round trip
        asm volatile("" : "+v"(e) : "v"(I));
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(need && (uint32_t)(e >> 32) != tag_in) != 0, 0)) {
            // The band above is not that far yet: poll, looking at the abort
            // flag and the clock every few rounds only (each is a memory
            // round trip of its own).
            unsigned long long t_start = 0;
            int ahead = slack;
#pragma nounroll
            for (int polls = 0; !dead; ++polls) {
                // a wave that shares its SIMD with other launches' waves
                // gives up its issue slots between polls
                if (A.poll_sleep) __builtin_amdgcn_s_sleep(2);
                e = ld_relaxed(Ein + min(c + ahead, nm1));
                if (__builtin_amdgcn_ballot_w64(need && (uint32_t)(e >> 32) != tag_in) == 0) {
                    if (ahead == 0) break;
                    ahead = 0;
                }
                if (polls % kRingPolls == 0) {
                    const unsigned long long now = __builtin_amdgcn_s_memrealtime();
                    if (polls == 0) t_start = now;
                    const bool late = A.timeout_ticks == 0 || now - t_start > A.timeout_ticks;
                    if (late) raise_abort(A.abort_flag);
                    dead = late || __builtin_amdgcn_readfirstlane(ld_flag(A.abort_flag)) != 0;
                }
            }
        }
        I = PAD && !need ? ~0u : (uint32_t)e;
    };
    // Linked bands: what a wave reads from LDS halfway through chunk j - 1
    // (the producer's progress, then the words of column chunk j; LDS runs a
    // wave's accesses in order, so the progress vouches for the words) and
    // checks when chunk j starts.
    [[maybe_unused]] int lk_prog = 0, lk_cons = 0;
    [[maybe_unused]] uint32_t lk_in = 0;
    [[maybe_unused]] const int lk_chunks = (n + C - 1) / C;   // column chunks that carry inputs
    auto link_read = [&](int j) {
        if (!K.first) {
            if (lane == 0) K.G->cons[K.w] = j - 1;   // the chunk before is in registers
            lk_prog = K.G->prog[K.w - 1];
            lk_in = K.in[(j & (kLinkSlots - 1)) * C + (lane & (C - 1))];
        }
        if (!K.last) lk_cons = K.G->cons[K.w + 1];
    };
    auto link_take = [&](int j, uint32_t &I) {
        if (__builtin_expect(__builtin_amdgcn_readfirstlane(lk_prog) < j, 0)) {
            lds_wait_ge(&K.G->prog[K.w - 1], j, K.G, A, dead);
            lk_in = K.in[(j & (kLinkSlots - 1)) * C + (lane & (C - 1))];
        }
        I = lk_in;
    };
    // the outputs of column chunk j, in lanes 64-C .. 63 of Ox
    auto link_put = [&](int j, uint32_t Ox) {
        if (__builtin_expect(__builtin_amdgcn_readfirstlane(lk_cons) < j - kLinkSlots, 0))
            lds_wait_ge(&K.G->cons[K.w + 1], j - kLinkSlots, K.G, A, dead);
        K.out[(j & (kLinkSlots - 1)) * C + (lane & (C - 1))] = both_halves(Ox);
        if (lane == 0) K.G->prog[K.w] = j;
    };
    uint32_t v = PAD ? ~0u : 0u, Q = 0, Osave = 0;
    int32_t bq = PAD ? pad : 0, IB = pB;
    if (!LK || K.first) {
        take_inputs(0, Q, std::false_type{});
    } else {
        link_read(0);
        link_take(0, Q);
        if (PAD && (lane & (C - 1)) >= n) Q = ~0u;
    }
    // One chunk: prefetch chunk k+1, then publish chunk k-1 (the wait for the
    // loads at the end then leaves the store in flight), comb C steps, take
    // the next inputs.  The chunks run in three phases (ramp-in, interior,
    // ramp-out) so the hot loop holds only the unmasked steps and no
    // register copies between masked and unmasked paths; the interior loop
    // takes two chunks per iteration, which lets the compiler close it
    // without copying the h registers (with one chunk it copied them).
    // Issuing the prefetch halfway through the chunk instead was measured no
    // faster.
    using Masked = std::integral_constant<bool, true>;
    using Full = std::integral_constant<bool, false>;
    auto chunk = [&](auto colmask, int k) {
        const int t0 = k * C;
        constexpr bool CM = decltype(colmask)::value && !PAD;   // masked steps
        if constexpr (S8) load_sym(psym, t0 + C);
        if constexpr (decltype(colmask)::value) {
            const int c = t0 + C + (lane & (C - 1));
            if constexpr (!S8) pB = load_b(c, std::false_type{});
            if (!LK || K.first) pE = ld_relaxed(Ein + min(c, nm1));
        } else {   // an interior chunk: the next chunk's columns are inside [0, n)
            const uint32_t c = (uint32_t)(t0 + C + (lane & (C - 1)));
            if constexpr (!S8) pB = load_b(c, std::true_type{});
            if (!LK || K.first) pE = ld_relaxed(Ein + c);
        }
        publish(Osave, t0 - C, std::integral_constant<bool, !decltype(colmask)::value>{});
        if constexpr (LK) {
            // two halves, the link's words read between them
            constexpr int H = C / 2;
            if constexpr (S8) {
                uint32_t lo[H / 4], hi[H / 4];
#pragma unroll
                for (int q = 0; q < H / 4; ++q) {
                    lo[q] = sym[q];
                    hi[q] = sym[H / 4 + q];
                }
                band_steps8<TM, H, ROWMASK, CM>(a, h, valid, v, Q, lo, t0, lane, n);
                link_read(k + 1);
                band_steps8<TM, H, ROWMASK, CM>(a, h, valid, v, Q, hi, t0 + H, lane, n);
            } else {
                band_steps<TM, H, ROWMASK, CM>(a, h, valid, v, bq, Q, IB, t0, lane, n);
                link_read(k + 1);
                band_steps<TM, H, ROWMASK, CM>(a, h, valid, v, bq, Q, IB, t0 + H, lane, n);
            }
        } else if constexpr (S8) {
            band_steps8<TM, C, ROWMASK, CM>(a, h, valid, v, Q, sym, t0, lane, n);
        } else {
            band_steps<TM, C, ROWMASK, CM, PK, OH>(a, h, valid, v, bq, Q, IB, t0, lane, n);
        }
        Osave = Q;
        if constexpr (LK) {
            // chunk k completes column chunk k - 64 / C; an interior chunk
            // always completes one that carries outputs
            const int jo = k - kWave / C;
            if (!K.last && (!decltype(colmask)::value || (jo >= 0 && jo < lk_chunks)))
                link_put(jo, Q);
        }
        if (!decltype(colmask)::value || k + 1 < nchunks) {   // an interior chunk is never the last
            if constexpr (S8) {
#pragma unroll
                for (int q = 0; q < C / 4; ++q) sym[q] = psym[q];
            }
            if constexpr (decltype(colmask)::value) IB = pad_past_n(pB, t0 + C + (lane & (C - 1)));
            else IB = pB;
            if (!LK || K.first) {
                take_inputs(t0 + C, Q, std::integral_constant<bool, !decltype(colmask)::value>{});
            } else if (!decltype(colmask)::value || k + 1 < lk_chunks) {
                link_take(k + 1, Q);
                if (PAD && decltype(colmask)::value && t0 + C + (lane & (C - 1)) >= n) Q = ~0u;
            } else {
                Q = ~0u;   // columns past n
            }
        }
    };
    // Interior chunks: no lane's column leaves [0, n) (t0 >= 63, t0 + C <= n),
    // the next chunk's prefetch stays inside (t0 + 2C <= n) and so does the
    // publish of the chunk before (columns t0 - 64 - C .. t0 - 65, so
    // t0 >= 64 + C).
    const int k_in = (kWave + C) / C;                      // first interior chunk
    const int k_out = max(k_in, min(n / C - 1, nchunks));  // first chunk after them
    int k = 0;
    for (; k < min(k_in, nchunks); ++k) chunk(Masked{}, k);
    for (; k + 1 < k_out; k += 2) {
        chunk(Full{}, k);
        chunk(Full{}, k + 1);
    }
    for (; k < k_out; ++k) chunk(Full{}, k);
    for (; k < nchunks; ++k) chunk(Masked{}, k);
    publish(Osave, (nchunks - 1) * C, std::false_type{});
    if constexpr (PK) {
#pragma unroll
        for (int k = 0; k < TM; ++k)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                if (r0 + k < P.m_[q]) P.h_out[q][P.m_[q] - 1 - (r0 + k)] = (int32_t)((h[k] >> (16 * q)) & 0xffffu);
    } else {
#pragma unroll
        for (int k = 0; k < TM; ++k)
            if (valid[k]) {
                const int l = m - 1 - (r0 + k);
                // ids are below m+n after a completed comb; the test keeps an
                // aborted one (whose strands are undefined) from writing out of range
                if (P.h_out) P.h_out[l] = (int32_t)h[k];
                if (P.perm && h[k] < (uint32_t)(m + n)) P.perm[h[k]] = n + l;
            }
    }
    if (A.trace && t_id < A.trace_cap && lane == 0) A.trace[2 * (size_t)t_id + 1] = __builtin_amdgcn_s_memrealtime();
    return !dead;
}

// One band of a pair, by what its column symbols are: bytes when the pair has
// byte copies and all of b fits in a byte, else 32-bit words.  A partial band
// (only a pair's last one) pads its rows; 32-bit words without a known absent
// symbol mask them, and as the chain's last band that one sets the pace of
// the whole launch.
template <int TM, int C, bool LK>
__device__ __forceinline__ bool band_dispatch(const ChainArgs &A, const PairDesc &P, int g, int lane, int t_id,
                                              const BandLink &K)
{
    const int flags = P.sym8 ? __builtin_amdgcn_readfirstlane(*P.sym8_flags) : kSym8Bad;
    if (!(flags & kSym8Bad)) {
        if (!(flags & kSym8Has255))
            return band_pass<TM, C, false, false, PairDesc, kSymBytesPadded, false, LK>(A, P, g, lane, t_id, K);
        return band_pass<TM, C, false, false, PairDesc, kSymBytes, false, LK>(A, P, g, lane, t_id, K);
    }
    // rows past m take a symbol that b does not hold, when the flags know one
    const uint32_t absent = P.sym8 ? ~(uint32_t)flags >> 8 : 0u;
    const bool rowmask = (long long)(g + 1) * (kWave * TM) > (long long)P.m && absent == 0;
    const int32_t row_pad = absent ? -1 - (int32_t)__builtin_ctz(absent) : 0;
    return rowmask ? band_pass<TM, C, true, false, PairDesc, kSymWords, false, LK>(A, P, g, lane, t_id, K)
                   : band_pass<TM, C, false, false, PairDesc, kSymWords, false, LK>(A, P, g, lane, t_id, K, row_pad);
}

// Tile p of a grid as a pair of its own.
__device__ __forceinline__ PairDesc tile_pair(const TileGrid &T, int p)
{
    PairDesc P = T.pair;
    if (T.GR * T.GC > 1) {
        const int i = p / T.GC, j = p - i * T.GC;
        P.a += (size_t)i * T.H;
        P.b += (size_t)j * T.W;
        P.m = T.rows(i);
        P.n = T.cols(j);
        P.E += (size_t)p * (2 * (size_t)T.W + 64);
        if (P.sym8) P.sym8 += (size_t)j * 4 * (size_t)P.sym8_stride;
        P.h_out = P.v_out = nullptr;
        P.perm = T.perm + T.perm_off(i, j);
        P.nbands = (P.m + kWave * P.tile_m - 1) / (kWave * P.tile_m);
    }
    return P;
}

// The pair of task t and its band (or group); a grid's last tile row may have
// fewer bands than the others (then P.nbands <= the band: no work).
__device__ __forceinline__ PairDesc task_pair(const ChainArgs &A, unsigned t, int &unit)
{
    if (A.pairs) {
        const int2 task = A.tasks[t];
        unit = task.y;
        return A.pairs[task.x];
    }
    const unsigned tiles = (unsigned)(A.grid.GR * A.grid.GC);
    unit = (int)(t / tiles);
    return tile_pair(A.grid, (int)(t % tiles));
}

template <int TM, int C>
__global__ __launch_bounds__(256) void comb_chain_kernel(ChainArgs A)
{
    const int lane = threadIdx.x & (kWave - 1);
    for (;;) {
        unsigned t = 0;
        if (lane == 0) t = atomicAdd(A.ticket, 1u);
        t = __builtin_amdgcn_readfirstlane(t);
        if ((int)t >= A.ntasks) break;
        if (__builtin_amdgcn_readfirstlane(ld_flag(A.abort_flag))) break;
        int g;
        const PairDesc P = task_pair(A, t, g);
        if (g >= P.nbands) continue;
        if (!band_dispatch<TM, C, false>(A, P, g, lane, (int)t, BandLink{})) break;
    }
}

// The packed chain: ticket t runs band tasks[t].y of couple tasks[t].x.
template <int TM, int C>
__global__ __launch_bounds__(256) void comb_chain16_kernel(ChainArgs A)
{
    const int lane = threadIdx.x & (kWave - 1);
    for (;;) {
        unsigned t = 0;
        if (lane == 0) t = atomicAdd(A.ticket, 1u);
        t = __builtin_amdgcn_readfirstlane(t);
        if ((int)t >= A.ntasks) break;
        if (__builtin_amdgcn_readfirstlane(ld_flag(A.abort_flag))) break;
        const int2 task = A.tasks[t];
        const CoupleDesc D = A.couples[task.x];
        const bool ok = __builtin_amdgcn_readfirstlane(D.onehot)
                            ? band_pass<TM, C, false, true, CoupleDesc, kSymWords, true>(A, D, task.y, lane, (int)t)
                            : band_pass<TM, C, false, true>(A, D, task.y, lane, (int)t);
        if (!ok) break;
    }
}

// ---- linked groups ----------------------------------------------------------
//
// kGroupW consecutive bands of one pair share a workgroup, one wave per band
// (one per SIMD of a CU), linked through LDS (band_pass, LK): three of four
// hand-offs go through LDS instead of memory.
// Ticket t runs band group tasks[t].y (bands W*y .. W*y+W-1) of pair
// tasks[t].x.  The only barriers are the three per task, which every wave
// passes whatever its band did.
template <int TM, int C>
__global__ __launch_bounds__(kWave * kGroupW) void comb_group_kernel(ChainArgs A)
{
    constexpr int W = kGroupW;
    __shared__ uint32_t links[W - 1][kLinkSlots * C];
    __shared__ GroupLds group;
    __shared__ unsigned s_task, s_stop;
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    lds_group *G = (lds_group *)&group;
    for (;;) {
        __syncthreads();  // every wave is done with the previous task's LDS
        if (threadIdx.x == 0) {
            const unsigned t = atomicAdd(A.ticket, 1u);
            s_task = t;
            s_stop = ((int)t >= A.ntasks || ld_flag(A.abort_flag)) ? 1u : 0u;
            for (int i = 0; i < W; ++i) {
                G->prog[i] = -1;
                G->cons[i] = -1;
            }
            G->stop = 0u;
        }
        __syncthreads();
        const unsigned t = __builtin_amdgcn_readfirstlane(s_task), stop = __builtin_amdgcn_readfirstlane(s_stop);
        __syncthreads();
        if (stop) break;
        int unit;
        const PairDesc P = task_pair(A, t, unit);
        const int g0 = unit * W;
        const int wact = min(W, P.nbands - g0);
        if (w < wact) {
            const int g = g0 + w, trace_id = (int)t * W + w;
            const BandLink K = {G, (lds_word *)&links[w > 0 ? w - 1 : 0][0], (lds_word *)&links[w < W - 1 ? w : 0][0], w,
                                w == 0, w == wact - 1};
            const bool ok = band_dispatch<TM, C, true>(A, P, g, lane, trace_id, K);
            if (!ok && lane == 0) G->stop = 1u;  // let the group's other waves stop waiting
        }
    }
}

// Byte symbols of a strip of ns columns at b (the layout lcsk_sym8_stride
// describes), one thread per word; copy 0 (which covers every column) raises
// *flags for a symbol outside [0, 255] or equal to the padding.
__device__ __forceinline__ void stage_sym8(const int32_t *b, int32_t ns, uint32_t *out, int32_t stride, int32_t *flags)
{
    const long long total = 4LL * stride;
    const long long step = (long long)gridDim.x * blockDim.x;
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += step) {
        const int j = (int)(q / stride);
        const long long x = 4 * (q - (long long)j * stride) + j - kSym8Pad;   // column of byte 0
        uint32_t word = 0;
        int seen = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const long long c = x + i;
            uint32_t sym = 255u;
            if (c >= 0 && c < ns) {
                sym = (uint32_t)b[c];
                seen |= sym > 255u ? kSym8Bad : sym == 255u ? kSym8Has255 : 0;
                if (~sym < (uint32_t)kSym8RowPads) seen |= 0x100 << ~sym;
            }
            word |= (sym & 0xffu) << (8 * i);
        }
        out[q] = word;
        if (seen && j == 0) atomicOr(flags, seen);
    }
}

__global__ void comb_sym8_kernel(const int32_t *b, int32_t n, uint32_t *out, int32_t stride, int32_t *flags)
{
    stage_sym8(b, n, out, stride, flags);
}

// Seeds the rings before a chain launch (blockIdx.y = pair): slot 0 holds
// the grid's top edge (v_in[c], or the ids m+c) under tag 0 for band 0,
// slot 1 holds a tag no band waits for.  A pair with no band (n == 0) gets
// its h_out here.  Block (0,0) clears the ticket and abort words, after
// folding the previous launch's abort flag into `sticky` (the context's
// status word, read and cleared by the host).  A kernel, not
// hipMemsetAsync, so the launch sequence can live inside a hipGraph.
__device__ __forceinline__ void prep_pair(const PairDesc &P, unsigned *ctrl, unsigned *sticky)
{
    // 64-bit indices: a grid-stride step past a size near 2^31 must not wrap
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < P.n; c += stride) {
        const uint32_t v0 = P.v_in ? (uint32_t)P.v_in[c] : (uint32_t)(P.m + c);
        P.E[c] = (unsigned long long)v0;                       // tag 0
        P.E[(size_t)P.n + c] = 0xffffffff00000000ull;          // no band has this tag
    }
    if (P.nbands == 0)
        for (long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x; r < P.m; r += stride)
            P.h_out[r] = P.h_in ? P.h_in[r] : (int32_t)r;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        if (sticky && ctrl[1]) *sticky = 1u;
        ctrl[0] = 0u;
        ctrl[1] = 0u;
    }
}

__global__ void comb_prep_kernel(const PairDesc *pairs, unsigned *ctrl, unsigned *sticky)
{
    prep_pair(pairs[blockIdx.y], ctrl, sticky);
}

// The tiles of a grid (blockIdx.y = tile): rings, control words and, from the
// first tile row, the byte copies of the strips.  The flags word is zero here:
// the extract kernel of the launch before left it so.
__global__ void comb_prep_grid_kernel(TileGrid T, unsigned *ctrl, unsigned *sticky)
{
    const PairDesc P = tile_pair(T, (int)blockIdx.y);
    prep_pair(P, ctrl, sticky);
    if (P.sym8 && (int)blockIdx.y < T.GC)
        stage_sym8(P.b, P.n, (uint32_t *)P.sym8, P.sym8_stride, T.sym8_flags);
}

// Seeds the rings of the packed chain (blockIdx.y = couple): column c of
// slot 0 carries both pairs' top-edge strands m + c (0xffff past a pair's
// n) under tag 0, slot 1 a tag no band waits for.  Block (0,0) clears the
// ticket and abort words after folding the abort flag into `sticky`.
__global__ void comb_prep16_kernel(const CoupleDesc *couples, unsigned *ctrl, unsigned *sticky)
{
    const CoupleDesc D = couples[blockIdx.y];
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < D.n; c += stride) {
        uint32_t v0 = 0;
        for (int q = 0; q < 2; ++q) v0 |= (c < D.n_[q] ? (uint32_t)(D.m_[q] + c) : 0xffffu) << (16 * q);
        D.E[c] = (unsigned long long)v0;                       // tag 0
        D.E[(size_t)D.n + c] = 0xffffffff00000000ull;          // no band has this tag
    }
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        if (sticky && ctrl[1]) *sticky = 1u;
        ctrl[0] = 0u;
        ctrl[1] = 0u;
    }
}

// Both pairs' v_out from the last band's slot (blockIdx.y = couple).
__global__ void comb_extract16_kernel(const CoupleDesc *couples)
{
    const CoupleDesc D = couples[blockIdx.y];
    const unsigned long long *slot = D.E + (size_t)(D.nbands & 1) * (size_t)D.n;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < D.n; c += stride) {
        const uint32_t w = (uint32_t)slot[c];
        for (int q = 0; q < 2; ++q)
            if (c < D.n_[q]) D.v_out[q][c] = (int32_t)((w >> (16 * q)) & 0xffffu);
    }
}

// Clears n words (a kernel, so the launch sequence can be captured).
__global__ void lcsk_zero_kernel(int32_t *x, int32_t n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = 0;
}

// Range check of the packed chain's symbols (blockIdx.y = string): bit 0 of
// bad[item] for a symbol outside [0, 0xfffd], bit 1 for one above 15 (the
// one-hot cells need every symbol in [0, 15]).
__global__ void check16_kernel(const SymbolRange *ranges, int32_t *bad)
{
    const SymbolRange R = ranges[blockIdx.y];
    bool out = false, wide = false;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < R.len;
         i += (long long)gridDim.x * blockDim.x) {
        const uint32_t x = (uint32_t)R.x[i];
        out = out || x > 0xfffdu;
        wide = wide || x > 15u;
    }
    const int flags = (__builtin_amdgcn_ballot_w64(out) != 0 ? 1 : 0) | (__builtin_amdgcn_ballot_w64(wide) != 0 ? 2 : 0);
    if (flags && (threadIdx.x & 63) == 0) atomicOr(&bad[R.item], flags);
}

// v_out = the strands the last band left in its slot (blockIdx.y = pair).
__device__ __forceinline__ void extract_pair(const PairDesc &P)
{
    const unsigned long long *slot = P.E + (size_t)(P.nbands & 1) * (size_t)P.n;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < P.n; c += stride) {
        const uint32_t id = (uint32_t)slot[c];
        if (P.v_out) P.v_out[c] = (int32_t)id;
        if (P.perm && id < (uint32_t)(P.m + P.n)) P.perm[id] = (int32_t)c;   // always, after a completed comb
    }
}
__global__ void comb_extract_kernel(const PairDesc *pairs) { extract_pair(pairs[blockIdx.y]); }
__global__ void comb_extract_grid_kernel(TileGrid T, const unsigned *abort_flag)
{
    extract_pair(tile_pair(T, (int)blockIdx.y));
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        if (T.sym8_flags) *T.sym8_flags = 0;
        if (T.status) *T.status = (int32_t)*abort_flag;
    }
}

// row_to_col of each pair's permutation (blockIdx.y = pair): the strand that
// leaves row l on the right goes to column n+l, the one leaving column j at
// the bottom to column j (permutation_matrix.hpp:88-115).
__global__ void from_strands_kernel(const PairDesc *pairs, int32_t *perm, const int64_t *perm_off)
{
    const PairDesc P = pairs[blockIdx.y];
    int32_t *r2c = perm + perm_off[blockIdx.y];
    const long long stride = (long long)gridDim.x * blockDim.x;
    const uint32_t size = (uint32_t)(P.m + P.n);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < (long long)size; i += stride) {
        // ids are always < m+n after a completed comb; the test keeps an
        // aborted one (whose strands are undefined) from writing out of range
        const uint32_t id = (uint32_t)(i < P.m ? P.h_out[i] : P.v_out[i - P.m]);
        if (id < size) r2c[id] = (int32_t)(i < P.m ? P.n + i : i - P.m);
    }
}

// h_out, v_out of a permutation: the strand that ends in column c < n leaves
// column c at the bottom, in column n + l row l on the right.
__global__ void strands_from_perm_kernel(const int32_t *r2c, int32_t m, int32_t n, int32_t *h_out, int32_t *v_out,
                                         int32_t *copy)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)m + n) return;
    const uint32_t c = (uint32_t)r2c[i];
    if (copy) copy[i] = (int32_t)c;
    if (c < (uint32_t)n) v_out[c] = (int32_t)i;
    else if (c < (uint32_t)(m + n)) h_out[c - (uint32_t)n] = (int32_t)i;
}

__global__ void copy_kernel(int32_t *dst, const int32_t *src, long long count)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) dst[i] = src[i];
}

// Identity strands for empty grids (m == 0 or n == 0).
__global__ void comb_identity_kernel(int32_t *h_out, int32_t m, int32_t *v_out, int32_t n, int32_t *perm)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) h_out[i] = (int32_t)i;
    if (i < n) v_out[i] = (int32_t)(m + i);
    if (perm && i < (long long)m + n) perm[i] = (int32_t)(i < m ? n + i : i - m);
}

}  // namespace lcsk

using namespace lcsk;

// Steps per chunk.  32 for both forms: against 16, half the per-chunk
// publish, prefetch and tag-check work outweighs the longer band-to-band lag
// (m=n=2^20 at TM=16: the register chain 143.9 against 145.6 ms, the LDS
// groups 154.7 against 166.0 ms; 8 and 64 steps are slower in both).
constexpr int kChainChunk = 32;

template <int TM>
static int launch_chain_tm(const ChainArgs &args, int grid_blocks, int block_threads, hipStream_t stream)
{
    if (args.group_w == 1) {
        comb_chain_kernel<TM, kChainChunk><<<dim3(grid_blocks), dim3(block_threads), 0, stream>>>(args);
        return 0;
    }
    if (args.group_w == kGroupW && block_threads == kGroupW * kWave) {
        comb_group_kernel<TM, kChainChunk><<<dim3(grid_blocks), dim3(block_threads), 0, stream>>>(args);
        return 0;
    }
    return -22;
}

static int launch_bands(const ChainArgs &args, int tile_m, int grid_blocks, int block_threads, hipStream_t stream)
{
    switch (tile_m) {
    case 1: return launch_chain_tm<1>(args, grid_blocks, block_threads, stream);
    case 2: return launch_chain_tm<2>(args, grid_blocks, block_threads, stream);
    case 4: return launch_chain_tm<4>(args, grid_blocks, block_threads, stream);
    case 8: return launch_chain_tm<8>(args, grid_blocks, block_threads, stream);
    case 16: return launch_chain_tm<16>(args, grid_blocks, block_threads, stream);
    case 32: return launch_chain_tm<32>(args, grid_blocks, block_threads, stream);
    default: return -22;
    }
}

int lcsk_launch_grid(const ChainArgs &args, int grid_blocks, int block_threads, hipStream_t stream)
{
    const TileGrid &T = args.grid;
    const unsigned tiles = (unsigned)(T.GR * T.GC);
    if (tiles < 1 || tiles > 65535 || args.ntasks <= 0) return -22;
    // one thread per ring column (and per word of the byte copies)
    const unsigned fill = (unsigned)std::min<long long>(1024, ((long long)T.W + 255) / 256);
    hipLaunchKernelGGL(comb_prep_grid_kernel, dim3(fill, tiles), dim3(256), 0, stream, T, args.ticket, args.sticky);
    const int rc = launch_bands(args, T.pair.tile_m, grid_blocks, block_threads, stream);
    if (rc) return rc;
    hipLaunchKernelGGL(comb_extract_grid_kernel, dim3(fill, tiles), dim3(256), 0, stream, T, args.abort_flag);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

int lcsk_launch_chain(const ChainArgs &args, const PairDesc *d_pairs, int npairs, int max_n, int tile_m,
                      int grid_blocks, int block_threads, hipStream_t stream)
{
    if (npairs <= 0) return 0;
    const int fill_blocks = (int)std::min<long long>(1024, std::max<long long>(1, ((long long)max_n + 255) / 256));
    hipLaunchKernelGGL(comb_prep_kernel, dim3(fill_blocks, npairs), dim3(256), 0, stream, d_pairs, args.ticket,
                       args.sticky);
    if (args.ntasks > 0) {
        const int rc = launch_bands(args, tile_m, grid_blocks, block_threads, stream);
        if (rc) return rc;
    }
    hipLaunchKernelGGL(comb_extract_kernel, dim3(fill_blocks, npairs), dim3(256), 0, stream, d_pairs);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

int lcsk_launch_sym8(const int32_t *b, int32_t n, uint32_t *out, int32_t stride, int32_t *flags, hipStream_t stream)
{
    if (n <= 0 || stride < lcsk_sym8_stride(n)) return -22;
    hipLaunchKernelGGL(lcsk_zero_kernel, dim3(1), dim3(64), 0, stream, flags, 1);
    const unsigned blocks = (unsigned)std::min<long long>((4LL * stride + 255) / 256, 8192);
    hipLaunchKernelGGL(comb_sym8_kernel, dim3(blocks), dim3(256), 0, stream, b, n, out, stride, flags);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

int lcsk_launch_check16(const SymbolRange *d_ranges, int32_t nranges, int32_t *d_bad, int32_t nitems,
                        hipStream_t stream)
{
    if (nranges <= 0) return 0;
    hipLaunchKernelGGL(lcsk_zero_kernel, dim3((unsigned)((nitems + 255) / 256)), dim3(256), 0, stream, d_bad, nitems);
    for (int32_t base = 0; base < nranges; base += 65535) {   // grid y is at most 65535
        const int32_t cnt = std::min<int32_t>(65535, nranges - base);
        hipLaunchKernelGGL(check16_kernel, dim3(4, (unsigned)cnt), dim3(256), 0, stream, d_ranges + base, d_bad);
    }
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

int lcsk_launch_chain16(const ChainArgs &args, const CoupleDesc *d_couples, int ncouples, int max_n, int tile_m,
                        int grid_blocks, int block_threads, hipStream_t stream)
{
    if (ncouples <= 0) return 0;
    const int fill_blocks = (int)std::min<long long>(1024, std::max<long long>(1, ((long long)max_n + 255) / 256));
    hipLaunchKernelGGL(comb_prep16_kernel, dim3(fill_blocks, ncouples), dim3(256), 0, stream, d_couples, args.ticket,
                       args.sticky);
    if (args.ntasks > 0) {
        const dim3 grid(grid_blocks), block(block_threads);
        switch (tile_m) {
        case 1: comb_chain16_kernel<1, kChainChunk><<<grid, block, 0, stream>>>(args); break;
        case 2: comb_chain16_kernel<2, kChainChunk><<<grid, block, 0, stream>>>(args); break;
        case 4: comb_chain16_kernel<4, kChainChunk><<<grid, block, 0, stream>>>(args); break;
        case 8: comb_chain16_kernel<8, kChainChunk><<<grid, block, 0, stream>>>(args); break;
        case 16: comb_chain16_kernel<16, kChainChunk><<<grid, block, 0, stream>>>(args); break;
        case 32: comb_chain16_kernel<32, kChainChunk><<<grid, block, 0, stream>>>(args); break;
        default: return -22;
        }
    }
    hipLaunchKernelGGL(comb_extract16_kernel, dim3(fill_blocks, ncouples), dim3(256), 0, stream, d_couples);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

int lcsk_launch_from_strands(const PairDesc *d_pairs, int npairs, int max_len, int32_t *perm,
                             const int64_t *d_perm_off, hipStream_t stream)
{
    if (npairs <= 0) return 0;
    const int blocks = (int)std::min<long long>(1024, std::max<long long>(1, ((long long)max_len + 255) / 256));
    hipLaunchKernelGGL(from_strands_kernel, dim3(blocks, npairs), dim3(256), 0, stream, d_pairs, perm, d_perm_off);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

int lcsk_launch_strands_from_perm(const int32_t *r2c, int32_t m, int32_t n, int32_t *h_out, int32_t *v_out,
                                  int32_t *copy, hipStream_t stream)
{
    const long long size = (long long)m + n;
    if (size == 0) return 0;
    hipLaunchKernelGGL(strands_from_perm_kernel, dim3((unsigned)((size + 255) / 256)), dim3(256), 0, stream, r2c, m, n,
                       h_out, v_out, copy);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

int lcsk_launch_copy(int32_t *dst, const int32_t *src, long long count, hipStream_t stream)
{
    if (count <= 0) return 0;
    const int blocks = (int)std::min<long long>(1024, (count + 255) / 256);
    hipLaunchKernelGGL(copy_kernel, dim3(blocks), dim3(256), 0, stream, dst, src, count);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}

int lcsk_launch_identity(int32_t *h_out, int32_t m, int32_t *v_out, int32_t n, hipStream_t stream, int32_t *perm)
{
    const long long mx = m > n ? m : n;
    if (mx == 0) return 0;
    hipLaunchKernelGGL(comb_identity_kernel, dim3((unsigned)((mx + 255) / 256)), dim3(256), 0, stream, h_out, m, v_out,
                       n, perm);
    return hipGetLastError() == hipSuccess ? 0 : -5;
}
