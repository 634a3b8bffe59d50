"""CPU emulation of the whole-GPU steady ant's index arithmetic
(platform-independent-lcs_amd/csrc/braid_kernels.hip, the "big cores" kernels:
big_split_count/scatter, the leaves' big_lift, big_hist_kernel, and
big_box_kernel with its line search, row rule, 64 x 64 steps of wider boxes
and lift into the parents), step for step in Python, checked against the
oracle's steady ant (orc_steady_ant, braid_multiplication.hpp:204-270).  The
leaves (one workgroup each on the GPU) are taken from the oracle here; the GPU
tests check the leaf kernel itself.  Small line, wave and block constants make
small cores exercise what only large cores meet on the GPU: several histogram
blocks per node, blocks of 512 entries, boxes wider than a wave."""
import numpy as np
import pytest

import oracle

LO = 1 << 31


def counted31(e, r):
    """counted<31>: bit 31 of e - r (numbers or arrays)."""
    return ((e - r) & 0xFFFFFFFF) >> 31


def w_log(e):
    wl = 1 + (e + 1) // 2
    return min(max(wl, 9), 13)


def depth(L, d, box_g, max_lines, w_fixed):
    s = 1 << (L - d)
    nb = min(s // box_g, max_lines)
    glog = (s // nb).bit_length() - 1
    w = min(s, w_fixed if w_fixed else 1 << w_log(L - d))
    return s, nb, glog, w, s // w


def partition(key, s, bit, cnt, tile=2048, next_bit=None):
    """big_split_scatter_kernel: stable partition of every segment of size s
    by `bit`, zeros first; par[pos] = old position.  cnt holds this depth's
    ones per tile; a block sums its segment's tiles itself.  With next_bit,
    it also returns the next depth's tile counts as the scatter accumulates
    them: each block counts the next bit of the keys it places per
    destination tile, its zeros and its ones each running into at most two
    tiles from their first destinations."""
    K = key.size
    new = np.empty_like(key)
    par = np.empty(K, np.int64)
    nxt = np.zeros(K // tile, np.int64)
    for blk in range(K // tile):
        seg = (blk * tile) & ~(s - 1)
        t0, nt = seg // tile, s // tile
        before_tiles = int(sum(cnt[t0:t0 + (blk - t0)]))
        ones_total = int(sum(cnt[t0:t0 + nt]))
        zeros_total = s - ones_total
        z0, o0 = blk * tile - before_tiles, seg + zeros_total + before_tiles
        zt, ot = z0 // tile, o0 // tile
        runs = {("z", 0): 0, ("z", 1): 0, ("o", 0): 0, ("o", 1): 0}
        before = before_tiles
        for x in range(blk * tile, (blk + 1) * tile):
            b = (int(key[x]) >> bit) & 1
            pos = seg + zeros_total + before if b else seg + (x - seg - before)
            before += b
            new[pos] = key[x]
            par[pos] = x
            if next_bit is not None and (int(key[x]) >> next_bit) & 1:
                idx = pos // tile - (ot if b else zt)
                assert idx in (0, 1)
                runs[("o" if b else "z", idx)] += 1
        if next_bit is not None:
            for (kind, idx), v in runs.items():
                if v:
                    nxt[(ot if kind == "o" else zt) + idx] += v
    return new, par, nxt


def tile_counts(key, bit, tile=2048):
    """big_split_count_kernel (depth 0): ones of `bit` per tile."""
    return np.array([int(((key[b * tile:(b + 1) * tile] >> bit) & 1).sum()) for b in range(key.size // tile)])


def block_search(Hj, Ht, nsegs, Yj):
    """Rounds of 64 blocks: the first block where Z + its own count of z_j
    entries reaches Y_j (the lanes' inclusive scan plus a carry)."""
    Z = 0
    for g0 in range(0, nsegs, 64):
        cs = []
        for g in range(g0, min(g0 + 64, nsegs)):
            P, T = Hj[g], Ht[g]
            cs.append((P & 0xFFFF) + (T >> 16) - (P >> 16))
        incl = np.cumsum(cs)
        hit = np.nonzero(Z + incl >= Yj)[0]
        if hit.size:
            l = int(hit[0])
            return g0 + l, Z + int(incl[l] - cs[l])
        Z += int(incl[-1])
    return nsegs - 1, Z


def select(counts, need):
    """Position of the need-th counted column of a row (select64), need >= 1."""
    return int(np.nonzero(np.cumsum(counts) == need)[0][0])


def box_rows(u, CI, r_lo, rho, cs, ce, col, wave):
    """The rows of a box of one wave that this piece decides, as (row, column)."""
    r = r_lo + np.arange(wave)
    m = counted31(u, cs)
    if col:
        m = m & (r < rho)
    need = int(col) + np.cumsum(m[::-1])[::-1]
    assert ce - cs <= wave
    out = []
    for i in range(wave):
        c = counted31(CI[cs:ce], int(r[i]))
        if (col and r[i] > rho) or need[i] > c.sum():
            continue
        T = cs + 1 + select(c, need[i]) if need[i] else cs
        out.append((int(r[i]), T - 1 if T > 0 and counted31(int(u[i]), T) else int(u[i]) & (LO - 1)))
    return out


def wide_box_rows(U, CI, r_lo, rho, cs, ce, col, wave):
    """The same in a box wider than a wave: `wave` rows at a time from rho
    upwards, the rows counted so far carried in `below`; `wave` columns at a
    time, the columns still needed carried in `need`."""
    out, below = [], int(col)
    for rb in range(rho & ~(wave - 1), r_lo - 1, -wave):
        r = rb + np.arange(wave)
        u = U[rb:rb + wave]
        m = counted31(u, cs)
        if col:
            m = m & (r < rho)
        need = below + np.cumsum(m[::-1])[::-1]
        below += int(m.sum())
        T = np.where(need > 0, -1, cs)
        for c0 in range(cs, ce, wave):
            e = np.full(wave, LO - 1, np.int64)   # past ce: counted at no line
            e[:min(wave, ce - c0)] = CI[c0:min(c0 + wave, ce)]
            for i in range(wave):
                c = counted31(e, int(r[i]))
                if T[i] < 0 and need[i] <= c.sum():
                    T[i] = c0 + 1 + select(c, need[i])
                need[i] -= c.sum()
        for i in range(wave):
            if (not col or r[i] <= rho) and T[i] >= 0:
                t = int(T[i])
                out.append((int(r[i]), t - 1 if t > 0 and counted31(int(u[i]), t) else int(u[i]) & (LO - 1)))
    return out


def emulate(P, Q, k, L, L0, box_g=64, max_lines=8192, w_fixed=None):
    """box_g: rows and columns of a wave (64 on the GPU)."""
    K = 1 << L
    d0 = L - L0
    keyP = np.array([P[x] if x < k else x for x in range(K)], np.int64)
    keyQ = np.arange(K, dtype=np.int64)
    for r in range(k):
        keyQ[Q[r]] = r
    parP, parQ = [], []
    cP, cQ = tile_counts(keyP, L - 1), tile_counts(keyQ, L - 1)
    for d in range(d0):
        nb = L - d - 2 if d + 1 < d0 else None
        keyP, pp, nP = partition(keyP, K >> d, L - d - 1, cP, next_bit=nb)
        keyQ, pq, nQ = partition(keyQ, K >> d, L - d - 1, cQ, next_bit=nb)
        if nb is not None:
            # the accumulated counts are the next depth's tile counts
            assert np.array_equal(nP, tile_counts(keyP, nb)) and np.array_equal(nQ, tile_counts(keyQ, nb))
            cP, cQ = nP, nQ
        parP.append(pp)
        parQ.append(pq)
    # U and CI alternate between two sets: a depth's boxes read one and lift
    # into the other
    U2, CI2 = [np.full(K, -1, np.int64) for _ in range(2)], [np.full(K, -1, np.int64) for _ in range(2)]

    def lift(d, v0, h, x, c):
        p_pos, q_pos = int(parP[d][x]), int(parQ[d][v0 + (c & (h - 1))])
        p0 = p_pos & ~(2 * h - 1)
        lo = 0 if x & h else LO
        U2[d & 1][p_pos] = (q_pos - p0) | lo
        CI2[d & 1][q_pos] = (p_pos - p0) | lo

    s0 = 1 << L0
    R = np.full(K, -1, np.int64)
    for v in range(K >> L0):
        kp = keyP[v * s0:(v + 1) * s0] & (s0 - 1)
        kq = keyQ[v * s0:(v + 1) * s0] & (s0 - 1)   # column -> shared row
        qr2c = np.empty(s0, np.int32)
        qr2c[kq] = np.arange(s0)
        for x, c in enumerate(oracle.steady_ant(kp.astype(np.int32), qr2c)):
            lift(d0 - 1, v * s0, s0, v * s0 + x, int(c))
    for d in range(d0 - 1, -1, -1):
        s, nb, glog, w, nsegs = depth(L, d, box_g, max_lines, w_fixed)
        g = 1 << glog
        nodes = K // s
        U, CI = U2[d & 1], CI2[d & 1]
        assert (U >= 0).all() and (CI >= 0).all()
        U2[1 - (d & 1)][:] = CI2[1 - (d & 1)][:] = -1   # what a depth reads was written for it
        # big_hist_kernel: per (y, node) an nb x nsegs prefix matrix, then totals
        H = {}
        for y, E in ((0, CI), (1, U)):
            for node in range(nodes):
                M = np.zeros((nb + 1, nsegs), np.int64)
                for gg in range(nsegs):
                    hh = np.zeros(nb, np.int64)
                    for i in range(w):
                        e = int(E[node * s + gg * w + i])
                        bk = (s - 1 - (e & 0x7FFFFFFF)) >> glog
                        hh[bk] += 1 if (e & LO) else 0x10000
                    M[:nb, gg] = np.concatenate([[0], np.cumsum(hh)[:-1]])
                    M[nb, gg] = hh.sum()
                H[(y, node)] = M
        # big_line: block_search + sweep_block
        T = {}
        for y, E in ((0, CI), (1, U)):
            for node in range(nodes):
                M = H[(y, node)]
                for j in range(nb):
                    Yj = int(sum(int(v) & 0xFFFF for v in M[j])) if j else 0
                    if Yj == 0:
                        T[(y, node, j)] = 0
                        continue
                    seg, Z = block_search(M[j], M[nb], nsegs, Yj)
                    need = Yj - Z
                    base = node * s + seg * w
                    for r in range(w):
                        e = int(E[base + r])
                        bk = (s - 1 - (e & 0x7FFFFFFF)) >> glog
                        if ((bk < j) if (e & LO) else (bk >= j)):
                            need -= 1
                            if need == 0:
                                T[(y, node, j)] = seg * w + r + 1
                                break
                    assert need == 0
        # big_box_kernel: one wave per piece (row lines, then column lines)
        seen = np.zeros(K, int)
        for t in range(2 * nodes * nb):
            col = t >= nodes * nb
            node, j = divmod(t - nodes * nb if col else t, nb)
            T0 = T[(int(col), node, j)] if j else 0
            if col and (j == 0 or T0 == 0):
                continue
            if col:
                rho, cs = T0 - 1, (nb - j) * g
                r_lo, ce = rho & ~(g - 1), cs + g
            else:
                r_lo, cs = s - (j + 1) * g, T0
                rho, ce = r_lo + g - 1, g if cs == 0 else (((cs - 1) >> glog) + 1) << glog
            v0 = node * s
            Un, CIn = U[v0:v0 + s], CI[v0:v0 + s]
            rows = (box_rows(Un[r_lo:r_lo + g], CIn, r_lo, rho, cs, ce, col, box_g) if g == box_g
                    else wide_box_rows(Un, CIn, r_lo, rho, cs, ce, col, box_g))
            for r, c in rows:
                seen[v0 + r] += 1
                if d:
                    lift(d - 1, v0, s, v0 + r, c)
                else:
                    R[r] = c
        assert (seen == 1).all()   # every row lies in exactly one piece's box
    return R[:k].astype(np.int32)


CASES = [
    # (k, L, L0, box side, max lines, fixed block width)
    (4096, 12, 10, 64, 8192, None),     # the library's constants: one block per node
    (4000, 12, 11, 64, 8192, None),     # padded core, leaves of 2^11
    (6000, 13, 11, 32, 8192, None),     # waves of 32
    (4096, 12, 10, 64, 16, 512),        # wide boxes (g = 256 at the top) and 8 blocks per node
    (4000, 12, 10, 32, 16, 512),        # boxes of 4 and 8 waves a side
    (8192, 13, 10, 16, 8192, 512),      # waves of 16, 16 blocks per node
    (16384, 14, 10, 32, 8192, None),    # four device-wide depths, 8 partition tiles per segment
]


@pytest.mark.parametrize("k,L,L0,box_g,max_lines,w", CASES)
def test_big_core_random(k, L, L0, box_g, max_lines, w):
    rng = np.random.default_rng(k + L0 + box_g)
    P = rng.permutation(k).astype(np.int32)
    Q = rng.permutation(k).astype(np.int32)
    assert np.array_equal(emulate(P, Q, k, L, L0, box_g, max_lines, w), oracle.steady_ant(P, Q))


def test_big_core_structured():
    """Identity, reversal, a shift and few swaps: paths hugging the box edges."""
    k = 4096
    rng = np.random.default_rng(1)
    ident = np.arange(k, dtype=np.int32)
    rev = ident[::-1].copy()
    shift = np.roll(ident, 123).astype(np.int32)
    near = ident.copy()
    for _ in range(50):
        i, j = rng.integers(0, k, 2)
        near[i], near[j] = near[j], near[i]
    for P, Q in ((ident, rev), (rev, rev), (shift, near), (rev, ident)):
        for box_g, max_lines, w in ((64, 8192, None), (64, 16, 512)):
            assert np.array_equal(emulate(P, Q, k, 12, 10, box_g, max_lines, w), oracle.steady_ant(P, Q))


def test_block_width_bounds():
    """Blocks are 512 .. 8192 entries, at most 1024 per node up to 2^22 points
    (what big_line's block search holds in registers)."""
    for e in range(11, 23):
        w = min(1 << e, 1 << w_log(e))
        assert 512 <= w <= 8192 and (1 << e) // w <= 1024
