"""Index arithmetic of the band chains' byte symbols, checked on the CPU.

Each strip of b (a tile column of a cut pair, or all of b) has four copies of
its own: stage_sym8 writes at byte x of copy j the symbol of the strip's
column x + j - 128, and 255 outside the strip's [0, n).  Lane L of a band
reads, for the chunk starting at step t, C/4 = 8 words of copy j = x0 % 4 from
word (x0 - j) / 4 + t / 4, x0 = 128 - L, and takes byte s % 4 of word s / 4 as
the symbol of step t + s.  This restates those formulas (comb_kernels.hip:
stage_sym8 and band_pass) and checks for every lane, every chunk up to the
last prefetch, several cuts and widths that each read stays inside its copy,
that each byte a combing lane uses is the symbol of the column it combs and
that a lane outside [0, n) holds 255, also where a neighbouring strip has
symbols there: the unmasked first and last chunks of a band rest on that.  It
runs no GPU code; the GPU parity tests compare the kernels themselves with the
oracle.
"""
import numpy as np
import pytest

PAD, C, WAVE = 128, 32, 64


def stride_words(n):
    return ((n + 2 * PAD + 15) // 16) * 4


def copies(strip):
    n = len(strip)
    st = stride_words(n)
    out = np.full((4, st * 4), 255, np.uint8)
    for j in range(4):
        x = np.arange(st * 4)
        c = x + j - PAD
        ok = (c >= 0) & (c < n)
        out[j, ok] = (strip[c[ok]] & 0xFF).astype(np.uint8)
    return out, st


@pytest.mark.parametrize("n,strips", [(1, 1), (63, 1), (64, 1), (97, 1), (1000, 1), (5003, 2), (5003, 3),
                                      (5003, 7), (4096, 4), (777, 5)])
def test_lane_windows_stay_inside_and_pick_their_columns(n, strips):
    rng = np.random.default_rng(n * 10 + strips)
    b = rng.integers(0, 255, n).astype(np.int64)   # 255 only as padding
    W = (n + strips - 1) // strips
    lanes = np.arange(WAVE)
    x0 = PAD - lanes
    j = x0 & 3
    word0 = (x0 - j) // 4
    for s0 in range(0, n, W):
        ns = min(W, n - s0)
        cp, st = copies(b[s0:s0 + ns])
        assert st * 4 >= ns + 2 * PAD and st % 4 == 0 and st <= stride_words(W)
        nchunks = (ns + WAVE + C - 1) // C
        for k in range(nchunks + 1):        # the last chunk prefetches chunk nchunks
            t = k * C
            first = word0 + t // 4
            last = first + C // 4 - 1
            assert (first >= 0).all() and (last < st).all(), (n, strips, s0, k)
            for L in range(WAVE):
                words = cp[j[L], 4 * first[L]: 4 * (last[L] + 1)]
                col = t + np.arange(C) - L
                inside = (col >= 0) & (col < ns)
                want = np.where(inside, b[s0 + np.clip(col, 0, ns - 1)], 255)
                assert np.array_equal(words, want), (n, strips, s0, k, L)


def test_copies_are_padded_outside_the_string():
    b = np.arange(1, 11, dtype=np.int64)
    cp, st = copies(b)
    for j in range(4):
        held = np.nonzero(cp[j] != 255)[0]
        assert held.min() == PAD - j and held.max() == PAD - j + 9 and held.size == 10
