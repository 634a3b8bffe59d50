"""The bit-parallel LCS kernel at the edges of its table and block rules:
alphabets around the two-column table's largest (9), blocks of two columns
(tall pairs) and of four (wide ones), column counts around the 32-column word,
batches; against the oracle's word-parallel recurrence."""
import numpy as np
import pytest

import lcs_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma", [1, 8, 9, 10, 200])
def test_words_bands_and_blocks(sigma):
    rng = np.random.default_rng(sigma)
    with lcs_amd.Context(0) as ctx:
        # rows (bands of 2048) x columns either way round: few bands and many
        for m, n in ((2048, 31), (2049, 32), (4096, 33), (2047, 2048), (40000, 3000), (30001, 257), (9000, 64),
                     (6145, 6143), (12289, 40001)):
            a = rng.integers(0, sigma, m).astype(np.int32)
            b = rng.integers(0, sigma, n).astype(np.int32)
            want = oracle.llcs_bitpar(a, b)
            assert ctx.llcs(a, b, sigma) == want, (m, n)
            assert ctx.llcs(b, a, sigma) == want, (n, m)


def test_symbols_outside_the_alphabet_next_to_the_table_rows():
    with lcs_amd.Context(0) as ctx:
        a = np.zeros(3000, np.int32)
        for sigma in (9, 10):
            for bad in (sigma, -1, 255, 1 << 30):
                for where in (0, 1, 2999):
                    b = a.copy()
                    b[where] = bad
                    for x, y in ((a, b), (b, a)):
                        with pytest.raises(lcs_amd.LcsError):
                            ctx.llcs(x, y, sigma)
            assert ctx.llcs(a, a, sigma) == 3000


@pytest.mark.parametrize("sigma", [4, 9, 10, 200])
def test_a_budget_without_room_for_codes(sigma):
    # the bands then read the symbols themselves; edges of the 32-column chunk
    # and of the string, unaligned starts of a pair's columns, and bad symbols
    rng = np.random.default_rng(sigma)
    sizes = [(0, 5), (5, 0), (1, 1), (31, 33), (2047, 65), (4097, 64), (70, 2049), (3000, 3001)]
    A = [rng.integers(0, sigma, m).astype(np.int32) for m, _ in sizes]
    B = [rng.integers(0, sigma, n).astype(np.int32) for _, n in sizes]
    want = [oracle.llcs_bitpar(a, b) if a.size and b.size else 0 for a, b in zip(A, B)]
    with lcs_amd.Context(0) as free:
        assert free.llcs_batch(A, B, sigma).tolist() == want
        budget = free.memory()[0] - 1024   # short by a part of the codes
    with lcs_amd.Context(0, hbm_budget=budget) as ctx:
        assert ctx.llcs_batch(A, B, sigma).tolist() == want
        assert ctx.memory()[0] < budget   # none kept
        B[4][7] = sigma
        with pytest.raises(lcs_amd.LcsError):
            ctx.llcs_batch(A, B, sigma)


@pytest.mark.parametrize("sigma", [4, 5, 9, 10])
@pytest.mark.parametrize("shape", ["tall", "many"])
def test_batches(sigma, shape):
    # tall: few pairs whose bands outnumber their words of columns, blocks of
    # two; many: more bands than the chip holds at once (of tables of column
    # pairs, and of four to a CU), blocks of four and, for 5 to 9 symbols, one
    # column a table row.  Word edges and empty strings among them.
    rng = np.random.default_rng(sigma)
    edges = [0, 1, 31, 32, 33]
    if shape == "tall":
        sizes = [(40000, 40000), (30001, 33000)] + [(20000 + n, n) for n in edges]
    else:
        sizes = [(int(m), int(n)) for m, n in rng.integers(1, 3000, (1300, 2))] + [(2049, n) for n in edges]
    A = [rng.integers(0, sigma, m).astype(np.int32) for m, _ in sizes]
    B = [rng.integers(0, sigma, n).astype(np.int32) for _, n in sizes]
    want = [oracle.llcs_bitpar(a, b) if a.size and b.size else 0 for a, b in zip(A, B)]
    with lcs_amd.Context(0) as ctx:
        assert ctx.llcs_batch(A, B, sigma).tolist() == want
        assert ctx.llcs_batch(B, A, sigma).tolist() == want
        B[1][5] = sigma
        with pytest.raises(lcs_amd.LcsError):
            ctx.llcs_batch(A, B, sigma)
        B[1][5] = 0
        want[1] = oracle.llcs_bitpar(A[1], B[1])
        assert ctx.llcs_batch(A, B, sigma).tolist() == want   # the error does not stay
