"""The unmasked first and last chunks of a band on the GPU: lanes outside the
grid carry a pad symbol, so a pair whose symbols come near the pad values (255
for byte symbols, -1 and below for 32-bit ones, the top of 16 bits for packed
couples) must still give the oracle's strands, at widths around the 32-step
chunk and the 64-lane skew.  Whole numbers: compared exactly."""
import numpy as np
import pytest

import lcs_amd
import oracle

pytestmark = pytest.mark.gpu

WIDTHS = [1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 161]
SYMBOLS = {
    "byte_255": [0, 1, 254, 255],        # b holds the byte copies' padding: masked steps
    "byte_254": [0, 1, 253, 254],        # a row may hold 255, b does not
    "minus": [-1, -2, -3, 0],            # the 32-bit path's first pad values are taken
    "int_min": [-(1 << 31), (1 << 31) - 1, 255, 256],
}


def pair(rng, m, n, symbols, extra_a=()):
    a = rng.choice(np.array(list(symbols) + list(extra_a), np.int64), m).astype(np.int32)
    b = rng.choice(np.array(symbols, np.int64), n).astype(np.int32)
    return a, b


@pytest.mark.parametrize("name", sorted(SYMBOLS))
@pytest.mark.parametrize("variant", [lcs_amd.VARIANT_CHAIN, lcs_amd.VARIANT_CHAIN_BYTES, lcs_amd.VARIANT_CHAIN_LDS])
def test_pad_symbols_never_match(name, variant):
    rng = np.random.default_rng(len(name))
    with lcs_amd.Context(0) as ctx:
        for tm in (1, 2, 4, 16):
            for n in WIDTHS:
                m = int(rng.integers(1, 64 * tm * 3))
                a, b = pair(rng, m, n, SYMBOLS[name], extra_a=(255,))
                h, v, _ = ctx.comb(a, b, lcs_amd.schedule(tm, 1, variant, 1))
                ho, vo = oracle.comb(a, b)
                assert np.array_equal(h, ho) and np.array_equal(v, vo), (name, variant, tm, m, n)


def test_pad_search_passes_a_full_band():
    # every value the search tries first is in the band: 64 rows hold -1 .. -64
    a = -np.arange(1, 65, dtype=np.int32)
    b = np.concatenate([a[::-1], a, [-65, -66]]).astype(np.int32)
    with lcs_amd.Context(0) as ctx:
        h, v, _ = ctx.comb(a, b, lcs_amd.schedule(1, 1, lcs_amd.VARIANT_CHAIN, 1))
    ho, vo = oracle.comb(a, b)
    assert np.array_equal(h, ho) and np.array_equal(v, vo)


@pytest.mark.parametrize("symbols", [[0, 15], [0, 16], [65532, 65533]])
def test_packed_couples_of_uneven_widths(symbols):
    rng = np.random.default_rng(symbols[1])
    a_list, b_list = [], []
    for n in WIDTHS:
        for other in (n, n + 1, 3 * n + 5):
            a, b = pair(rng, int(rng.integers(1, 600)), other, symbols)
            a_list.append(a)
            b_list.append(b)
    with lcs_amd.Context(0) as ctx:
        for tm in (1, 4, 8):
            scheds = [lcs_amd.schedule(tm, 1, lcs_amd.VARIANT_PACKED16, 1)] * len(a_list)
            h, v = ctx.batch_comb(a_list, b_list, scheds)
            for p in range(len(a_list)):
                ho, vo = oracle.comb(a_list[p], b_list[p])
                assert np.array_equal(h[p], ho) and np.array_equal(v[p], vo), (tm, p, a_list[p].size, b_list[p].size)


def test_strips_pad_their_own_edges():
    # byte copies are padded per strip: the columns left of a strip belong to
    # its neighbour and must not reach its first band's ramp
    rng = np.random.default_rng(3)
    a, b = rng.integers(0, 4, 500).astype(np.int32), rng.integers(0, 4, 1000).astype(np.int32)
    ho, vo = oracle.comb(a, b)
    with lcs_amd.Context(0) as ctx:
        for strips in (2, 3, 7):
            h, v, _ = ctx.comb(a, b, lcs_amd.schedule(2, 1, lcs_amd.VARIANT_CHAIN_BYTES, strips))
            assert np.array_equal(h, ho) and np.array_equal(v, vo), strips
