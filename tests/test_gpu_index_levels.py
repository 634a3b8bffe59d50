"""The dominance index where its layout changes: one and two bits in the last
level, edges of records, of a workgroup's rows, of superblocks (2^20 rows) and
of workgroups with several tiles (from 2^22 rows), against direct counts."""
import numpy as np
import pytest

import lcs_amd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with lcs_amd.Context(0) as c:
        yield c


@pytest.mark.parametrize("size", [1, 2, 3, 31, 32, 33, 63, 64, 65, 2047, 2048, 2049, 4095, 4096, (1 << 20) - 1, 1 << 20,
                                  (1 << 20) + 1, (1 << 21) + 5, (1 << 22) - 1, 1 << 22, (1 << 22) + 4097])
def test_index_matches_direct_counts(ctx, size):
    rng = np.random.default_rng(size)
    p = rng.permutation(size).astype(np.int32)
    p[rng.integers(0, size, size // 50)] = -1
    idx = lcs_amd.DominanceIndex(ctx, p)
    nq = 60
    r = rng.integers(0, size + 2, nq).astype(np.int32)
    c = rng.integers(-1, size + 2, nq).astype(np.int32)
    edges = np.array([0, 1, size - 1, size, size // 2], np.int32)
    r, c = np.concatenate([r, np.repeat(edges, 5)]), np.concatenate([c, np.tile(edges, 5)])
    got = idx.query(size, 0, lcs_amd.SEMI_DOMINANCE, r, c)
    idx.close()
    assert got.tolist() == [int((p[i:] < j).sum()) for i, j in zip(r, c)]


@pytest.mark.parametrize("shape", ["sorted", "reversed", "equal", "unset"])
def test_index_of_uneven_values(ctx, shape):
    size = 70001
    up = np.arange(size, dtype=np.int32)
    p = {"sorted": up, "reversed": up[::-1].copy(), "equal": np.full(size, 4097, np.int32),
         "unset": np.full(size, -1, np.int32)}[shape]
    idx = lcs_amd.DominanceIndex(ctx, p)
    r = np.arange(0, size, 997, dtype=np.int32)
    for j in (0, 1, 4097, 4098, 65536, size):
        got = idx.query(size, 0, lcs_amd.SEMI_DOMINANCE, r, np.full(r.size, j, np.int32))
        assert got.tolist() == [int((p[i:] < j).sum()) for i in r]
    idx.close()
