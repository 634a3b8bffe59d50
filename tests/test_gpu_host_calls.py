"""Host calls: the staging limit of their copies, and device memory that is
kept between calls against the budget, bit for bit against the oracle."""
import numpy as np
import pytest

import lcs_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with lcs_amd.Context(0) as c:
        yield c


def wide(m, n):
    return lcs_amd.gen_uniform(1, m, 4), lcs_amd.gen_uniform(2, n, 4)


# strings and results together: the last size that is staged (4 MiB of words:
# 16 + n in, 16 + 8 + n or, with row_to_col, 16 + 2 * (8 + n) out) and the next
@pytest.mark.parametrize("n", [524268, 524269])
def test_strands_at_the_staging_limit(ctx, n):
    a, b = wide(8, n)
    h, v, score = ctx.comb(a, b)
    ho, vo = oracle.comb(a, b, order="mt")
    assert np.array_equal(h, ho) and np.array_equal(v, vo) and score == int((vo < 8).sum())


@pytest.mark.parametrize("m,n", [(0, 0), (0, 5), (5, 0), (1, 1), (17, 3), (8, 349509), (8, 349510)])
def test_permutation_at_the_staging_limit(ctx, m, n):
    a, b = wide(m, n)
    r2c, c2r, score = ctx.comb_permutation(a, b)
    ho, vo = oracle.comb(a, b, order="mt")
    ro, co = oracle.from_strands(ho, vo)
    assert np.array_equal(r2c, ro) and np.array_equal(c2r, co) and score == int((vo < m).sum())


@pytest.mark.parametrize("size", [262144, 262145])   # 4 * size - 1 words; the next size is over the limit
def test_product_at_the_staging_limit(ctx, size):
    rng = np.random.default_rng(size)
    p, q = (rng.permutation(size).astype(np.int32) for _ in range(2))
    for glue in (False, True):
        assert np.array_equal(ctx.braid_multiply(p, q, 1, glue), oracle.staggered_multiply(p, q, 1, glue))


def test_results_outlive_the_next_call(ctx):
    a, b = wide(300, 400)
    first = ctx.comb(a, b)
    ctx.comb(b, a)
    ho, vo = oracle.comb(a, b)
    assert np.array_equal(first[0], ho) and np.array_equal(first[1], vo)


def test_kept_memory_gives_way_to_the_budget():
    a, b = wide(300, 20000)
    with lcs_amd.Context(0) as c:
        c.comb(a, b)
        budget = c.memory()[0]
    p = np.random.default_rng(3).permutation(2000).astype(np.int32)
    with lcs_amd.Context(0, hbm_budget=budget) as c:
        for _ in range(2):
            assert np.array_equal(c.braid_multiply(p, p, 1000, True), oracle.staggered_multiply(p, p, 1000, True))
            idx = lcs_amd.DominanceIndex(c, p)
            assert idx.query(2000, 0, lcs_amd.SEMI_DOMINANCE, [5], [7])[0] == int((p[5:] < 7).sum())
            idx.close()
        assert c.memory()[0] > 0   # kept
        h, v, _ = c.comb(a, b)
        assert c.memory()[0] <= budget
    ho, vo = oracle.comb(a, b)
    assert np.array_equal(h, ho) and np.array_equal(v, vo)


def test_an_index_reuses_memory_of_a_larger_one(ctx):
    rng = np.random.default_rng(9)
    for size in (5000, 4200, 70, 5000, 9000):
        p = rng.permutation(size).astype(np.int32)
        r, c = rng.integers(0, size + 1, 50).astype(np.int32), rng.integers(0, size + 1, 50).astype(np.int32)
        idx = lcs_amd.DominanceIndex(ctx, p)
        got = idx.query(size, 0, lcs_amd.SEMI_DOMINANCE, r, c)
        idx.close()
        assert got.tolist() == [int((p[i:] < j).sum()) for i, j in zip(r, c)]


def test_an_index_may_outlive_its_context():
    c = lcs_amd.Context(0)
    idx = lcs_amd.DominanceIndex(c, np.arange(100, dtype=np.int32))
    c.close()
    idx.close()
