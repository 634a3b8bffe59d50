"""Requests without a schedule: one tile height for a micro-batch, whatever
its mix of lengths, with requests that bring their own, against the oracle."""
import numpy as np
import pytest

import lcs_amd
import oracle

pytestmark = pytest.mark.gpu


# one short; many short; one band beside many; a batch that favours few rows
# per lane; empty strings
@pytest.mark.parametrize("shapes", [[(1, 1)], [(63, 900)] * 40, [(64, 20000), (5000, 300)], [(64, 60000), (6000, 6000)], [(20000, 30000)],
                                    [(65, 65), (513, 7), (30000, 4000), (4000, 30000), (0, 9), (9, 0), (0, 0)]])
@pytest.mark.parametrize("own", [0, 8])
def test_mixed_requests(shapes, own):
    with lcs_amd.Context(0) as c:
        srv = lcs_amd.Server(c, hbm_budget=64 << 20, max_inflight=2)
        pairs = [(lcs_amd.gen_uniform(2 * i, m, 4), lcs_amd.gen_uniform(2 * i + 1, n, 4)) for i, (m, n) in enumerate(shapes)]
        ids = [srv.submit(a, b, lcs_amd.schedule(own, 1, lcs_amd.VARIANT_CHAIN, 1) if own and i % 2 else None)
               for i, (a, b) in enumerate(pairs)]
        for rid, (a, b) in zip(ids, pairs):
            h, v = srv.wait(rid)
            ho, vo = oracle.comb(a, b, order="mt")
            assert np.array_equal(h, ho) and np.array_equal(v, vo)
        srv.close()
