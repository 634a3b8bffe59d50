"""Times of the band chain against each other, from its events (medians, one
launch alone on the GPU): what makes a chain's step longer than its VALU work
shows as a ratio between two chains of the same width."""
import statistics

import pytest

import lcs_amd

pytestmark = pytest.mark.gpu

N = 100000


def chain_ms(ctx, bands, tile_m, alphabet):
    a, b = lcs_amd.gen_uniform(1, 64 * tile_m * bands, alphabet), lcs_amd.gen_uniform(2, N, alphabet)
    sched = lcs_amd.schedule(tile_m, 1, lcs_amd.VARIANT_CHAIN, 1)
    times = []
    for _ in range(9):
        ctx.comb(a, b, sched)
        times.append(ctx.chain_ms())
    return statistics.median(times[2:])


def test_wide_symbols_wait_for_no_load_before_the_steps():
    # one band, one row per lane: 32-bit symbols move between lanes and bytes
    # do not, 18 against 12.5 ns a step; with a wait for the next chunk's
    # symbols before the steps, 20
    with lcs_amd.Context(0) as ctx:
        assert chain_ms(ctx, 1, 1, 300) < 1.5 * chain_ms(ctx, 1, 1, 4)


@pytest.mark.parametrize("bands", [16, 32])
def test_a_chain_of_bands_keeps_the_pace_of_one(bands):
    # 32 bands add 31 lags of about 162 steps to 100064: 1.05 of one band's
    # time; in step with the stores of the band above them 1.4 to 2.0
    with lcs_amd.Context(0) as ctx:
        assert chain_ms(ctx, bands, 1, 4) < 1.3 * chain_ms(ctx, 1, 1, 4)
