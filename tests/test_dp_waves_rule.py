"""The rule for phase 1's wavefronts per pair counts the compute units of the
device: a pair's share of them decides, not the number of pairs alone."""
import pytest

import cother_amd


def _waves(*args):
    return cother_amd.lib().cth_selftest_dp_waves(*args)


@pytest.mark.parametrize("trace", [0, 1])
@pytest.mark.parametrize("lq,ltmean,ltmax", [(130, 180, 400), (372, 235, 700), (600, 230, 1300), (2000, 2000, 4500)])
def test_pairs_and_units_in_proportion(lq, ltmean, ltmax, trace):
    for np in (64, 300, 1500, 6000):
        of = {ncu: _waves(lq, ltmean, ltmax, np * ncu // 64, trace, ncu) for ncu in (64, 128, 256, 304)}
        assert len(set(of.values())) == 1, (np, of)
        assert 1 <= of[64] <= 8


def test_more_units_take_more_wavefronts_a_pair():
    assert _waves(372, 235, 700, 1500, 1, 32) < _waves(372, 235, 700, 1500, 1, 2048)
