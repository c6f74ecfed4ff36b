"""The autotuner's choice: thresholds between the measured sizes, levels weighted by their call, and the rule that
names the kernel of a level (no GPU needed)."""

import itertools
import random

import pytest

from torchhull_amd import tuning


def _samples(levels, seed):
    rng = random.Random(seed)
    return {g: [(n, rng.uniform(0.1, 1.0)) for n in levels] for g in (64, 16, 4, 2, 1)}


@pytest.mark.parametrize("seed", range(8))
def test_choice_is_the_best_of_all_cuts(seed):
    rng = random.Random(100 + seed)
    levels = [rng.choice((1, 8, 60, 400, 3000, 20000, 150000)) for _ in range(14)]
    weights = [rng.uniform(0.2, 2.0) for _ in levels]
    samples = _samples(levels, seed)
    chosen, cost = tuning.choose_thresholds(samples, weights)

    def total(thresholds):
        return sum(w * samples[tuning.split_for(n, thresholds)][i][1] for i, (n, w) in enumerate(zip(levels, weights)))

    cuts = sorted({0, tuning._MAX} | set(levels))
    best = min(total(t) for t in itertools.combinations_with_replacement(cuts, 4))
    assert cost == pytest.approx(best) and total(chosen) == pytest.approx(best)
    assert chosen == sorted(chosen)


def test_present_thresholds_stay_where_they_cost_next_to_nothing():
    sizes = [1000, 30000, 300000, 3000000]
    fast = dict(zip(sizes, (64, 16, 4, 1)))
    samples = {g: [(n, 1.0 if g == fast[n] else 2.0) for n in sizes] for g in (64, 16, 4, 2, 1)}
    # the last two cut the same sizes as the choice does, the first ones do not
    chosen, cost = tuning.choose_thresholds(samples, present=[100, 20000, 310000, 2900000])
    assert cost == 4.0
    assert chosen[2:] == [310000, 2900000]
    assert 1000 <= chosen[0] < 30000 <= chosen[1] < 300000
    # a level that hardly counts may go to the present threshold's lanes
    weights = [1.0, 1.0, 1.0, 1e-4]
    chosen, cost = tuning.choose_thresholds(samples, weights, [1000, 30000, 300000, 3000000])
    assert chosen == [1000, 30000, 300000, 3000000] and cost == pytest.approx(3.0002)


def test_thresholds_lie_between_the_measured_sizes():
    sizes = [1000, 30000, 31000, 900000]
    fast = dict(zip(sizes, (64, 16, 4, 1)))
    samples = {g: [(n, 1.0 if g == fast[n] else 2.0) for n in sizes] for g in (64, 16, 4, 2, 1)}
    chosen, cost = tuning.choose_thresholds(samples)
    assert cost == 4.0
    assert chosen[0] == 5500  # sqrt(1000 * 30000) to two digits
    assert 30000 <= chosen[1] < 31000 <= chosen[2] <= chosen[3] < 900000


def test_a_level_counts_by_its_share_of_the_call():
    # one level of a short call against a longer one of a long call
    samples = {g: [(100, 0.1), (110, 3.0)] for g in (64, 16, 4, 2, 1)}
    samples[64] = [(100, 0.05), (110, 3.2)]  # better for the short call
    samples[16] = [(100, 0.1), (110, 3.0)]
    assert tuning.choose_thresholds(samples, [1 / 0.3, 1 / 30.0])[0][0] >= 100
    both = tuning.choose_thresholds({g: [(100, a[1]), (100, b[1])] for g, (a, b) in samples.items()}, [1.0, 1.0])
    assert both[0][0] == 0  # by milliseconds the long call decides


@pytest.mark.parametrize("n, cameras, kernel", [
    (8192, 8, 8), (8193, 8, 16), (8192, 3, 8), (8193, 3, 4), (4096, 16, 8), (4097, 16, 16), (4096, 9, 8),
    (1024, 64, 8), (1025, 64, 64), (1024, 1100, 8), (2048, 32, 8), (2049, 32, 64), (2049, 17, 64),
])
def test_kernel_of_the_levels_with_64_lanes(n, cameras, kernel):
    assert tuning.split_for(n, (10000, 10000, 10000, 10000), cameras) == kernel


def test_kernel_of_larger_levels():
    t = (100, 1000, 10000, 100000)
    assert [tuning.split_for(n, t, 4) for n in (1000, 10000, 100000, 100001)] == [4, 4, 2, 1]
    assert [tuning.split_for(n, t, 5) for n in (1000, 10000, 100000, 100001)] == [16, 4, 2, 1]


def test_the_stored_file_says_how_it_was_made():
    import json

    v = json.loads(tuning.DEFAULT_PATH.read_text())
    assert tuning.load() == v["max_parents"]
    # chosen on its own draw, and no worse than what it replaced on another one
    assert v["shares"] <= v["default_shares"] and v["other_draw"]["shares"] <= v["other_draw"]["default_shares"]
    assert v["workloads"] > 100
