"""Tuned entries for the sizes of the one-wave passes (host only): an entry
that shapes the 4096-point passes is used in their place, the tuner tries such
entries, and none that ships takes the one-wave passes away."""
import os

import pytest

SMALL_POINTS = 18  # log2


@pytest.fixture
def tune():
    from boojum_cuda_amd import autotune
    autotune.clear()
    yield autotune
    autotune.clear()


def threads(log_n, cols, bitrev=False):
    from boojum_cuda_amd import ntt
    return {p["workgroup_threads"] for p in ntt.describe_plan(log_n, cols, bitrev, bitrev)}


@pytest.mark.parametrize("bitrev", [False, True])
@pytest.mark.parametrize("log_n", [13, 14, 15])
def test_entries_shape_the_passes(tune, log_n, bitrev):
    from boojum_cuda_amd import ntt
    P = tune.TuneParams
    most = 1 << (SMALL_POINTS - log_n)
    assert threads(log_n, 1, bitrev) == threads(log_n, most, bitrev) == {64}
    assert threads(log_n, most + 1, bitrev) == {256}
    lc = most.bit_length() - 1
    tune.set_entry(log_n, lc, P(9, 1))
    plan = ntt.describe_plan(log_n, most, bitrev, bitrev)
    assert {(p["contiguous"], p["log_h"]) for p in plan} == {(1, 9), (0, log_n - 9)} and threads(log_n, most) == {256}
    assert threads(log_n, 1, bitrev) == {256}  # the nearest bucket's
    tune.set_entry(log_n, lc, P(0, 0, 3))
    strided = [p for p in ntt.describe_plan(log_n, most, bitrev, bitrev) if not p["contiguous"]]
    assert [p["pairs_per_workgroup"] for p in strided] == [3]
    tune.set_entry(log_n, lc, P(0, 0, 0, 64))
    assert threads(log_n, most, bitrev) == {256}
    tune.set_entry(log_n, lc, P(0, 0, 0, 0, 0, 0, 12))
    assert threads(log_n, most, bitrev) == {256}
    tune.set_entry(log_n, lc, P(0, 0, 0, 0, 4, 4))  # ragged units only
    assert threads(log_n, most, bitrev) == {64}
    with pytest.raises(RuntimeError):
        tune.set_entry(log_n, lc, P(0, 0, 0, 0, 0, 0, 8))


def test_2_16_keeps_its_rule(tune):
    for params in ((), (10, 1), (0, 0, 3), (0, 0, 0, 64)):
        tune.set_entry(16, 2, tune.TuneParams(*params))
        assert threads(16, 1) == threads(16, 4) == {64} and threads(16, 5) == {256}
    tune.set_entry(16, 2, tune.TuneParams(0, 0, 0, 0, 0, 0, 12))
    assert threads(16, 4) == {256}


def test_shipped_database_keeps_the_one_wave_passes(tune):
    from boojum_cuda_amd._lib import LIB_PATH
    tune.load(os.path.join(os.path.dirname(LIB_PATH), "tuning", "mi355x.txt"))
    for log_n in (13, 14, 15, 16):
        for cols in range(1, (1 << (SMALL_POINTS - log_n)) + 1):
            assert threads(log_n, cols) == {64}, (log_n, cols)


@pytest.mark.parametrize("wins", [(9, 1, 0, 0, 0, 0, 0), (0, 0, 2, 0, 0, 0, 0), (0, 0, 0, 1024, 0, 0, 0),
                                  (0, 0, 0, 0, 0, 0, 12), None])
def test_tuner_tries_them(tune, monkeypatch, wins):
    """tune_shape on stand-in timings in which one entry beats the built-in plan."""
    class Bench:
        import torch

        def __init__(self, log_n, num_cols, reps):
            self.shape = log_n, num_cols

        def outputs(self):
            return self.torch.zeros(1), self.torch.zeros(1)

        def warm(self):
            pass

        def time_ms(self):
            return 1.0 if tune.get_entry(*self.shape).key() == wins else 2.0

    monkeypatch.setattr(tune, "_Bench", Bench)
    monkeypatch.setattr(tune, "_time_ragged", lambda *a: 1.0)
    best = tune.tune_shape(14, 0, log=lambda m: None)[0]
    assert best.key() == (wins or (0,) * 7)
