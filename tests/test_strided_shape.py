"""Launch shapes of the strided passes (host only): the groups cover every
(column, block) pair exactly once at any column count, and full rounds of
resident workgroups are taken where the planner's rule says so."""
import pytest


@pytest.mark.parametrize("bitrev", [False, True])
@pytest.mark.parametrize("log_n", [14, 17, 18, 19, 21, 24])
def test_groups_cover_the_pairs(log_n, bitrev):
    from boojum_cuda_amd import autotune, ntt
    autotune.clear()
    for cols in [*range(1, 130), 255, 256, 1000, 70001]:
        for p in ntt.describe_plan(log_n, cols, bitrev, bitrev):
            if p["contiguous"] or p["workgroup_threads"] == 64:
                continue
            assert 1 <= p["groups"] <= 65535 and p["pairs_per_workgroup"] >= 1
            assert (p["groups"] - 1) * p["pairs_per_workgroup"] < p["work_items"] <= \
                p["groups"] * p["pairs_per_workgroup"]


def test_full_rounds():
    from boojum_cuda_amd import autotune, ntt
    autotune.clear()

    def pairs(log_n, cols, bitrev):
        return [p["pairs_per_workgroup"] for p in ntt.describe_plan(log_n, cols, bitrev, bitrev)
                if not p["contiguous"]]
    assert pairs(17, 100, False) == pairs(17, 100, True) == [7]  # 15 x 32 workgroups
    assert pairs(18, 40, False) == [5]                           # 8 x 64
    assert pairs(19, 6, False) == pairs(19, 6, True) == [1]      # 768 workgroups; b2n: 2 would fill 384 of 512
    assert pairs(16, 100, False) == [1]                          # 4 bits: little setup
    assert pairs(20, 256, True) == [16]                          # more than 8 pairs a round
