"""The 64-bit sums of the 16-lane Poseidon partial round (coop_mul_add): with
the column entries the library derives, no sum passes 64 bits at the largest
S-box output and the largest terms."""
import numpy as np
import pytest

import oracle


@pytest.mark.parametrize("seed", [None, 1])
def test_sums_stay_below_2_64(seed):
    from boojum_cuda_amd import poseidon
    rc = oracle.pos_grain_constants() if seed is None else \
        np.random.default_rng(seed).integers(0, 2**64, 360, dtype=np.uint64)
    top, word, term = 2**64 - 1, 2**32 - 1, 2 * (2**32 - 1)  # any u64; two 32-bit terms
    entries = [int(w) for w in np.ravel(poseidon.fused_table(rc)["w_hats"])]
    for a, lo in [(w, term) for w in entries] + [(1, 2**52 - 1)]:
        a0, a1 = a & word, a >> 32
        p = a0 * word + lo
        t = a0 * word + lo + (p >> 32)
        t2 = a1 * word + (t & top)
        q = a1 * word + (t2 >> 32 & word)
        assert max(p, t, q) <= top and t2 <= 2 * top + 1
        assert a * top + lo + (lo << 32) < 2**128
    assert all(w & word != word for w in entries)
