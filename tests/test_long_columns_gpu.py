"""Columns longer than a buffer descriptor reaches (beyond 2^28 points the
passes address by pointer): a sparse input's transform is known in closed form
at any output, and the inverse gives the input back."""
import numpy as np
import pytest

from pyref import P, brev, omega

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n", [28, 29])
def test_sparse_column(gpu_ctx, log_n):
    import torch
    from boojum_cuda_amd import ntt
    n = 1 << log_n
    rng = np.random.default_rng(log_n)
    at = [0, 1, n // 2 + 3, n - 1] + [int(i) for i in rng.integers(0, n, 4)]
    values = {i: int(v) for i, v in zip(at, rng.integers(1, P, len(at), dtype=np.uint64))}
    idx = torch.tensor(list(values), device="cuda")
    val = torch.from_numpy(np.array(list(values.values()), dtype=np.uint64).view(np.int64)).to("cuda")
    x = torch.zeros(n, dtype=torch.int64, device="cuda")
    x[idx] = val
    y = torch.empty_like(x)
    ntt.batch_ntt_out_of_place(x, y, log_n, 1, 0, 0, n, n, False, False, 0, 0)
    w = omega(log_n)
    for k in [0, 1, n - 1, n // 2] + [int(i) for i in rng.integers(0, n, 12)]:
        want = sum(v * pow(w, i * k, P) for i, v in values.items()) % P
        assert int(np.uint64(y[brev(k, log_n)].item() & (2**64 - 1))) == want, k
    ntt.batch_ntt_in_place(y, log_n, 1, 0, n, True, True, 0, 0)
    assert torch.equal(y, x)
