"""GPU parity of the one-wave transforms: 2..128 points (several columns to a
wave, one or four waves to a workgroup) in every direction, order and coset, at
column counts around a wave's and a workgroup's share, and the latency path of
2^13..2^16 points on either side of its column count; with padded strides and
in place, bit for bit against the oracle."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n", range(1, 8))
@pytest.mark.parametrize("bitrev", [False, True])
@pytest.mark.parametrize("inverse", [False, True])
def test_short_columns(gpu_ctx, log_n, bitrev, inverse):
    import torch
    from boojum_cuda_amd import ntt
    n, per_wave = 1 << log_n, 1 << (8 - log_n)
    for cols, log_ext, coset in ((1, 0, 0), (per_wave, 2, 3), (per_wave + 1, 0, 0), (3 * per_wave - 1, 1, 0),
                                 (4097 * per_wave - 1, 0, 0), (4098 * per_wave + 1, 1, 1)):
        si, so = n + 1, n + 2
        x = oracle.fill_raw(cols * si, 7 * log_n + cols, 0)
        want = np.full(cols * so, 5, dtype=np.uint64)
        oracle.batch_ntt(x, log_n, cols, si, so, bitrev, inverse, log_ext, coset, out=want, threads=8)
        d = torch.from_numpy(x.view(np.int64)).to("cuda")
        out = torch.full((cols * so,), 5, dtype=torch.int64, device="cuda")
        ntt.batch_ntt_out_of_place(d, out, log_n, cols, 0, 0, si, so, bitrev, inverse, log_ext, coset)
        got = out.cpu().numpy().view(np.uint64).reshape(cols, so)
        assert np.array_equal(got, want.reshape(cols, so))
        ntt.batch_ntt_in_place(d, log_n, cols, 0, si, bitrev, inverse, log_ext, coset)
        ip = d.cpu().numpy().view(np.uint64).reshape(cols, si)
        assert np.array_equal(ip[:, :n], got[:, :n]) and np.array_equal(ip[:, n:], x.reshape(cols, si)[:, n:])


@pytest.mark.parametrize("log_n", range(13, 17))
@pytest.mark.parametrize("bitrev", [False, True])
@pytest.mark.parametrize("inverse", [False, True])
def test_latency_path(gpu_ctx, log_n, bitrev, inverse):
    import torch
    from boojum_cuda_amd import ntt
    n = 1 << log_n
    most = 1 << (18 - log_n)
    for cols in (1, most - 1, most, most + 1):
        si, so = n + 1, n + 2
        x = oracle.fill_raw(cols * si, 7 * log_n + cols, 0)
        want = np.full(cols * so, 5, dtype=np.uint64)
        oracle.batch_ntt(x, log_n, cols, si, so, bitrev, inverse, 0, 0, out=want, threads=8)
        d = torch.from_numpy(x.view(np.int64)).to("cuda")
        out = torch.full((cols * so,), 5, dtype=torch.int64, device="cuda")
        ntt.batch_ntt_out_of_place(d, out, log_n, cols, 0, 0, si, so, bitrev, inverse, 0, 0)
        assert np.array_equal(out.cpu().numpy().view(np.uint64), want), cols
        ntt.batch_ntt_in_place(d, log_n, cols, 0, si, bitrev, inverse, 0, 0)
        ip = d.cpu().numpy().view(np.uint64).reshape(cols, si)
        assert np.array_equal(ip[:, :n], want.reshape(cols, so)[:, :n])
