"""GPU check of the batched-coset LDE: batch_lde against its definition through
the plain entry points (one inverse transform, then one forward coset
transform per coset), bit for bit, over one- to three-pass sizes, both orders,
blowups, column counts and padded strides, and a captured graph of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def brev(x, bits):
    return int(format(x, f"0{bits}b")[::-1], 2) if bits else 0


def reference(x, log_n, cols, si, sc, so, k, bitrev):
    import torch
    from boojum_cuda_amd import ntt
    n = 1 << log_n
    coeffs = torch.zeros(cols * sc, dtype=torch.int64, device="cuda")
    out = torch.zeros(cols * so, dtype=torch.int64, device="cuda")
    ntt.batch_ntt_out_of_place(x, coeffs, log_n, cols, 0, 0, si, sc, bitrev, True, 0, 0)
    for c in range(1 << k):
        blk = brev(c, k) if bitrev else c
        ntt.batch_ntt_out_of_place(coeffs, out, log_n, cols, 0, blk * n, sc, so, not bitrev, False, k, c)
    return coeffs, out


@pytest.mark.parametrize("bitrev", [True, False])
@pytest.mark.parametrize("log_n,cols,k,pad", [
    (11, 3, 2, 0), (12, 1, 1, 0), (12, 5, 3, 7), (13, 2, 1, 0), (14, 3, 2, 1), (15, 1, 4, 0), (16, 9, 2, 16),
    (17, 2, 3, 3), (19, 3, 1, 0), (20, 2, 2, 5), (21, 1, 2, 0), (22, 2, 1, 1)])
def test_batched_cosets_match_single_transforms(gpu_ctx, log_n, cols, k, pad, bitrev):
    import torch
    from boojum_cuda_amd import lde
    n = 1 << log_n
    si, sc, so = n + pad, n + 2 * pad, (n << k) + 3 * pad
    g = torch.Generator(device="cuda").manual_seed(log_n * 100 + cols)
    x = torch.randint(-2**63, 2**63 - 1, (cols * si,), dtype=torch.int64, device="cuda", generator=g)
    want_c, want = reference(x, log_n, cols, si, sc, so, k, bitrev)
    coeffs, out = torch.zeros_like(want_c), torch.zeros_like(want)
    lde.batch_lde(x, coeffs, out, log_n, cols, si, sc, so, k, bitrev)
    assert torch.equal(coeffs, want_c) and torch.equal(out, want)


@pytest.mark.parametrize("bitrev", [True, False])
def test_graph_replays_match(gpu_ctx, bitrev):
    import torch
    from boojum_cuda_amd import lde
    log_n, cols, k = 14, 3, 2
    n = 1 << log_n
    x = torch.randint(0, 2**62, (cols * n,), dtype=torch.int64, device="cuda")
    coeffs, out = torch.zeros_like(x), torch.zeros(cols * (n << k), dtype=torch.int64, device="cuda")
    graph = lde.LdeGraph(x, coeffs, out, log_n, cols, n, n, n << k, k, bitrev)
    for i in range(4):
        x.copy_(torch.randint(0, 2**62, (cols * n,), dtype=torch.int64, device="cuda"))
        out.zero_()
        graph.launch()
        torch.cuda.synchronize()
        want_c, want = reference(x, log_n, cols, n, n, n << k, k, bitrev)
        assert torch.equal(coeffs, want_c) and torch.equal(out, want), f"replay {i}"
    graph.destroy()
