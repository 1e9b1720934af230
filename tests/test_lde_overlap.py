"""Coefficients that lie inside the LDE's outputs: the cosets then have to run
one after the other, so that the last one may be transformed in place.  Host
code with a recorded runtime on the CPU; results on the GPU."""
import pytest

import fake_hip

LOG_N, COLS, K = 13, 3, 2


def test_launches_by_overlap(tmp_path):
    got = fake_hip.run(tmp_path, f"""
        log_n, cols, k = {LOG_N}, {COLS}, {K}
        n = 1 << log_n
        base = 1 << 40
        def lde(coeffs, sc, outputs, so, bitrev=1):
            fake.fake_reset()
            assert lib.bc_batch_lde(1 << 41, coeffs, outputs, log_n, cols, n, sc, so, k, bitrev, None) == 0
            return len(launches())
        so = (n << k) + n
        done(dict(
            apart=lde(base, n, base + 8 * cols * n, n << k),
            last_block=lde(base + 8 * 3 * n, n << k, base, n << k),
            last_block_natural=lde(base + 8 * 3 * n, n << k, base, n << k, 0),
            first_block=lde(base, n << k, base, n << k),
            between_rows=lde(base + 8 * (n << k), so, base, so),
            row_before=lde(base - 8 * n, so, base, so),
            straddles=lde(base + 8 * ((n << k) - 1), so, base, so),
            runs_into_next_row=lde(base + 8 * ((n << k) + 1), so, base, so),
            other_stride=lde(base + 8 * (n << k), n, base, so),
            touches_end=lde(base + 8 * cols * (n << k), n, base, n << k),
            touches_start=lde(base - 8 * cols * n, n, base, n << k),
        ))
    """)
    # two launches of the inverse transform, then two for all cosets or two for each
    together, apart = 4, 2 + (2 << K)
    for name in ("apart", "between_rows", "row_before", "touches_end", "touches_start"):
        assert got[name] == together, (name, got)
    for name in ("last_block", "last_block_natural", "first_block", "straddles", "runs_into_next_row", "other_stride"):
        assert got[name] == apart, (name, got)


@pytest.mark.gpu
@pytest.mark.parametrize("bitrev", [True, False])
@pytest.mark.parametrize("log_n,cols,k", [(11, 3, 2), (12, 1, 1), (13, 3, 2), (17, 2, 3), (20, 5, 1)])
def test_coefficients_in_the_last_block(gpu_ctx, log_n, cols, k, bitrev):
    import torch
    from boojum_cuda_amd import lde
    n = 1 << log_n
    so = n << k
    x = torch.randint(-2**63, 2**63 - 1, (cols * n,), dtype=torch.int64, device="cuda")
    coeffs, want = torch.zeros_like(x), torch.zeros(cols * so, dtype=torch.int64, device="cuda")
    lde.batch_lde(x, coeffs, want, log_n, cols, n, n, so, k, bitrev)
    out = torch.zeros_like(want)
    lde.batch_lde(x, out[so - n:], out, log_n, cols, n, so, so, k, bitrev)
    assert torch.equal(out, want)
    graph = lde.LdeGraph(x, out[so - n:], out, log_n, cols, n, so, so, k, bitrev)
    for _ in range(3):
        out.zero_()
        graph.launch()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    graph.destroy()
