"""Launch shapes of columns of 2..128 points (host code with a recorded
runtime): every column is covered once, and no launch asks for more than the
2^32 - 1 threads along x that the runtime takes.  2^34 points in place are
128 GiB and fit the card."""
import pytest

import fake_hip


@pytest.mark.parametrize("log_n,cols", [
    (1, 1), (1, 2**32 - 1), (2, 2**32 - 1), (3, 2**31), (4, 2**30), (5, 2**29 - 1), (5, 2**29), (6, 2**28 + 1),
    (7, 2**27 - 2), (7, 2**27), (7, 2**28), (7, 3 * 2**26 + 5), (4, 4096 * 16), (4, 4096 * 16 + 1)])
def test_columns_covered(tmp_path, log_n, cols):
    got = fake_hip.run(tmp_path, f"""
        n, pad = 1 << {log_n}, 3
        rc = lib.bc_batch_ntt_internal(1 << 40, 1 << 50, {log_n}, {cols}, n, n + pad, 0, 0, 0, 0, None)
        done(dict(rc=rc, kernels=kernels(), shapes=[(g, b) for _, g, b in launches()],
                  args=[[fake.fake_arg_word(i, w) for w in range(4)] for i in range(fake.fake_launches())]))
    """)
    assert got["rc"] == 0
    n, col = 1 << log_n, 0
    for (grid, block), (src, dst, stride_in, stride_out) in zip(got["shapes"], got["args"]):
        assert grid[0] * block[0] < 2**32 and grid[1:] == block[1:] == [1, 1]
        assert (stride_in, stride_out) == (n, n + 3)
        assert src == 2**40 + 8 * n * col and dst == 2**50 + 8 * (n + 3) * col
        col += grid[0] * block[0] // 64 << (8 - log_n)
    assert set(got["kernels"]) == {"ntt_short_kernel"}
    assert cols <= col < cols + (4 << (8 - log_n))  # less than a workgroup more
