"""GPU parity of barycentric evaluation over short columns on either side of the
choice of kernel: one thread a column, one workgroup a column, tiles with
partial sums.  Raw u64 inputs, aligned and not, bit for bit against the
oracle's sum."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("log_count,num_polys", [(1, 3), (4, 5), (5, 1), (5, 65), (6, 8192), (6, 8193), (7, 8193),
                                                 (9, 7), (10, 33), (11, 5)])
def test_short_columns(gpu_ctx, kind, log_count, num_polys):
    import torch
    from boojum_cuda_amd import barycentric as b
    count, coef_width, planes = 1 << log_count, 1 if kind == 0 else 2, 2 if kind == 2 else 1
    ys = oracle.fill_raw(num_polys * planes * count, 31 * log_count + num_polys, 0)
    coeffs = oracle.fill_raw(coef_width * count, 32 * log_count + num_polys, 1)
    want = oracle.bary_batch_eval(ys, kind == 2, coeffs, kind != 0, count, num_polys)
    partial_elems, final_bytes = b.get_batch_eval_temp_storage_sizes(kind, count, num_polys)
    partial = torch.empty(max(1, partial_elems * coef_width), dtype=torch.int64, device="cuda")
    final = torch.empty(max(1, final_bytes), dtype=torch.uint8, device="cuda")
    for shift in (0, 1):
        def dev(a):
            return torch.from_numpy(np.concatenate([np.zeros(shift, np.uint64), a]).view(np.int64)).to("cuda")[shift:]
        evals = torch.empty(num_polys * coef_width, dtype=torch.int64, device="cuda")
        b.batch_eval(kind, dev(ys), count, num_polys, dev(coeffs), partial, final, evals)
        assert np.array_equal(evals.cpu().numpy().view(np.uint64), want), shift
