"""Evaluations that are written over the columns or coefficients they are
computed from.  Host code with a recorded runtime on the CPU; results on the
GPU."""
import pytest

import fake_hip


def test_launches_by_overlap(tmp_path):
    got = fake_hip.run(tmp_path, """
        rows, polys, ys, co, part = 256, 20, 1 << 40, 1 << 41, 1 << 42
        def run(evals, rows=rows, kind=1):
            fake.fake_reset()
            assert lib.bc_batch_eval(kind, ys, rows, polys, co, part, 1 << 20, None, 0, evals, None) == 0
            return [k[5:] for k in kernels()]
        done(dict(
            apart=run(1 << 43), behind_ys=run(ys + 8 * rows * polys), before_ys=run(ys - 16 * polys),
            behind_coeffs=run(co + 16 * rows), over_ys=run(ys), end_of_ys=run(ys + 8 * rows * polys - 8),
            into_ys=run(ys - 16 * polys + 8), over_coeffs=run(co), end_of_coeffs=run(co + 16 * rows - 8),
            end_of_pairs=run(ys + 16 * rows * polys - 8, kind=2), base_coeffs=run(co + 8 * rows, kind=0),
            longer=run(ys, rows=2048), shorter=run(ys, rows=64)))
    """)
    one, two = ["eval_column_kernel"], ["eval_column_kernel", "eval_final_kernel"]
    for name in ("apart", "behind_ys", "before_ys", "behind_coeffs", "base_coeffs"):
        assert got[name] == one, (name, got)
    for name in ("over_ys", "end_of_ys", "into_ys", "over_coeffs", "end_of_coeffs", "end_of_pairs"):
        assert got[name] == two, (name, got)
    assert got["longer"] == ["eval_tiles_kernel", "eval_final_kernel"]
    assert got["shorter"] == one  # below 128 rows no room for partial sums is asked for


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("log_rows,polys", [(7, 1), (7, 300), (8, 33), (10, 20), (11, 20)])
@pytest.mark.parametrize("over", ["ys", "coeffs"])
def test_evaluations_over_their_inputs(gpu_ctx, kind, log_rows, polys, over):
    import torch
    from boojum_cuda_amd import barycentric as b
    rows, ext = 1 << log_rows, kind != 0
    y_len, c_len, e_len = (2 if kind == 2 else 1) * rows * polys, (2 if ext else 1) * rows, (2 if ext else 1) * polys
    g = torch.Generator(device="cuda").manual_seed(log_rows + polys)
    ys, coeffs = (torch.randint(-2**63, 2**63 - 1, (k,), dtype=torch.int64, device="cuda", generator=g)
                  for k in (max(y_len, e_len), max(c_len, e_len)))
    partial, _ = b.get_batch_eval_temp_storage_sizes(kind, rows, polys)
    temp = torch.zeros(partial * (2 if ext else 1), dtype=torch.int64, device="cuda")
    want = torch.zeros(e_len, dtype=torch.int64, device="cuda")
    b.batch_eval(kind, ys[:y_len], rows, polys, coeffs[:c_len], temp, None, want)
    evals = (ys if over == "ys" else coeffs)[:e_len]
    b.batch_eval(kind, ys[:y_len], rows, polys, coeffs[:c_len], temp, None, evals)
    assert torch.equal(evals, want)
