"""Room of the allocation-free ragged call (recorded runtime, CPU): batches
whose plans filled its static array to the last bytes when work units were 32
tiles or pairs (fewer units, so a shorter index of them) are still taken, and
much larger ones still refused."""
import pytest

import fake_hip

BC_ERROR_OUT_OF_MEMORY = 2
NTT, LDE = 0, 2


@pytest.mark.parametrize("cosets,log_n,op,log_blowup,cols", [
    (False, 8, NTT, 0, 524256), (False, 10, NTT, 0, 524244), (False, 11, NTT, 0, 524228), (False, 12, NTT, 0, 523748),
    (False, 14, NTT, 0, 261104), (False, 9, LDE, 2, 104841), (True, 8, NTT, 0, 445733), (True, 12, NTT, 0, 445301),
    (True, 14, NTT, 0, 221995)])
def test_full_batches_fit(tmp_path, cosets, log_n, op, log_blowup, cols):
    got = fake_hip.run(tmp_path, f"""
        class Job(ctypes.Structure):
            _fields_ = [(k, ctypes.c_void_p) for k in ("inputs", "outputs", "coeffs")] + \\
                       [(k, ctypes.c_uint32) for k in ("log_n", "num_cols", "stride_in", "stride_out",
                                                       "stride_coeffs", "op", "log_blowup")]
        def job(i, log_n, cols, op, k):
            n, at = 1 << log_n, (i + 1) << 44
            return Job(at, at + (1 << 42), at + (1 << 43), log_n, cols, n, n << k, n, op, k)
        def run(cols):
            jobs = [job(100, {log_n}, cols, {op}, {log_blowup})]
            if {cosets}:  # all 256 cosets of 14 sizes: many segments
                jobs += [job(i, 8 + i, 1, {LDE}, 8) for i in range(14)]
            return lib.bc_ragged_run_no_alloc(ctypes.cast((Job * len(jobs))(*jobs), ctypes.c_void_p), len(jobs), None)
        done([run({cols}), run({cols} + {cols} // 32)])
    """)
    assert got == [0, BC_ERROR_OUT_OF_MEMORY]
