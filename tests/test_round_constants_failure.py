"""A replacement of the Poseidon round constants that fails part way (recorded
runtime, CPU): the hashes are then not available, rather than run on a mixture
of old and new tables."""
import fake_hip

BC_ERROR_NOT_INITIALIZED = 3


def test_failed_copy_leaves_no_mixture(tmp_path):
    got = fake_hip.run(tmp_path, """
        def constants(k):
            return lib.bc_poseidon_set_round_constants((ctypes.c_uint64 * 360)(*range(k, k + 360)))
        def hashes():
            v, r = 1 << 40, 1 << 41
            return [lib.bc_poseidon_leaves(v, 8 << 15, r, 4 << 15, 0, 0, 0, None),
                    lib.bc_poseidon_nodes(v, 800, r, 400, None),
                    lib.bc_poseidon_build_merkle_tree(v, 8 << 10, r, 8 << 10, 0, 3, None),
                    lib.bc_poseidon2_leaves_cooperative(v, 800, r, 400, 0, 0, 0, None),
                    lib.bc_poseidon2_build_merkle_tree_nodes(v, 1 << 10, r, 1 << 10, 2, None)]
        out = dict(before=hashes(), first=constants(1), usable=hashes(), failures=[])
        copies, k = 0, 0
        while True:
            fake.fake_reset()
            fake.fake_fail_symbol_copy(k)
            rc = constants(1000 + k)
            if rc == 0:
                break
            fake.fake_reset()
            after = hashes()
            out["failures"].append((rc, after, len(launches())))
            fake.fake_fail_symbol_copy(-1)
            assert constants(2000 + k) == 0 and hashes() == [0] * 5
            k += 1
        done(out)
    """)
    assert got["before"] == [BC_ERROR_NOT_INITIALIZED] * 5
    assert got["first"] == 0 and got["usable"] == [0] * 5
    assert got["failures"]
    for rc, after, launched in got["failures"]:
        assert rc != 0 and after == [BC_ERROR_NOT_INITIALIZED] * 5 and launched == 0
