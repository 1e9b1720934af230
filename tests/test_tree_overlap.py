"""Tree inputs that lie where the tree's later layers go: they are read before
those layers are written only if each layer has a launch of its own.  Host
code with a recorded runtime on the CPU; results on the GPU."""
import pytest

import fake_hip
from test_poseidon_gpu import HASHES, consts  # noqa: F401


def test_launches_by_overlap(tmp_path):
    got = fake_hip.run(tmp_path, """
        rc = (ctypes.c_uint64 * 360)(*range(1, 361))
        assert lib.bc_poseidon_set_round_constants(rc) == 0
        leaves, base = 1 << 10, 1 << 40
        def tree(values, cols, layers=11):
            fake.fake_reset()
            assert lib.bc_poseidon2_build_merkle_tree(values, leaves * cols, base, 8 * leaves, 0, layers, None) == 0
            return [k[9:] for k in kernels()]
        def nodes(values, layers=6):
            fake.fake_reset()
            assert lib.bc_poseidon_build_merkle_tree_nodes(values, 8 * leaves, base, 8 * leaves, layers, None) == 0
            return len(launches())
        done(dict(
            tree_apart=tree(base + 64 * leaves, 4), tree_before=tree(base - 32 * leaves, 4),
            tree_in_nodes=tree(base + 32 * leaves, 4), tree_last_word=tree(base + 64 * leaves - 8, 8),
            tree_into_nodes=tree(base - 32 * leaves + 8, 8), tree_leaves_only=tree(base + 32 * leaves, 4, 1),
            nodes_apart=nodes(base + 64 * leaves), nodes_into_first_layer=nodes(base - 32 * leaves),
            nodes_in_second=nodes(base + 32 * leaves), nodes_last_word=nodes(base + 64 * leaves - 8),
            nodes_one_layer=nodes(base + 32 * leaves, 1)))
    """)
    fused, plain = ["leaves_coop_kernel"] + ["nodes_coop_kernel"], ["leaves_coop_kernel"] + 2 * ["nodes_coop_kernel"]
    assert got["tree_apart"] == got["tree_before"] == fused
    assert got["tree_in_nodes"] == got["tree_last_word"] == got["tree_into_nodes"] == plain
    assert got["tree_leaves_only"] == ["leaves_coop_kernel"]
    assert got["nodes_apart"] == got["nodes_into_first_layer"] == 1
    assert got["nodes_in_second"] == got["nodes_last_word"] == 2  # the first layer alone, then the others
    assert got["nodes_one_layer"] == 1


@pytest.mark.gpu
@pytest.mark.parametrize("p", HASHES)
@pytest.mark.parametrize("log_leaves,cols", [(1, 1), (5, 4), (6, 2), (11, 3), (13, 4), (14, 4)])
def test_tree_of_values_among_its_nodes(gpu_ctx, consts, p, log_leaves, cols):
    import torch
    from boojum_cuda_amd import poseidon
    leaves = 1 << log_leaves
    values = torch.randint(-2**63, 2**63 - 1, (leaves * cols,), dtype=torch.int64, device="cuda")
    want, tree = (torch.zeros(8 * leaves, dtype=torch.int64, device="cuda") for _ in range(2))
    poseidon.build_merkle_tree(values, want, 0, layers_count=log_leaves + 1, p=p)
    inside = tree[4 * leaves:4 * leaves + leaves * cols]
    inside.copy_(values)
    poseidon.build_merkle_tree(inside, tree, 0, layers_count=log_leaves + 1, p=p)
    assert torch.equal(tree[:8 * leaves - 4], want[:8 * leaves - 4])


@pytest.mark.gpu
@pytest.mark.parametrize("p", HASHES)
@pytest.mark.parametrize("log_nodes", [1, 5, 6, 9, 14])
def test_nodes_of_values_among_later_layers(gpu_ctx, consts, p, log_nodes):
    import torch
    from boojum_cuda_amd import poseidon
    nodes = 1 << log_nodes
    values = torch.randint(-2**63, 2**63 - 1, (8 * nodes,), dtype=torch.int64, device="cuda")
    want = torch.zeros_like(values)
    poseidon.build_merkle_tree_nodes(values, want, log_nodes + 1, p=p)
    both = torch.zeros(12 * nodes, dtype=torch.int64, device="cuda")
    both[4 * nodes:].copy_(values)
    poseidon.build_merkle_tree_nodes(both[4 * nodes:], both[:8 * nodes], log_nodes + 1, p=p)
    assert torch.equal(both[:8 * nodes - 4], want[:8 * nodes - 4])
