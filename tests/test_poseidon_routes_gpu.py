"""GPU parity of the two hashing routes on either side of their switch: leaf
sets and node layers of at most 2^14 take 16
lanes a state (several node layers to a launch), larger ones one lane.
Bit-exact against the oracle."""
import numpy as np
import pytest

import oracle
from test_poseidon_gpu import HASHES, consts, oracle_leaves, oracle_nodes, to_dev, to_host  # noqa: F401

pytestmark = pytest.mark.gpu
EDGES = np.array([0, 1, 2**32 - 1, 2**32, 2**64 - 2**32, 2**64 - 2**32 + 1, 2**64 - 1], dtype=np.uint64)


def values(count, seed):
    """Raw u64 draws, one in eight an edge value."""
    r = np.random.default_rng(seed)
    v = r.integers(0, 2**64, count, dtype=np.uint64)
    at = r.random(count) < 0.125
    v[at] = EDGES[r.integers(0, len(EDGES), int(at.sum()))]
    return v


@pytest.mark.parametrize("p", HASHES)
@pytest.mark.parametrize("count", [1, 31, 33, 1 << 14, (1 << 14) + 1, (1 << 15) + 1])
@pytest.mark.parametrize("log_rows,cols", [(0, 1), (0, 13), (1, 8), (2, 3), (3, 5)])
def test_leaves_either_side_of_the_switch(consts, p, count, log_rows, cols):  # noqa: F811
    import torch
    from boojum_cuda_amd import poseidon
    rows = 1 << log_rows
    vals = values(rows * cols * count, count * 16 + cols)
    res = torch.zeros(4 * count, dtype=torch.int64, device="cuda")
    poseidon.launch_single_thread_leaves_kernel(to_dev(vals), res, log_rows, p=p)
    assert np.array_equal(to_host(res), oracle_leaves(vals, rows, cols, count, consts, p))


@pytest.mark.parametrize("p", HASHES)
@pytest.mark.parametrize("count", [(1 << 14) - 1, (1 << 14) + 3, (1 << 15) + 3])
def test_checkpoints_across_the_switch(consts, p, count):  # noqa: F811
    """Capacity stored by one route's kernel and loaded by the other's."""
    import torch
    from boojum_cuda_amd import poseidon
    c1, c2 = 16, 5
    vals = values((c1 + c2) * count, count)
    first, second = to_dev(vals[:c1 * count]), to_dev(vals[c1 * count:])
    one = poseidon.launch_single_thread_leaves_kernel
    coop = poseidon.launch_cooperative_leaves_kernel
    want = oracle_leaves(vals, 1, c1 + c2, count, consts, p)
    for a, b in ((one, one), (one, coop), (coop, one)):
        res = torch.zeros(4 * count, dtype=torch.int64, device="cuda")
        a(first, res, 0, False, True, p=p)
        b(second, res, 0, True, False, p=p)
        assert np.array_equal(to_host(res), want)


@pytest.mark.parametrize("p", HASHES)
@pytest.mark.parametrize("log_children,layers", [(1, 1), (4, 4), (6, 1), (6, 5), (6, 6), (7, 7), (13, 6), (13, 13),
                                                 (15, 3), (16, 2), (16, 16)])
def test_fused_node_layers(consts, p, log_children, layers):  # noqa: F811
    """layers_count node layers: whole launches of six, remainders, layers that
    start above 2^14 nodes and trees narrower than a workgroup."""
    import torch
    from boojum_cuda_amd import poseidon
    n = 1 << log_children
    vals = values(4 * n, n + layers)
    guard = 0x5A5A5A5A
    res = torch.full((4 * n,), guard, dtype=torch.int64, device="cuda")
    poseidon.build_merkle_tree_nodes(to_dev(vals), res, layers, p=p)
    got, layer, at = to_host(res), vals, 0
    for l in range(layers):
        count = n >> (l + 1)
        layer = oracle_nodes(layer, count, consts, p)
        assert np.array_equal(got[at:at + 4 * count], layer), f"layer {l}"
        at += 4 * count
    assert (got[at:] == guard).all()


@pytest.mark.parametrize("log_leaves", [1, 4, 5, 6, 11, 13, 14, 15])
@pytest.mark.parametrize("p", [0, 1])
def test_tree_equals_leaves_and_nodes(gpu_ctx, p, log_leaves):
    """build_merkle_tree (whose leaves' launch climbs the first node layers when
    they are few) against the leaves and nodes entry points, for every number
    of layers."""
    import torch
    from boojum_cuda_amd import poseidon
    kind = (poseidon.POSEIDON, poseidon.POSEIDON2)[p]
    leaves = 1 << log_leaves
    g = torch.Generator(device="cuda").manual_seed(log_leaves)
    values = torch.randint(-2**63, 2**63 - 1, (leaves * 2 * 9,), dtype=torch.int64, device="cuda", generator=g)
    for layers in range(1, log_leaves + 2):
        want = torch.full((8 * leaves,), -1, dtype=torch.int64, device="cuda")
        got = want.clone()
        poseidon.build_merkle_tree_leaves(values, want[:4 * leaves], 1, p=kind)
        poseidon.build_merkle_tree_nodes(want[:4 * leaves], want[4 * leaves:], layers - 1, p=kind)
        poseidon.build_merkle_tree(values, got, 1, layers_count=layers, p=kind)
        assert torch.equal(got, want), layers
