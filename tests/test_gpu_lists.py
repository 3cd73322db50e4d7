"""The K-nearest lists where their kernels change course, against the oracle's rebuild, bit
for bit: equal distances (by id then), lists just below and above 24 and 32 candidates (the
row, its tail, the buffers cut back), nodes that lie on each other, waves and blocks that
are not full, and a grid with cells smaller than the bars reach.
"""
import dataclasses

import numpy as np
import pytest

from conftest import Fixture
from oracle import orc
from trussnet_amd._abi import Nodes, RelaxParams

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tn():
    from trussnet_amd import relax

    if relax.device_count() < 1:
        pytest.fail("no HIP device visible")
    return relax


def nodes_at(grid, P, types=(0,), seed=0):
    """Nodes at P with the labels of their voxels and types drawn from `types`"""
    rng = np.random.default_rng(seed)
    P = np.asarray(P, np.float32).reshape(-1, 3)
    v = np.clip((P / np.asarray(grid.vs, np.float32)).astype(int), 0, np.array([grid.nx, grid.ny, grid.nz]) - 1)
    lab = grid.L.reshape(grid.nz, grid.ny, grid.nx)[v[:, 2], v[:, 1], v[:, 0]]
    n = len(P)
    part = np.zeros((n, 2), np.uint16)
    return Nodes(P, lab, rng.choice(np.array(types, np.uint8), n), part)


def lattice(step, n, rng):
    """n points of a lattice, in a shuffled order: equal distances everywhere"""
    e = int(np.ceil(n ** (1 / 3)))
    P = np.stack(np.meshgrid(*[np.arange(e)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * step + 9.0
    return P[rng.permutation(n)]


def same_lists(tn, grid, nodes, prm=RelaxParams()):
    want = orc.rebuild(grid, nodes, prm)
    with tn.Plan(grid, nodes, prm) as plan:
        got = plan.rebuild()
    for k in ("key", "sorted", "cstart", "nnb"):
        assert np.array_equal(got[k], want[k]), k
    listed = np.arange(24)[None, :] < want["nnb"][:, None]   # (what lies past a list's end is nobody's)
    assert np.array_equal(got["nbr"].reshape(-1, 24)[listed], want["nbr"].reshape(-1, 24)[listed])
    return want["nnb"]


# bars a node in the lattice's middle (h = 3, reach 4.8): 6, 18, 26, 56; 179 and more
@pytest.mark.parametrize("step,most", [(4.5, 6), (3.0, 18), (2.5, 24), (2.0, 24), (1.25, 24)])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 257, 1000])
def test_equal_distances(tn, step, most, n):
    grid = Fixture("jitter64").grid
    nnb = same_lists(tn, grid, nodes_at(grid, lattice(step, n, np.random.default_rng(n))))
    assert nnb.max() <= most and (n < 1000 or nnb.max() == most)


@pytest.mark.parametrize("per", [24, 25, 31, 32, 33, 34, 200])
def test_nodes_on_each_other(tn, per):
    """`per` nodes at each of a few places out of each other's reach (per - 1 bars, all of
    length 0), beside scattered ones"""
    grid = Fixture("jitter64").grid
    rng = np.random.default_rng(per)
    places = np.array([[9.0, 9, 9], [9, 9, 30.5], [40, 30, 9.25]], np.float32)
    P = np.concatenate([np.repeat(places, per, 0), rng.uniform(35, 60, (300, 3)).astype(np.float32)])
    nnb = same_lists(tn, grid, nodes_at(grid, P[rng.permutation(len(P))]))
    assert np.sum(nnb == min(per - 1, 24)) >= 3 * per


@pytest.mark.parametrize("name", ["sectors48", "aniso40"])
@pytest.mark.parametrize("density", [0.02, 0.06, 0.2, 1.0])
def test_scattered_of_all_types_and_labels(tn, name, density):
    """Labels side by side (no bar between interior nodes of two), sizes of several levels and
    all node types, from sparse to a dozen times what the lists hold"""
    grid = Fixture(name).grid
    rng = np.random.default_rng(7)
    ext = np.array([grid.nx, grid.ny, grid.nz]) * np.asarray(grid.vs)
    P = rng.uniform(0, 1, (int(density * 20000), 3)) * ext * [1, 1, 0.5]
    same_lists(tn, grid, nodes_at(grid, P, types=(0, 0, 0, 1, 2, 3)))


@pytest.mark.parametrize("hmax", [1.2, 2.0])
@pytest.mark.parametrize("density", [0.03, 0.5])
def test_reach_beyond_the_cells(tn, hmax, density):
    """A grid whose stated largest size is below its largest h: the reference searches only
    the cells around the node's own, which then miss bars"""
    base = Fixture("sectors48").grid
    grid = dataclasses.replace(base, hmax=hmax)
    assert float(np.max(grid.h)) > hmax
    rng = np.random.default_rng(11)
    P = rng.uniform(0, 48, (int(density * 20000), 3))
    same_lists(tn, grid, nodes_at(grid, P, types=(0, 1)))
