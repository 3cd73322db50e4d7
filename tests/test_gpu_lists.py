"""The K-nearest lists where their kernels change course, against the oracle's rebuild, bit
for bit: equal distances (by id then), lists just below and above 24 and 32 candidates (the
row, its tail, the buffers cut back), nodes that lie on each other, waves and blocks that
are not full, a grid with cells smaller than the bars reach, and bars that end past the cells
the reference visits by a rounding; in any unit of length.
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


def past_the_region(hmin, prm, want, seed):
    """(size, place, place of the other) along an axis with voxels of 1: two nodes in the first
    and the third row of cells of the lowest level, the lower one of that size, the upper one of
    size hmin, such that they are a bar by the 32-bit test while the upper one's cell lies just
    past the lower one's scan region: rounding puts the bar's reach (t + skin) (h_i + h_j) / 2 two
    units above the region's ((t + skin) h_i + b) / 2, b the edge of the cells."""
    f = np.float32
    T = f(prm.t) + f(prm.skin)
    half, b = T * f(0.5), T * hmin

    def cell(x):
        return int(np.floor((x + f(0.5)) / b))

    edge = f(2) * b - f(0.5)   # the first place of the third row
    while cell(edge) >= 2:
        edge = np.nextafter(edge, f(-1))
    while cell(edge) < 2:
        edge = np.nextafter(edge, f(9))
    rng = np.random.default_rng(seed)
    out = []
    while len(out) < want:
        hi = hmin * f(rng.uniform(1.05, 1.5))
        r, rj = f(0.5) * (T * hi + b), half * (hi + hmin)
        if (rj - r) / np.spacing(r) < 2:
            continue
        p = f(np.float64(edge) - np.float64(r) - np.float64(np.spacing(r)))
        e = edge - p
        if e * e < rj * rj and cell(p + r) < 2:
            out.append((hi, p, edge))
    return out


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_bars_just_past_the_scan_region(tn, axis):
    """A candidate that passes the test of distance by its last bit, in a cell that the
    reference does not visit for the node: not in the list"""
    prm = RelaxParams()
    hmin = np.float32(1.0129207)
    pairs = past_the_region(hmin, prm, 12, axis)
    base = Fixture("jitter64").grid
    grid = dataclasses.replace(base, hmin=float(hmin), hmax=float(2 * hmin), h=np.full(base.h.size, hmin, np.float32))
    h = grid.h.reshape(grid.nz, grid.ny, grid.nx)
    P, low, up = [], [], []
    for k, (hi, lo, hi_place) in enumerate(pairs):
        a, b = 6.0 + 9.0 * (k % 4), 8.0 + 9.0 * (k // 4)   # (out of the other pairs' reach)
        for place, size in ((lo, hi), (hi_place, hmin), (np.float32(1.6), hi)):   # the third: scans that cell for its own list
            p = np.insert(np.array([a, b], np.float32), axis, place)
            if size == hmin:
                up.append(len(P))
            elif place == lo:
                low.append(len(P))
            if place == np.float32(1.6):
                p[(axis + 1) % 3] += np.float32(1.0)
            x, y, z = np.floor(p + 0.5).astype(int)
            h[z, y, x] = size
            P.append(p)
    nodes = nodes_at(grid, P)
    nodes.lab[:] = 1
    want = orc.rebuild(grid, nodes, prm)
    for i, j in zip(low, up):   # a bar by its length, and not in the list
        assert j not in want["nbr"].reshape(-1, 24)[i][: want["nnb"][i]]
        assert i in want["nbr"].reshape(-1, 24)[j][: want["nnb"][j]]
    same_lists(tn, grid, nodes, prm)


@pytest.mark.parametrize("power", [-62, -40, 40, 49, 54])
@pytest.mark.parametrize("per", [20, 100])
def test_any_unit_of_length(tn, power, per):
    """Lengths scaled by a power of two: the same lists, down to squares near the smallest
    normal number and up to squares near the largest; 20 nodes a place fill no buffer, 100 do"""
    u = np.float32(2.0 ** power)
    base = Fixture("jitter64").grid
    grid = dataclasses.replace(base, vs=tuple(float(u * v) for v in base.vs), h=base.h * u, hmin=float(u * np.float32(base.hmin)),
                               hmax=float(u * np.float32(base.hmax)))
    rng = np.random.default_rng(per)
    P = np.concatenate([np.repeat(rng.uniform(8, 14, (7, 3)), per, 0), rng.uniform(6, 20, (333, 3)), rng.uniform(40, 50, (5, 3))])
    nodes = nodes_at(base, P[rng.permutation(len(P))])
    nodes.P *= u
    assert same_lists(tn, grid, nodes).max() == 24


@pytest.mark.parametrize("counts", [(127, 128, 129), (255, 1, 256), (383, 384, 385), (640, 641), (2000, 3000, 700)])
@pytest.mark.parametrize("ahead", [0, 1, 200])
def test_cells_longer_than_a_block(tn, counts, ahead):
    """Cells of so many nodes that renumbering reads them past a block's window, to one side or
    both, in a row and from any place in a block (`ahead` nodes in cells before them)"""
    grid = Fixture("jitter64").grid
    b = float(np.float32(1.6) * np.float32(grid.hmin))
    rng = np.random.default_rng(sum(counts) + ahead)
    cell = [rng.uniform(0.02, 0.98, (c, 3)) * b + [(4 + k) * b - 0.5, 6 * b - 0.5, 6 * b - 0.5] for k, c in enumerate(counts)]
    P = np.concatenate([rng.uniform(0.5, 2 * b, (ahead, 3)), *cell])
    same_lists(tn, grid, nodes_at(grid, P[rng.permutation(len(P))]))


def test_renumbering_a_long_cell_costs_less_than_its_search(tn):
    """100 k nodes in a few cells: both grow with the square of a cell's nodes, the search with
    by far the larger factor"""
    grid = Fixture("jitter64").grid
    P = 30.0 + 4.0 * np.random.default_rng(1).uniform(0, 1, (100000, 3))
    with tn.Plan(grid, nodes_at(grid, P), RelaxParams(max_iters=0)) as plan:
        plan.set_timing(True)
        plan.run()
        ms = {k: v[1] for k, v in plan.timings().items()}
    assert ms["permute"] < 0.2 * ms["neighbors"], ms
