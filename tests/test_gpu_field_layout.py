"""The label fields' device layout (9^3 corner values a slot, a record a brick) against
the oracle, which reads the stored layout voxel by voxel: every query the same bits at
points in brick interiors, on brick faces and edges, at the grid's sides and outside it,
for labels the cell's brick lists and labels it does not.
"""
import dataclasses

import numpy as np
import pytest

from conftest import Fixture, bits
from trussnet_amd._abi import Nodes, RelaxParams

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tn():
    from trussnet_amd import relax

    if relax.device_count() < 1:
        pytest.fail("no HIP device visible")
    return relax


def _points(shape, vs, seed):
    """Uniform points reaching out of the grid, and points whose coordinates sit at and
    beside brick faces (voxels 8 k - 1 .. 8 k + 1, half voxels between)."""
    rng = np.random.default_rng(seed)
    n = np.array(shape[::-1])
    free = rng.uniform(-2.5, n + 1.5, (6000, 3))
    near = 8 * rng.integers(0, np.maximum(2, n // 8 + 1), (6000, 3)) + rng.choice(
        [-1.5, -1.0, -0.75, -0.5, -0.25, 0.0, 0.3, 0.5, 1.0], (6000, 3))
    ends = rng.choice([-1.0, -0.5, 0.0, 1.0], (500, 3)) + rng.integers(0, 2, (500, 3)) * (n - 1)
    return (np.concatenate([free, near, ends]) * np.array(vs)).astype(np.float32)


@pytest.mark.parametrize("shape,vs,blocks,nlab", [
    ((24, 16, 32), (1.0, 1.0, 1.0), 6, 3),      # whole bricks
    ((17, 9, 25), (0.9, 1.1, 1.3), 5, 4),       # one voxel over a brick along each axis
    ((7, 8, 15), (2.0, 0.5, 1.0), 3, 5),        # less than a brick
    ((1, 1, 1), (1.0, 1.0, 1.0), 1, 2),
    ((20, 23, 31), (1.0, 1.0, 1.0), 2, 60),     # more labels near a brick than it lists
])
def test_queries_equal_the_oracle(tn, oracle_lib, shape, vs, blocks, nlab):
    from trussnet_amd import gridbuild

    rng = np.random.default_rng(7)
    cells = [(s + blocks - 1) // blocks for s in shape]
    lab = rng.integers(0, nlab, cells).astype(np.uint16)
    for ax in range(3):
        lab = np.repeat(lab, blocks, axis=ax)
    lab = np.ascontiguousarray(lab[:shape[0], :shape[1], :shape[2]])
    grid = gridbuild.build(lab, vs, device=0)
    X = _points(shape, vs, 3)
    one = Nodes(np.zeros((1, 3)), np.zeros(1), np.zeros(1), np.full((1, 2), 0xFFFF))
    with tn.Plan(grid, one, RelaxParams()) as plan:
        for a, b in ((0, 1), (1, 2), (nlab - 1, 0), (nlab + 5, 1), (0xFFFE, 0)):
            got = plan.field_points(a, b, X)
            want = oracle_lib.field_points(grid, a, b, X)
            for g, w, name in zip(got, want, ("phi", "psi", "grad", "label", "second")):
                assert np.array_equal(bits(g), bits(w)), (shape, a, b, name)


@pytest.mark.parametrize("name,voxel", [("sectors48", False), ("sectors48", True), ("aniso40", False), ("aniso40", True),
                                        ("gray40", False), ("tpm32", False)])
def test_points_far_out(tn, oracle_lib, name, voxel):
    """Points whose voxel coordinates leave the range of an integer along any of the axes, as a
    corner's Newton steps can: outside the grid, in the slots and in the stored layout (which a
    voxel-trap plan reads)"""
    case = Fixture(name)
    grid = case.grid
    rng = np.random.default_rng(2)
    near = rng.uniform(0, 1, (4000, 3)) * np.array([grid.nx, grid.ny, grid.nz]) * np.array(grid.vs)
    far = rng.choice([2.0 ** 31, 2.0 ** 31 - 128, 2.0 ** 32, 1e10, 1e20, -2.0 ** 31, -1e10, -1e20], (4000, 3)) * rng.choice([1.0, 1.5], (4000, 3))
    X = np.where(rng.random((4000, 3)) < 0.6, far, near).astype(np.float32)
    with tn.Plan(grid, case.seeds, RelaxParams(voxel_trap=voxel)) as plan:
        for a, b in ((0, 1), (1, 0), (1, 2)):
            for g, w, what in zip(plan.field_points(a, b, X), oracle_lib.field_points(grid, a, b, X),
                                  ("phi", "psi", "grad", "label", "second")):
                assert np.array_equal(g, w), (a, b, what)


@pytest.mark.parametrize("name", ["sectors48", "ellipsoids56"])
def test_bricks_that_share_slots(tn, oracle_lib, name):
    """A grid whose bricks of the same labels refer to one brick's slots: the values beyond a
    slot's upper faces are each brick's own, so such a grid is read as stored. The same nodes
    as of the grid that holds the shared values once for every brick."""
    case = Fixture(name)
    grid = case.grid
    slot, phi, first = grid.bl_slot.copy(), grid.phi.reshape(-1, 512).copy(), {}
    lab = grid.bl_lab.reshape(-1, 16)
    for b in np.flatnonzero(slot >= 0):
        n = int(grid.bl_cnt[b])
        a = first.setdefault(tuple(lab[b, :n].tolist()), b)
        phi[grid.bl_slot[b]:grid.bl_slot[b] + n] = phi[grid.bl_slot[a]:grid.bl_slot[a] + n]
        slot[b] = grid.bl_slot[a]
    assert (slot != grid.bl_slot).sum() > 10
    shared, own = dataclasses.replace(grid, bl_slot=slot), dataclasses.replace(grid, phi=phi.ravel())
    X = _points((grid.nz, grid.ny, grid.nx), grid.vs, 3)
    with tn.Plan(shared, case.seeds, RelaxParams()) as plan:
        for a, b in ((0, 1), (1, 2)):
            for g, w in zip(plan.field_points(a, b, X), oracle_lib.field_points(shared, a, b, X)):
                assert np.array_equal(bits(g), bits(w))
    prm = RelaxParams(max_iters=30, dptol=0.0)
    want = oracle_lib.relax(shared, case.seeds, prm)[0]
    for g in (shared, own):
        assert tn.relax(g, case.seeds, prm, device=0)[0].equal(want)
    assert tn.seed(shared, prm, device=0).equal(tn.seed(own, prm, device=0))


def test_stored_layout_where_the_slots_do_not_fit(tn):
    """A relaxation that just fits the no-allocation entry point's memory has no room left
    for the slots and reads the stored layout: the same bits."""
    case = Fixture("spheres64")
    s = case.seeds
    reps = 90
    P, lab, typ, part = np.tile(s.P, (reps, 1)), np.tile(s.lab, reps), np.tile(s.typ, reps), np.tile(s.part, (reps, 1))
    prm = RelaxParams(max_iters=3, dptol=0.0)

    def run(n):
        try:
            return tn.relax_noalloc(case.grid, Nodes(P[:n], lab[:n], typ[:n], part[:n]), prm, device=0)
        except tn.DeviceError:
            return None

    lo, hi = 1000, s.n * reps
    assert run(hi) is None
    while hi - lo > 500:   # the largest count that fits, to 0.25 MB
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if run(mid) is not None else (lo, mid)
    # 500 nodes more were refused: less is left than these take (328 bytes each, about 50 buffers
    # in steps of 256), and the slots take more than that
    assert 4 * 736 * case.grid.nslot > 500 * 400 + 50 * 256
    got, _ = run(lo)
    want, _ = tn.relax(case.grid, Nodes(P[:lo], lab[:lo], typ[:lo], part[:lo]), prm, device=0)
    assert got.equal(want)


@pytest.mark.parametrize("shape,nlab,blocks,vs,seed", [
    ((23, 27, 45), 3, 2, (0.976, 0.993, 1.223), 1168), ((15, 36, 21), 3, 2, (0.596, 1.492, 1.432), 1173)])
def test_corner_steps_that_run_away(tn, shape, nlab, blocks, vs, seed):
    """Volumes of small blocks, among whose corners are some with nearly dependent gradients:
    their Newton steps go 3e9 and 8e9 voxels out (with the voxel sizes' further digits) and are
    then dropped for the vertex itself"""
    from trussnet_amd import gridbuild
    from trussnet_amd._abi import GridParams

    rng = np.random.default_rng(seed)
    assert shape == tuple(int(v) for v in rng.integers(5, 56, 3))
    assert nlab == int(rng.integers(1, 6)) and blocks == int(rng.choice([2, 3, 5, 9, 16]))
    lab = rng.integers(0, nlab + 1, [(s + blocks - 1) // blocks for s in shape]).astype(np.uint16)
    for ax in range(3):
        lab = np.repeat(lab, blocks, axis=ax)
    lab = np.ascontiguousarray(lab[:shape[0], :shape[1], :shape[2]])
    rng.random()
    size = tuple(float(v) for v in rng.uniform(0.5, 2, 3))
    assert np.allclose(size, vs, atol=1e-3)
    h = float(rng.uniform(0.8, 2.5)) * min(size)
    grid = gridbuild.build(lab, size, GridParams(hbase=h, hmin=h, hmax=h), device=0)
    seeds = tn.seed(grid, RelaxParams(), device=0)
    corner = seeds.P[seeds.typ == 3] / np.array(size, np.float32)
    off = corner - (np.floor(corner) + 0.5)
    assert len(corner) > 100 and (off ** 2).sum(1).max() < 0.76 and ((off ** 2).sum(1) <= 0.2501).mean() > 0.9
    assert tn.seed(grid, RelaxParams(), device=0).equal(seeds)
