"""The list of nodes past a full skin, which the statistics kernel gathers block by block:
with a skin near zero almost every node is on it at every iteration, and with few blocks
(TN_STATS_BLOCKS) each walks so many chunks of 256 nodes that it writes its list out more
than once on the way (as blocks do by themselves from 4.2 M nodes on). Node counts on and
beside the chunks at which it does. Against the oracle: the number listed, the nodes and
the statistics, bit for bit.
"""
import numpy as np
import pytest

from conftest import Fixture
from trussnet_amd._abi import Nodes, RelaxParams

pytestmark = pytest.mark.gpu

STAT_KEYS = ["iters", "rebuilds", "last_move", "last_p99", "fire_resets", "fire_dt", "n_interior", "n_interface",
             "n_junction", "n_corner"]
ITERS = 8


@pytest.fixture(scope="module")
def tn():
    from trussnet_amd import relax

    if relax.device_count() < 1:
        pytest.fail("no HIP device visible")
    return relax


def first(nodes, n):
    return Nodes(nodes.P[:n], nodes.lab[:n], nodes.typ[:n], nodes.part[:n])


def params(fire, skin):
    return RelaxParams(max_iters=ITERS, dptol=0.0, fire=fire, skin=skin)


def same(got, st, want, sw):
    assert got.equal(want), int((got.P != want.P).any(axis=1).sum())
    for k in STAT_KEYS:
        assert np.float32(st[k]) == np.float32(sw[k]), (k, st[k], sw[k])


@pytest.mark.parametrize("fire", [True, False])
@pytest.mark.parametrize("skin", [0.0, 1e-3])
@pytest.mark.parametrize("blocks,n", [(1, 255), (1, 2047), (1, 2048), (1, 2049), (1, 2304), (1, 4096), (1, 4097),
                                      (2, 4096), (2, 4100), (3, 9000), (3, 50000)])
def test_listed_over_many_chunks(tn, oracle_lib, monkeypatch, blocks, n, skin, fire):
    monkeypatch.setenv("TN_STATS_BLOCKS", str(blocks))
    case = Fixture("ellipsoids56")
    seeds = case.seeds
    if n > seeds.n:   # more of them, each a little off its first
        P = np.concatenate([seeds.P + np.float32(0.01 * k) for k in range(-(-n // seeds.n))])
        reps = len(P) // seeds.n
        seeds = Nodes(P, np.tile(seeds.lab, reps), np.tile(seeds.typ, reps), np.tile(seeds.part, (reps, 1)))
    seeds, prm = first(seeds, n), params(fire, skin)
    want, sw, trace = oracle_lib.relax(case.grid, seeds, prm, trace=True)
    listed = sum(t["nrefresh"] for t in trace if not t["rebuilt"])
    assert listed > (0.3 if skin == 0.0 else 0.1) * n * ITERS   # most of them, time and again
    with tn.Plan(case.grid, seeds, prm) as plan:
        plan.set_timing(("refresh",))
        st = plan.run()
        got = plan.download()
        items = plan.timings()["refresh"][2]
    same(got, st, want, sw)
    assert items == listed


def test_listed_in_a_batch(tn, oracle_lib, monkeypatch):
    monkeypatch.setenv("TN_STATS_BLOCKS", "1")
    cases = [Fixture("ellipsoids56"), Fixture("spheres64"), Fixture("sectors48")]
    grids, nodes, prms = [c.grid for c in cases], [c.seeds for c in cases], [params(k != 1, 0.0) for k in range(3)]
    assert max(s.n for s in nodes) > 2048
    for g, s, p, (got, st) in zip(grids, nodes, prms, tn.relax_batch(grids, nodes, prms, device=0)):
        same(got, st, *oracle_lib.relax(g, s, p))
