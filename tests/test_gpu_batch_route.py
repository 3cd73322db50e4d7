"""Which layout of the fields a batch's moves read (TN_BATCH_VERBOSE names it): the corner
slots where every volume that has nodes to move smoothly has them, whatever else is in the
batch; the stored layout beside a gray-scale volume. The nodes are the single runs' ones.
"""
import pytest

from conftest import Fixture
from trussnet_amd._abi import Nodes, RelaxParams

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tn():
    from trussnet_amd import relax

    if relax.device_count() < 1:
        pytest.fail("no HIP device visible")
    return relax


def part(case, n):
    s = case.seeds
    return Nodes(s.P[:n], s.lab[:n], s.typ[:n], s.part[:n])


@pytest.mark.parametrize("more,layout", [
    (None, "corner slots"),
    (("spheres64", 0, False), "corner slots"),     # no nodes
    (("gray40", 0, False), "corner slots"),        # no nodes of a gray-scale volume
    (("sectors48", 500, True), "corner slots"),    # the voxel trap's moves read the labels
    (("gray40", 500, False), "stored layout"),
])
def test_layout_of_a_batch(tn, monkeypatch, capfd, more, layout):
    names = [("spheres64", 800, False), ("jitter64", 300, False)] + ([more] if more else [])
    cases = [Fixture(n) for n, _, _ in names]
    nodes = [part(c, n) for c, (_, n, _) in zip(cases, names)]
    prms = [RelaxParams(max_iters=5, dptol=0.0, voxel_trap=v) for _, _, v in names]
    monkeypatch.setenv("TN_BATCH_VERBOSE", "1")
    out = tn.relax_batch([c.grid for c in cases], nodes, prms, device=0)
    assert f"moves over the {layout}\n" in capfd.readouterr().err
    for c, s, p, (got, _) in zip(cases, nodes, prms, out):
        assert got.equal(tn.relax(c.grid, s, p, device=0)[0])
