"""Plans that follow each other on one device share streams, events, pinned blocks and
buffers that earlier ones left: their results stay their own, in turn, overlapping in
time and from several threads, and whatever was done with a plan before a run.
"""
import threading

import pytest

from conftest import Fixture

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tn():
    from trussnet_amd import relax

    if relax.device_count() < 1:
        pytest.fail("no HIP device visible")
    return relax


@pytest.mark.parametrize("before", ["nothing", "step", "rebuild", "force", "download", "run"])
def test_run_starts_from_the_seeds(tn, before):
    case = Fixture("sectors48")
    prm, want, stats = case.runs()[1]
    with tn.Plan(case.grid, case.seeds, prm) as plan:
        if before != "nothing":
            {"step": lambda: plan.step(3), "rebuild": plan.rebuild, "force": plan.force, "download": plan.download,
             "run": plan.run}[before]()
        st = plan.run()
        assert plan.download().equal(want)
        assert st["rebuilds"] == int(stats["rebuilds"]) and st["iters"] == int(stats["iters"])


def test_plans_from_several_threads(tn):
    cases = [Fixture(n) for n in ("sectors48", "jitter64", "aniso40", "gray40")]
    wrong = []

    def work(case):
        for _ in range(3):
            for prm, want, _ in case.runs()[:2]:
                got, _ = tn.relax(case.grid, case.seeds, prm)
                if not got.equal(want):
                    wrong.append(case.name)

    threads = [threading.Thread(target=work, args=(c,)) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_more_plans_alive_than_are_kept(tn):
    case = Fixture("jitter64")
    prm, want, _ = case.runs()[0]
    plans = [tn.Plan(case.grid, case.seeds, prm) for _ in range(40)]
    for p in plans[::3]:
        p.run()
        assert p.download().equal(want)
    for p in plans:
        p.close()
    got, _ = tn.relax(case.grid, case.seeds, prm)
    assert got.equal(want)
