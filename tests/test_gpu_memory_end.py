"""Where device memory ends (TN_MEM_LIMIT_MB stands in for a small device): the corner slots
that the queries can do without give way to what a call needs, so that a call that fits at
one limit fits at every larger one, and gives the same nodes with the slots and without.
"""
import numpy as np
import pytest

from trussnet_amd._abi import GridParams, RelaxParams

pytestmark = pytest.mark.gpu

STEP = 4   # MiB between the limits tried


@pytest.fixture(scope="module")
def tn():
    from trussnet_amd import relax

    if relax.device_count() < 1:
        pytest.fail("no HIP device visible")
    return relax


@pytest.fixture(scope="module")
def volume():
    """A grid of many labels a brick: its slots take more than everything else of a seeding"""
    from trussnet_amd import gridbuild

    lab = np.random.default_rng(5).integers(1, 40, (30, 30, 30)).astype(np.uint16)
    for ax in range(3):
        lab = np.repeat(lab, 4, axis=ax)
    grid = gridbuild.build(lab, prm=GridParams(hbase=5.0, hmin=5.0, hmax=5.0), device=0)
    assert grid.nslot * 736 * 4 > 100 << 20
    return grid


def smallest_limit(tn, monkeypatch, call, same, beyond):
    """The smallest limit (MiB) that call() runs at; it runs at all tried from there on, to
    `beyond` above it, and gives the same"""
    monkeypatch.delenv("TN_MEM_LIMIT_MB", raising=False)
    want, fits, limit = call(), {}, 0
    while not any(fits.values()) or limit < min(k for k in fits if fits[k]) + beyond:
        limit += STEP
        monkeypatch.setenv("TN_MEM_LIMIT_MB", "1")   # (the buffers kept from the call before, given back)
        with pytest.raises(tn.DeviceError):
            call()
        monkeypatch.setenv("TN_MEM_LIMIT_MB", str(limit))
        try:
            assert same(call(), want), limit
            fits[limit] = True
        except tn.DeviceError as e:
            assert e.code == 3 and "memory" in str(e), e
            fits[limit] = False
        assert limit < 4096
    first = min(k for k in fits if fits[k])
    print(f"[memory] from {first} MiB on; refused above it: {[k for k in fits if k > first and not fits[k]]}", flush=True)
    assert not fits[STEP] and all(fits[k] for k in fits if k >= first)
    return first


def test_seeding(tn, monkeypatch, volume):
    smallest_limit(tn, monkeypatch, lambda: tn.seed(volume, RelaxParams(), device=0), lambda a, b: a.equal(b), 300)


def test_plan(tn, monkeypatch, volume):
    seeds, prm = tn.seed(volume, RelaxParams(), device=0), RelaxParams(max_iters=3, dptol=0.0)
    smallest_limit(tn, monkeypatch, lambda: tn.relax(volume, seeds, prm, device=0)[0], lambda a, b: a.equal(b), 300)


def test_batch(tn, monkeypatch, volume):
    """Three volumes take no more than three times what one takes alone, and the batch's tables"""
    seeds, prm = tn.seed(volume, RelaxParams(), device=0), RelaxParams(max_iters=3, dptol=0.0)

    def batch(count):
        return [x for x, _ in tn.relax_batch([volume] * count, [seeds] * count, [prm] * count, device=0)]

    def same(a, b):
        return all(x.equal(y) for x, y in zip(a, b))

    one = smallest_limit(tn, monkeypatch, lambda: batch(1), same, 40)
    three = smallest_limit(tn, monkeypatch, lambda: batch(3), same, 600)
    assert three <= 3 * one + STEP
