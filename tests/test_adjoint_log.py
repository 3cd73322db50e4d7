"""The adjoint's logarithm log(1 + x) on [0, 1], its coefficients as the source holds them:
the largest relative error of the polynomial itself, and of the 32-bit evaluation in units
in the last place, which the source states."""
import os
import re

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def coefficients():
    """From the lowest order on"""
    with open(os.path.join(ROOT, "trussnet_amd", "csrc", "tn_adjoint.hpp")) as f:
        body = f.read().split("float log1p_unit(float x) {")[1].split("\n}")[0]
    return [float.fromhex(h) for h in re.findall(r"(-?0x[0-9a-f.]+p[-+]?\d+)f", body)][::-1]


def test_polynomial():
    c = coefficients()
    assert len(c) == 10 and all(float(np.float32(v)) == v for v in c)
    x = np.unique(np.concatenate([0.5 + 0.5 * np.cos(np.linspace(0, np.pi, 20001)), np.logspace(-6, 0, 4000)]))
    x = x[x > 1e-7].astype(np.longdouble)
    p = np.zeros_like(x)
    for v in reversed(c):
        p = p * x + np.longdouble(v)
    assert np.max(np.abs((x + x * x * p) / np.log1p(x) - 1)) < 1.3e-9


def test_as_computed():
    def fma(a, b, c):   # (a product of 32-bit values is exact in 64 bits)
        return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(np.float32)

    x = np.unique(np.concatenate([np.linspace(0, 1, 200001), np.logspace(-30, 0, 50001)]).astype(np.float32))
    x = x[x > 0]
    c = coefficients()
    p = np.full(x.shape, np.float32(c[-1]))
    for v in c[-2::-1]:
        p = fma(p, x, np.full(x.shape, np.float32(v)))
    y = fma((p * x).astype(np.float32), x, x)
    want = np.log1p(x.astype(np.longdouble))
    off = np.abs((y.astype(np.longdouble) - want) / np.spacing(want.astype(np.float32)).astype(np.longdouble))
    assert off.max() < 1.2 and off.mean() < 0.225, (float(off.max()), float(off.mean()))
