"""The broadphase's integer grids (host build): quantised boxes against the double-precision ones."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def grids(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("grids") / "grids_harness.so")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-fno-fast-math", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas",
                    "-o", out, os.path.join(ROOT, "tests", "native", "grids_harness.cpp")], check=True)
    return ctypes.CDLL(out)


SPREADS = {
    "plain": lambda rng, n: rng.normal(size=n),
    "fine": lambda rng, n: rng.integers(0, 65536, size=n) / 65535.0,
    "flat": lambda rng, n: np.zeros(n),
    "flat_nonfinite": lambda rng, n: rng.choice([0.0, 0.0, np.inf, -np.inf, np.nan], size=n),
    "nonfinite": lambda rng, n: rng.choice([0.0, 0.3, 1.0, np.inf, -np.inf, np.nan], size=n),
    "huge": lambda rng, n: rng.choice([-1.7e308, -1e308, 0.0, 0.5e308, 1.2e308, 1.7e308], size=n),
    "huge_nonfinite": lambda rng, n: rng.choice([-1.7e308, 1.0, 1.2e308, 1.7e308, np.inf, -np.inf, np.nan], size=n),
    "tiny": lambda rng, n: rng.choice([0.0, 5e-324, 1e-320, 1e-310, 1e-300], size=n),
}


@pytest.mark.parametrize("name", sorted(SPREADS))
@pytest.mark.parametrize("order", ["bounds", "any"])
def test_quantised_boxes(grids, name, order):
    """Boxes that overlap still do when quantised; boxes two quanta into each other overlap."""
    rng = np.random.default_rng(len(name))
    n = 400
    a, b = SPREADS[name](rng, n), SPREADS[name](rng, n)
    lo, hi = (np.fmin(a, b), np.fmax(a, b)) if order == "bounds" else (a, b)
    qlo, qhi = np.zeros(n, np.uint16), np.zeros(n, np.uint16)
    p = lambda x: x.ctypes.data_as(ctypes.c_void_p)   # noqa: E731
    grids.quantise_axis(p(lo), p(hi), ctypes.c_int64(n), p(qlo), p(qhi))
    reaches = ~(hi[:, None] < lo[None, :])   # (a NaN separates nothing)
    ql, qh = qlo.astype(int), qhi.astype(int)
    assert (qh[:, None] >= ql[None, :])[reaches].all()
    sure = np.array([[grids.surely_reaches(int(h), int(l)) for l in np.unique(ql)] for h in np.unique(qh)], bool)
    sure = sure[np.searchsorted(np.unique(qh), qh)][:, np.searchsorted(np.unique(ql), ql)]
    assert reaches[sure].all()


def test_cell_bits(grids):
    """Enough for every cell coordinate and the one after it, and no more; an extent that is no number ends too."""
    f = grids.cell_bits
    f.argtypes = [ctypes.c_double, ctypes.c_double]
    rng = np.random.default_rng(0)
    for n in [1, 2, 3, 4, 7, 8, 9, 1023, 1024, 2**20 - 1, 2**20] + rng.integers(1, 2**20, size=50).tolist():
        for extent, inv in ((float(n), 1.0), (float(n) * 0.37, 1.0 / 0.37), (n - 1e-9, 1.0)):
            assert f(extent, inv) == (int(extent * inv) + 1).bit_length()
    for extent in (0.0, float("nan"), -1.0, 5e-324):
        assert f(extent, 10.0) == 1
    assert f(float("inf"), 1.0) == f(1e300, 1e10) == 21
