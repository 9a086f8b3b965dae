"""Diagnostics of a field that has blown up."""
import numpy as np
import pytest

from gturbo_amd.solver import Solver
from helpers import params_for, random_spectral

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("part", [0, 1])
@pytest.mark.parametrize("n", [16, 256, 2048])
def test_infinite_mode_beside_a_nan(n, part):
    """One mode with an infinite and a NaN part: its modulus is infinite, and so
    are its shell and the sums over all modes; the other shells are untouched."""
    s = Solver(params_for(n, famp=0.0))
    z = random_spectral(n, 7)
    kx, ky = 3, 1
    with np.errstate(all="ignore"):
        b = z.copy()
        b[ky, 2 * kx + part], b[ky, 2 * kx + 1 - part] = -np.inf, np.nan
    for a in (z, b):
        s.enter_data(a)
    ib = s.shell_index()[ky, kx]
    for got, want in zip(s.spectrum(b), s.spectrum(z)):
        assert got[ib - 1] == np.inf
        keep = np.arange(n // 2) != ib - 1
        assert np.array_equal(got[keep], want[keep])
    assert np.all(s.glob(b)[:4] == np.inf)
    s.close()
