"""Single-run passes of the small grids (a column's or row's fields side by
side): line lengths below, at and above a wave, both ka sources, both
rectangles, and columns with more forced modes than a workgroup stages."""
import numpy as np
import pytest

from gturbo_amd.solver import Solver

from helpers import params_for, random_spectral

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _steps(oracle_mod, p, nsteps):
    s, o = Solver(p), oracle_mod.Oracle(p)
    z = random_spectral(p.n, 17 + p.n, truncated=p.truncate == 1)
    zg = z.copy()
    znl, znew, u, v = (s.field() for _ in range(4))
    s.enter_data(zg)
    for a in (znl, znew, u, v):
        s.enter_data(a, copyin=False)
    sg = so = 90017
    for _ in range(nsteps):
        if s.rko == 4:
            s.step4(zg, znl, znew, u, v)
            o.step4(z)
        else:
            s.step(zg, znl, u, v)
            o.step(z)
        sg, so = s.forcing(zg, sg), o.forcing(z, so)
    s.update_host(zg)
    s.close()
    assert sg == so
    return _rel(zg, z)


@pytest.mark.parametrize("n", [16, 32, 64, 128, 512, 1024])
@pytest.mark.parametrize("alpv,truncate", [(2.0, 1), (1.5, 1), (1.5, 0)])
def test_forced_steps(oracle_mod, n, alpv, truncate):
    """Step, forcing, step (fused boundary) three times.  The ring reaches
    from k = 1 to min(N/5, 34): at N >= 256 its middle columns hold up to 68
    modes.  Tolerance as for the other three-step comparisons (1e-12)."""
    p = params_for(n, alpv=alpv, truncate=truncate, rko=2 if n in (32, 512) else 4,
                   ring=(1.0, min(n / 5.0, 34.0)))
    assert _steps(oracle_mod, p, 3) < 1e-12


def test_forcing_phase_ring_wraps(oracle_mod):
    """150 forced steps: every slot of the phase ring is used again.  A step
    adds round-off of order 1e-16; 1e-12 over 150 steps."""
    assert _steps(oracle_mod, params_for(64), 150) < 1e-12
