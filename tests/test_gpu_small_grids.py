"""Single-run passes of the small grids (a column's or row's fields side by
side): line lengths below, at and above a wave, both ka sources, both
rectangles, and columns with more forced modes than a workgroup stages."""
import numpy as np
import pytest

from gturbo_amd import ic
from gturbo_amd.adjoint import Adjoint
from gturbo_amd.ensemble import SPECTRAL, Ensemble, solo_run
from gturbo_amd.params import InitialSpectrum
from gturbo_amd.solver import Solver
from helpers import params_for, random_spectral
from test_gpu_adjoint import _tlm

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


@pytest.mark.parametrize("n", [16, 128, 2048])
def test_consumers_of_fft_dir(oracle_mod, n):
    """fft_dir leaves its spectrum on the whole half-spectrum: trunc of it, a
    step of it without trunc (modes outside the 2/3 rectangle), the same of a
    copy, fft_inv of each, and trunc of an array that was transformed before
    it served as the accumulator.  1e-12 as for the other comparisons."""
    p = params_for(n)
    s, o = Solver(p), oracle_mod.Oracle(p)
    rng = np.random.default_rng(n)
    w = np.zeros((n, n + 2))
    w[:, :n] = rng.standard_normal((n, n)) * (4.0 / n)
    a, b, c = w.copy(), w.copy(), w.copy()
    ag, bg, cg = w.copy(), s.field(), w.copy()
    znl, u, v = (s.field() for _ in range(3))
    for x in (ag, bg, cg, znl, u, v):
        s.enter_data(x)

    def same(xg, x):
        s.update_host(xg)
        assert _rel(xg, x) < 1e-12

    for x in (a, b, c):
        o.fft_dir(x)
    s.fft_dir(ag)
    s.copy(bg, ag)
    s.trunc(ag)
    o.trunc(a)
    s.fft_dir(cg)
    s.step4(bg, znl, cg, u, v)  # cg: accumulator from here on
    o.step4(b)
    same(ag, a)
    same(bg, b)
    s.step4(ag, znl, cg, u, v)
    o.step4(a)
    s.synchronize()
    s.trunc(cg)
    s.update_host(cg)
    assert cg[0, 0] == 0.0 and cg[0, 1] == 0.0
    kc = s.rect[0]
    assert not np.any(np.ascontiguousarray(cg).view(np.complex128)[:, kc + 1:])
    for xg, x in ((ag, a), (bg, b)):
        s.fft_inv(xg)
        o.fft_inv(x)
        same(xg, x)
    s.close()


@pytest.mark.parametrize("n,alpv,rko,nsteps,kchk", [
    (16, 2.0, 4, 5, 2), (32, 1.5, 2, 6, 4), (512, 1.5, 4, 3, 2), (1024, 2.0, 4, 3, 3)])
def test_adjoint_dot_product(oracle_mod, n, alpv, rko, nsteps, kchk):
    """Adjoint passes at the ends of their sizes, with a partial last segment
    (5 = 2 + 2 + 1): <gT, M' dw0> = <M'^T gT, dw0> as in test_gpu_adjoint."""
    p = params_for(n, alpv=alpv, rko=rko, famp=1.0)
    rng = np.random.default_rng(n + nsteps)
    w0 = ic.physical_field(p, InitialSpectrum(seed=11, p=4.0, k0=max(n / 16.0, 2.0), energy=0.5))
    dw0, gT = rng.standard_normal((n, n)), rng.standard_normal((n, n))
    o = oracle_mod.Oracle(p)
    wT_o, dwT = _tlm(o, w0.astype(np.float64), dw0, nsteps, 481929)
    with Adjoint(p, nsteps, kchk) as adj:
        wT, _ = adj.forward(w0.astype(np.float64), 481929)
        g0 = adj.backward(gT)
    assert _rel(wT, wT_o) < 1e-11
    lhs, rhs = float(np.sum(gT * dwT)), float(np.sum(g0 * dw0))
    assert abs(lhs - rhs) <= 1e-10 * abs(lhs)


@pytest.mark.parametrize("n,truncate,lx", [(32, 1, 1), (64, 0, 2), (2048, 1, 1), (8192, 0, 1)])
def test_shell_sums(n, truncate, lx):
    """Spectrum and fluxes of a random spectrum against numpy: runs of shells
    across chunks and waves, several columns per shell, the most LDS bins
    (8192 untruncated).  Sums of up to 1e5 terms a shell: 1e-12 of each sum's
    absolute terms."""
    p = params_for(n, truncate=truncate, xlx=2 * np.pi * lx, ring=(3.0, 5.0))
    s = Solver(p)
    nh, nb = n // 2 + 1, n // 2
    z, q = (random_spectral(n, k, truncated=bool(truncate)) for k in (1, 2))
    s.enter_data(z)
    s.enter_data(q)
    sp, sz = s.spectrum(z)
    fle, flz = s.fluxes(z, q)
    ib = s.shell_index()
    s.close()
    zc, qc = (np.ascontiguousarray(a).view(np.complex128).reshape(n, nh) for a in (z, q))
    kx = np.arange(nh) * s.dkx
    ky = np.where(np.arange(n) <= n // 2, np.arange(n), np.arange(n) - n) * s.dky
    k2 = kx[None, :] ** 2 + ky[:, None] ** 2
    k2[0, 0] = 1.0
    ok = (ib < nb) & (ib > 0)
    fac = np.ones((1, nh))
    fac[0, 0] = fac[0, -1] = 0.5

    def bins(v):
        return np.bincount(ib[ok] - 1, weights=v[ok], minlength=nb)

    a2 = fac * np.abs(zc) ** 2
    fz = 2 * fac * (zc.real * qc.real + zc.imag * qc.imag)
    for got, v in ((sp, a2 / k2 / s.dkx), (sz, a2 / s.dkx)):
        assert np.all(np.abs(got - bins(v)) <= 1e-12 * bins(np.abs(v)))
    for got, v in ((fle, fz / k2), (flz, fz)):
        assert np.max(np.abs(got - np.cumsum(bins(v)[::-1])[::-1])) <= 1e-12 * np.abs(v[ok]).sum()


@pytest.mark.parametrize("n,alpv,truncate", [(2048, 2.0, 1), (2048, 1.5, 0), (2048, 1.5, 1),
                                             (4096, 1.5, 1)])
def test_forced_steps_large(oracle_mod, n, alpv, truncate):
    """The in-place y passes and the ka table at 2048 and 4096: two forced RK4
    steps with the fused boundary between them (1e-12 as above)."""
    p = params_for(n, alpv=alpv, truncate=truncate, ring=(10.0, 20.0))
    assert _steps(oracle_mod, p, 2) < 1e-12


@pytest.mark.parametrize("sizes", [(128, 512, 1024), (256,), (256, 2048)])
def test_default_ensemble_schedule_matches_solo_runs(sizes):
    """The schedule an ensemble starts with (256-thread y passes up to N =
    1024, 512 with a member of 2048) keeps every member's arithmetic."""
    ps = [params_for(n, alpv=(0.5, 1.0, 2.0)[m % 3], ring=(n / 8 - 1.0, n / 8 + 1.0))
          for m, n in enumerate(sizes)]
    fields = [ic.physical_field(p, InitialSpectrum(seed=70 + p.n, p=4.0, k0=p.n / 16.0,
                                                   energy=0.5)) for p in ps]
    ens = Ensemble(ps, seeds=[5 + m for m in range(len(ps))])
    for m, w in enumerate(fields):
        ens.set_field(m, w)
    ens.run(11)
    ens.synchronize()
    for m, (p, w) in enumerate(zip(ps, fields)):
        z, seed = solo_run(p, w, 5 + m, 11)
        assert ens.get_seed(m) == seed
        assert np.array_equal(ens.get_field(m, SPECTRAL), z), p.n
    ens.close()
