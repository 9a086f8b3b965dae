"""Mapped device arrays (gt_map_data): their owner writes the next frame into one
that was transformed, or takes its spectrum (gt_sync_ref) and writes to that."""
import numpy as np
import pytest
import torch  # first: the library then binds to torch's HIP runtime

from gturbo_amd.solver import Solver
from helpers import params_for

pytestmark = pytest.mark.gpu


def _frame(n, seed):
    w = np.zeros((n, n + 2))
    w[:, :n] = np.random.default_rng(seed).standard_normal((n, n)) * (4.0 / n)
    return w


@pytest.mark.parametrize("n", [16, 64, 2048, 4096])
def test_frames_written_one_after_the_other(oracle_mod, n):
    """A spectrum per frame, each frame put into the mapped array in place of
    the one before; then one transformed twice, whose second transform is that
    of its spectrum (1e-12 as for the other spectra)."""
    p = params_for(n)
    s, o = Solver(p), oracle_mod.Oracle(p)
    t = torch.zeros((n, n + 2), dtype=torch.float64, device="cuda")
    s.map_data(t)
    for seed, times in ((1, 1), (1, 1), (2, 2), (3, 1)):
        w = _frame(n, seed)
        t.copy_(torch.from_numpy(w))
        torch.cuda.synchronize()
        for _ in range(times):
            s.fft_dir(t)
            got = s.spectrum(t)
            o.fft_dir(w)
            for g, e in zip(got, o.spectrum(w)):
                assert np.max(np.abs(g - e)) <= 1e-12 * np.max(np.abs(e))
    s.close()


@pytest.mark.parametrize("written", [False, True])
def test_unmapped_after_fft_dir(oracle_mod, written):
    """The spectrum, or what its owner has put into the memory since."""
    n = 64
    p = params_for(n)
    s, o = Solver(p), oracle_mod.Oracle(p)
    w = _frame(n, 9)
    t = torch.from_numpy(w).cuda()
    torch.cuda.synchronize()
    s.map_data(t)
    s.fft_dir(t)
    s.synchronize()
    if written:
        t.fill_(2.5)
        torch.cuda.synchronize()
        w[:] = 2.5
    else:
        o.fft_dir(w)
    s.unmap_data(t)
    s.close()
    assert np.linalg.norm(t.cpu().numpy() - w) <= 1e-12 * np.linalg.norm(w)


@pytest.mark.parametrize("n", [64, 2048])
@pytest.mark.parametrize("then", ["step4", "fft_inv"])
def test_spectrum_written_by_its_owner(oracle_mod, n, then):
    """fft_dir, sync_ref, the spectrum scaled by its owner, then a step or the
    way back (1e-12 as for the other comparisons)."""
    p = params_for(n)
    s, o = Solver(p), oracle_mod.Oracle(p)
    w = _frame(n, 5)
    t = torch.from_numpy(w).cuda()
    a = [torch.zeros_like(t) for _ in range(4)]
    torch.cuda.synchronize()
    for x in (t, *a):
        s.map_data(x)
    s.fft_dir(t)
    s.sync_ref(t)
    t *= 0.5
    torch.cuda.synchronize()
    o.fft_dir(w)
    w *= 0.5
    if then == "step4":
        s.step4(t, *a)
        o.step4(w)
    else:
        s.fft_inv(t)
        o.fft_inv(w)
    s.sync_ref(t)
    got = t.cpu().numpy()
    assert np.linalg.norm(got - w) < 1e-12 * np.linalg.norm(w)
    s.close()
