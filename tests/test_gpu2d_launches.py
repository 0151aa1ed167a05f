"""The 2D stepper's launches at the sizes where their work lists end: the
DFT fold's frequency chunks and cell chunks, against the oracle."""
import numpy as np
import pytest

from conftest import check, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("polarization", ["tez", "tmz"])
@pytest.mark.parametrize("nx,nfreq", [(64, 1), (255, 8), (257, 9), (96, 33)])
def test_fold_chunks(polarization, nx, nfreq):
    """Spectra of a line for nfreq frequencies over nx cells: chunks of 8
    frequencies and 256 cells, full and partial, a partial block of steps at
    the end (FP64, the parity bar)."""
    import oracle
    from fdtd_amd import sim2d

    spec = sim2d.sweep_instance(np.random.default_rng(nx), side=96, nsteps=101, nfreq=nfreq, polarization=polarization)
    spec["grid"]["nx"] = nx
    gs, gi, _ = sim2d.make_simulation2d(spec, precision="fp64")
    os_, oi, _ = oracle.make_simulation2d(spec)
    gs.step(101)
    os_.step(101)
    comps = (sim2d.EZ2, sim2d.HX2) if polarization == "tmz" else (sim2d.EX2, sim2d.HZ2)
    for c in comps:
        for a, b in zip(gs.dft(gi[0], c), os_.dft(oi[0], c)):
            check(f"fold {polarization} {nx} {nfreq} {c}", relerr(a, b), 1e-12)
    gs.close()
    os_.close()
