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


@pytest.mark.parametrize("polarization", ["tez", "tmz"])
@pytest.mark.parametrize("tfsf", [False, True])
def test_dispersive_cells_and_monitors_on_shared_rows(polarization, tfsf):
    """Gold cells on the line source's row, on a TFSF row and on the
    monitors' rows, monitors on the first and last rows of tiles and of
    wavefront strips, probes at tile corners and in gold: the rows where the
    E launch's dispersive cells and the H launch's samples take part (FP64
    against the oracle, the parity bar)."""
    import oracle
    from fdtd_amd import sim2d

    spec = sim2d.sweep_instance(np.random.default_rng(7), side=130, nsteps=150, npml=8, polarization=polarization)
    nx, ny = 130, 130
    om = spec["dft"][0]["omega"][:6]
    spec["materials"] = [spec["materials"][0],
                         {"type": "drude2cp", "region": sim2d.box2((1, 20), (70, 40))},
                         {"type": "drude2cp", "region": sim2d.box2((60, 60), (nx, 66))}]
    spec["sources"][0]["j"] = 24
    spec["dft"] = [{"j": j, "omega": om} for j in (16, 33, 64, 9)]
    spec["probes"] = [[1, 16], [64, 17], [65, 33], [nx, 64], [65, 62], [5, 30]]
    if tfsf:
        pul = {k: spec["sources"][0][k] for k in ("t0", "st", "w0")}
        spec["tfsf"] = [dict(lo=28, hi=90, src_index=20, npml=8, **pul)]
    gs, gi, gp = sim2d.make_simulation2d(spec, precision="fp64")
    os_, oi, op = oracle.make_simulation2d(spec)
    for n in (1, 32, 117):
        gs.step(n)
        os_.step(n)
    comps = (sim2d.EZ2, sim2d.HX2, sim2d.HY2, sim2d.DZ2) if polarization == "tmz" else \
        (sim2d.EX2, sim2d.EY2, sim2d.HZ2, sim2d.DX2, sim2d.DY2)
    for c in comps:
        check(f"rows {polarization} {tfsf} {c}", relerr(gs.field(c), os_.field(c)), 1e-12)
    for a, b in zip(gi, oi):
        for c in comps[:1] + ((sim2d.HX2,) if polarization == "tmz" else (sim2d.HZ2,)):
            for x, y in zip(gs.dft(a, c), os_.dft(b, c)):
                check(f"rows dft {polarization} {tfsf} {c}", relerr(x, y), 1e-12)
    for a, b in zip(gp, op):
        check(f"rows probe {polarization} {tfsf}", relerr(gs.probe(a), os_.probe(b)), 1e-12)
    gs.close()
    os_.close()


@pytest.mark.parametrize("polarization", ["tez", "tmz"])
@pytest.mark.parametrize("nx,nfreq", [(96, 1), (511, 3), (512, 70), (513, 2), (1030, 5)])
def test_flux_is_the_sum_of_the_read_spectra(polarization, nx, nfreq):
    """A line's flux, bit for bit the products of its two spectra added cell
    after cell from zero in FP64: rows below, at and past the 512 cells a
    wavefront takes at a time."""
    from fdtd_amd import sim2d

    spec = sim2d.sweep_instance(np.random.default_rng(nx), side=96, nsteps=101, nfreq=nfreq, polarization=polarization)
    spec["grid"]["nx"] = nx
    s, ids, _ = sim2d.make_simulation2d(spec, precision="fp32")
    s.step(101)
    e, h, sign = (sim2d.EZ2, sim2d.HX2, 1.0) if polarization == "tmz" else (sim2d.EX2, sim2d.HZ2, -1.0)
    for a in ids:
        (er, ei), (hr, hi) = s.dft(a, e), s.dft(a, h)
        p = sign * ((hr * er + hi * ei) * spec["grid"]["ds"])
        want = np.cumsum(np.concatenate([np.zeros((1, nfreq)), p]), axis=0)[-1]
        assert np.any(want != 0)
        assert np.array_equal(s.flux(a), want)
    s.close()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("polarization", ["tez", "tmz"])
def test_marked_d(polarization, precision, monkeypatch):
    """The E launch with D marked nontemporal (what a batch past the
    memory-side cache runs; FDTD_NT forces a side): the same bits."""
    from fdtd_amd import sim2d

    spec = sim2d.sweep_instance(np.random.default_rng(4), side=130, nsteps=150, polarization=polarization)
    comps = (sim2d.EZ2, sim2d.HX2, sim2d.HY2, sim2d.DZ2) if polarization == "tmz" else \
        (sim2d.EX2, sim2d.EY2, sim2d.HZ2, sim2d.DX2, sim2d.DY2)
    got = []
    for nt in "01":
        monkeypatch.setenv("FDTD_NT", nt)
        s, ids, _ = sim2d.make_simulation2d(spec, precision=precision)
        s.step(150)
        got.append([s.field(c) for c in comps] + [s.flux(a) for a in ids])
        s.close()
    assert np.any(got[0][0] != 0)
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("polarization", ["tez", "tmz"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_monitors_of_one_strip(polarization, precision):
    """Four lines and eight probes on the rows of one wavefront strip (21-24
    of interior cells), the rows beside it and a row alone, lines of both
    components, of E and of H alone, with a gate: simulations in a batch and
    alone give the same bits, and hold the oracle's samples."""
    import oracle
    from fdtd_amd import sim2d

    tm = polarization == "tmz"
    spec = sim2d.sweep_instance(np.random.default_rng(3), side=96, nsteps=80, npml=8, polarization=polarization)
    spec["grid"]["nx"] = 150
    spec["materials"] = spec["materials"][:1]
    spec["sources"][0]["j"] = 18
    om = spec["dft"][0]["omega"][:9]
    e, h = (sim2d.DFT_EZ, sim2d.DFT_HX) if tm else (sim2d.DFT_EX, sim2d.DFT_HZ)
    spec["dft"] = [{"j": 21, "omega": om}, {"j": 22, "omega": om, "mask": e, "n_begin": 20, "n_end": 70},
                   {"j": 24, "omega": om, "mask": h}, {"j": 21, "omega": om, "mask": e | h, "n_begin": 33}]
    spec["probes"] = [[1, 21], [64, 22], [65, 23], [150, 24], [128, 24], [129, 20], [5, 25], [70, 60]]
    other = dict(spec, dft=spec["dft"][:1], probes=[])
    sims = [sim2d.make_simulation2d(s, precision=precision) for s in (spec, other, spec)]
    alone = sim2d.make_simulation2d(spec, precision=precision)
    batch = sim2d.Batch2D([s[0] for s in sims])
    ref = oracle.make_simulation2d(spec)
    for n in (1, 32, 47):
        batch.run([n, n // 2, n])
        alone[0].step(n)
        ref[0].step(n)
    batch.sync()
    tol = 1e-12 if precision == "fp64" else 1e-4
    for x, y, z, d in zip(sims[0][1], alone[1], ref[1], spec["dft"]):
        for c in [(sim2d.EZ2 if tm else sim2d.EX2)] * bool(d.get("mask", e) & e) + \
                 [(sim2d.HX2 if tm else sim2d.HZ2)] * bool(d.get("mask", h) & h):
            for u, v, w, o in zip(sims[0][0].dft(x, c), sims[2][0].dft(x, c), alone[0].dft(y, c), ref[0].dft(z, c)):
                assert np.array_equal(u, v) and np.array_equal(u, w)
                check(f"strip dft {polarization} {precision} {c}", relerr(u, o), tol)
    for x, y, z in zip(sims[0][2], alone[2], ref[2]):
        u = sims[0][0].probe(x)
        assert np.array_equal(u, sims[2][0].probe(x)) and np.array_equal(u, alone[0].probe(y))
        check(f"strip probe {polarization} {precision}", relerr(u, ref[0].probe(z)), tol)
    batch.close()
    for s in (*sims, alone, ref):
        s[0].close()
