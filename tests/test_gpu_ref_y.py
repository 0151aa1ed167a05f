"""The reference-order step beside the y-slab PML, through the C ABI against
the oracle: what writes fields next to a slab between two steps (the
caller, a TFSF wave's terms), and its parts in one launch and apart.

Tolerance, normwise, FP64 against the oracle: 1e-12.  FP32 fields 2e-4."""
import math

import numpy as np
import pytest

from conftest import check, relerr
from test_oracle_tfsf import tfsf_box

pytestmark = pytest.mark.gpu
P = 8


def _slabs(spec):
    spec["pml"] = {"mode": "ref_y", "npml": [0, P, 0], "order": 3.0, "R0": math.exp(-16.0),
                   "eps_low": 1.0, "eps_high": 2.25}
    return spec


def _field_err(g, o):
    return max(relerr(np.stack([g.field(q) for q in c]), np.stack([o.field(q) for q in c]))
               for c in ((0, 1, 2), (3, 4, 5)))


def _along_y(comp, lo=25, hi=55):
    """A TFSF wave along y between the slabs, ny = 64 + 2 P."""
    spec = tfsf_box(1, comp, True, n_axis=64 + 2 * P, nsteps=130)
    spec["tfsf"][0].update(lo=lo, hi=hi)
    return _slabs(spec)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("comp,lo,hi", [(0, 25, 63 + P), (2, 25, 63 + P), (2, P + 2, 55), (0, P + 2, 63 + P),
                                        (0, 64 + P, 0), (2, 20, 0)])
def test_tfsf_terms_beside_the_slabs(comp, lo, hi, precision):
    """The TFSF planes nearest to the slabs that a handle takes: the terms on
    H on row lo-1 = P+1 and on row hi = ny-P-1, one and two sided."""
    import fdtd_amd
    import oracle

    spec = _along_y(comp, lo, hi)
    g, _, _ = fdtd_amd.make_simulation(spec, precision=precision)
    o, _, _ = oracle.make_simulation(spec)
    for n in (1, 64, 65):
        g.step(n)
        o.step(n)
    assert max(np.abs(o.field(c)).max() for c in range(3)) > 1e-3
    check(f"ref-y tfsf comp {comp} lo {lo} hi {hi} {precision}", _field_err(g, o),
          1e-12 if precision == "fp64" else 2e-4)


@pytest.mark.parametrize("axis,lo,hi", [(0, 25, 55), (2, 25, 55), (1, 25, 64 + P), (1, P + 1, 55), (1, 65 + P, 0)])
def test_tfsf_planes_refused_beside_the_slabs(axis, lo, hi):
    """Waves across the slabs, and planes one row nearer to a slab than those
    above: refused at commit."""
    import fdtd_amd

    spec = _along_y(0, lo, hi)
    spec["tfsf"][0].update(axis=axis, comp=2 if axis == 0 else 0)
    if axis != 1:
        spec["grid"].update({"nx" if axis == 0 else "nz": 80})
    g, _, _ = fdtd_amd.make_simulation(spec)
    with pytest.raises(fdtd_amd.FdtdError):
        g.commit()


@pytest.mark.parametrize("before,between", [((), (3, 5)), ((3, 5), ()), ((3, 4, 5), (3, 5)), ((0, 2, 6, 8), (0, 1, 2)),
                                            ((3,), (6, 7, 8))])
def test_fields_set_beside_the_slabs(before, between):
    """Components set by the caller before the first step and between steps,
    noise on the rows inside both slabs' edges and one past them."""
    import fdtd_amd
    import oracle

    spec = _along_y(0)
    spec.pop("tfsf")
    spec["grid"].update(nx=11, nz=9, periodic=[1, 0, 0])
    spec["materials"][0]["region"]["hi"] = [11, 64 + 2 * P, 9]
    rows = [P - 1, P, P + 1, spec["grid"]["ny"] - P - 1, spec["grid"]["ny"] - P]
    sims = (fdtd_amd.make_simulation(spec)[0], oracle.make_simulation(spec)[0])

    def put(comps, seed):
        rng = np.random.default_rng(seed)
        for c in comps:
            noise = rng.standard_normal((sims[0].shape[0], len(rows), sims[0].shape[2]))
            for s in sims:
                f = s.field(c)
                f[:, rows, :] = noise
                s.set_field(c, f)

    put(before, 1)
    for n, seed in ((1, 2), (7, 3), (32, 4)):
        for s in sims:
            s.step(n)
        if seed < 4:
            put(between, seed)
    g, o = sims
    assert np.abs(o.field(3)).max() > 0 and np.abs(o.field(5)).max() > 0
    check(f"ref-y fields set {before} {between}", _field_err(g, o), 1e-12)


def test_parts_together_and_apart():
    """Six dispersive groups (a launch takes four), a source plane through
    one of them, eleven DFT planes, probes and a TFSF wave, in calls across a
    DFT block: one launch a half step against a launch of its own for every
    part (profiling), bit for bit, and the oracle."""
    import fdtd_amd
    import oracle
    from test_gpu_launches import _same, _spec

    spec = _slabs(_spec())
    ny = spec["grid"]["ny"]
    spec["sources"].append(dict(spec["sources"][0], axis=1, index=14, comp=0))
    spec["tfsf"] = [dict(tfsf_box(1, 0)["tfsf"][0], lo=P + 2, hi=ny - P - 1, src_index=5, npml=2)]
    steps = (1, 63, 1, 25)
    runs = []
    for prof in (False, True):
        s, ids, pids = fdtd_amd.make_simulation(spec, engine="staged")
        s.set_profiling(prof)
        for q in steps:
            s.step(q)
        runs += [s, ids, pids]
    _same(*runs, spec)
    for c in range(6, 9):
        assert np.array_equal(runs[0].field(c), runs[3].field(c)), c
    o, io, po = oracle.make_simulation(spec)
    o.step(sum(steps))
    check("ref-y parts fields", _field_err(runs[0], o), 1e-12)
    for x, y, d in zip(runs[1], io, spec["dft"]):
        for c in d["comps"]:
            for u, v in zip(runs[0].dft(x, c), o.dft(y, c)):
                check(f"ref-y parts dft {c}", relerr(u, v), 1e-12)
    for x, y in zip(runs[2], po):
        check("ref-y parts probe", relerr(runs[0].probe(x), o.probe(y)), 1e-12)
