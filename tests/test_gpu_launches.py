"""The FUSED engine's launches at the sizes where their parts end: more
dispersive groups and monitor planes than a launch takes along, calls of
one step, grids whose lists leave the E launch, and the parts together
(no profiling) against each in a launch of its own (profiling)."""
import numpy as np
import pytest

from conftest import check, relerr

pytestmark = pytest.mark.gpu


def _spec(n=(41, 36, 34), groups=6, planes=11, nsteps=90):
    """Gold-like boxes of `groups` different parameter sets, `planes` DFT
    planes over the three axes with unlike gates, probes in and beside them."""
    from fdtd_amd import box, gold_params_dict, workloads

    spec = workloads.c1_gold_sphere(nsteps=nsteps, n=32)
    spec["grid"].update(nx=n[0], ny=n[1], nz=n[2])
    spec["pml"]["npml"] = [5, 4, 6]
    mats = [{"type": "dielectric", "region": box((1, 1, 1), n), "eps": 1.0},
            {"type": "dielectric", "region": box((1, 1, n[2] - 9), n), "eps": 2.25}]
    for g in range(groups):
        q = gold_params_dict()
        q["gamma"] *= 1.0 + 0.1 * g
        lo = (8 + 4 * g, 10 + g, 12)
        mats.append({"type": "drude2cp", "region": box(lo, (lo[0] + 2, lo[1] + 8, 20)), "params": q})
    spec["materials"] = mats
    spec["sources"][0]["index"] = 9
    om = spec["dft"][0]["omega"][:3]
    spec["dft"] = [{"axis": q % 3, "index": 8 + q, "omega": om, "n_begin": 1 + 7 * (q % 4),
                    "comps": [[1, 2, 4, 5], [0, 2, 3, 5], [0, 1, 3, 4], [2, 3]][q % 4] if q % 4 < 3 else [2, 3]}
                   for q in range(planes)]
    spec["probes"] = [[9, 12, 15], [1, 1, 1], list(n), [20, 18, 10]]
    return spec


def _run(spec, precision, steps, profiling=False):
    import fdtd_amd

    sim, ids, pids = fdtd_amd.make_simulation(spec, precision=precision, engine="fused")
    sim.set_profiling(profiling)
    for n in steps:
        sim.step(n)
    return sim, ids, pids


def _same(a, ia, pa, b, ib, pb, spec):
    for c in range(6):
        assert np.array_equal(a.field(c), b.field(c)), c
    for x, y, d in zip(ia, ib, spec["dft"]):
        for c in d["comps"]:
            for u, v in zip(a.dft(x, c), b.dft(y, c)):
                assert np.array_equal(u, v)
    for x, y in zip(pa, pb):
        assert np.array_equal(a.probe(x), b.probe(y))


@pytest.mark.parametrize("form", [{"FDTD_ONEPASS": "0"}, {"FDTD_ONEPASS": "0", "FDTD_ZMARCH": "4"},
                                  {"FDTD_ONEPASS": "1", "FDTD_ONEPASS_BY": "2", "FDTD_ONEPASS_KC": "8"}])
def test_groups_and_planes_past_one_list(form, monkeypatch):
    """Six dispersive groups (a launch takes four), eleven planes (a launch
    takes eight), calls of 1, 63, 1 and 25 steps across a DFT block: FP64
    against the oracle at the parity bar, and bit for bit the run whose
    parts are launches of their own."""
    import oracle

    for k, v in form.items():
        monkeypatch.setenv(k, v)
    spec = _spec()
    steps = (1, 63, 1, 25)
    a, ia, pa = _run(spec, "fp64", steps)
    b, ib, pb = _run(spec, "fp64", steps, profiling=True)
    _same(a, ia, pa, b, ib, pb, spec)
    o, io, po = oracle.make_simulation(spec)
    for n in steps:
        o.step(n)
    for c in range(6):
        check(f"lists field {c}", relerr(a.field(c), o.field(c)), 1e-12)
    for x, y, d in zip(ia, io, spec["dft"]):
        for c in d["comps"]:
            for u, v in zip(a.dft(x, c), o.dft(y, c)):
                check(f"lists dft {c}", relerr(u, v), 1e-12)
    for x, y in zip(pa, po):
        check("lists probe", relerr(a.probe(x), o.probe(y)), 1e-12)
    for s in (a, b, o):
        s.close()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n,apart", [((9, 362, 362), False), ((9, 363, 363), True)])
def test_lists_beside_the_rows_and_apart(n, apart, precision, monkeypatch):
    """Grids on both sides of the line from which the lists of the two-kernel
    E half have a launch of their own (32,768 workgroups of rows; 9 cells a
    row leave lanes idle): the same bits as the one-pass step."""
    assert (n[1] * n[2] >= 4 * 32768) == apart
    spec = _spec(n, groups=0, planes=2, nsteps=6)
    spec["pml"]["npml"] = [2, 6, 6]
    spec["probes"] = [[5, 110, 15], [1, 1, 1], list(n)]
    monkeypatch.setenv("FDTD_ONEPASS", "0")
    from fdtd_amd import box, gold_params_dict

    spec["materials"].append({"type": "drude2cp", "region": box((4, 100, 9), (6, 140, 30)),
                              "params": gold_params_dict()})
    spec["dft"] = [{"axis": 2, "index": 12, "omega": spec["dft"][0]["omega"], "comps": [0, 1, 3, 4]}]
    a, ia, pa = _run(spec, precision, (6,))
    monkeypatch.setenv("FDTD_ONEPASS", "1")
    b, ib, pb = _run(spec, precision, (6,))
    _same(a, ia, pa, b, ib, pb, spec)
    a.close()
    b.close()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("by,kc", [("2", "16"), ("4", "200"), ("8", "2")])
@pytest.mark.parametrize("case", ["gold_sphere", "periodic_box"])
def test_marked_stores_of_the_march(case, by, kc, precision, monkeypatch):
    """The one-pass step with its stores marked nontemporal (what a grid past
    the memory-side cache runs; FDTD_NT forces a side), a wavefront marching
    4 planes, all of the grid's, or 1: the same bits."""
    from test_gpu_onepass import _cases, _run as run, _same as same

    spec = _cases()[case]
    env = {"FDTD_ONEPASS": "1", "FDTD_ONEPASS_BY": by, "FDTD_ONEPASS_KC": kc}
    got = [run(spec, precision, dict(env, FDTD_NT=nt), monkeypatch) for nt in "01"]
    same(*got[0], *got[1])


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("case", ["ref_graphene_small", "periodic_box"])
def test_marked_d_of_the_reference_order(case, precision, golden, monkeypatch):
    """The same of the staged engine's D, y-slab PML and periodic axes."""
    import fdtd_amd
    from test_gpu_onepass import _cases

    spec = _cases()[case] if case == "periodic_box" else golden(case)[0]
    got = []
    for nt in "01":
        monkeypatch.setenv("FDTD_NT", nt)
        sim, _, _ = fdtd_amd.make_simulation(spec, precision=precision, engine="staged")
        sim.step(min(spec["nsteps"], 130))
        got.append(sim)
    assert np.abs(got[0].field(0)).max() > 0
    for c in range(9):
        assert np.array_equal(got[0].field(c), got[1].field(c)), c


@pytest.mark.parametrize("nfreq", [1, 16, 17, 33, 49, 64, 65, 130])
def test_fold_tiles(nfreq):
    """Spectra at nfreq frequencies (16 a tile, 64 a pass) over planes whose
    cells end inside a tile of 16, folded over blocks of 1, 3, 63, 64 and 5
    samples: FP64 against the oracle at the parity bar."""
    import oracle
    from fdtd_amd import workloads

    n = (33, 35, 38)
    spec = _spec(n, groups=1, planes=3)
    spec["pml"]["npml"] = [4, 4, 6]
    om = workloads.wavelength_frequencies(400e-9, 900e-9, nfreq)
    for d in spec["dft"]:
        d.update(omega=list(om), n_begin=1)
    a, ia, _ = _run(spec, "fp64", (1, 3, 63, 64, 5))
    o, io, _ = oracle.make_simulation(spec)
    o.step(136)
    for x, y, d in zip(ia, io, spec["dft"]):
        for c in d["comps"]:
            for u, v in zip(a.dft(x, c), o.dft(y, c)):
                check(f"fold {nfreq} {c}", relerr(u, v), 1e-12)


@pytest.mark.parametrize("n", [(204, 205, 16), (409, 411, 16)])
def test_large_reads_from_two_threads(n):
    """Spectra of 10 and 43 MB an array, read through the pinned slots (from
    16 MiB on, 2 MiB a slice, the last one short) by two threads from two
    handles at once: the bytes of the same frequencies on planes of two
    frequencies each, whose reads stay below the line."""
    import threading

    import fdtd_amd
    from fdtd_amd import workloads

    nf = 32
    om = list(workloads.wavelength_frequencies(400e-9, 900e-9, nf))
    sims = []
    for q in range(2):
        spec = workloads.c1_gold_sphere(nsteps=8, n=16)
        spec["grid"].update(nx=n[0], ny=n[1], nz=n[2])
        spec["pml"]["npml"] = [2, 2, 2]
        spec["materials"] = [{"type": "dielectric", "region": fdtd_amd.box((1, 1, 1), n), "eps": 1.0 + q}]
        spec["sources"][0]["index"] = 7
        spec["dft"] = [{"axis": 2, "index": 8, "omega": w, "comps": [0, 4]}
                       for w in [om] + [om[f:f + 2] for f in range(0, nf, 2)]]
        spec["probes"] = []
        s, i, _ = fdtd_amd.make_simulation(spec, precision="fp32", engine="fused")
        s.step(8)
        sims.append((s, i))
    got = [None, None]

    def read(q):
        s, i = sims[q]
        got[q] = [s.dft(i[0], c) for c in (0, 4)]

    th = [threading.Thread(target=read, args=(q,)) for q in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for (s, i), g in zip(sims, got):
        for c, parts in zip((0, 4), g):
            assert np.any(parts[0] != 0) and np.any(parts[1] != 0)
            for k in range(nf // 2):
                for u, v in zip(parts, s.dft(i[1 + k], c)):
                    assert np.array_equal(u[:, :, 2 * k:2 * k + 2], v)
        s.close()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n", [(1, 5, 3), (63, 7, 5), (64, 4, 9), (129, 3, 2), (2049, 1025, 3)])
def test_packed_field_reads(n, precision):
    """A field read back equals the field set: rows of 1, 63, 64 and 129
    cells, and one plane a pass where two exceed the device's buffer (17 MB
    a plane)."""
    import fdtd_amd

    sim = fdtd_amd.Simulation(n[0], n[1], n[2], 1e-9, 0.5, precision=precision, engine="fused")
    rng = np.random.default_rng(n[0])
    for c in (0, 4):
        f = rng.standard_normal(n).astype(np.float32).astype(np.float64)
        sim.set_field(c, f)
        assert np.array_equal(sim.field(c), f), c
    sim.close()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("zm", ["1", "4"])
def test_incident_line_beside_the_h_half(zm, precision, monkeypatch):
    """The incident line's E half step as a block of the H launch (one TFSF)
    and as a launch of its own (profiling): the same bits, line included."""
    from test_gpu_tfsf import _tfsf_through_pml

    monkeypatch.setenv("FDTD_ONEPASS", "0")
    monkeypatch.setenv("FDTD_ZMARCH", zm)
    spec = dict(_tfsf_through_pml(nsteps=150), dft=[])
    a, ia, pa = _run(spec, precision, (1, 85, 64))
    b, ib, pb = _run(spec, precision, (1, 85, 64), profiling=True)
    assert np.abs(a.field(0)).max() > 0 or np.abs(a.field(2)).max() > 0
    _same(a, ia, pa, b, ib, pb, spec)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_reads_leave_the_device_memory_as_it_was(precision):
    """A field read takes no device memory beyond its own time; the buffer of
    the energy and flux sums is replaced where a larger one is needed, so the
    handle holds the larger one alone."""
    import fdtd_amd
    from fdtd_amd import workloads

    spec = workloads.c1_gold_sphere(nsteps=8, n=32)
    om = list(workloads.wavelength_frequencies(400e-9, 900e-9, 4096))
    spec["dft"] = [dict(spec["dft"][0], omega=om)]
    sim, ids, _ = fdtd_amd.make_simulation(spec, precision=precision, engine="fused")
    sim.step(4)
    m0 = sim.memory_bytes()
    f = [sim.field(c) for c in range(6)]
    assert sim.memory_bytes() == m0
    we = sim.energy()
    m1 = sim.memory_bytes()
    flux = sim.flux(ids[0])
    assert sim.memory_bytes() - m0 == 8 * 4096 and m1 - m0 <= 8 * 4096
    assert sim.energy() == we and np.array_equal(sim.flux(ids[0]), flux)
    assert all(np.array_equal(sim.field(c), f[c]) for c in range(6))
    assert sim.memory_bytes() - m0 == 8 * 4096
    sim.close()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("form", [{"FDTD_ONEPASS": "0"}, {"FDTD_ONEPASS": "1", "FDTD_ONEPASS_BY": "2"}, "staged"])
def test_samples_beside_the_launches_and_alone(form, precision, monkeypatch):
    """Eleven planes and four probes sampled beside the step's launches, in
    calls that end before, at and behind a DFT block: the same bits as
    sampled by a launch at each step's end (FDTD_DFT_FUSE=0), and as with
    every part in a launch of its own (profiling)."""
    import fdtd_amd

    spec = _spec(groups=2)
    if form == "staged":
        spec["pml"].update(mode="ref_y", npml=[0, 5, 0])
    else:
        for k, v in form.items():
            monkeypatch.setenv(k, v)
    runs = []
    for fuse, prof in (("1", False), ("0", False), ("1", True)):
        monkeypatch.setenv("FDTD_DFT_FUSE", fuse)
        sim, ids, pids = fdtd_amd.make_simulation(spec, precision=precision)
        sim.set_profiling(prof)
        for n in (1, 62, 1, 1, 64, 2):
            sim.step(n)
        runs.append((sim, ids, pids))
    for r in runs[1:]:
        _same(*runs[0], *r, spec)
    assert all(np.abs(runs[0][0].dft(i, d["comps"][-1])[0]).max() > 0 for i, d in zip(runs[0][1], spec["dft"]))
    for r in runs:
        r[0].close()


@pytest.mark.parametrize("precision,n", [("fp64", (256, 128, 3)), ("fp64", (255, 128, 3)), ("fp32", (256, 512, 6)),
                                         ("fp32", (257, 511, 6))])
def test_field_reads_at_the_packing_line(precision, n):
    """Fields of 768 KiB (FP64) and 6 MiB (FP32) of results, from which on
    they are packed on the device, and just below: the field set, and the
    device memory as it was."""
    import fdtd_amd

    sim = fdtd_amd.Simulation(*n, 1e-9, 0.5, precision=precision, engine="fused")
    f = np.random.default_rng(n[0]).standard_normal(n).astype(np.float32).astype(np.float64)
    sim.set_field(2, f)
    m = sim.memory_bytes()
    assert np.array_equal(sim.field(2), f) and sim.memory_bytes() == m
    sim.close()


@pytest.mark.parametrize("bx", ["2", "4"])
def test_marked_stores_of_the_x_face_tiles(bx, monkeypatch):
    """The x-face tiles of 2 rows (in the march's launch) and of 4 (their
    own), stores marked and not: the same bits."""
    from test_gpu_onepass import _cases, _run as run, _same as same

    spec = _cases()["x_edges"]
    env = {"FDTD_ONEPASS": "1", "FDTD_ONEPASS_BY": "4", "FDTD_ONEPASS_KC": "16", "FDTD_XFACE_BY": bx}
    got = [run(spec, "fp32", dict(env, FDTD_NT=nt), monkeypatch) for nt in "01"]
    same(*got[0], *got[1])


def test_packed_reads_from_more_threads_than_buffers():
    """Six threads, a handle each, reading fields of 0.8-2 MiB (the four
    shared buffers) and of 2.7 MiB (buffers of their own) while handles come
    and go: the fields set, every time, and no device memory of the handles."""
    import threading

    import fdtd_amd

    bad = []

    def work(q):
        try:
            rng = np.random.default_rng(q)
            for r in range(6):
                n = [(48, 48, 48), (61, 64, 64), (40, 90, 60), (70, 70, 72)][(q + r) % 4]
                sim = fdtd_amd.Simulation(*n, 1e-9, 0.5, precision="fp64", engine="fused")
                f = rng.standard_normal(n)
                sim.set_field(r % 6, f)
                m = sim.memory_bytes()
                for _ in range(8):
                    if not np.array_equal(sim.field(r % 6), f):
                        bad.append((q, r))
                if sim.memory_bytes() != m:
                    bad.append((q, r, "memory"))
                sim.close()
        except Exception as e:  # noqa: BLE001 - reported below
            bad.append((q, repr(e)))

    th = [threading.Thread(target=work, args=(q,)) for q in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
