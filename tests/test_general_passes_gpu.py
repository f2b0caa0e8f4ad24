"""The passes that read a cell's CPML memory face by face after its curl, which
plans with overlapping slabs of one axis take (a descriptor can ask for them;
grids built by Simulation are always wider than their slabs), and CPML
with kappa other than 1 on every pass: forward against the float64 oracle
and one another, reverse by the transpose identity and against the batched
reverse passes.

Tolerance of a float32 run against the oracle: 40 steps of some 10 roundings of
6e-8 each, growing linearly at worst, is 2.4e-5 of a series' size."""
import copy

import numpy as np
import pytest

from oracle import cstep
from oracle import fdtd_np as o
from tests import cases
from tests.test_resident_gpu import _outputs, _spec

pytestmark = pytest.mark.gpu
STEPS = 40
TOL = 2.5e-5


def _setup(n, cpml, layers, kappa=1.0, mag=False, lane="run", monitors=False):
    """Problem and oracle configuration of a grid with `layers` deep faces."""
    from rfx_amd.cpml import face_tables
    spec = dict(_spec(n, cpml, mag), lane=lane, kappa_max=kappa)
    if not monitors:
        spec.update(dft_planes=[], flux_monitors=[])
    sim = cases.to_sim(spec)
    grid, prob, _ = sim._build_problem(STEPS, lane)
    g, cfg = o.build_uniform(spec, STEPS)
    assert tuple(cfg.shape) == tuple(prob.shape)
    if layers != cpml:
        prob.faces = face_tables(layers, prob.dt, grid.face_cell_sizes(), kappa)
        b, c, k = o.cpml_profile(layers, cfg.dt, g.dx, kappa)
        cfg.cpml_n = layers
        cfg.cpml_profiles = {(ax, side): (b, c, k) if side == 0 else (b[::-1], c[::-1], k[::-1])
                             for ax in range(3) for side in range(2)}
    return sim, prob, cfg


OVERLAPS = [
    ((3, 17, 40), 6, 9, False),      # 16 x 30 x 53: x
    ((16, 3, 4), 6, 9, True),        # 29 x 16 x 17: y and z
    ((4, 5, 6), 3, 7, False),        # 11 x 12 x 13: all, most cells in two slabs of an axis
    ((4, 5, 6), 3, 9, True),
]


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _run(torch, dr, v):
    from rfx_amd import autotune as at
    at.set_variant(dr, *v)
    dr.reset()
    dr.run(0, STEPS)
    torch.cuda.synchronize()
    return _outputs(dr)


def _against_oracle(dr, cfg, outs):
    ref = cstep.run_c(cfg, STEPS)
    ts = outs[0].cpu().numpy()
    assert np.abs(ts).max() > 0
    assert cases.rel_l2(ts, ref.time_series) < TOL
    size = max(np.abs(ref.fields[c]).max() for c in ("ex", "ey", "ez"))
    hsize = max(np.abs(ref.fields[c]).max() for c in ("hx", "hy", "hz"))
    for c, x in zip(("ex", "ey", "ez", "hx", "hy", "hz"), outs[3:9]):
        err = np.abs(x.cpu().numpy() - ref.fields[c]).max()
        assert err <= TOL * (size if c[0] == "e" else hsize), c


@pytest.mark.parametrize("n, cpml, layers, mag", OVERLAPS)
def test_overlapping_slabs(torch, n, cpml, layers, mag):
    from rfx_amd import _lib
    from rfx_amd import autotune as at
    from rfx_amd.engine import DeviceRun
    _, prob, cfg = _setup(n, cpml, layers, mag=mag)
    assert any(2 * layers > m for m in prob.shape)
    dr = DeviceRun(prob, STEPS, "cuda", two_sets=True)
    assert at.get_variant(dr) == (0, 1)
    for refused in (8, 9):
        with pytest.raises(_lib.RfxHipError):
            at.set_variant(dr, refused, 0)
    res = {}
    for v in ((0, 1), (0, 0), (4, 1), (6, 1), (5, 0), (1, 0)):
        print("[gpu-case] overlapping slabs", n, layers, v, flush=True)
        res[v] = _run(torch, dr, v)
    dr.close()
    _against_oracle(dr, cfg, res[(0, 1)])
    for v in ((0, 0), (4, 1), (6, 1), (5, 0)):
        assert all(torch.equal(a, b) for a, b in zip(res[(0, 1)], res[v])), v
    assert torch.equal(res[(0, 1)][0], res[(1, 0)][0])


def test_overlapping_slabs_with_poles_and_graded_cells(torch):
    """The general passes' other instances: dispersive against the numpy
    oracle, graded against the fused step."""
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] overlapping slabs, poles", flush=True)
    _, prob, cfg = _setup((4, 5, 6), 3, 7)
    w = 2 * np.pi * 11e9
    poles, lor = [(2.0, 6e-12)], [(w, 2e9, 1.1 * w * w)]
    spec = dict(_spec((4, 5, 6), 3), dft_planes=[], flux_monitors=[], debye={"d": poles},
                lorentz={"d": lor})
    _, prob_d, _ = cases.to_sim(spec)._build_problem(STEPS, "run")
    _, cfg_d = o.build_uniform(spec, STEPS)
    prob_d.faces, cfg_d.cpml_n, cfg_d.cpml_profiles = prob.faces, cfg.cpml_n, cfg.cpml_profiles
    dr = DeviceRun(prob_d, STEPS, "cuda", two_sets=False)
    got = _run(torch, dr, (0, 1))
    dr.close()
    ref = o.run_loop(cfg_d, STEPS)
    assert cases.rel_l2(got[0].cpu().numpy(), ref.time_series) < TOL
    print("[gpu-case] overlapping slabs, graded", flush=True)
    spec = dict(cases.mixed_graded_case())
    sim = cases.to_sim(spec)
    grid, prob, _ = sim._build_problem(STEPS, "run", s11_freqs=np.asarray(spec["s11_freqs"], np.float32))
    from rfx_amd.cpml import face_tables
    prob.faces = face_tables(min(prob.shape), prob.dt, grid.face_cell_sizes())
    dr = DeviceRun(prob, STEPS, "cuda", two_sets=True)
    res = {v: _run(torch, dr, v) for v in ((0, 1), (4, 1), (1, 0))}
    dr.close()
    assert float(res[(0, 1)][0].abs().max()) > 0
    assert all(torch.equal(a, b) for a, b in zip(res[(0, 1)], res[(4, 1)]))
    assert all(torch.equal(a, b) for a, b in zip(res[(0, 1)][:2], res[(1, 0)][:2]))


def _identity(torch, prob):
    """<F x0, w> = <x0, F^T w> for random states, memory and probe weights."""
    import ctypes as C
    from rfx_amd import _lib
    from rfx_amd.adjoint import AdjointRunner
    prob = copy.copy(prob)
    prob.sources = []
    run = AdjointRunner(prob, STEPS, "cuda")
    dr = run.dr
    gen = torch.Generator(device="cpu").manual_seed(7)
    x0 = [torch.randn(prob.shape, generator=gen).cuda() for _ in range(6)]
    psi0 = torch.randn(dr.psis[0].numel(), generator=gen).cuda()
    dr.load_state(x0, psi0)
    ts = run.forward()
    w = torch.randn(ts.shape, generator=gen).cuda()
    lhs = float((ts.double() * w.double()).sum())
    adj = [torch.zeros(prob.shape, device="cuda") for _ in range(6)]
    adj_psi, gbar = torch.zeros_like(psi0), torch.zeros_like(psi0)
    d = _lib.AdjointDesc()
    for c in range(6):
        d.d_adj[c] = adj[c].data_ptr()
    d.d_adj_psi, d.d_gbar, d.d_probe_adj = adj_psi.data_ptr(), gbar.data_ptr(), w.data_ptr()
    _lib.check(dr.lib.rfxh_adjoint(dr.plan, C.byref(d), 0, STEPS, dr.stream_ptr()))
    torch.cuda.synchronize()
    rhs = sum(float((a.double() * x.double()).sum()) for a, x in zip(adj, x0))
    rhs += float((adj_psi.double() * psi0.double()).sum())
    scale = float(ts.double().norm() * w.double().norm())
    assert scale > 0 and abs(lhs - rhs) <= 1e-5 * scale
    run.dr.close()


def _against_batched(torch, make):
    from rfx_amd.adjoint import AdjointRunner, BatchAdjointRunner
    r = AdjointRunner(make(), STEPS, "cuda")
    ts = r.forward()
    g = r.backward(2.0 * ts).cpu().numpy().copy()
    ts = ts.cpu().numpy().copy()
    r.dr.close()
    b = BatchAdjointRunner([make()], [STEPS], "cuda")
    tb = b.forward()
    gb = b.backward([2.0 * t for t in tb])[0].cpu().numpy().copy()
    tb = tb[0].cpu().numpy().copy()
    b.close()
    assert cases.rel_l2(tb, ts) < 1e-6
    assert np.isfinite(g).all() and np.abs(g).max() > 0
    np.testing.assert_allclose(gb, g, rtol=1e-5, atol=1e-6 * np.abs(g).max())


@pytest.mark.parametrize("n, cpml, layers, mag", OVERLAPS)
@pytest.mark.parametrize("lane", ["run", "forward"])
def test_overlapping_slabs_reverse(torch, n, cpml, layers, mag, lane):
    print("[gpu-case] overlapping slabs, reverse", n, layers, lane, flush=True)
    _identity(torch, _setup(n, cpml, layers, mag=mag, lane=lane)[1])
    _against_batched(torch, lambda: _setup(n, cpml, layers, mag=mag, lane=lane)[1])


KAPPA = [((19, 23, 30), 6, 6, False), ((12, 9, 40), 8, 8, True), ((3, 17, 40), 6, 9, False)]


@pytest.mark.parametrize("n, cpml, layers, mag", KAPPA)
def test_kappa(torch, n, cpml, layers, mag):
    from rfx_amd import _lib
    from rfx_amd import autotune as at
    from rfx_amd.batch import Batch
    from rfx_amd.engine import DeviceRun
    sim, prob, cfg = _setup(n, cpml, layers, kappa=4.0, mag=mag)
    assert any((f[3] != 0).any() for f in prob.faces)
    dr = DeviceRun(prob, STEPS, "cuda", two_sets=True)
    assert at.get_variant(dr) == (0, 1)
    with pytest.raises(_lib.RfxHipError):     # (the resident step's corrections assume kappa = 1)
        at.set_variant(dr, 9, 0)
    variants = [(0, 1), (4, 1), (6, 1), (5, 1), (1, 0)]
    if layers == cpml:
        variants += [(2, 0), (7, 0), (8, 0)]
    res = {}
    for v in variants:
        print("[gpu-case] kappa", n, layers, v, flush=True)
        res[v] = _run(torch, dr, v)
    dr.close()
    _against_oracle(dr, cfg, res[(0, 1)])
    for v in variants[1:]:
        assert cases.rel_l2(res[v][0].cpu().numpy(), res[(0, 1)][0].cpu().numpy()) < 1e-6, v
    if layers == cpml:
        b = Batch([sim], STEPS)
        b.run()
        assert cases.rel_l2(b.runs[0].probe_out.cpu().numpy(),
                            res[(0, 1)][0].cpu().numpy()) < 1e-6
        b.close()


@pytest.mark.parametrize("n, cpml, layers, mag", KAPPA)
def test_kappa_reverse(torch, n, cpml, layers, mag):
    print("[gpu-case] kappa, reverse", n, layers, flush=True)
    for lane in ("run", "forward"):
        _identity(torch, _setup(n, cpml, layers, 4.0, mag, lane)[1])
    _against_batched(torch, lambda: _setup(n, cpml, layers, 4.0, mag, "forward")[1])


def _poles_first(mat, points):
    """Renumber a material map so that the ids with poles follow the first one."""
    from rfx_amd import _lib
    for idx in points:                   # (DeviceRun's own flags: no new ids after this)
        mat.set_cell(tuple(idx), add_flags=_lib.RFXH_POINT)
    order = sorted(range(1, len(mat.table)), key=lambda q: (int(mat.table[q][3]) >> 16) == 0)
    order = np.array([0] + order)
    new = np.empty(len(order), np.uint16)
    new[order] = np.arange(len(order))
    mat.ids = new[mat.ids]
    mat.table = [mat.table[q] for q in order]
    mat._lookup = {key: int(new[q]) for key, q in mat._lookup.items()}


@pytest.mark.parametrize("nd, nl, before, after", [
    (1, 1, 0, 0), (3, 2, 0, 0), (2, 1, 70, 0),
    (1, 1, 0, 140),       # pole ids within one 64-bit word, other ids past it
])
def test_pole_loads_against_the_general_pass(torch, nd, nl, before, after):
    """The one-cell dispersive pass against the batched pass that reads poles
    and CPML memory after the curl, which a batch of uniform and graded
    instances takes."""
    from rfx_amd.batch import Batch
    from rfx_amd.engine import DeviceRun
    from tests.test_pole_loads_gpu import DEBYE, LORENTZ
    print("[gpu-case] poles, general pass", nd, nl, before, after, flush=True)
    spec = dict(_spec((29, 24, 21), 6), dft_planes=[], flux_monitors=[],
                debye={"d": DEBYE[:nd]}, lorentz={"d": LORENTZ[:nl]})
    dx = 1e-3
    spec["materials"] = dict(spec["materials"])

    def boxes(count, tag, z):
        out = []
        for q in range(count):
            spec["materials"][f"{tag}{q}"] = (2.0 + 0.05 * q, 0.0, 1.0)
            lo = ((q % 14 + 0.5) * dx, (q // 14 + 0.5) * dx, z * dx)
            out.append((lo, tuple(v + 0.9 * dx for v in lo), f"{tag}{q}"))
        return out

    # (the later boxes lie beside the pole material and within its box of state)
    spec["geometry"] = boxes(before, "x", 1.5) + spec["geometry"] + boxes(after, "y", 10.5)
    sim = cases.to_sim(spec)
    if after:
        build = sim._build_problem

        def poles_first(*a, **k):
            g, p, ports = build(*a, **k)
            _poles_first(p.mat, [op[0] for op in p.sources + p.probes])
            return g, p, ports
        sim._build_problem = poles_first
    _, prob, _ = sim._build_problem(STEPS, "run")
    dr = DeviceRun(prob, STEPS, "cuda", two_sets=False)
    ids = np.nonzero(dr.flags >> 16)[0]
    assert len(ids) and (len(dr.flags) > 64) == (before + after > 0)
    if after:
        assert ids.max() < 64
    alone = _run(torch, dr, (0, 1))
    dr.close()
    graded = dict(cases.mixed_graded_case())
    b = Batch([sim, cases.to_sim(graded)], STEPS)
    assert {bool(p.graded) for p in b.problems} == {False, True}
    b.run()
    both = _outputs(b.runs[0])
    b.close()
    assert float(alone[0].abs().max()) > 0
    assert all(torch.equal(x, y) for x, y in zip(alone, both))
