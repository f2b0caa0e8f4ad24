"""The resident step (a whole run of a small grid in one launch) against the
one-cell two-pass step on the same plan: the arithmetic is the same product
for product, so fields, CPML memory, probe and port samples and every
accumulator are equal bit for bit.  Sizes at the edges of its blocks (one
block, partial last blocks on each axis, every number of planes per thread
that the cut uses), an odd number of steps, runs in pieces, staging rings
shorter than a run, and two plans on two streams."""
import numpy as np
import pytest

from oracle import fdtd_np as o
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import rfx_amd
    return rfx_amd


def _spec(n, cpml, mag=False):
    dx = 1e-3
    dom = tuple((v - 0.5) * dx for v in n)
    c = [v * dx for v in (n[0] // 2, n[1] // 2, n[2] // 2)]
    mats = {"d": (3.0, 0.02, 1.0), "m": (1.0, 1e8, 1.0)}
    if mag:
        mats["mag"] = (1.5, 0.0, 2.0)
    geom = [(tuple(0.3 * v for v in dom), tuple(0.8 * v for v in dom), "mag" if mag else "d"),
            ((0.1 * dom[0], 0.2 * dom[1], c[2] - 1.2e-3), (0.6 * dom[0], 0.9 * dom[1], c[2] - 0.8e-3),
             "m")]
    src = tuple(c[a] + dx * (1 if n[a] > 4 else 0) for a in range(3))
    return dict(freq_max=25e9, domain=dom, dx=dx, boundary="cpml" if cpml else "pec",
                cpml_layers=cpml, materials=mats, geometry=geom,
                ports=[(tuple(c), "ez", 0.0, o.Pulse(12e9, 0.9), True),
                       (src, "ex", 0.0, o.Pulse(9e9, 0.8), True)],
                probes=[(tuple(c), "ez"), (src, "hx"), ((0.0, 0.0, 0.0), "ey")],
                dft_planes=[("z", c[2], "ez", np.array([5e9, 9e9, 12e9, 14e9, 20e9]), 5),
                            ("x", c[0], "hy", np.array([8e9]), 1)],
                flux_monitors=[("x", c[0], np.array([8e9, 9e9]), 2, None, None, "rect", 0.25),
                               ("y", c[1], np.array([7e9]), 1, None, None, "hann", 0.25),
                               ("z", 0.0, np.array([7e9]), 1, None, None, "rect", 0.25)],
                lane="run")


def _outputs(dr):
    out = [dr.probe_out, dr.port_out, dr.psi, *dr.fields, *dr.plane_acc, *dr.flux_acc]
    return [x.clone() for x in out + [f for box in dr.ntff_acc for f in box]]


def _same(dr, n, pieces=None):
    """Both steps over n steps (the resident one in the given pieces)."""
    import torch
    from rfx_amd import autotune as at
    res = {}
    for v, cut in (((0, 1), [n]), ((9, 0), pieces or [n])):
        at.set_variant(dr, *v)
        assert at.get_variant(dr) == v
        dr.reset()
        lo = 0
        for m in cut:
            dr.run(lo, m)
            lo += m
        assert lo == n
        torch.cuda.synchronize()
        res[v] = _outputs(dr)
    for a, b in zip(res[(0, 1)], res[(9, 0)]):
        assert torch.equal(a, b)
    assert float(res[(9, 0)][0].abs().max()) > 0


@pytest.mark.parametrize("n, cpml, steps", [
    ((3, 3, 3), 0, 9),                   # one block, smaller than a wavefront
    ((6, 5, 40), 0, 33),
    ((11, 12, 13), 6, 41),               # slabs on most cells
    ((40, 30, 9), 8, 60),
    ((70, 30, 25), 8, 37),               # the README quick start's grid
    ((5, 150, 17), 6, 30),               # flat, many rows
    ((96, 80, 63), 8, 24),               # near the most cells
    ((200, 21, 37), 6, 24),
])
def test_equals_the_two_pass_step(R, n, cpml, steps):
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] resident", n, cpml, flush=True)
    sim = cases.to_sim(_spec(n, cpml))
    _, prob, _ = sim._build_problem(steps, "run")
    for two in (True, False):
        dr = DeviceRun(prob, steps, "cuda", two_sets=two)
        _same(dr, steps)
        dr.close()


def test_pieces_ports_and_graded(R):
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] resident, graded mixed case in pieces", flush=True)
    spec = dict(cases.mixed_graded_case())
    spec["materials"] = {k: (e, s, 1.0) for k, (e, s, _) in spec["materials"].items()}
    sim = cases.to_sim(spec)
    _, prob, _ = sim._build_problem(71, "run", s11_freqs=np.asarray(spec["s11_freqs"], np.float32))
    dr = DeviceRun(prob, 71, "cuda")
    _same(dr, 71, [5, 17, 3, 46])        # (3 steps take the two-pass kernels)
    dr.close()
    print("[gpu-case] resident, lumped port", flush=True)
    sim = cases.to_sim(cases.S11_CASE)
    _, prob, _ = sim._build_problem(50, "forward",
                                    s11_freqs=np.asarray(cases.S11_CASE["s11_freqs"], np.float32))
    dr = DeviceRun(prob, 50, "cuda")
    _same(dr, 50)
    dr.close()


def test_rings_shorter_than_the_run(R):
    """Enough monitors that a launch stages fewer steps than the run has."""
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] resident, several launches", flush=True)
    spec = _spec((60, 60, 60), 6)
    spec["flux_monitors"] = [(ax, (4 + q) * 3e-3, np.array([8e9]), 1, None, None, "rect", 0.25)
                             for q in range(8) for ax in "xyz"]
    sim = cases.to_sim(spec)
    sim.add_ntff_box((5e-3,) * 3, (50e-3,) * 3, freqs=np.array([6e9, 9e9]))
    steps = 95
    _, prob, _ = sim._build_problem(steps, "run")
    assert len(prob.fluxes) + 6 * len(prob.ntff) + len(prob.planes) == 32
    per_step = 16 * 24 * 73 * 73 + 8 * 73 * 73 + 16 * 6 * 45 * 45
    assert (64 << 20) // per_step < steps
    dr = DeviceRun(prob, steps, "cuda")
    _same(dr, steps)
    dr.close()


def test_refused_and_default(R):
    from rfx_amd import _lib
    from rfx_amd import autotune as at
    from rfx_amd.engine import DeviceRun
    small = DeviceRun(cases.to_sim(_spec((12, 12, 12), 6))._build_problem(8, "run")[1], 8, "cuda")
    assert at.get_variant(small) == (9, 0)
    at.set_variant(small, 4, 1)
    assert at.get_variant(small) == (4, 1)
    with pytest.raises(_lib.RfxHipError):
        at.set_variant(small, 9, 1)
    small.close()
    mag = DeviceRun(cases.to_sim(_spec((12, 12, 12), 6, True))._build_problem(8, "run")[1], 8, "cuda")
    assert at.get_variant(mag) != (9, 0)          # several mu_r
    mag.close()
    big = DeviceRun(cases.to_sim(_spec((150, 150, 80), 0))._build_problem(8, "run")[1], 8, "cuda")
    with pytest.raises(_lib.RfxHipError):
        at.set_variant(big, 9, 0)
    big.close()


def test_two_plans_on_two_streams(R):
    """Launches of two plans on two streams: each gets its own results."""
    import torch
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] resident, two plans on two streams", flush=True)
    steps = 200
    runs = [DeviceRun(cases.to_sim(_spec(n, 6))._build_problem(steps, "run")[1], steps, "cuda")
            for n in ((30, 31, 32), (44, 20, 25))]
    want = []
    for dr in runs:
        dr.run()
        torch.cuda.synchronize()
        want.append(_outputs(dr))
        dr.reset()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in runs]
    for _ in range(2):
        for s, dr in zip(streams, runs):
            with torch.cuda.stream(s):
                dr.reset()
                dr.run()
    torch.cuda.synchronize()
    for dr, w in zip(runs, want):
        assert all(torch.equal(a, b) for a, b in zip(_outputs(dr), w))
        dr.close()


def test_device_held_by_another_process(R):
    """While somebody else holds the device for resident launches, runs take
    the two-pass step (the holder is played by a socket of this process)."""
    import gc
    import socket
    import torch
    from rfx_amd import autotune as at
    from rfx_amd.engine import DeviceRun
    gc.collect()                          # no plan of this process holds it
    p = torch.cuda.get_device_properties(0)
    name = f"{p.pci_domain_id:04x}:{p.pci_bus_id:02x}:{p.pci_device_id:02x}.0"
    _, prob, _ = cases.to_sim(_spec((20, 21, 22), 6))._build_problem(40, "run")
    want = DeviceRun(prob, 40, "cuda")
    want.run()
    torch.cuda.synchronize()
    ref = _outputs(want)
    want.close()
    with socket.socket(socket.AF_UNIX, socket.SOCK_DGRAM) as s:
        s.bind("\0rfxhip-resident-" + name)
        dr = DeviceRun(prob, 40, "cuda")
        dr.run()
        torch.cuda.synchronize()
        assert at.get_variant(dr) != (9, 0)
        assert all(torch.equal(a, b) for a, b in zip(_outputs(dr), ref))
        dr.close()
