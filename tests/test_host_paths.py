"""Host paths of the C ABI library that need a device to fail: run on the CPU
against a HIP runtime of its own (fake_hip.c), which keeps device memory on
the host, logs the launches instead of running them, and fails allocations on
request.  Each case runs in a process of its own that loads nothing else of
HIP."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "rfx_amd", "librfxhip.so")

PRELUDE = """
import ctypes as C, importlib.util, os, sys, types
import numpy as np
F = C.CDLL(os.environ["FAKE_HIP_SO"], mode=C.RTLD_GLOBAL)
F.fake_log.restype = C.c_char_p
F.fake_limit.argtypes = [C.c_longlong]
F.fake_live.restype = F.fake_peak.restype = C.c_longlong
F.fake_pinned.restype = C.POINTER(C.c_uint32)
sys.modules["torch"] = types.ModuleType("torch")     # (_lib imports it to share its runtime)
spec = importlib.util.spec_from_file_location("_lib", os.path.join(os.environ["ROOT"], "rfx_amd/_lib.py"))
L = importlib.util.module_from_spec(spec)
spec.loader.exec_module(L)
lib = L.load()
keep = []

def f32(a):
    a = np.ascontiguousarray(a, np.float32)
    keep.append(a)
    return a.ctypes.data_as(C.POINTER(C.c_float))

def buf(n, dt=np.float32):
    a = np.zeros(n, dt)
    keep.append(a)
    return a.ctypes.data

def desc(n, steps=100, two=True, cpml=(0,) * 6, planes=0, mem=None):
    # mem: cells that exist (grids whose kernels the fake runtime does not run)
    d = L.Desc()
    d.nx, d.ny, d.nz = n
    cells = mem or int(np.prod(n))
    for a in range(3):
        d.inv_e[a] = f32(np.full(n[a], 1e3))
        d.inv_h[a] = f32(np.full(n[a], 1e3))
    d.dt = 1e-12
    d.d_mat, d.n_mat = buf(cells, np.uint16), 1
    d.mat_coef = f32([1.0, 0.5, 0.5, 0.5])
    fl = np.zeros(1, np.uint32)
    keep.append(fl)
    d.mat_flags = fl.ctypes.data_as(C.POINTER(C.c_uint32))
    for c in range(6):
        d.d_f[c] = buf(cells)
        if two:
            d.d_f2[c] = buf(cells)
    for f in range(6):
        d.cpml_n[f] = cpml[f]
        if cpml[f]:
            for t in (d.cpml_b, d.cpml_c, d.cpml_km1):
                t[f] = f32(np.zeros(cpml[f]))
            d.cpml_inv_d[f] = 1e3
    if any(cpml):
        npsi = cells if mem else lib.rfxh_psi_floats(C.byref(d))
        d.d_psi, d.d_psi2 = buf(npsi), buf(npsi)
    d.max_steps = steps
    if planes:
        fr = np.array([1e9])
        keep.append(fr)
        pl = (L.Plane * planes)()
        for q in range(planes):
            pl[q].axis, pl[q].index, pl[q].comp, pl[q].n_freq = 0, q, 2, 1
            pl[q].freqs = fr.ctypes.data_as(C.POINTER(C.c_double))
            pl[q].d_acc = buf(2 * n[1] * n[2], np.float64)
        keep.append(pl)
        d.n_plane, d.planes = planes, pl
    return d

def create(d):
    p = C.c_void_p()
    L.check(lib.rfxh_plan_create(C.byref(d), C.byref(p)))
    return p

def variant(p):
    k, q = C.c_int(), C.c_int()
    L.check(lib.rfxh_get_variant(p, C.byref(k), C.byref(q)))
    return k.value

def run(p, lo=0, n=20):
    F.fake_clear()
    rc = lib.rfxh_run(p, lo, n, None, 1)
    return rc, [l.split() for l in F.fake_log().decode().splitlines()]

def resident(log):
    return [l for l in log if "k_resident" in l[0]]

def two_pass(log):
    return [l for l in log if "k_update_h" in l[0] or l[0] == "graph"]
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if not os.path.exists(LIB):
        pytest.skip("librfxhip.so not built")
    out = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", out, os.path.join(HERE, "fake_hip.c")],
                   check=True)

    def case(body, **env):
        e = dict(os.environ, FAKE_HIP_SO=out, ROOT=ROOT, FAKE_HIP_BUS=f"test-{os.getpid()}", **env)
        r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body)], env=e,
                           capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return case


def test_resident_workspace_is_whole_or_absent(fake):
    """Whichever allocation of a resident run's set-up fails, the run takes
    the two-pass step, no launch ever gets a missing parameter block, and
    nothing is left over."""
    fake("""
    start = F.fake_live()
    for nth in range(4):
        p = create(desc((12, 13, 14), planes=3))
        assert variant(p) == 9
        F.fake_fail_at(nth)
        for _ in range(2):
            rc, log = run(p)
            assert rc == 0, (nth, lib.rfxh_last_error())
            assert all(l[4] != "(nil)" for l in resident(log)), (nth, log)
            assert bool(resident(log)) != bool(two_pass(log)), (nth, log)
            if nth == 0 and _ == 0:
                assert two_pass(log)
        F.fake_fail_at(-1)
        L.check(lib.rfxh_plan_destroy(p))
        assert F.fake_live() == start
    """)


def test_a_resident_run_that_gave_up_is_reported(fake):
    """Every resident run ends with the kernel that looks at its stop word, and
    the word that kernel leaves for the host becomes an error of whichever
    call comes first; after it the plan takes the two-pass step until it is
    told otherwise."""
    fake("""
    for first in ("status", "run", "record", "batch"):
        p = create(desc((12, 13, 14), planes=2))
        b = C.c_void_p()
        L.check(lib.rfxh_batch_create(C.byref(p), 1, C.byref(b)))
        rc, log = run(p)
        assert rc == 0 and resident(log) and "k_res_check" in log[-1][0], log
        assert lib.rfxh_status(p) == 0
        F.fake_pinned()[0] = 1                       # as k_res_check does
        region = L.Region(0, 0, 0, 2, 2, 2)
        rec = buf(9 * 8 * 20)
        one, n = (C.c_int64 * 1)(0), (C.c_int64 * 1)(20)
        rc = {"status": lambda: lib.rfxh_status(p), "run": lambda: run(p)[0],
              "record": lambda: lib.rfxh_run_record(p, 0, 20, C.byref(region), rec, None),
              "batch": lambda: lib.rfxh_batch_run(b, one, n, None, 0)}[first]()
        assert rc < 0 and b"gave up" in lib.rfxh_last_error(), (first, rc)
        assert lib.rfxh_status(p) == 0 and variant(p) != 9
        rc, log = run(p)
        assert rc == 0 and two_pass(log) and not resident(log), log
        L.check(lib.rfxh_set_variant(p, 9, 0))
        rc, log = run(p)
        assert rc == 0 and resident(log), log
        L.check(lib.rfxh_batch_destroy(b))
        L.check(lib.rfxh_plan_destroy(p))
    """)


def test_resident_step_needs_a_unit_for_every_block(fake):
    """On a stream (or in a process) whose compute-unit mask has fewer units
    than the grid has blocks a run takes the two-pass step; on the next
    stream without one it is resident again."""
    body = """
    p = create(desc((40, 41, 42)))
    rc, log = run(p)
    assert rc == 0
    if os.environ.get("HSA_CU_MASK"):
        assert two_pass(log) and not resident(log)
        sys.exit(0)
    blocks = int(resident(log)[0][1])
    for units, res in ((blocks - 1, False), (blocks, True), (8, False), (-1, True)):
        F.fake_mask(units)
        rc, log = run(p)
        assert rc == 0 and bool(resident(log)) == res and bool(two_pass(log)) != res, (units, log)
        assert variant(p) == 9
    """
    fake(body)
    fake(body, HSA_CU_MASK="0:0-15")


def test_a_momentary_holder_costs_the_resident_step_for_its_time_only(fake):
    """Runs take the two-pass step while somebody else holds the device (or its
    memory), say so, and the resident step again when it is free."""
    fake("""
    import socket
    p = create(desc((12, 13, 14)))
    for _ in range(2):
        with socket.socket(socket.AF_UNIX, socket.SOCK_DGRAM) as s:
            s.bind("\\0rfxhip-resident-" + os.environ["FAKE_HIP_BUS"])
            rc, log = run(p)
            assert rc == 0 and two_pass(log) and not resident(log) and variant(p) != 9, log
        if _ == 0:
            L.check(lib.rfxh_set_variant(p, 9, 0))     # accepted, and what the plan is set to
            assert variant(p) == 9
    F.fake_limit(1)
    rc, log = run(p)
    assert rc == 0 and two_pass(log) and variant(p) != 9
    F.fake_limit(-1)
    rc, log = run(p)
    assert rc == 0 and resident(log) and variant(p) == 9, log
    """)


def test_a_run_allocates_nothing_that_ends_a_capture_elsewhere(fake):
    """The first resident run's allocations are made in the relaxed capture
    mode, and the thread's own mode is back afterwards; a run on a stream
    under capture allocates nothing and takes the two-pass step."""
    fake("""
    p = create(desc((12, 13, 14), planes=2))
    F.fake_capture(1)
    rc, log = run(p, n=5)
    assert rc == 0 and two_pass(log) and not resident(log)
    F.fake_capture(0)
    live = F.fake_live()
    rc, log = run(p)
    assert rc == 0 and resident(log) and F.fake_live() > live
    assert not any(l[0].startswith("malloc") for l in log), log
    F.fake_clear()
    create(desc((4, 4, 4)))
    assert "malloc-global" in F.fake_log().decode()
    """)


def test_resident_workspace_is_bounded(fake):
    """However many samples a step stages, the workspace stays within 100 MB:
    the rings hold fewer steps, and where they would hold fewer than four the
    plan does not take the resident step."""
    fake("""
    for n, faces, res in (((8, 352, 352), 32, True), ((8, 352, 352), 7, True),
                          ((3, 352, 352), 32, True), ((8, 352, 352), 1, True),
                          ((8, 352, 352), -32, False),
                          ((8, 352, 352), -8, True)):
        d = desc(n, steps=100, planes=max(faces, 0), mem=1)
        for q in range(faces):
            d.planes[q].index = q % n[0]
        if faces < 0:                                # flux monitors: four samples a point
            fr = np.array([1e9])
            fl = (L.Flux * -faces)()
            for f in fl:
                f.axis, f.index, f.lo1, f.n1, f.lo2, f.n2, f.n_freq = 0, 1, 0, n[1], 0, n[2], 1
                f.freqs, f.d_acc = fr.ctypes.data_as(C.POINTER(C.c_double)), buf(8)
            d.n_flux, d.flux = -faces, fl
        p = create(d)
        assert (variant(p) == 9) == res, (n, faces)
        F.fake_peak()
        rc, log = run(p, n=100)
        assert rc == 0 and bool(resident(log)) == res, (n, faces)
        assert F.fake_peak() <= 100e6, (n, faces)
    """)


def test_what_the_resident_step_leaves_takes_the_two_pass_step(fake):
    """Short and timed runs of a plan set to the resident step, whatever it was
    set to before."""
    fake("""
    for before in (1, 2, 3, 4, 7, 8):
        p = create(desc((12, 13, 14)))
        L.check(lib.rfxh_set_variant(p, before, 0))
        rc, log = run(p, n=3)
        assert rc == 0
        cur = lib.rfxh_state_set(p)
        L.check(lib.rfxh_set_variant(p, 9, 0))
        rc, log = run(p, n=3)
        assert rc == 0 and len(two_pass(log)) == 3 and not resident(log), (before, log)
        L.check(lib.rfxh_set_timing(p, 1))
        rc, log = run(p)
        assert rc == 0 and two_pass(log) and lib.rfxh_state_set(p) == cur, (before, log)
        L.check(lib.rfxh_set_timing(p, 0))
        rc, log = run(p)
        assert rc == 0 and resident(log) and lib.rfxh_state_set(p) == cur
    """)


@pytest.mark.parametrize("size, nf, n_theta, n_phi", [
    ((480, 470, 300), 4, 181, 72),       # 816 direction tiles
    ((1000, 990, 40), 4, 120, 133),
    ((86, 85, 84), 4, 37, 72),
    ((300, 300, 300), 1, 2, 3),
])
def test_far_field_scratch_is_bounded_and_dispensable(fake, size, nf, n_theta, n_phi):
    """The transform's scratch stays within 48 MiB and the tables, forward and
    reverse (whose own sums it cannot do without), and where the device has
    room for those alone the transform runs without the rest."""
    fake(f"""
    size, nf, nt, nph = {size}, {nf}, {n_theta}, {n_phi}
    th, ph, fr = (np.linspace(1.0, 2.0, k) for k in (nt, nph, nf))
    ptr = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
    tabs = [np.ones(s + 5) for s in size]
    d = L.FarFieldDesc()
    for a in range(3):
        d.lo[a], d.hi[a], d.n_axis[a] = 2, 2 + size[a], size[a] + 5
        d.pos[a] = d.width[a] = ptr(tabs[a])
    d.n_freq, d.freqs, d.c0, d.eta0 = nf, ptr(fr), 3e8, 377.0
    for f in range(6):
        d.d_acc[f] = buf(1)
    out = (C.c_void_p * 6)(*[buf(1)] * 6)
    table = 8 * (9 * nt * nph + nf + 2 * sum(size) + 32)
    sums = 8 * 24 * nf * nt * nph
    def forward():
        return lib.rfxh_ntff_far_field(C.byref(d), nt, ptr(th), nph, ptr(ph), buf(1), buf(1), None)
    def reverse():
        return lib.rfxh_ntff_far_field_adjoint(C.byref(d), nt, ptr(th), nph, ptr(ph), buf(1), buf(1),
                                               C.cast(out, C.POINTER(C.c_void_p)), None)
    for call, need, split in ((forward, table, "k_far_field_sum"),
                              (reverse, table + sums, "k_far_field_adj_sum")):
        F.fake_clear()
        F.fake_peak()
        assert call() == 0
        log = F.fake_log().decode()
        assert F.fake_peak() <= (48 << 20) + need, call
        F.fake_limit(need)
        F.fake_clear()
        assert call() == 0, lib.rfxh_last_error()
        assert split not in F.fake_log().decode() and "k_far_field" in F.fake_log().decode()
        F.fake_limit(1)
        assert call() == -3, lib.rfxh_last_error()
        F.fake_limit(-1)
    """)


def test_launches_of_single_step_runs(fake):
    """A run of one step is four launches (the step counter, H, E, the counter),
    of n two-pass steps 2 n + 2, whatever the plan runs otherwise."""
    fake("""
    p = create(desc((12, 13, 14)))
    for v in (0, 4, 9):
        L.check(lib.rfxh_set_variant(p, v, 0))
        for n in (1, 2, 3):
            rc, log = run(p, n=n)
            assert rc == 0 and len(log) == 2 * n + 2, (v, n, log)
    """)


def test_a_lacking_launch_is_one_workgroup_short(fake):
    body = """
    p = create(desc((40, 41, 42)))
    rc, log = run(p)
    print("BLOCKS", resident(log)[0][1])
    """
    assert int(fake(body).split("BLOCKS ")[1].split()[0]) == 1 + int(
        fake(body, RFXH_RESIDENT_LACKING="1").split("BLOCKS ")[1].split()[0])
