"""The default step of very large grids with DFT planes, in pieces whose
two-pass tails (up to three steps) begin and end anywhere in the 16-step groups
of the planes' folds, eagerly and from graphs: accumulators, CPML memory, fields
and samples equal the two-pass step's bit for bit, as the same samples are
added in the same order."""
import numpy as np
import pytest

from tests import cases
from tests.test_resident_gpu import _spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, cpml", [((624, 255, 255), 0), ((604, 236, 236), 10)])
def test_planes_and_memory(n, cpml):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from rfx_amd import autotune as at
    from rfx_amd.engine import DeviceRun
    steps = 75
    spec = dict(_spec(n, cpml), flux_monitors=[])
    c = n[0] // 2 * 1e-3
    spec["dft_planes"] = spec["dft_planes"] + [("y", n[1] // 2 * 1e-3, "ex", np.array([9e9]), 1),
                                               ("x", c, "ez", np.array([8e9, 12e9]), 2)]
    _, prob, _ = cases.to_sim(spec)._build_problem(steps, "run")
    assert len(prob.planes) == 4
    dr = DeviceRun(prob, steps, "cuda", two_sets=True)
    assert at.get_variant(dr)[0] == 8
    # (the tails start at 4, 11, 16, 18, 27, 30, 41 and 74)
    pieces = {"eager": (7, 5, 6, 1, 11, 3, 9, 33), "graph": (75,), "two-pass": (75,)}
    res = {}
    for how, cut in pieces.items():
        print("[gpu-case] default sweep with planes", n, cpml, how, flush=True)
        if how == "two-pass":
            at.set_variant(dr, 0, 1)
        dr.reset()
        lo = 0
        for m in cut:
            dr.run(lo, m, use_graph=how != "eager")
            lo += m
        assert lo == steps
        torch.cuda.synchronize()
        assert dr.state_set() == 0
        res[how] = [x.clone() for x in (dr.probe_out, *dr.plane_acc, dr.psi, *dr.fields)]
    dr.close()
    assert all(float(x.abs().max()) > 0 for x in res["two-pass"][:4])
    for how in ("eager", "graph"):
        for q, (a, b) in enumerate(zip(res[how], res["two-pass"])):
            assert torch.equal(a, b), (how, q)
