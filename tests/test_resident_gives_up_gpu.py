"""A resident run whose workgroups give up waiting (forced by leaving out the
last one, with a small poll limit, so that every kernel still ends) hands out
nothing that could be taken for a result: its fields, samples and accumulators
are NaN, the error is raised, and the plan goes on with the two-pass step."""
import numpy as np
import pytest

from tests import cases
from tests.test_resident_gpu import _outputs, _spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, cpml, faces, steps", [
    ((40, 30, 9), 8, 0, 40),
    ((96, 80, 63), 8, 0, 40),
    ((60, 60, 60), 6, 24, 95),            # several launches a run
])
def test_outputs_are_nan_and_the_error_is_raised(n, cpml, faces, steps, monkeypatch):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from rfx_amd import _lib
    from rfx_amd import autotune as at
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] resident run that gives up", n, flush=True)
    spec = _spec(n, cpml)
    if faces:
        spec["flux_monitors"] = [(ax, (4 + q) * 3e-3, np.array([8e9]), 1, None, None, "rect", 0.25)
                                 for q in range(faces // 3) for ax in "xyz"]
        per_step = faces * 16 * 73 * 73
        assert (64 << 20) // per_step < steps
    _, prob, _ = cases.to_sim(spec)._build_problem(steps, "run")
    monkeypatch.setenv("RFXH_RESIDENT_LACKING", "1")
    dr = DeviceRun(prob, steps, "cuda")
    monkeypatch.delenv("RFXH_RESIDENT_LACKING")
    ref = DeviceRun(prob, steps, "cuda")
    at.set_variant(ref, 0, 1)
    ref.run()
    ref.check()
    want = _outputs(ref)
    for _ in range(2):
        dr.reset()
        at.set_variant(dr, 9, 0)
        dr.run()
        torch.cuda.synchronize()
        outs = [dr.probe_out, *dr.fields, *dr.plane_acc, *dr.flux_acc]
        assert all(bool(torch.isnan(torch.view_as_real(x) if x.is_complex() else x).all())
                   for x in outs)
        with pytest.raises(_lib.RfxHipError, match="gave up"):
            dr.check()
        dr.check()
        assert at.get_variant(dr) != (9, 0)
        dr.reset()
        dr.run()
        dr.check()
        assert all(torch.equal(a, b) for a, b in zip(_outputs(dr), want))
    dr.close()
    ref.close()
    # through the user's call: no result is handed out
    monkeypatch.setenv("RFXH_RESIDENT_LACKING", "1")
    with pytest.raises(_lib.RfxHipError, match="gave up"):
        cases.to_sim(spec).run(n_steps=steps)
