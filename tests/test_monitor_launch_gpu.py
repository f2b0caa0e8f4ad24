"""All DFT planes, flux monitors and NTFF faces of a plan go in one launch:
each accumulator has to be, bit for bit, the one of a plan that holds its
monitor alone (one entry, no search among block starts), on both field sets,
in pieces, and with faces of fewer than 256 points, of a multiple of 256 and
of ragged sizes."""
import numpy as np
import pytest

from tests import cases
from tests.test_resident_gpu import _spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, cpml", [((6, 5, 4), 0), ((32, 16, 16), 0), ((37, 21, 29), 6)])
@pytest.mark.parametrize("variant", [(0, 1), (4, 0), (1, 0)])
def test_each_monitor_equals_its_own_plan(n, cpml, variant):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from rfx_amd import autotune as at
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] monitors", n, cpml, variant, flush=True)
    steps = 31

    def accs(spec):
        _, prob, _ = cases.to_sim(spec)._build_problem(steps, "run")
        dr = DeviceRun(prob, steps, "cuda", two_sets=True)
        at.set_variant(dr, *variant)
        dr.reset()
        lo = 0
        for m in (6, 1, 13, 11):
            dr.run(lo, m)
            lo += m
        torch.cuda.synchronize()
        out = [x.clone() for x in [*dr.plane_acc, *dr.flux_acc]]
        dr.close()
        return out

    spec = _spec(n, cpml)
    together = accs(spec)
    alone = []
    for key in ("dft_planes", "flux_monitors"):
        for m in spec[key]:
            alone += accs(dict(spec, dft_planes=[], flux_monitors=[]) | {key: [m]})
    assert len(together) == len(alone) == 5
    assert all(torch.equal(a, b) for a, b in zip(together, alone))
    assert sum(float(np.abs(a.cpu().numpy()).max()) > 0 for a in together) >= 3
