"""The dispersive one-cell E pass (first pole of each kind loaded with the
fields, cells with poles found by a bit of their material id) against the
batched E pass (poles read after the curl): equal bit for bit, for none, one
and several poles of each kind and for pole materials whose ids do not fit
one 64-bit word."""
import numpy as np
import pytest

from tests import cases
from tests.test_resident_gpu import _outputs, _spec

pytestmark = pytest.mark.gpu

DEBYE = [(2.0, 6e-12), (0.7, 2e-11), (0.3, 4e-12)]
# (omega_0, delta, kappa = delta_eps omega_0^2)
LORENTZ = [(w, d, de * w * w) for de, w, d in ((1.1, 2 * np.pi * 11e9, 2e9),
                                               (0.4, 2 * np.pi * 17e9, 5e9))]


@pytest.mark.parametrize("nd, nl, extra", [(1, 0, 0), (0, 1, 0), (1, 1, 0), (3, 2, 0), (2, 1, 70)])
def test_equals_the_batched_pass(nd, nl, extra):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from rfx_amd import autotune as at
    from rfx_amd.batch import Batch
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] poles", nd, nl, extra, flush=True)
    steps = 40
    spec = _spec((29, 24, 21), 6)
    spec.update(dft_planes=[], flux_monitors=[], debye={"d": DEBYE[:nd]}, lorentz={"d": LORENTZ[:nl]})
    dx = 1e-3
    spec["materials"] = dict(spec["materials"])
    boxes = []
    for q in range(extra):      # one cell each, before the pole material
        name = f"x{q}"
        spec["materials"][name] = (2.0 + 0.05 * q, 0.0, 1.0)
        lo = ((q % 14 + 0.5) * dx, (q // 14 + 0.5) * dx, 1.5 * dx)
        boxes.append((lo, tuple(v + 0.9 * dx for v in lo), name))
    spec["geometry"] = boxes + spec["geometry"]
    sim = cases.to_sim(spec)
    _, prob, _ = sim._build_problem(steps, "run")
    dr = DeviceRun(prob, steps, "cuda", two_sets=False)
    assert (len(dr.flags) > 64) == (extra > 0)
    at.set_variant(dr, 0, 1)
    dr.reset()
    dr.run(0, steps)
    torch.cuda.synchronize()
    alone = _outputs(dr)
    dr.close()
    # (the second instance's slabs meet, so the batch takes the general pass)
    b = Batch([sim, cases.to_sim(_spec((3, 17, 40), 6))], steps)
    b.run()
    both = _outputs(b.runs[0])
    b.close()
    assert float(alone[0].abs().max()) > 0
    assert all(torch.equal(x, y) for x, y in zip(alone, both))
