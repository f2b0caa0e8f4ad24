"""The default step of very large grids (two steps a sweep): a run equals the
two-pass step's in probes and fields, in pieces,
captured by the caller and replayed, and leaves the state in the same field
set; a smaller or a flatter grid or deeper slabs keep the two-pass step."""
import pytest

from tests import cases
from tests.test_resident_gpu import _spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, cpml, sweep", [
    ((624, 255, 255), 0, True),
    ((604, 236, 236), 10, True),
    ((600, 234, 234), 11, False),   # z slabs deeper than the sweep's edge tiles
    ((620, 254, 260), 0, False),    # short rows of planes
    ((600, 255, 255), 0, False),    # fewer cells
])
def test_default(n, cpml, sweep):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from rfx_amd import autotune as at
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] default sweep", n, cpml, flush=True)
    steps = 24
    spec = dict(_spec(n, cpml), dft_planes=[], flux_monitors=[])
    _, prob, _ = cases.to_sim(spec)._build_problem(steps, "run")
    dr = DeviceRun(prob, steps, "cuda", two_sets=True)
    print("[gpu-case] shape", prob.shape, at.get_variant(dr), flush=True)
    assert at.get_variant(dr)[0] == (8 if sweep else 0)
    if sweep:
        res = []
        for how in ("pieces", "captured", "two-pass"):
            if how == "two-pass":
                at.set_variant(dr, 0, 1)
            dr.reset()
            lo = 0
            for m in ((7, 1, 2, 4) if how != "captured" else ()):
                dr.run(lo, m)
                lo += m
            if how == "captured":
                dr.run(0, 4)
                torch.cuda.synchronize()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g):       # steps 4 .. 13
                    dr.run(4, 10, use_graph=False)
                g.replay()
            torch.cuda.synchronize()
            assert dr.state_set() == 0
            res.append([x.clone() for x in (dr.probe_out, *dr.fields)])
        assert float(res[0][0].abs().max()) > 0
        for r in res[:2]:
            assert all(torch.equal(a, b) for a, b in zip(r, res[2]))
    dr.close()
