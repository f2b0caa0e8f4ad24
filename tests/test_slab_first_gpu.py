"""The two-pass kernels that load a cell's CPML memory before its fields are
waited for, at every column width and workgroup order, against the fused step
(each face's memory loaded after the curl): fields, memory and samples are
equal bit for bit.  Sizes: planes that columns do not divide (with and without
CPML), slabs that touch, and slabs of one axis that overlap (the plan then
keeps the general kernels)."""
import pytest

from tests import cases
from tests.test_resident_gpu import _outputs, _spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, cpml", [
    ((7, 5, 6), 0),
    ((29, 18, 35), 0),
    ((9, 12, 7), 3),
    ((19, 23, 70), 6),
    ((3, 17, 40), 6),       # slabs of x meet
    ((31, 2, 9), 8),        # of y and z
    ((70, 66, 33), 8),
])
def test_equals_the_fused_step(n, cpml):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from rfx_amd import autotune as at
    from rfx_amd.engine import DeviceRun
    steps = 23
    _, prob, _ = cases.to_sim(_spec(n, cpml))._build_problem(steps, "run")
    dr = DeviceRun(prob, steps, "cuda", two_sets=True)
    res = {}
    for v in ((1, 0), (0, 1), (0, 0), (4, 1), (6, 1), (5, 1), (5, 0)):
        print("[gpu-case] slab first", n, cpml, v, flush=True)
        at.set_variant(dr, *v)
        dr.reset()
        dr.run(0, steps)
        torch.cuda.synchronize()
        res[v] = _outputs(dr)
    dr.close()
    assert float(res[(1, 0)][0].abs().max()) > 0
    for v, out in res.items():
        for name, a, b in zip(("probes", "ports"), res[(1, 0)], out):
            assert torch.equal(a, b), (v, name)
        if v != (1, 0):     # (the fused step leaves its state in the other set)
            for q, (a, b) in enumerate(zip(res[(0, 1)], out)):
                assert torch.equal(a, b), (v, q)
