"""A plan's first resident run, whose workspace is allocated then, while the
same thread captures a graph on another stream: both come out right."""
import pytest

from tests import cases
from tests.test_resident_gpu import _outputs, _spec

pytestmark = pytest.mark.gpu


def test_first_run_beside_a_capture():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from rfx_amd import autotune as at
    from rfx_amd.engine import DeviceRun
    print("[gpu-case] resident, first run beside a capture", flush=True)
    steps = 30
    _, prob, _ = cases.to_sim(_spec((40, 30, 9), 8))._build_problem(steps, "run")
    ref, dr = (DeviceRun(prob, steps, "cuda") for _ in range(2))
    at.set_variant(ref, 0, 1)
    ref.run()
    x = torch.zeros(1000, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x += 1.0
        with torch.cuda.stream(side):
            dr.run()
        x *= 2.0
    assert at.get_variant(dr) == (9, 0)
    dr.check()
    assert all(torch.equal(a, b) for a, b in zip(_outputs(dr), _outputs(ref)))
    for n in (2.0, 6.0, 14.0):
        graph.replay()
        torch.cuda.synchronize()
        assert bool((x == n).all())
    dr.close()
    ref.close()
