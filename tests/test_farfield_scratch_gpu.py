"""The far-field transform where its partial sums are at their bound, so that a
row segment is longer than the 32 rows that LDS holds: against the float64
oracle, with the tolerance of test_farfield_tiles_gpu.py (the sums here have
up to 5e3 terms with phases below 100 rad)."""
import numpy as np
import pytest

from oracle import fdtd_np as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size, nf, n_theta, n_phi, rows", [
    ((333, 2, 3), 20, 25, 129, 167),     # 1020 direction tiles, two segments
    ((110, 3, 2), 16, 41, 96, 55),       # odd last chunks of rows
])
def test_long_row_segments(size, nf, n_theta, n_phi, rows):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import rfx_amd as R
    from rfx_amd import farfield as F
    one = 6 * 4 * nf * n_theta * n_phi * 16
    assert -(-n_theta * n_phi // 64) * nf < 1024          # the faces are split
    assert -(-size[0] // 32) * one > 48 << 20              # by 32 rows it would pass the bound
    assert -(-size[0] // ((48 << 20) // one)) == rows > 32
    print("[gpu-case] far field, long segments", size, nf, n_theta, n_phi, flush=True)
    rng = np.random.default_rng(sum(size) + nf)
    lo, dx = (3, 2, 4), 1e-3
    hi = tuple(a + n for a, n in zip(lo, size))
    grid = R.Grid(25e9, tuple((h + 2.5) * dx for h in hi), dx, 0)
    freqs = np.linspace(3e9, 14e9, nf).astype(np.float32)
    box = F.NTFFBox(lo[0], hi[0], lo[1], hi[1], lo[2], hi[2], freqs)
    theta, phi = np.linspace(0.0, np.pi, n_theta), np.linspace(0.1, 5.0, n_phi)
    x = {name: rng.standard_normal((nf,) + s + (4,)) + 1j * rng.standard_normal((nf,) + s + (4,))
         for name, s in zip(o.NTFF_FACES, o.ntff_face_shapes(lo, hi))}
    pos, width = o.ntff_axis_tables(grid.shape, dx)
    et, ep = o.far_field(x, lo, hi, freqs, pos, width, theta, phi)
    big = max(np.abs(et).max(), np.abs(ep).max())
    got = F.compute_far_field(F.NTFFData(*[x[n] for n in o.NTFF_FACES]), box, grid, theta, phi)
    assert np.abs(got.E_theta - et).max() <= 1e-11 * big
    assert np.abs(got.E_phi - ep).max() <= 1e-11 * big
