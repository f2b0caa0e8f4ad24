"""The far-field transform and its reverse mode at the edges of their tiles
(64 directions, 32 rows in segments of at least 4, 8 columns; 64 columns x 16
rows and 32 directions in reverse; one segment or several, one workgroup for
all faces where directions x frequencies fill the device): E_theta, E_phi
against the float64 oracle, the face gradients by the dot-product identity
Re <G, A x> = Re <A^H G, x> with the oracle's A x.  float64 sums of up to 1e4
unit-size terms with phases below 100 rad: 1e4 x 2^-53 x 100 = 1e-10 relative
at worst, a few 1e-14 expected; held to 1e-11."""
import numpy as np
import pytest

from oracle import fdtd_np as o

pytestmark = pytest.mark.gpu
TOL = 1e-11


@pytest.fixture(scope="module")
def F():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from rfx_amd import farfield
    return farfield


@pytest.mark.parametrize("size, nf, n_theta, n_phi", [
    ((1, 1, 1), 1, 1, 1),
    ((2, 1, 9), 1, 8, 8),                # 64 directions exactly, one column tile and a bit
    ((33, 32, 8), 2, 13, 5),             # 65 directions, 32 / 33 rows
    ((5, 16, 65), 1, 4, 16),
    ((17, 64, 7), 3, 3, 11),
    ((70, 13, 31), 1, 129, 1),
    ((6, 5, 4), 70, 32, 32),             # 1120 direction tiles: every face in one workgroup
])
def test_tiles(F, size, nf, n_theta, n_phi):
    import torch
    import rfx_amd as R
    print("[gpu-case] far field", size, nf, n_theta, n_phi, flush=True)
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
    plain = F.compute_far_field(F.NTFFData(*[x[n] for n in o.NTFF_FACES]), box, grid, theta, phi)
    faces = [torch.from_numpy(x[n]).cuda().requires_grad_(True) for n in o.NTFF_FACES]
    ff = F.compute_far_field(F.NTFFData(*faces), box, grid, theta, phi)
    for got in ((plain.E_theta, plain.E_phi), (ff.E_theta.detach().cpu().numpy(),
                                               ff.E_phi.detach().cpu().numpy())):
        assert np.abs(got[0] - et).max() <= TOL * big
        assert np.abs(got[1] - ep).max() <= TOL * big
    gt = rng.standard_normal(et.shape) + 1j * rng.standard_normal(et.shape)
    gp = rng.standard_normal(et.shape) + 1j * rng.standard_normal(et.shape)
    torch.autograd.backward([ff.E_theta, ff.E_phi],
                            [torch.from_numpy(gt).cuda(), torch.from_numpy(gp).cuda()])
    # face by face: the oracle's transform of one face alone
    for q, name in enumerate(o.NTFF_FACES):
        one = {n: x[n] if n == name else np.zeros_like(x[n]) for n in o.NTFF_FACES}
        at, ap = o.far_field(one, lo, hi, freqs, pos, width, theta, phi)
        left = np.sum((gt.conj() * at + gp.conj() * ap).real)
        g = faces[q].grad.cpu().numpy()
        right = np.sum((g.conj() * x[name]).real)
        scale = np.sum(np.abs(gt) * np.abs(at)) + np.sum(np.abs(gp) * np.abs(ap))
        assert abs(left - right) <= TOL * scale, name
