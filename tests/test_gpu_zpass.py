"""GPU test of the fused z pass against the stand-alone scalar sum: the same
potential, energy and virial for orthorhombic and triclinic boxes over the
factor pairs' edges.  Both evaluate the influence function by the same FP32
expressions, on spectra of the same transform up to rounding, so the potential
differs by FP32 transform rounding (3e-6, the transform tests' bound) and the
sums, quadratic in the spectrum, by less than twice that."""
import numpy as np
import pytest

from gpu_recip_amd import _lib as L
from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip
from gpu_util import rel_err, rel_fro, rel_rms, run_solve, say, to_dev, torch_dev

pytestmark = pytest.mark.gpu

SHAPES = [
    (12, 10, 16),   # 4 * 4: the shortest pair, even in every axis (Nyquist planes)
    (9, 15, 25),    # 5 * 5: odd in every axis
    (10, 9, 27),    # 3 * 9
    (15, 12, 75),   # 5 * 15
    (18, 20, 96),   # 8 * 12, last tile of lines not full
    (12, 10, 125),  # 5 * 25: the longest codelet
    (20, 9, 162),   # 9 * 18
    (8, 6, 192),    # 12 * 16: the longest pair
]


def _parts(nfft, recip, x, fused):
    torch, dev = torch_dev()
    nx, ny, nz = nfft
    ev = CudaEnergyVirial()
    pme = CudaPMERecip(nx, ny, nz, 4, ev)
    c = torch.empty((nx // 2 + 1) * ny * nz * 2, dtype=torch.float32, device=dev)
    g = torch.empty(nx * ny * nz, dtype=torch.float32, device=dev)
    ev.clear()
    pme.spread_charge(to_dev(x), len(x), recip)
    pme.r2c_fft()
    if not fused:  # completes the spectrum, so the stand-alone scalar sum runs
        pme.copy_grid(L.GRID_SPECTRUM, c)
    pme.scalar_sum(recip, 0.34, True, True)
    pme.c2r_fft()
    pme.copy_grid(L.GRID_REAL, g)
    ev.copyToHost()
    torch.cuda.synchronize()
    e, v, pot = ev.getEnergy("recip"), np.array(ev.getVirial()), g.cpu().numpy().astype(np.float64)
    # the solved spectrum as the second sum leaves it (a triclinic one is unscaled on both routes)
    pme.spread_charge(to_dev(x), len(x), recip)
    pme.r2c_fft()
    if not fused:
        pme.copy_grid(L.GRID_SPECTRUM, c)
    pme.scalar_sum(recip, 0.34, False, False)
    pme.copy_grid(L.GRID_SPECTRUM, c)
    torch.cuda.synchronize()
    return pot, e, v, c.cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("tric", [False, True])
@pytest.mark.parametrize("nfft", SHAPES)
def test_fused_z_pass_matches_stand_alone_sum(nfft, tric):
    say(f"  z pass {nfft} triclinic={tric}")
    box = [0.9 * n for n in nfft]
    H = np.diag(box)
    if tric:
        H[0, 1], H[0, 2], H[1, 2] = 0.15 * box[0], -0.1 * box[0], 0.2 * box[1]
    recip = np.linalg.inv(H).reshape(9)
    rng = np.random.default_rng(sum(nfft))
    x = np.empty((300, 4), np.float32)
    x[:, :3] = rng.random((300, 3)) @ H.T
    x[:, 3] = rng.standard_normal(300)
    p0, e0, v0, c0 = _parts(nfft, recip, x, False)
    p1, e1, v1, c1 = _parts(nfft, recip, x, True)
    assert rel_rms(p1, p0) < 3e-6
    assert rel_err(e1, e0) < 6e-6 and rel_fro(v1, v0) < 6e-6
    if tric:
        assert rel_rms(c1, c0) < 3e-6


@pytest.mark.parametrize("nz", [125, 162])
def test_long_codelets_in_a_batch_match_single(nz):
    from gpu_recip_amd import systems
    from gpu_recip_amd.pme import PmeBatch, force_stride
    torch, dev = torch_dev()
    nfft, box = (20, 18, nz), (18.0, 16.0, 0.9 * nz)
    x = systems.triplets(200, box, seed=nz)
    n, st = len(x), force_stride(len(x))
    recip = [1 / box[0], 0, 0, 0, 1 / box[1], 0, 0, 0, 1 / box[2]]
    b = PmeBatch(1 << 30)
    xd, f = to_dev(x), torch.zeros(3 * st, dtype=torch.float32, device=dev)
    sid = b.add(PmeBatch.desc(nfft, 4, 0.34, recip, xd, n, f, L.FORCE_FLOAT, st, True), keep=(xd, f))
    b.solve()
    e, v = b.results([sid])
    fh = f.cpu().numpy()
    one = run_solve(nfft, 4, 0.34, box, x)
    assert np.array_equal(np.stack([fh[:n], fh[st:st + n], fh[2 * st:2 * st + n]], 1).astype(np.float64), one["force"])
    assert rel_err(e[0], one["energy"]) < 1e-12 and rel_fro(v[0], one["virial"]) < 1e-12
