"""Split-precision y axes inside the register four-step planes: every codelet
beside the 16-point one, even and odd x, lengths that keep the other planes or
passes, and batches with FP32 systems beside them."""
import numpy as np
import pytest

import oracle as O
from gpu_recip_amd import _lib as L
from gpu_recip_amd import systems
from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip, PmeBatch
from gpu_util import rel_rms, to_dev, torch_dev

pytestmark = pytest.mark.gpu

# relative RMS of a spectrum against the FP64 FFT of the same grid, as the other
# split-precision tests have it
SPEC_TOL = {L.PREC_BF16X3: 5e-5, L.PREC_FP16X3: 5e-6}


@pytest.mark.parametrize("prec", [L.PREC_BF16X3, L.PREC_FP16X3])
@pytest.mark.parametrize("nfft", [
    (24, 32, 18), (25, 48, 20), (32, 64, 12), (45, 80, 10), (48, 96, 8), (30, 128, 9), (54, 144, 15), (27, 160, 8),
    (160, 192, 6),              # the largest plane: 192 = 16 x 12
    (20, 16, 24), (16, 240, 8), (12, 256, 8),  # no such pair: stages
])
def test_split_plane_spectrum_and_roundtrip(nfft, prec):
    torch, dev = torch_dev()
    box = tuple(0.9 * n for n in nfft)
    s = systems.PmeSystem("t", systems.triplets(999, box, 5), box, nfft, 4, 0.34)
    nx, ny, nz = nfft
    pme = CudaPMERecip(*nfft, 4, CudaEnergyVirial())
    pme.set_precision(prec)
    g = torch.empty(nx * ny * nz, dtype=torch.float32, device=dev)
    c = torch.empty((nx // 2 + 1) * ny * nz * 2, dtype=torch.float32, device=dev)
    pme.spread_charge(to_dev(s.xyzq), s.natom, s.recip)
    pme.copy_grid(L.GRID_REAL, g)
    pme.r2c_fft()
    pme.copy_grid(L.GRID_SPECTRUM, c)
    torch.cuda.synchronize()
    grid = g.cpu().numpy().astype(np.float64).reshape(nz, ny, nx)
    spec = c.cpu().numpy().astype(np.float64).view(np.complex128).reshape(nz, ny, nx // 2 + 1)
    assert rel_rms(spec, O.fft3d_r2c(grid)) < SPEC_TOL[prec]
    pme.c2r_fft()
    pme.copy_grid(L.GRID_REAL, g)
    torch.cuda.synchronize()
    back = g.cpu().numpy().astype(np.float64).reshape(nz, ny, nx)
    assert rel_rms(back, grid * (nx * ny * nz)) < 2 * SPEC_TOL[prec]


def test_split_planes_in_a_batch_match_single():
    torch, dev = torch_dev()
    b = PmeBatch(2 << 30)
    kept = []
    for k, (nfft, prec) in enumerate([((40, 48, 64), L.PREC_BF16X3), ((45, 80, 36), L.PREC_FP16X3),
                                      ((40, 48, 64), L.PREC_FP32), ((144, 144, 30), L.PREC_BF16X3),
                                      ((150, 160, 20), L.PREC_FP16X3), ((30, 30, 32), L.PREC_BF16X3)]):
        box = tuple(0.9 * n for n in nfft)
        s = systems.PmeSystem("t", systems.triplets(3000, box, 31 + k), box, nfft, 6, 0.34)
        x = to_dev(s.xyzq)
        f = torch.zeros(s.natom, 3, device=dev)
        i = b.add(PmeBatch.desc(nfft, 6, s.kappa, s.recip, x, s.natom, f, L.FORCE_FLOAT3, s.natom, precision=prec),
                  keep=(x, f))
        kept.append((s, x, f, prec, i))
    torch.cuda.synchronize()
    b.solve()
    e, _ = b.results([k[4] for k in kept])
    for n, (s, x, f, prec, _) in enumerate(kept):
        ev = CudaEnergyVirial()
        pme = CudaPMERecip(*s.nfft, 6, ev)
        pme.set_precision(prec)
        fs = torch.zeros(s.natom, 3, device=dev)
        ev.clear()
        pme.solve(x, s.natom, s.recip, s.kappa, True, True, s.natom, fs, L.FORCE_FLOAT3)
        ev.copyToHost()
        torch.cuda.synchronize()
        assert torch.equal(f, fs), (s.nfft, prec)
        assert abs(e[n] - ev.getEnergy("recip")) <= 1e-12 * abs(e[n])
