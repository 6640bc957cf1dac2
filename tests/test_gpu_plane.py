"""GPU test of the register four-step plane passes: forward spectrum and round
trip against the FP64 FFT at the edges of their range.  Tolerance: FP32
transforms of up to 2^22 points through about 12 radix steps round to a few
1e-7 relative RMS; 3e-6 is the bound of the other transform tests."""
import numpy as np
import pytest

import oracle as O
from gpu_recip_amd import _lib as L
from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip
from gpu_util import rel_rms, say, to_dev, torch_dev

pytestmark = pytest.mark.gpu

SHAPES = [
    (8, 4, 4),        # shortest lines: x 2*2, y 2*2
    (12, 9, 5),       # x 2*3, y 3*3
    (18, 6, 8),       # odd half length (no self-paired column)
    (9, 15, 6),       # odd nx and ny: paired rows, last row alone
    (25, 36, 4),      # odd nx, even ny
    (30, 150, 6),     # x 3*5, y 10*15
    (150, 20, 6),     # x 5*15
    (135, 135, 4),    # the largest odd plane (two LDS buffers)
    (180, 180, 4),    # y 12*15
    (192, 192, 4),    # the largest plane of one buffer
    (16, 192, 4),     # long y, short x
    (40, 256, 4),     # y 16*16 is beyond the pair passes: Stockham planes
]


@pytest.mark.parametrize("nfft", SHAPES)
def test_plane_spectrum_and_roundtrip(nfft):
    torch, dev = torch_dev()
    nx, ny, nz = nfft
    say(f"  plane passes {nfft}")
    rng = np.random.default_rng(nx * ny + nz)
    box = [0.9 * n for n in nfft]
    n = 400
    x = np.empty((n, 4), np.float32)
    x[:, :3] = rng.random((n, 3)) * box
    x[:, 3] = rng.standard_normal(n)
    pme = CudaPMERecip(nx, ny, nz, 4, CudaEnergyVirial())
    g = torch.empty(nx * ny * nz, dtype=torch.float32, device=dev)
    c = torch.empty((nx // 2 + 1) * ny * nz * 2, dtype=torch.float32, device=dev)
    pme.spread_charge(to_dev(x), n, [1 / box[0], 0, 0, 0, 1 / box[1], 0, 0, 0, 1 / box[2]])
    pme.copy_grid(L.GRID_REAL, g)
    pme.r2c_fft()
    pme.copy_grid(L.GRID_SPECTRUM, c)
    torch.cuda.synchronize()
    grid = g.cpu().numpy().astype(np.float64).reshape(nz, ny, nx)
    spec = c.cpu().numpy().astype(np.float64).view(np.complex128).reshape(nz, ny, nx // 2 + 1)
    assert rel_rms(spec, O.fft3d_r2c(grid)) < 3e-6
    pme.c2r_fft()
    pme.copy_grid(L.GRID_REAL, g)
    torch.cuda.synchronize()
    back = g.cpu().numpy().astype(np.float64).reshape(nz, ny, nx)
    assert rel_rms(back, grid * (nx * ny * nz)) < 3e-6
