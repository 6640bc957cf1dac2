"""FP16x3 solves whose influence function falls below the smallest exponent that a
column can be scaled by: a fine grid with a small kappa leaves columns near the
Nyquist edges of x and y below 2^-114.  Forces and energy stay finite and as close
to the FP64 oracle as the FP32 transforms' (the bound of the 144^3 test)."""
import numpy as np
import pytest

import oracle as O
from gpu_recip_amd import _lib as L
from gpu_recip_amd import systems
from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip
from gpu_util import rel_err, rel_rms, to_dev, torch_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfft,spacing,kappa", [
    ((96, 96, 96), 0.80, 0.30),
    ((96, 96, 96), 0.87, 0.28),
    ((64, 80, 128), 0.80, 0.28),
    ((48, 64, 240), 0.78, 0.28),  # z in Stockham stages
])
def test_small_columns_stay_finite(nfft, spacing, kappa):
    torch, dev = torch_dev()
    box = tuple(spacing * n for n in nfft)
    s = systems.PmeSystem("t", systems.triplets(int(0.1 * box[0] * box[1] * box[2] / 3), box, 29), box, nfft, 4, kappa)
    natom = s.natom
    o = O.solve(O.OracleParams(*nfft, 4, kappa, box, index_mode=O.INDEX_F32), s.xyzq)
    x = to_dev(s.xyzq)
    res = {}
    for prec in (L.PREC_FP32, L.PREC_FP16X3):
        ev = CudaEnergyVirial()
        pme = CudaPMERecip(*nfft, 4, ev)
        pme.set_precision(prec)
        f = torch.zeros(natom, 3, dtype=torch.float32, device=dev)
        ev.clear()
        pme.solve(x, natom, s.recip, kappa, True, True, natom, f, L.FORCE_FLOAT3)
        ev.copyToHost()
        torch.cuda.synchronize()
        fr = f.cpu().numpy().astype(np.float64)
        assert np.isfinite(fr).all() and np.isfinite(ev.getEnergy("recip"))
        res[prec] = rel_rms(fr, o["force"]), rel_err(ev.getEnergy("recip"), o["energy"])
    assert res[L.PREC_FP16X3][0] < 2 * res[L.PREC_FP32][0] + 1e-6
    assert res[L.PREC_FP16X3][1] < 1e-5
