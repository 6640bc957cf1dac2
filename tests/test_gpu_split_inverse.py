"""The split-precision z pass runs its hi-lo 16-point DFTs ahead of the other factor
in both directions: 250,002 atoms at 144^3 are then 3.79e-5 (relative RMS of the
forces) from the FP64 oracle, as in Stockham stages with the radix-16 stage first, and
3.83e-5 with the 16-point DFT behind the other factor in the inverse.  The batched z
pass gives the same forces."""
import pytest

import oracle as O
from gpu_recip_amd import _lib as L
from gpu_recip_amd import systems
from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip, PmeBatch
from gpu_util import rel_rms, to_dev, torch_dev

pytestmark = pytest.mark.gpu


def test_bf16_force_error_at_144():
    torch, dev = torch_dev()
    s = systems.config_split_precision()
    n = s.natom
    o = O.solve(O.OracleParams(*s.nfft, s.order, s.kappa, s.box, index_mode=O.INDEX_F64), s.xyzq)
    x = to_dev(s.xyzq)
    pme = CudaPMERecip(*s.nfft, s.order, CudaEnergyVirial())
    pme.set_precision(L.PREC_BF16X3)
    f = torch.zeros(n, 3, dtype=torch.float32, device=dev)
    pme.solve(x, n, s.recip, s.kappa, False, False, n, f, L.FORCE_FLOAT3)
    b = PmeBatch(2 << 30)
    fb = torch.zeros(n, 3, dtype=torch.float32, device=dev)
    b.add(PmeBatch.desc(list(s.nfft), s.order, s.kappa, s.recip, x, n, fb, L.FORCE_FLOAT3, n,
                        precision=L.PREC_BF16X3), keep=(x, fb))
    torch.cuda.synchronize()
    b.solve()
    torch.cuda.synchronize()
    err = rel_rms(f.cpu().numpy().astype("float64"), o["force"])
    assert err < 3.80e-5, err
    assert torch.equal(f, fb)
