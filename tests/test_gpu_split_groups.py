"""Split-precision planes with several z planes per workgroup: batches with 2 and 4
planes per item for at least two items per CU (256 CUs), even and odd nx, planes that
fit the group once, twice or four times, nz not a multiple of the group.  Forces equal
the single-system solver's, which transforms one plane per workgroup, bit for bit."""
import pytest

from gpu_recip_amd import _lib as L
from gpu_recip_amd import systems
from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip, PmeBatch
from gpu_util import to_dev, torch_dev

pytestmark = pytest.mark.gpu

GRIDS = [(24, 32, 27), (25, 48, 30), (32, 64, 25), (45, 80, 45), (90, 96, 54), (20, 160, 27)]


@pytest.mark.parametrize("group,reps", [(2, 6), (4, 11)])
def test_split_plane_groups_match_single(group, reps):
    torch, dev = torch_dev()
    assert 2 * 256 * group <= reps * sum(n[2] for n in GRIDS) < 2 * 256 * (group + 1)
    b = PmeBatch(8 << 30)
    kept = []
    for rep in range(reps):
        for k, nfft in enumerate(GRIDS):
            box = tuple(0.9 * n for n in nfft)
            s = systems.PmeSystem("t", systems.triplets(200, box, 500 + 10 * rep + k), box, nfft, 4, 0.34)
            prec = (L.PREC_BF16X3, L.PREC_FP16X3)[(rep + k) % 2]
            x = to_dev(s.xyzq)
            f = torch.zeros(s.natom, 3, device=dev)
            i = b.add(PmeBatch.desc(nfft, 4, s.kappa, s.recip, x, s.natom, f, L.FORCE_FLOAT3, s.natom,
                                    precision=prec), keep=(x, f))
            kept.append((s, x, f, prec, i))
    torch.cuda.synchronize()
    b.solve()
    e, _ = b.results([k[4] for k in kept])
    for n, (s, x, f, prec, _) in enumerate(kept):
        ev = CudaEnergyVirial()
        pme = CudaPMERecip(*s.nfft, 4, ev)
        pme.set_precision(prec)
        fs = torch.zeros(s.natom, 3, device=dev)
        ev.clear()
        pme.solve(x, s.natom, s.recip, s.kappa, True, True, s.natom, fs, L.FORCE_FLOAT3)
        ev.copyToHost()
        torch.cuda.synchronize()
        assert torch.equal(f, fs), (s.nfft, prec)
        assert abs(e[n] - ev.getEnergy("recip")) <= 1e-12 * abs(e[n])
