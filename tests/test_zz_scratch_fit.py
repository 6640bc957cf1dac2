"""GPU test of pme_recip_solve_noalloc at the edge of its 64 MiB scratch: 64^3, order 6,
403,000 atoms (394 chunks of 1,024) fit with the 64 bricks of 16 points per edge but
not with the 252 that a solve with buffers of its own takes.  The call takes the fewer
bricks and gives the other solve's results bit for bit, and the handle's own plan is
in use again afterwards."""
import numpy as np
import pytest

from gpu_recip_amd import _lib as L
from gpu_recip_amd import systems
from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip
from gpu_util import to_dev, torch_dev

pytestmark = pytest.mark.gpu


def test_noalloc_takes_fewer_bricks_at_the_edge():
    torch, dev = torch_dev()
    n, nfft, box = 403000, (64, 64, 64), (150.0, 160.0, 155.0)
    s = systems.PmeSystem("t", systems.triplets(n // 3 + 1, box, 41), box, nfft, 6, 0.34)
    x = to_dev(s.xyzq)

    def run(pme, ev, fn):
        f = torch.zeros(n, 3, dtype=torch.float32, device=dev)
        ev.clear()
        fn(x, n, s.recip, s.kappa, True, True, n, f, L.FORCE_FLOAT3)
        ev.copyToHost()
        torch.cuda.synchronize()
        return f, ev.getEnergy("recip"), np.array(ev.getVirial())

    ev_a, ev_b = CudaEnergyVirial(), CudaEnergyVirial()
    pa, pb = CudaPMERecip(*nfft, 6, ev_a), CudaPMERecip(*nfft, 6, ev_b)
    want = run(pa, ev_a, pa.solve)
    for fn in (pb.solve_noalloc, pb.solve, pb.solve_noalloc):
        got = run(pb, ev_b, fn)
        assert torch.equal(got[0], want[0]) and got[1] == want[1] and np.array_equal(got[2], want[2])
    # 409,000 atoms (400 chunks) do not fit with any plan
    with pytest.raises(L.PmeError) as e:
        pb.solve_noalloc(to_dev(np.tile(s.xyzq, (2, 1))), 409000, s.recip, s.kappa, True, True, 409000,
                         torch.zeros(409000, 3, dtype=torch.float32, device=dev), L.FORCE_FLOAT3)
    assert e.value.status == 4  # PME_ERR_BUDGET
