"""Brick plans of single-system solves: small and uneven grids take bricks
narrower than 16 points, larger ones an uneven number per axis.  Integer grid
accumulation and per-atom gather sums make the forces independent of the plan, so
the solve must equal a batched one planned with bricks of 16 bit for bit; the
smallest also against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natom,nfft,order", [
    (30, (8, 8, 8), 4),       # one brick, or two of four points
    (301, (24, 27, 25), 4),
    (2001, (32, 32, 32), 4),
    (2001, (30, 36, 40), 6),  # narrowest bricks of order 6: five points
    (1501, (32, 45, 40), 8),  # seven points and up at order 8
    (23559, (64, 64, 64), 6),
    (60000, (144, 125, 108), 4),
])
def test_brick_plan_does_not_change_results(natom, nfft, order):
    import torch

    import oracle as O
    from gpu_recip_amd import _lib as L
    from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip, PmeBatch

    rng = np.random.default_rng(natom)
    box = np.array(nfft) * 0.9
    x = np.empty((natom, 4), np.float32)
    x[:, :3] = (rng.random((natom, 3)) * 1.4 - 0.2) * box  # some outside the box
    x[:, 3] = rng.uniform(-1, 1, natom)
    recip = list(np.diag(1.0 / box).reshape(-1))
    xd = torch.from_numpy(x).cuda()
    ev = CudaEnergyVirial()
    pme = CudaPMERecip(*nfft, order, ev)
    f = torch.zeros(natom, 3, device="cuda")
    ev.clear()
    pme.solve(xd, natom, recip, 0.34, True, True, natom, f, L.FORCE_FLOAT3)
    ev.copyToHost()
    torch.cuda.synchronize()
    b = PmeBatch(1 << 30)
    b.set_tuning(16, 16, 0)
    fb = torch.zeros(natom, 3, device="cuda")
    k = b.add(PmeBatch.desc(list(nfft), order, 0.34, recip, xd, natom, fb, L.FORCE_FLOAT3, natom,
                            calc_energy_virial=True), keep=(xd, fb))
    torch.cuda.synchronize()
    b.solve()
    e, _ = b.results([k])
    assert torch.equal(f, fb)
    assert abs(ev.getEnergy("recip") - e[0]) <= 1e-12 * abs(e[0])
    if natom <= 2001:
        o = O.solve(O.OracleParams(*nfft, order, 0.34, tuple(box), index_mode=O.INDEX_F32), x)
        d = f.cpu().numpy().astype(np.float64) - o["force"]
        # FP32 sums of order^3 terms on either side of the transforms: 1e-5 of the rms
        # force, the bound of the other single-solve tests
        assert np.sqrt((d ** 2).sum() / (o["force"] ** 2).sum()) < 1e-5
