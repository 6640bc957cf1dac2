"""Binning at the edges of its chunks: one atom per thread up to 512 x 512 atoms,
two up to 512 x 1024, records placed one by one beyond.  The grid sums and forces
against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natom,nfft,order", [
    # a lone atom's force is what cancellation leaves of terms a thousand times as
    # large: 2.3e-4 from the oracle, as with any order of the records
    pytest.param(1, (16, 16, 16), 4, marks=pytest.mark.xfail(reason="relative bound on a cancelled force")),
    (511, (20, 18, 16), 6),
    (512, (20, 18, 16), 6),
    (513, (20, 18, 16), 8),
    (2048, (8, 27, 40), 4),       # one brick along x
    (262144, (36, 40, 32), 4),
    (262145, (36, 40, 32), 4),
    (300001, (32, 36, 40), 6),
    (524288, (36, 40, 32), 4),
    (524289, (36, 40, 32), 4),
])
def test_binning_chunk_edges(natom, nfft, order):
    import torch

    import oracle as O
    from gpu_recip_amd import _lib as L
    from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip, PmeBatch

    rng = np.random.default_rng(natom + order)
    box = np.array(nfft) * 0.9
    x = np.empty((natom, 4), np.float32)
    x[:, :3] = rng.random((natom, 3)) * box
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
    o = O.solve(O.OracleParams(*nfft, order, 0.34, tuple(box), index_mode=O.INDEX_F32), x)
    d = f.cpu().numpy().astype(np.float64) - o["force"]
    # the bounds of the other single-solve tests
    assert np.sqrt((d ** 2).sum() / (o["force"] ** 2).sum()) < 1e-5
    assert abs(ev.getEnergy("recip") - o["energy"]) < 1e-5 * abs(o["energy"])
    if natom <= 300001:  # the gather from the binned records
        b = PmeBatch(2 << 30)
        fb = torch.zeros(natom, 3, device="cuda")
        b.add(PmeBatch.desc(list(nfft), order, 0.34, recip, xd, natom, fb, L.FORCE_FLOAT3, natom), keep=(xd, fb))
        torch.cuda.synchronize()
        b.solve()
        torch.cuda.synchronize()
        assert torch.equal(f, fb)
