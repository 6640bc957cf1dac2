"""One atom, the smallest input of the binning.  Its force is what is left when the
terms of its stencil cancel, so the bound is absolute: 1e-6 (16 FP32 roundings of
2^-24) of the sum of the terms' sizes, formed from the FP64 oracle's potential.
Energy as in the other single solves, batch equal to the single solve bit for bit."""
import numpy as np
import pytest

import oracle as O
from gpu_recip_amd import _lib as L
from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip, PmeBatch

pytestmark = pytest.mark.gpu
CCELEC = 332.0716


@pytest.mark.parametrize("order", [4, 6, 8])
def test_lone_atom(order):
    import torch

    nfft = (16, 16, 16)
    rng = np.random.default_rng(1 + order)
    box = np.array(nfft) * 0.9
    x = np.empty((1, 4), np.float32)
    x[:, :3] = rng.random((1, 3)) * box
    x[:, 3] = rng.uniform(-1, 1, 1)
    recip = list(np.diag(1.0 / box).reshape(-1))
    p = O.OracleParams(*nfft, order, 0.34, tuple(box), index_mode=O.INDEX_F32)
    o = O.solve(p, x, want_grids=True)
    # sum over the stencil of |q dtheta theta theta phi| n/L, per component
    idx, fr = O.index_f32(x, [recip[0], recip[4], recip[8]], nfft)
    th, dth = zip(*(O.bspline(order, fr[0][a]) for a in range(3)))
    at = [(idx[0][a] + np.arange(order)) % nfft[a] for a in range(3)]
    phi = np.abs(o["phi"][np.ix_(at[2], at[1], at[0])])
    size = np.empty(3)
    for a in range(3):
        w = [np.abs(dth[c] if c == a else th[c]) for c in range(3)]
        size[a] = CCELEC * abs(x[0, 3]) * nfft[a] / box[a] * np.einsum("zyx,z,y,x->", phi, w[2], w[1], w[0])
    assert (np.abs(o["force"][0]) < 1e-2 * size).all()  # the terms do cancel
    xd = torch.from_numpy(x).cuda()
    ev = CudaEnergyVirial()
    pme = CudaPMERecip(*nfft, order, ev)
    f = torch.zeros(1, 3, device="cuda")
    ev.clear()
    pme.solve(xd, 1, recip, 0.34, True, True, 1, f, L.FORCE_FLOAT3)
    ev.copyToHost()
    b = PmeBatch(1 << 30)
    fb = torch.zeros(1, 3, device="cuda")
    i = b.add(PmeBatch.desc(list(nfft), order, 0.34, recip, xd, 1, fb, L.FORCE_FLOAT3, 1), keep=(xd, fb))
    torch.cuda.synchronize()
    b.solve()
    e, _ = b.results([i])
    torch.cuda.synchronize()
    assert (np.abs(f.cpu().numpy()[0] - o["force"][0]) < 1e-6 * size).all()
    assert abs(ev.getEnergy("recip") - o["energy"]) < 1e-5 * abs(o["energy"])
    assert torch.equal(f, fb) and abs(e[0] - ev.getEnergy("recip")) <= 1e-12 * abs(e[0])
