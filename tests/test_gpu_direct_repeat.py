"""The direct term's energy and shift forces are the same bits on every run, also where
the sums need more than 53 bits of their fixed point (charges of one sign: some 1e8
kcal/mol in all, where a 2^32 fixed-point sum of 2^21 fills an FP64 mantissa)."""
import numpy as np
import pytest

import oracle as O
from gpu_recip_amd import nlist, systems
from gpu_recip_amd.direct import CudaPMEDirectForce, DeviceTileList
from gpu_recip_amd.pme import CudaEnergyVirial, force_stride
from gpu_util import rel_err, rel_rms, torch_dev

pytestmark = pytest.mark.gpu


def test_large_sums_repeat_bit_for_bit():
    torch, dev = torch_dev()
    boxl, roff = 50.0, 9.0
    box = (boxl, boxl, boxl)
    x = systems.triplets(4000, box, seed=77)
    x[:, :3] = np.mod(x[:, :3].astype(np.float64), boxl).astype(np.float32)
    x[:, 3] = np.random.default_rng(7).uniform(6.0, 10.0, len(x)).astype(np.float32)
    water = nlist.water_exclusions(len(x))
    tl = nlist.build(x, box, roff, excl_pairs=water)
    ev = CudaEnergyVirial()
    dr = CudaPMEDirectForce(ev)
    dr.setup(*box, 0.34, roff, roff - 1.0, 1.0)
    dl = DeviceTileList(tl, dev)
    stride = force_stride(tl.npad, 8)
    o = O.direct_ewald(x, box, 0.34, roff, excl=water)
    runs = []
    for _ in range(8):
        f = torch.zeros(3, stride, dtype=torch.int64, device=dev)
        ev.clear()
        dr.calc_force(dl.xyzq, dl, True, True, stride, f)
        ev.copyToHost()
        torch.cuda.synchronize()
        runs.append((f.cpu().numpy(), ev.getEnergy("elec"), np.array(ev.getSforce())))
    f, e, sf = runs[0]
    assert rel_rms(f[:, tl.sorted_index()].T / 2.0 ** 40, o["force"]) < 1e-5
    assert e > 2.0 ** 24 and rel_err(e, o["energy"]) < 1e-5
    for g in runs[1:]:
        assert np.array_equal(g[0], f) and g[1] == e and np.array_equal(g[2], sf)
