"""GPU test of the pair kernel's tile queue at the edges of its range: lists of
one tile, of an odd number of tiles, of fewer and of more tiles than the launch
has waves.  Tolerance: the pair term is good to a few 1e-7, forces are sums of a
few hundred of them; 1e-5 relative RMS is the bound of the other direct tests."""
import numpy as np
import pytest

import oracle as O
from gpu_recip_amd import nlist, systems
from gpu_recip_amd.direct import CudaPMEDirectForce, DeviceTileList
from gpu_recip_amd.pme import CudaEnergyVirial, force_stride
from gpu_util import rel_err, rel_rms, say, torch_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntrip,boxl,roff", [(4, 19.0, 9.0), (11, 19.0, 9.0), (60, 20.0, 6.0), (4000, 50.0, 9.0)])
def test_direct_list_sizes(ntrip, boxl, roff):
    torch, dev = torch_dev()
    box = (boxl, boxl, boxl)
    x = systems.triplets(ntrip, box, seed=40 + ntrip)
    x[:, :3] = np.mod(x[:, :3].astype(np.float64), boxl).astype(np.float32)
    water = nlist.water_exclusions(len(x))
    tl = nlist.build(x, box, roff, excl_pairs=water)
    say(f"  {len(x)} atoms, {len(tl.ientry)} i entries, {len(tl.tile_indj)} j tiles")
    ev = CudaEnergyVirial()
    dr = CudaPMEDirectForce(ev)
    dr.setup(*box, 0.34, roff, roff - 1.0, 1.0)
    dl = DeviceTileList(tl, dev)
    stride = force_stride(tl.npad, 8)
    o = O.direct_ewald(x, box, 0.34, roff, excl=water)
    raw = []
    for _ in range(2):  # the queues are cleared by every call
        f = torch.zeros(3, stride, dtype=torch.int64, device=dev)
        ev.clear()
        dr.calc_force(dl.xyzq, dl, True, True, stride, f)
        ev.copyToHost()
        torch.cuda.synchronize()
        raw.append(f.cpu().numpy())
        force = raw[-1][:, tl.sorted_index()].T / 2.0 ** 40
        assert rel_rms(force, o["force"]) < 1e-5
        assert rel_err(ev.getEnergy("elec"), o["energy"]) < 1e-5
    assert np.array_equal(raw[0], raw[1])
