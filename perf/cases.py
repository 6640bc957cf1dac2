"""The work a user of this engine has it do, as measurable cases.

listed() names the cases, draw() gives more of the same ranges, prepare() makes
what a program holds before the call (device inputs, solver handles, resident
systems, tile lists), run() is one pass through the public entry points and
exact() the same results in 64 bits by plain numpy and torch.

Kinds of case:
  solve   one system through CudaPMERecip: the five stage calls or solve(),
          with or without energy and virial (with them the step ends in the
          host readback an MD program does), any force layout, order 4/6/8,
          orthorhombic or triclinic box, FP32 or split-precision transforms
  batch   many resident systems per pass through PmeBatch
  serve   a burst of requests of uneven sizes through PmeServer
  direct  the direct-space Ewald term on a tile list, with the exclusion
          corrections, through CudaPMEDirectForce

Systems are boxes of water-like triplets at 0.1 atoms per cubic Angstrom with
a grid spacing of about 0.9 to 1 Angstrom.  Fixed-point (2^40) forces are
returned as float32, as an integrator reads them; energies and virials come
as one float32 tensor per call.
"""
import math

import numpy as np
import torch

CCELEC = 332.0716
Q_O, Q_H, R_OH, THETA = -0.834, 0.417, 0.9572, math.radians(104.52)
TRICLINIC = (0.13, -0.08, 0.11)  # tilts xy, xz, yz of a triclinic box, in units of the tilted-to edge


def _solve(name, natom, n, order, kappa, spacing, calls="five", ev=True, force="float", tric=False, prec="fp32",
           self_energy=False):
    return {"name": name, "kind": "solve", "natom": natom, "nx": n[0], "ny": n[1], "nz": n[2], "order": order,
            "kappa": kappa, "lx": round(n[0] * spacing, 4), "ly": round(n[1] * spacing, 4),
            "lz": round(n[2] * spacing, 4), "calls": calls, "ev": ev, "force": force, "tric": tric, "prec": prec,
            "self": self_energy}


def listed():
    return [
        # the smallest call: an MD step of a solvated peptide-sized box, forces only
        _solve("small-2k-32c-p4", 2001, (32, 32, 32), 4, 0.34, 0.85, calls="solve", ev=False),
        # the small benchmark solve, five stage calls, energy and virial read back every step
        _solve("small-8k-48c-p4-ev", 8001, (48, 48, 48), 4, 0.34, 40.0 / 48),
        # the drop-in sequence at the size of the reference's test system: fixed-point
        # forces added to an array shared with other terms, reciprocal and self energy
        _solve("dropin-24k-64c-p6-int64", 23559, (64, 64, 64), 6, 0.32, 62.23 / 64, force="int64", self_energy=True),
        # odd and uneven edges, no factor of two on two axes; AoS forces, an MD step
        _solve("ragged-50k-81x75x125-p6", 50001, (81, 75, 125), 6, 0.34, 0.87, calls="solve", ev=False,
               force="float3"),
        # a triclinic cell, energy and virial (constant-pressure runs)
        _solve("triclinic-54k-90x80x96-p6-ev", 54000, (90, 80, 96), 6, 0.32, 0.92, tric=True),
        # the production solve with everything read back
        {"name": "plain-96k-108x100x96-p6-ev", "kind": "solve", "natom": 96000, "nx": 108, "ny": 100, "nz": 96,
         "order": 6, "kappa": 0.32, "lx": 100.0, "ly": 96.0, "lz": 90.0, "calls": "five", "ev": True,
         "force": "float", "tric": False, "prec": "fp32", "self": False},
        # a large system's MD step, forces only
        _solve("md-250k-144c-p4", 250002, (144, 144, 144), 4, 0.30, 135.0 / 144, calls="solve", ev=False),
        # the same system with the transforms on the matrix cores
        _solve("split-250k-144c-p4-ev", 250002, (144, 144, 144), 4, 0.30, 135.0 / 144, prec="bf16x3"),
        # the largest single system
        _solve("large-400k-160c-p6-ev", 399999, (160, 160, 160), 6, 0.34, 1.0),
        # 64 uneven systems per launch, under the kind of plan the autotuner stores for them
        {"name": "batch-64-2k-40k-p4-ev", "kind": "batch", "nsys": 64, "mix": 2, "nmin": 2000, "nmax": 40000,
         "order": 4, "kappa": 0.34, "ev": True, "plan": "tuned"},
        # a burst of requests from 5k to 400k atoms, orders 4 and 6
        {"name": "serve-24-5k-400k", "kind": "serve", "nreq": 24, "mix": 4, "nmin": 5000, "nmax": 400000,
         "kappa": 0.34},
        # the direct-space half of a step, with the exclusion corrections
        {"name": "direct-24k-roff9-ev", "kind": "direct", "natom": 24000, "roff": 9.0, "kappa": 0.34, "ev": True},
    ]


def _smooth_near(x):
    """The 2/3/5-smooth integer nearest to x."""
    best = None
    for n in range(max(2, int(x * 0.8)), int(x * 1.25) + 3):
        m = n
        for f in (2, 3, 5):
            while m % f == 0:
                m //= f
        if m == 1 and (best is None or abs(n - x) < abs(best - x)):
            best = n
    return best


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choices(["solve", "batch", "serve", "direct"], [10, 3, 2, 2])[0]
    if kind == "solve":
        order = rng.choices([4, 6, 8], [5, 5, 2])[0]
        natom = 3 * int(_log_uniform(rng, 500, {4: 130000, 6: 120000, 8: 60000}[order]))
        edge = (natom / 0.1) ** (1.0 / 3.0)
        spacing = rng.uniform(0.87, 1.0)
        n = [min(180, max(24, _smooth_near(edge * rng.uniform(0.8, 1.2) / spacing))) for _ in range(3)]
        tric = rng.random() < 0.2
        prec = rng.choice(["bf16x3", "fp16x3"]) if rng.random() < 0.15 else "fp32"
        return {"kind": "solve", "natom": natom, "nx": n[0], "ny": n[1], "nz": n[2], "order": order,
                "kappa": round(rng.uniform(0.30, 0.36), 3), "lx": round(n[0] * spacing, 3),
                "ly": round(n[1] * spacing, 3), "lz": round(n[2] * spacing, 3),
                "calls": rng.choice(["five", "solve"]), "ev": rng.random() < 0.5,
                "force": rng.choice(["float", "float3", "int64"]), "tric": tric, "prec": prec,
                "self": rng.random() < 0.3}
    if kind == "batch":
        return {"kind": "batch", "nsys": rng.randint(4, 48), "mix": rng.randrange(1 << 20), "nmin": 1500,
                "nmax": int(_log_uniform(rng, 5000, 40000)), "order": rng.choice([4, 4, 6]), "kappa": 0.34,
                "ev": rng.random() < 0.7, "plan": rng.choice(["tuned", "default"])}
    if kind == "serve":
        return {"kind": "serve", "nreq": rng.randint(4, 16), "mix": rng.randrange(1 << 20), "nmin": 5000,
                "nmax": int(_log_uniform(rng, 20000, 300000)), "kappa": 0.34}
    return {"kind": "direct", "natom": 3 * int(_log_uniform(rng, 2000, 8000)), "roff": round(rng.uniform(8.0, 12.0), 2),
            "kappa": round(rng.uniform(0.30, 0.36), 3), "ev": rng.random() < 0.5}


# ---- inputs ------------------------------------------------------------------

def _triplets(natom, box, rng):
    """(natom, 4) float32: O, H, H triplets, centres uniform in the box (rows of
    `box` are the cell vectors), random orientations."""
    nt = (natom + 2) // 3
    centres = rng.random((nt, 3)) @ box
    q = rng.standard_normal((nt, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    w, x, y, z = q.T
    ex = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y + z * w), 2 * (x * z - y * w)], 1)
    ey = np.stack([2 * (x * y - z * w), 1 - 2 * (x * x + z * z), 2 * (y * z + x * w)], 1)
    s, c = R_OH * math.sin(THETA / 2), R_OH * math.cos(THETA / 2)
    out = np.empty((nt, 3, 4), np.float32)
    out[:, 0, :3] = centres
    out[:, 1, :3] = centres + s * ex + c * ey
    out[:, 2, :3] = centres - s * ex + c * ey
    out[:, 0, 3] = Q_O
    out[:, 1:, 3] = Q_H
    return out.reshape(-1, 4)[:natom]


def _cell(case):
    """The cell vectors of a solve case, one per row."""
    box = np.diag([case["lx"], case["ly"], case["lz"]])
    if case["tric"]:
        xy, xz, yz = TRICLINIC
        box[1, 0], box[2, 0], box[2, 1] = xy * case["lx"], xz * case["lx"], yz * case["ly"]
    return box


def _recip(box):
    """9 floats, row a = the reciprocal vector of cell vector a."""
    return [float(v) for v in np.linalg.inv(box).T.reshape(-1)]


def _systems(case):
    """Sizes of the systems of a batch or serve case: (natom, box, n, order)."""
    rng = np.random.default_rng(case["mix"])
    out = []
    if case["kind"] == "batch":
        for _ in range(case["nsys"]):
            natom = 3 * max(1, round(math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]))) / 3))
            # edges of 30 to 75 A, grid edges at most 0.9 A per point
            box = [float(v) for v in rng.uniform(30.0, 75.0, 3)]
            out.append((natom, box, [_smooth_up(v / 0.9) for v in box], case["order"]))
    else:
        for _ in range(case["nreq"]):
            natom = 3 * max(1, round(math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]))) / 3))
            edge = (natom / 0.1) ** (1.0 / 3.0)
            out.append((natom, [edge] * 3, [_smooth_up(edge)] * 3, int(rng.choice([4, 6]))))
    return out


def _smooth_up(x):
    n = max(8, math.ceil(x - 1e-9))
    while True:
        m = n
        for f in (2, 3, 5):
            while m % f == 0:
                m //= f
        if m == 1:
            return n
        n += 1


def _inputs(case, seed):
    """Host coordinates of every system of the case, from the seed alone."""
    rng = np.random.default_rng([seed, 77])
    if case["kind"] == "solve":
        return [_triplets(case["natom"], _cell(case), rng)]
    if case["kind"] == "direct":
        edge = (case["natom"] / 0.1) ** (1.0 / 3.0)
        x = _triplets(case["natom"], np.diag([edge] * 3), rng)
        x[:, :3] = np.mod(x[:, :3], np.float32(edge))  # wrapped, as the tile list holds them
        x[:, :3][x[:, :3] >= np.float32(edge)] = 0.0
        return [x]
    return [_triplets(s[0], np.diag(s[1]), rng) for s in _systems(case)]


# ---- the program around the calls -------------------------------------------

def prepare(case, seed):
    return {"solve": _prepare_solve, "batch": _prepare_batch, "serve": _prepare_serve,
            "direct": _prepare_direct}[case["kind"]](case, _inputs(case, seed))


def _prepare_solve(case, xs):
    from gpu_recip_amd import _lib as L
    from gpu_recip_amd.pme import CudaEnergyVirial, CudaPMERecip, force_stride

    dev = torch.device("cuda")
    ev = CudaEnergyVirial()
    pme = CudaPMERecip(case["nx"], case["ny"], case["nz"], case["order"], ev)
    if case["prec"] != "fp32":
        pme.set_precision({"bf16x3": L.PREC_BF16X3, "fp16x3": L.PREC_FP16X3}[case["prec"]])
    n = case["natom"]
    if case["force"] == "float3":
        ft, stride, f = L.FORCE_FLOAT3, n, torch.zeros(n, 3, dtype=torch.float32, device=dev)
    elif case["force"] == "int64":
        stride = force_stride(n, 8)
        ft, f = L.FORCE_INT64, torch.zeros(3, stride, dtype=torch.int64, device=dev)
    else:
        stride = force_stride(n)
        ft, f = L.FORCE_FLOAT, torch.zeros(3, stride, dtype=torch.float32, device=dev)
    return {"case": case, "ev": ev, "pme": pme, "x": torch.from_numpy(xs[0]).to(dev), "n": n,
            "recip": _recip(_cell(case)), "stride": stride, "ft": ft, "f": f}


def _prepare_batch(case, xs):
    from gpu_recip_amd import _lib as L
    from gpu_recip_amd.pme import PmeBatch

    dev = torch.device("cuda")
    # on a stream of the program's own, as an MD engine would run it
    stream = torch.cuda.Stream()
    b = PmeBatch(16 << 30, stream=stream)
    if case["plan"] == "tuned":
        b.set_half_bricks(True)
        b.set_tuning(32, 32, 0)
        b.set_chains(1)
    total = sum(len(x) for x in xs)
    f = torch.zeros(total, 3, dtype=torch.float32, device=dev)
    x = torch.from_numpy(np.concatenate(xs)).to(dev)
    ids, at = [], 0
    for (natom, box, n, order), xi in zip(_systems(case), xs):
        d = PmeBatch.desc(n, order, case["kappa"], _recip(np.diag(box)), x[at:at + natom], natom, f[at:at + natom],
                          L.FORCE_FLOAT3, natom, calc_energy_virial=case["ev"])
        ids.append(b.add(d, keep=(x, f)))
        at += natom
    torch.cuda.synchronize()
    return {"case": case, "b": b, "stream": stream, "ids": ids, "x": x, "f": f}


def _prepare_serve(case, xs):
    from gpu_recip_amd import _lib as L
    from gpu_recip_amd.pme import PmeBatch, PmeServer

    dev = torch.device("cuda")
    srv = PmeServer(8 << 30, nlanes=2)
    reqs = []
    for (natom, box, n, order), xi in zip(_systems(case), xs):
        x = torch.from_numpy(xi).to(dev)
        f = torch.zeros(natom, 3, dtype=torch.float32, device=dev)
        d = PmeBatch.desc(n, order, case["kappa"], _recip(np.diag(box)), x, natom, f, L.FORCE_FLOAT3, natom)
        reqs.append((d, x, f))
    torch.cuda.synchronize()
    return {"case": case, "srv": srv, "reqs": reqs}


def _prepare_direct(case, xs):
    from gpu_recip_amd import nlist
    from gpu_recip_amd.direct import CudaPMEDirectForce, DeviceTileList
    from gpu_recip_amd.pme import CudaEnergyVirial, force_stride

    dev = torch.device("cuda")
    edge = (case["natom"] / 0.1) ** (1.0 / 3.0)
    tl, ex14 = nlist.water_box(xs[0], (edge,) * 3, case["roff"])
    ev = CudaEnergyVirial()
    dr = CudaPMEDirectForce(ev)
    dr.setup(edge, edge, edge, case["kappa"], case["roff"], case["roff"] - 1.0, 1.0)
    dr.set_14_list(np.zeros((0, 3), np.int32), ex14)
    dl = DeviceTileList(tl, dev)
    stride = force_stride(tl.npad, 8)
    f = torch.zeros(3, stride, dtype=torch.int64, device=dev)
    return {"case": case, "ev": ev, "dr": dr, "dl": dl, "stride": stride, "f": f,
            "at": torch.from_numpy(tl.sorted_index()).to(dev)}


def run(state):
    return {"solve": _run_solve, "batch": _run_batch, "serve": _run_serve,
            "direct": _run_direct}[state["case"]["kind"]](state)


def _run_solve(s):
    c, pme, ev = s["case"], s["pme"], s["ev"]
    n, recip, kappa = s["n"], s["recip"], c["kappa"]
    if c["force"] == "int64":
        s["f"].zero_()  # the array the terms of a step add to
    if c["ev"] or c["self"]:
        ev.clear()
    if c["calls"] == "solve":
        pme.solve(s["x"], n, recip, kappa, c["ev"], c["ev"], s["stride"], s["f"], s["ft"])
    else:
        pme.spread_charge(s["x"], n, recip)
        pme.r2c_fft()
        pme.scalar_sum(recip, kappa, c["ev"], c["ev"])
        pme.c2r_fft()
        pme.gather_force(s["x"], n, recip, s["stride"], s["f"], s["ft"])
    if c["self"]:
        pme.calc_self_energy(s["x"], n, kappa)
    out = {}
    if c["ev"] or c["self"]:
        ev.copyToHost()
        torch.cuda.current_stream().synchronize()
        if c["ev"]:
            out["ev"] = torch.tensor([ev.getEnergy("recip"), *ev.getVirial()], dtype=torch.float32)
        if c["self"]:
            out["self"] = torch.tensor([ev.getEnergy("self")], dtype=torch.float32)
    out["force"] = s["f"][:, :n].float() * 2.0 ** -40 if c["force"] == "int64" else s["f"]
    return out


def _run_batch(s):
    s["b"].solve()
    if not s["case"]["ev"]:
        torch.cuda.current_stream().wait_stream(s["stream"])
        return {"force": s["f"]}
    e, v = s["b"].results(s["ids"])
    return {"force": s["f"], "energy": e.astype(np.float32), "virial": v.astype(np.float32)}


def _run_serve(s):
    srv = s["srv"]
    tickets = [srv.submit(k, d) for k, (d, x, f) in enumerate(s["reqs"])]
    got = [srv.wait(t) for t in tickets]
    return {"force": [f for d, x, f in s["reqs"]],
            "ev": torch.tensor([[g[0], *g[1]] for g in got], dtype=torch.float32)}


def _run_direct(s):
    c, dr, ev = s["case"], s["dr"], s["ev"]
    s["f"].zero_()
    if c["ev"]:
        ev.clear()
    dr.calc_force(s["dl"].xyzq, s["dl"], c["ev"], c["ev"], s["stride"], s["f"])
    dr.calc_14_force(s["dl"].xyzq, c["ev"], c["ev"], s["stride"], s["f"])
    out = {}
    if c["ev"]:
        ev.copyToHost()
        torch.cuda.current_stream().synchronize()
        out["energy"] = torch.tensor([ev.getEnergy("elec"), ev.getEnergy("excl")], dtype=torch.float32)
        out["shift"] = torch.tensor(ev.getSforce(), dtype=torch.float32)
    out["force"] = s["f"][:, s["at"]].float() * 2.0 ** -40  # in the program's own order of the atoms
    return out


# ---- what cannot be done without -----------------------------------------------

def _solve_work(natom, n, order, ev, force_bytes=12):
    # coordinates and charges in, forces out; per atom two operations a stencil
    # point in the spread and four in the gather, a real transform each way, and
    # the influence function with (or without) energy and virial
    g = n[0] * n[1] * n[2]
    gc = (n[0] // 2 + 1) * n[1] * n[2]
    flops = natom * (6 * order ** 3 + 12 * order ** 2) + 5.0 * g * math.log2(g) + (30 if ev else 12) * gc
    return (16 + force_bytes) * natom, flops


def work(case):
    if case["kind"] == "direct":
        n, r, k = case["natom"], case["roff"], 0.1
        pairs = n * (4.0 / 3.0 * math.pi * r ** 3 * k) / 2
        return {"bytes": 40.0 * n, "flops": 28.0 * pairs}
    if case["kind"] == "solve":
        b, f = _solve_work(case["natom"], (case["nx"], case["ny"], case["nz"]), case["order"], case["ev"],
                           24 if case["force"] == "int64" else 12)
        return {"bytes": float(b), "flops": float(f)}
    got = [_solve_work(s[0], s[2], s[3], True) for s in _systems(case)]
    return {"bytes": float(sum(g[0] for g in got)), "flops": float(sum(g[1] for g in got))}


# ---- the same in 64 bits --------------------------------------------------------

def _spline(w, order):
    """theta[j] = M_order(w + order-1-j) and its derivative, per atom: (order, N) each."""
    th = [1.0 - w, w]
    for k in range(3, order + 1):
        prev = [None] + th + [None]
        dth, new = [], []
        for j in range(k):
            a, b = prev[j], prev[j + 1]
            a = torch.zeros_like(w) if a is None else a
            b = torch.zeros_like(w) if b is None else b
            u = w + (k - 1 - j)
            new.append((u * a + (k - u) * b) / (k - 1))
            dth.append(a - b)
        th = new
    return th, dth


def _bsp_mod(order, n):
    w = torch.zeros(1, dtype=torch.float64)
    th = [float(t) for t in _spline(w, order)[0]]
    k = np.arange(n)
    s = sum(t * np.exp(2j * math.pi * ((j + 1) * k % n) / n) for j, t in enumerate(th))
    return torch.from_numpy(1.0 / np.abs(s) ** 2)


def _exact_recip(x, n, order, kappa, recip):
    """(force (N, 3), [energy, virial 9]) of one system in FP64."""
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    x = torch.from_numpy(x).to(dev).double()
    R = torch.tensor(recip, dtype=torch.float64, device=dev).reshape(3, 3)
    q = x[:, 3]
    idx, th, dth = [], [], []
    for a in range(3):
        t = x[:, :3] @ R[a] + 0.5
        fr = n[a] * (t - torch.floor(t))
        i = torch.floor(fr)
        t, d = _spline(fr - i, order)
        idx.append(i.long() % n[a])
        th.append(t)
        dth.append(d)
    nx, ny, nz = n
    grid = torch.zeros(nz * ny * nx, dtype=torch.float64, device=dev)
    rows = [[((idx[2] + jz) % nz * ny + (idx[1] + jy) % ny) * nx for jy in range(order)] for jz in range(order)]
    cols = [(idx[0] + jx) % nx for jx in range(order)]
    for jz in range(order):
        for jy in range(order):
            w = q * th[1][jy] * th[2][jz]
            for jx in range(order):
                grid.index_add_(0, rows[jz][jy] + cols[jx], w * th[0][jx])
    S = torch.fft.rfftn(grid.reshape(nz, ny, nx))

    def wave(k, size):
        return torch.where(k >= size // 2 + size % 2, k - size, k).double()

    k1, k2, k3 = (torch.arange(s, device=dev) for s in (nx // 2 + 1, ny, nz))
    det = float(torch.linalg.det(R.cpu()))
    fac = math.pi ** 2 / kappa ** 2
    pf = [_bsp_mod(order, s).to(dev) for s in n]

    def eterm(i1, i2, i3):
        """eterm and m at every (k3, k2, k1) for index vectors per axis."""
        m1 = wave(i1, nx)[None, None, :]
        m2 = wave(i2, ny)[None, :, None]
        m3 = wave(i3, nz)[:, None, None]
        m = [m1 * R[0, c] + m2 * R[1, c] + m3 * R[2, c] for c in range(3)]
        msq = m[0] ** 2 + m[1] ** 2 + m[2] ** 2
        inv = torch.where(msq > 0, 1.0 / msq, torch.zeros_like(msq))
        e = torch.exp(-fac * msq) * inv * det / math.pi
        return e * pf[0][i1][None, None, :] * pf[1][i2][None, :, None] * pf[2][i3][:, None, None], m, inv

    e0, m0, inv0 = eterm(k1, k2, k3)
    q2 = S.real ** 2 + S.imag ** 2
    acc = [0.0] * 10
    # every point, and the mirror of each with k1 >= 1
    for mirror in (False, True):
        e, m, inv = eterm((nx - k1) % nx, (ny - k2) % ny, (nz - k3) % nz) if mirror else (e0, m0, inv0)
        t = e * q2
        if mirror:
            t = t.clone()
            t[:, :, 0] = 0.0
        v = 2.0 * (fac + inv)
        acc[0] += 0.5 * CCELEC * float(t.sum())
        for a in range(3):
            for b in range(a, 3):
                s = -0.5 * CCELEC * float((t * (v * m[a] * m[b] - (1.0 if a == b else 0.0))).sum())
                acc[1 + 3 * a + b] += s
                if a != b:
                    acc[1 + 3 * b + a] += s
    phi = torch.fft.irfftn(S * e0, s=(nz, ny, nx), norm="forward").reshape(-1)
    g = [torch.zeros_like(q) for _ in range(3)]
    for jz in range(order):
        for jy in range(order):
            a = torch.zeros_like(q)
            b = torch.zeros_like(q)
            for jx in range(order):
                p = phi[rows[jz][jy] + cols[jx]]
                a += th[0][jx] * p
                b += dth[0][jx] * p
            g[0] += b * th[1][jy] * th[2][jz]
            g[1] += a * dth[1][jy] * th[2][jz]
            g[2] += a * th[1][jy] * dth[2][jz]
    g = torch.stack([g[a] * q * CCELEC * n[a] for a in range(3)], 1)
    return (g @ R).cpu(), acc


def _exact_direct(x, edge, kappa, roff):
    """(force (N, 3), [elec, excl]) of the direct term in FP64: atoms sorted by
    z, each block against the atoms within roff in z."""
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    p = torch.from_numpy(x).to(dev).double()
    n = len(p)
    order = torch.argsort(p[:, 2])
    s, mol = p[order], order // 3
    force = torch.zeros(n, 3, dtype=torch.float64, device=dev)
    elec = 0.0

    def pair(d, r2, qq, f):
        r = torch.sqrt(r2)
        e = qq * (torch.special.erfc(kappa * r) + f) / r
        g = (-qq * 2.0 / math.sqrt(math.pi) * kappa * torch.exp(-kappa * kappa * r2) - e) / r2
        return e, g[:, None] * d

    step = 256
    z = s[:, 2].contiguous()
    for a in range(0, n, step):
        b = min(a + step, n)
        dz = z[None, :] - z[a:b, None]
        dz = dz - edge * torch.round(dz / edge)
        near = torch.nonzero((dz.abs() < roff).any(0)).reshape(-1)
        d = s[a:b, None, :3] - s[None, near, :3]
        d = d - edge * torch.round(d / edge)
        r2 = (d * d).sum(-1)
        ok = (r2 < roff * roff) & (mol[a:b, None] != mol[None, near])
        i, j = torch.nonzero(ok, as_tuple=True)
        e, g = pair(d[i, j], r2[i, j], CCELEC * s[a + i, 3] * s[near[j], 3], 0.0)
        elec += 0.5 * float(e.sum())
        force.index_add_(0, order[a + i], g)
    o = torch.arange(0, n - n % 3, 3, device=dev)
    i, j = torch.cat([o, o, o + 1]), torch.cat([o + 1, o + 2, o + 2])
    d = p[i, :3] - p[j, :3]
    d = d - edge * torch.round(d / edge)
    e, g = pair(d, (d * d).sum(-1), CCELEC * p[i, 3] * p[j, 3], -1.0)
    force.index_add_(0, i, g)
    force.index_add_(0, j, -g)
    return force.cpu(), [elec, float(e.sum())]


def exact(case, seed):
    xs = _inputs(case, seed)
    if case["kind"] == "direct":
        edge = (case["natom"] / 0.1) ** (1.0 / 3.0)
        f, e = _exact_direct(xs[0], edge, case["kappa"], case["roff"])
        out = {"energy": torch.tensor(e, dtype=torch.float64), "shift": None} if case["ev"] else {}
        out["force"] = f.T.contiguous()
        return out
    if case["kind"] == "solve":
        x = xs[0]
        f, ev = _exact_recip(x, (case["nx"], case["ny"], case["nz"]), case["order"], case["kappa"],
                             _recip(_cell(case)))
        out = {}
        if case["ev"]:
            out["ev"] = torch.tensor(ev, dtype=torch.float64)
        if case["self"]:
            q = x[:, 3].astype(np.float64)
            out["self"] = torch.tensor([-case["kappa"] * CCELEC / math.sqrt(math.pi) * float((q * q).sum())],
                                       dtype=torch.float64)
        if case["force"] == "float3":
            out["force"] = f
        elif case["force"] == "int64":
            out["force"] = f.T.contiguous()
        else:
            n = len(x)
            stride = -(-(n - 1 + 32) * 4 // 256) * 64  # rows padded to 256 bytes
            out["force"] = torch.zeros(3, stride, dtype=torch.float64)
            out["force"][:, :n] = f.T
        return out
    got = [_exact_recip(x, s[2], s[3], case["kappa"], _recip(np.diag(s[1])))
           for s, x in zip(_systems(case), xs)]
    if case["kind"] == "serve":
        return {"force": [g[0] for g in got], "ev": torch.tensor([g[1] for g in got], dtype=torch.float64)}
    out = {"force": torch.cat([g[0] for g in got])}
    if case["ev"]:
        out["energy"] = torch.tensor([g[1][0] for g in got], dtype=torch.float64)
        out["virial"] = torch.tensor([g[1][1:] for g in got], dtype=torch.float64)
    return out
