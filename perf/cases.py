"""Performance cases: the molecular-dynamics work this engine is used for,
through its public Python classes, with inputs made here from a seed and an
independent 64-bit torch evaluation of what each pass computes.

Kinds of case:
  lj       CbnMD.run on a Lennard-Jones box (the main loop: integrate, wrap,
           ghosts, list rebuild every 20 steps, force, thermo)
  modules  the reference's module calls by hand: exchange, binning, halo,
           list, force, energy, virial
  nnp      CbnMD.run with the neural-network potential
  batch    Batch.run: many independent boxes stepped together
  serve    Server: a group of jobs submitted, run and collected

Engine state lives in device memory behind handles and a program reads it
back when it wants a snapshot, not after every run() call; so the outputs of
the MD kinds are mappings that download the state when an entry is read
(atoms ordered by id, positions unwrapped).  A server's results are host
arrays and are collected inside the pass.
"""
import math

import numpy as np
import torch

import cabanamd_amd as M

EVERY = 20  # steps between list rebuilds
SKIN = 0.3
LJ_CUT = 2.5
DT = 0.005
NNP_DT = 0.0005
PREC = {"fp64": M.PREC_FP64, "mixed": M.PREC_MIXED}
# pair coefficients (i, j, eps, sigma) of the one- and two-type fluids
COEFF = {1: [(1, 1, 1.0, 1.0)],
         2: [(1, 1, 1.0, 1.0), (1, 2, 0.9, 0.975), (2, 2, 0.8, 0.95)]}


# ---- the cases ---------------------------------------------------------------

def listed():
    def lj(name, nx, ny, nz, **kw):
        c = dict(name=name, kind="lj", nx=nx, ny=ny, nz=nz, rho=0.8442,
                 temp=1.44, types=1, half=False, prec="fp64", steps=100)
        c.update(kw)
        return c

    return [
        # the smallest box a deck runs (the golden 256-atom case): every step
        # is launches and latency
        lj("lj_256_fp64", 4, 4, 4),
        # the reference's own CPU deck size, 32,000 atoms, in double
        lj("lj_32k_fp64", 20, 20, 20),
        # a two-component fluid in an uneven box, mixed precision
        lj("lj_48k_two_type_mixed", 17, 23, 31, rho=0.78, temp=1.1, types=2,
           prec="mixed"),
        # the headline size, mixed precision (the production setting)
        lj("lj_2m_mixed", 80, 80, 80, prec="mixed"),
        # a large box in double
        lj("lj_864k_fp64", 60, 60, 60),
        # newton on: half lists with the reaction added to the partner
        lj("lj_500k_half_fp64", 50, 50, 50, half=True),
        # a program that drives the modules itself, as the reference's loop does
        dict(name="modules_256k_fp64", kind="modules", nx=40, ny=40, nz=40,
             rho=0.8442, half=False, prec="fp64"),
        # two elements, 70 symmetry functions each, BF16 matrix layers: small
        # (latency) and large (throughput) boxes
        dict(name="nnp_3000_mixed", kind="nnp", model="two", nx=10, ny=15,
             nz=20, prec="mixed", steps=20),
        dict(name="nnp_192k_mixed", kind="nnp", model="two", nx=40, ny=60,
             nz=80, prec="mixed", steps=20),
        # one metal, 27 functions over three etas, FP32 layers
        dict(name="nnp_metal_19k_fp32", kind="nnp", model="metal", nx=17,
             ny=17, nz=17, prec="fp64", steps=20),
        # an ensemble of 512 boxes of 500 to 20,000 atoms
        dict(name="batch_512_mixed", kind="batch", nsys=512, lo=500, hi=20000,
             prec="mixed", steps=40),
        # served jobs, 70 % LJ and 30 % NNP, submitted, run and collected
        dict(name="serve_12_jobs", kind="serve", njobs=12, lo=1000, hi=20000,
             slo=60, shi=160),
    ]


def _logu(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def _cells(rng, n, least):
    """Uneven cell counts nx, ny, nz with nx ny nz near n."""
    side = n ** (1.0 / 3.0)
    nx = max(least, round(side * rng.uniform(0.7, 1.3)))
    ny = max(least, round(math.sqrt(n / nx) * rng.uniform(0.8, 1.25)))
    return nx, ny, max(least, round(n / (nx * ny)))


def draw(rng):
    kind = rng.choice(["lj", "lj", "lj", "lj", "modules", "nnp", "nnp",
                       "batch", "serve"])
    if kind == "lj":
        nx, ny, nz = _cells(rng, _logu(rng, 256, 1.0e6) / 4, 4)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz,
                    rho=round(rng.uniform(0.70, 0.90), 3),
                    temp=round(rng.uniform(0.8, 2.0), 2),
                    types=rng.choice([1, 1, 2]),
                    half=rng.random() < 0.25,
                    prec=rng.choice(["fp64", "mixed"]), steps=100)
    if kind == "modules":
        nx, ny, nz = _cells(rng, _logu(rng, 256, 5.0e5) / 4, 4)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz,
                    rho=round(rng.uniform(0.70, 0.90), 3),
                    half=rng.random() < 0.5,
                    prec=rng.choice(["fp64", "mixed"]))
    if kind == "nnp":
        model = rng.choice(["two", "metal"])
        if model == "two":
            nx, ny, nz = _cells(rng, _logu(rng, 500, 1.0e5), 6)
        else:
            nx, ny, nz = _cells(rng, _logu(rng, 500, 1.0e5) / 4, 3)
        return dict(kind=kind, model=model, nx=nx, ny=ny, nz=nz,
                    prec=rng.choice(["fp64", "mixed"]), steps=20)
    if kind == "batch":
        return dict(kind=kind, nsys=round(_logu(rng, 8, 256)), lo=500,
                    hi=round(_logu(rng, 2000, 20000)),
                    prec=rng.choice(["fp64", "mixed"]), steps=40)
    return dict(kind=kind, njobs=rng.randint(6, 12), lo=1000,
                hi=round(_logu(rng, 4000, 20000)), slo=60, shi=160)


# ---- inputs ------------------------------------------------------------------

def _rng(seed, salt=0):
    return np.random.default_rng([int(seed), salt])


def _fcc(nx, ny, nz, a):
    g = np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz),
                             indexing="ij"), -1).reshape(-1, 1, 3)
    b = np.array([[0, 0, 0], [0, .5, .5], [.5, 0, .5], [.5, .5, 0]]) + 0.25
    return a * (g + b).reshape(-1, 3), a * np.array([nx, ny, nz], float)


def _velocities(rng, n, temp):
    v = rng.standard_normal((n, 3)) * math.sqrt(temp)
    return v - v.mean(axis=0)


def _lj_box(nx, ny, nz, rho, temp, types, seed, salt=0):
    """A warm fcc crystal about to melt: sites displaced by up to 0.05,
    Gaussian velocities, types at random (one third type 1)."""
    rng = _rng(seed, salt)
    x, L = _fcc(nx, ny, nz, (4.0 / rho) ** (1.0 / 3.0))
    x = np.mod(x + rng.uniform(-0.05, 0.05, x.shape), L)
    t = (rng.random(len(x)) < (types - 1) / 3.0).astype(np.int32)
    return dict(x=x, v=_velocities(rng, len(x), temp), t=t, L=L)


def _nnp_box(model, nx, ny, nz, seed, salt=0):
    rng = _rng(seed, salt)
    if model == "two":  # jittered simple cubic, one third element 1
        x = 2.5 * (np.stack(np.meshgrid(np.arange(nx), np.arange(ny),
                                        np.arange(nz), indexing="ij"),
                            -1).reshape(-1, 3) + 0.5)
        L = 2.5 * np.array([nx, ny, nz], float)
        amp, frac = 0.25, 1.0 / 3.0
    else:  # fcc metal at thermal displacements
        x, L = _fcc(nx, ny, nz, 6.65)
        amp, frac = 0.3, 0.0
    x = np.mod(x + rng.uniform(-amp, amp, x.shape), L)
    t = (rng.random(len(x)) < frac).astype(np.int32)
    return dict(x=x, v=_velocities(rng, len(x), 0.05), t=t, L=L)


def _near_cube(n):
    nx = max(4, round(n ** (1.0 / 3.0)))
    ny = max(4, round((n / nx) ** 0.5))
    return nx, ny, max(4, round(n / (nx * ny)))


def _batch_boxes(case, seed):
    """The ensemble's boxes; sizes, densities and temperatures are the case's
    own and the atoms the seed's."""
    rng = _rng(case["nsys"] + 131 * case["hi"], 1)
    out = []
    for k in range(case["nsys"]):
        n = math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))
        out.append(_lj_box(*_near_cube(n / 4.0), float(rng.uniform(0.70, 0.90)),
                           float(rng.uniform(0.8, 2.0)), 1, seed, 10 + k))
    return out


def _serve_jobs(case, seed):
    """(is NNP, steps, box) of each job; three in ten are NNP jobs, of a
    quarter of the atoms.  The sizes and steps are the case's own and the
    atoms the seed's."""
    rng = _rng(case["njobs"] + 131 * case["hi"], 2)
    out = []
    for k in range(case["njobs"]):
        n = math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))
        rho, temp = float(rng.uniform(0.70, 0.90)), float(rng.uniform(0.8, 2.0))
        steps = int(rng.integers(case["slo"], case["shi"] + 1))
        if k % 10 in (1, 4, 7):
            c = [max(6, m) for m in _near_cube(n / 4.0)]
            out.append((True, steps, _nnp_box("two", *c, seed, 10 + k)))
        else:
            out.append((False, steps, _lj_box(*_near_cube(n / 4.0), rho, temp,
                                              1, seed, 10 + k)))
    return out


# ---- NNP models --------------------------------------------------------------

def _model(kind):
    """Two-element model: 15 radial etas per neighbour element, 5 angular etas
    x 4 zetas x 2 lambdas, network 70-25-25-1, cutoff 6.  Metal model: 3
    radial and 3 x 8 angular functions, network 27-24-24-1, cutoff 7.37."""
    if kind == "two":
        m = dict(nelem=2, rc=6.0, hidden=[25, 25], any_pair=True,
                 reta=[0.01 * 200.0 ** (k / 14.0) for k in range(15)],
                 aeta=[0.001 * 50.0 ** (k / 4.0) for k in range(5)])
    else:
        m = dict(nelem=1, rc=7.37, hidden=[24, 24], any_pair=False,
                 reta=[0.01, 0.02, 0.05], aeta=[0.01, 0.02, 0.05])
    m["pl"] = [(z, lam) for z in (1.0, 2.0, 4.0, 16.0) for lam in (-1.0, 1.0)]
    nsf = len(m["reta"]) * m["nelem"] + len(m["aeta"]) * len(m["pl"])
    rng = _rng(87287, nsf)
    sizes = [nsf] + m["hidden"] + [1]
    m["W"] = [[rng.standard_normal((sizes[l + 1], sizes[l])) /
               math.sqrt(sizes[l]) for l in range(3)] for _ in range(m["nelem"])]
    m["b"] = [[0.1 * rng.standard_normal(sizes[l + 1]) for l in range(3)]
              for _ in range(m["nelem"])]
    # min-max scaling ranges from a small frame
    box = _nnp_box(kind, *((8, 8, 8) if kind == "two" else (5, 5, 5)), 5)
    x, L = _dev(box["x"]), _dev(box["L"]).expand(len(box["x"]), 3)
    t = _dev(box["t"])
    one = torch.zeros(len(x), dtype=torch.long, device=x.device)
    i, j = _pairs(x, one, L[:1], m["rc"] + SKIN)
    G = torch.cat([g for _, _, g in _sf_chunks(m, x, t, L, i, j)]).cpu().numpy()
    m["gmin"] = [G[box["t"] == e].min(0) for e in range(m["nelem"])]
    m["gmax"] = [G[box["t"] == e].max(0) for e in range(m["nelem"])]
    return m


def _engine_model(m):
    nn = M.NNPModel.create(m["nelem"], m["hidden"], "ttl")
    nn.set_scaling(True, 0.0, 1.0)
    for e in range(m["nelem"]):
        sf = [(2, ne, -1, eta, 0.0, 0.0, 0.0) for eta in m["reta"]
              for ne in range(m["nelem"])]
        pair = (-1, -1) if m["any_pair"] else (0, 0)
        sf += [(3, *pair, eta, 0.0, lam, z) for eta in m["aeta"]
               for z, lam in m["pl"]]
        for k, s in enumerate(sf):
            nn.add_sf(e, *s, m["rc"], gmin=float(m["gmin"][e][k]),
                      gmax=float(m["gmax"][e][k]))
        for l in range(3):
            nn.set_layer(e, l, m["W"][e][l], m["b"][e][l])
    return nn


# ---- outputs -----------------------------------------------------------------

class Snapshot(dict):
    """Outputs in device memory: an entry is downloaded when it is read."""

    def __init__(self, keys, read):
        super().__init__((k, None) for k in keys)
        self._read, self._got = read, None

    def __getitem__(self, k):
        if self._got is None:
            self._got = self._read()
        return self._got[k]

    def get(self, k, default=None):
        return self[k] if k in self else default

    def items(self):
        return [(k, self[k]) for k in self]

    def values(self):
        return [self[k] for k in self]


def _unwrap(x, x0, L):
    return x - L * np.round((x - x0) / L)


def _by_id(x, v, f, i, n, box):
    o = np.argsort(i[:n], kind="stable")
    return dict(x=_unwrap(x[:n][o], box["x"], box["L"]), v=v[:n][o], f=f[:n][o])


# ---- prepare and run ---------------------------------------------------------

def _lj_params(case, steps):
    types = case.get("types", 1)
    p = M.lattice_params(cutoff=LJ_CUT, skin=SKIN, every=EVERY, dt=DT,
                         half=case.get("half", False), nsteps=steps,
                         thermo=steps)
    p.ntypes = types
    for k in range(types):
        p.mass[k] = 1.0
    p.ncoeff = len(COEFF[types])
    for k, (i, j, eps, sig) in enumerate(COEFF[types]):
        p.coeff_i[k], p.coeff_j[k] = i, j
        p.coeff_eps[k], p.coeff_sigma[k], p.coeff_cut[k] = eps, sig, LJ_CUT
    return p


def _nnp_params(m, steps):
    return M.nnp_params(ntypes=m["nelem"], cutoff=m["rc"], skin=SKIN,
                        dt=NNP_DT, nsteps=steps, thermo=steps, every=EVERY,
                        mass=(1.0,) * m["nelem"])


ZERO = [0.0, 0.0, 0.0]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("lj", "nnp"):
        if kind == "lj":
            box = _lj_box(case["nx"], case["ny"], case["nz"], case["rho"],
                          case["temp"], case["types"], seed)
            md = M.CbnMD(_lj_params(case, case["steps"]),
                         precision=PREC[case["prec"]])
        else:
            box = _nnp_box(case["model"], case["nx"], case["ny"], case["nz"],
                           seed)
            m = _model(case["model"])
            md = M.CbnMD(_nnp_params(m, case["steps"]),
                         precision=PREC[case["prec"]])
            md.set_nnp_model(_engine_model(m))
        md.set_initial_state(box["x"], box["t"], ZERO, list(box["L"]),
                             v=box["v"])
        md.init()
        return dict(case=case, box=box, md=md)
    if kind == "modules":
        box = _lj_box(case["nx"], case["ny"], case["nz"], case["rho"], 1.44, 1,
                      seed)
        s = M.System(1)
        s.create_domain(ZERO, list(box["L"]), LJ_CUT + SKIN)
        s.resize(int(1.5 * len(box["x"])) + 1024)
        s.upload(box["x"], box["v"], None, box["t"], None)
        F = M.ForceLJ(s, PREC[case["prec"]])
        F.init_coeff([["pair_coeff", "1", "1", "1.0", "1.0", str(LJ_CUT)]])
        return dict(case=case, box=box, s=s, F=F, comm=M.Comm(s, LJ_CUT + SKIN),
                    binning=M.Binning(s),
                    nl=M.NeighborVerlet(LJ_CUT + SKIN, case["half"], 100))
    if kind == "batch":
        boxes = _batch_boxes(case, seed)
        B = M.Batch(_lj_params(case, 100), PREC[case["prec"]])
        hs = [B.add(b["x"], b["t"], ZERO, list(b["L"]), v=b["v"])
              for b in boxes]
        B.run(0)  # the systems join
        return dict(case=case, boxes=boxes, B=B, hs=hs)
    jobs = _serve_jobs(case, seed)
    m = _model("two")
    S = M.Server(_lj_params(case, 100), _nnp_params(m, 100), _engine_model(m))
    return dict(case=case, jobs=jobs, S=S)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("lj", "nnp"):
        md, box = state["md"], state["box"]
        md.run(case["steps"])  # ends with a thermo row

        def read():
            x, v, f, _, i = md.arrays()
            out = _by_id(x, v, f, i, md.n_local, box)
            out["thermo"] = md.thermo()[-1, 1:]
            return out
        return Snapshot(["x", "v", "f", "thermo"], read)
    if kind == "modules":
        s, F, nl = state["s"], state["F"], state["nl"]
        state["comm"].exchange()
        state["binning"].create_binning(*[LJ_CUT + SKIN] * 3)
        state["comm"].exchange_halo()
        nl.create(s)
        F.compute(s, nl)
        if case["half"]:
            state["comm"].update_force()
        pe = F.compute_energy(s, nl)
        w = F.compute_virial(s, nl)

        def read():
            x, v, f, _, i = s.download()
            out = _by_id(x, v, f, i, s.N_local, state["box"])
            out.update(pe=np.float64(pe), w=np.float64(w))
            return out
        return Snapshot(["f", "pe", "w"], read)
    if kind == "batch":
        B = state["B"]
        B.run(case["steps"])

        def read():
            got = []
            for h, b in zip(state["hs"], state["boxes"]):
                x, v, f, _, i = B.download(h)
                got.append(_by_id(x, v, f, i, len(x), b))
            return {k: np.concatenate([g[k] for g in got]) for k in "xvf"}
        return Snapshot(["x", "v", "f"], read)
    S = state["S"]
    ids = [S.submit(S.NNP if nnp else S.LJ, b["x"], b["t"], ZERO, list(b["L"]),
                    steps, v=b["v"]) for nnp, steps, b in state["jobs"]]
    S.drain(600.0)
    out = {}
    for name, want in (("lj", False), ("nnp", True)):
        got = [S.result(j)[:2] + (b,) for j, (nnp, _, b)
               in zip(ids, state["jobs"]) if nnp == want]
        if got:
            out[name + "_x"] = np.concatenate([_unwrap(x, b["x"], b["L"])
                                               for x, _, b in got])
            out[name + "_v"] = np.concatenate([v for _, v, _ in got])
    return out


# ---- what a pass cannot do without -------------------------------------------

LJ_PAIR_FLOPS = 23.0  # distance 8, test 1, pair 8, one force update 6


def _lj_work(n, rho, steps):
    """Every pair inside the cutoff once a step; state in and out once."""
    pairs = n * rho * (2.0 / 3.0) * math.pi * LJ_CUT ** 3
    return 128.0 * n, steps * (pairs * LJ_PAIR_FLOPS + 18.0 * n)


def _nnp_work(model, n, steps):
    """Neighbours, triplets (both sides and the third inside the cutoff) and
    layers; per-term flops of the symmetry functions and their forces."""
    if model == "two":
        rho, rc, ng, npl, nr, net = 0.064, 6.0, 5, 8, 30, 70 * 25 + 650
    else:
        rho, rc, ng, npl, nr, net = 4 / 6.65 ** 3, 7.37, 3, 8, 3, 27 * 24 + 600
    nb = rho * 4.0 / 3.0 * math.pi * rc ** 3
    trip = nb * nb / 2 * 15.0 / 32.0
    per = (trip * (120 + 13 * ng + 9 * npl + 6 * ng * npl) +
           nb * (50 + 20 * nr) + 6.0 * net)
    return 128.0 * n, steps * n * per


def work(case):
    kind = case["kind"]
    if kind == "lj":
        b, f = _lj_work(4 * case["nx"] * case["ny"] * case["nz"], case["rho"],
                        case["steps"])
    elif kind == "modules":  # a list build and force, energy and virial
        b, f = _lj_work(4 * case["nx"] * case["ny"] * case["nz"], case["rho"],
                        2)
    elif kind == "nnp":
        per = 1 if case["model"] == "two" else 4
        b, f = _nnp_work(case["model"],
                         per * case["nx"] * case["ny"] * case["nz"],
                         case["steps"])
    elif kind == "batch":
        lo, hi = case["lo"], case["hi"]
        n = case["nsys"] * (hi - lo) / math.log(hi / lo)
        b, f = _lj_work(n, 0.8, case["steps"])
    else:
        lo, hi = case["lo"], case["hi"]
        n = (hi - lo) / math.log(hi / lo)
        steps = (case["slo"] + case["shi"]) / 2
        b1, f1 = _lj_work(0.7 * case["njobs"] * n, 0.8, steps)
        b2, f2 = _nnp_work("two", 0.075 * case["njobs"] * n, steps)
        b, f = b1 + b2, f1 + f2
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the difference seen against exact().  In the
    trajectories a rounding difference of one force evaluation (1e-16 in
    double, a few 1e-6 in mixed precision) grows with the liquid's Lyapunov
    exponent, by 5 to 10 times in 100 steps; two passes on one state are 200.
    Measured at T = 2: 9e-13 (largest 2e-11) in double and 2e-4 (largest
    8e-3) in mixed precision after 200 steps; boxes of up to two million
    atoms have larger extremes than the 14,000 atoms measured."""
    kind, double = case["kind"], case.get("prec") == "fp64"
    if kind == "lj":
        return ({"rel": 5e-12, "max": 5e-10} if double
                else {"rel": 1e-3, "max": 0.2})
    if kind == "modules":  # one force: 8e-15 and 5e-7, cancelling near sites
        return ({"rel": 5e-14, "max": 1e-12} if double
                else {"rel": 2e-6, "max": 1e-4})
    if kind == "nnp":  # FP32 symmetry functions: 1.8e-6, largest 3e-5
        return {"rel": 8e-6, "max": 1.5e-4}
    if kind == "batch":  # 80 steps
        return ({"rel": 1e-12, "max": 1e-10} if double
                else {"rel": 3e-5, "max": 1e-2})
    return {"rel": 1e-4, "max": 0.05}  # jobs of up to 160 steps, mixed


# ---- the same passes in 64-bit torch -----------------------------------------

def _dev(a):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    return torch.as_tensor(a, device=dev)


def _pairs(x, sysid, Ls, rl):
    """Pairs i < j of one system whose nearest images lie within rl: i, j as
    int64.  sysid (n) says which periodic box of Ls (nsys, 3) an atom is in;
    boxes start at 0 and are wider than 2 rl."""
    dev = x.device
    nc = torch.clamp((Ls / rl).floor().long(), min=1).cpu().numpy()
    base = np.concatenate([[0], np.cumsum(nc.prod(1))])
    ncell = int(base[-1])
    nbr = np.full((27, ncell), -1, np.int64)
    for s, (a, b, c) in enumerate(nc):
        g = np.stack(np.meshgrid(np.arange(a), np.arange(b), np.arange(c),
                                 indexing="ij"), -1).reshape(-1, 3)
        offs = [{1: (0,), 2: (0, 1)}.get(int(k), (-1, 0, 1)) for k in (a, b, c)]
        m = 0
        for dx in offs[0]:
            for dy in offs[1]:
                for dz in offs[2]:
                    h = (g + (dx, dy, dz)) % (a, b, c)
                    nbr[m, base[s]:base[s + 1]] = (
                        base[s] + (h[:, 0] * b + h[:, 1]) * c + h[:, 2])
                    m += 1
    n3 = _dev(nc).to(dev)[sysid]
    L = Ls[sysid]
    u = x / L
    u = u - u.floor()
    c3 = torch.minimum((u * n3).long(), n3 - 1)
    cell = (_dev(base[:-1]).to(dev)[sysid] +
            (c3[:, 0] * n3[:, 1] + c3[:, 1]) * n3[:, 2] + c3[:, 2])
    order = torch.argsort(cell, stable=True)
    count = torch.bincount(cell, minlength=ncell)
    start = torch.cumsum(count, 0) - count
    width = int(count.max())
    slot = torch.arange(len(x), device=dev) - start[cell[order]]
    table = torch.full((ncell + 1, width), -1, dtype=torch.long, device=dev)
    table[cell[order], slot] = order
    nbr = _dev(nbr).to(dev)
    gi, gj = [], []
    step = max(1, 40_000_000 // (width * width))
    for lo in range(0, ncell, step):
        a = table[lo:min(lo + step, ncell)]
        for k in range(27):
            b = table[nbr[k, lo:lo + len(a)]]
            ok = ((a[:, :, None] >= 0) & (b[:, None, :] > a[:, :, None]) &
                  (nbr[k, lo:lo + len(a)] >= 0)[:, None, None])
            p = ok.nonzero()
            i, j = a[p[:, 0], p[:, 1]], b[p[:, 0], p[:, 2]]
            d = x[i] - x[j]
            d = d - L[i] * torch.round(d / L[i])
            near = (d * d).sum(1) <= rl * rl
            gi.append(i[near])
            gj.append(j[near])
    return torch.cat(gi), torch.cat(gj)


def _lj_force(x, t, L, i, j, types):
    """Forces, energy (shifted at the cutoff) and virial of the listed pairs."""
    eps = torch.zeros((types, types), dtype=x.dtype, device=x.device)
    sig = eps.clone()
    for a, b, e, s in COEFF[types]:
        eps[a - 1, b - 1] = eps[b - 1, a - 1] = e
        sig[a - 1, b - 1] = sig[b - 1, a - 1] = s
    f = torch.zeros_like(x)
    pe = torch.zeros((), dtype=x.dtype, device=x.device)
    w = pe.clone()
    for lo in range(0, len(i), 20_000_000):
        a, b = i[lo:lo + 20_000_000], j[lo:lo + 20_000_000]
        d = x[a] - x[b]
        d = d - L[a] * torch.round(d / L[a])
        r2 = (d * d).sum(1)
        near = r2 < LJ_CUT * LJ_CUT
        a, b, d, r2 = a[near], b[near], d[near], r2[near]
        e, s6 = eps[t[a], t[b]], sig[t[a], t[b]] ** 6
        u = s6 / r2 ** 3
        fp = 24.0 * e * u * (2.0 * u - 1.0) / r2
        uc = s6 / LJ_CUT ** 6
        pe += (4.0 * e * (u * (u - 1.0) - uc * (uc - 1.0))).sum()
        w += (fp * r2).sum()
        d = d * fp[:, None]
        f.index_add_(0, a, d)
        f.index_add_(0, b, -d)
    return f, pe, w


def _sf_chunks(m, x, t, L, i, j):
    """Symmetry functions of every atom, some atoms at a time: yields (atoms,
    their neighbour tables and displacements, G)."""
    n, dev, rc = len(x), x.device, m["rc"]
    a, b = torch.cat([i, j]), torch.cat([j, i])
    d = x[b] - x[a]
    d = d - L[a] * torch.round(d / L[a])
    near = (d * d).sum(1) < rc * rc
    a, b, d = a[near], b[near], d[near]
    order = torch.argsort(a, stable=True)
    a, b, d = a[order], b[order], d[order]
    count = torch.bincount(a, minlength=n)
    start = torch.cumsum(count, 0) - count
    width = int(count.max())
    slot = torch.arange(len(a), device=dev) - start[a]
    # empty slots lie beyond the cutoff, and beyond it from one another
    D = torch.zeros((n, width, 3), dtype=x.dtype, device=dev)
    D[:, :, 0] = 100.0 + 10.0 * torch.arange(width, device=dev)
    J = torch.full((n, width), -1, dtype=torch.long, device=dev)
    D[a, slot], J[a, slot] = d, b
    tj = torch.where(J >= 0, t.long()[J.clamp(min=0)], -1)
    p, q = torch.triu_indices(width, width, 1, device=dev)

    def fcut(r):
        return torch.where(r < rc, 0.5 * (torch.cos(math.pi * r / rc) + 1), 0.0)

    reta = torch.tensor(m["reta"], dtype=x.dtype, device=dev)
    aeta = torch.tensor(m["aeta"], dtype=x.dtype, device=dev)
    step = max(1, 4_000_000 // max(1, len(p)))
    for lo in range(0, n, step):
        s = slice(lo, min(lo + step, n))
        dd = D[s].clone().requires_grad_(True)
        r = dd.norm(dim=2)
        fc = fcut(r)
        ex = torch.exp(-reta * (r * r)[..., None]) * fc[..., None]
        rad = torch.stack([(ex * (tj[s] == e)[..., None]).sum(1)
                           for e in range(m["nelem"])], 2)
        A, B = dd[:, p], dd[:, q]
        r1, r2, r3 = r[:, p], r[:, q], (B - A).norm(dim=2)
        cs = (A * B).sum(2) / (r1 * r2)
        F = fc[:, p] * fc[:, q] * fcut(r3)
        P = torch.stack([2.0 ** (1 - z) * (1 + lam * cs) ** z * F
                         for z, lam in m["pl"]], 1)
        E = torch.exp(-aeta * (r1 * r1 + r2 * r2 + r3 * r3)[..., None])
        ang = torch.matmul(P, E).transpose(1, 2)
        G = torch.cat([rad.flatten(1), ang.flatten(1)], 1)
        if not torch.is_grad_enabled():
            G = G.detach()
        yield s, (dd, J[s]), G.detach() if "gmin" not in m else G


def _nnp_force(m, x, t, L, i, j):
    f = torch.zeros_like(x)
    cst = [[torch.as_tensor(v[e], device=x.device) for v in
            (m["gmin"], m["gmax"])] for e in range(m["nelem"])]
    net = [[(torch.as_tensor(W, device=x.device),
             torch.as_tensor(b, device=x.device))
            for W, b in zip(m["W"][e], m["b"][e])] for e in range(m["nelem"])]
    for s, (dd, J), G in _sf_chunks(m, x, t, L, i, j):
        total = 0.0
        for e in range(m["nelem"]):
            h = G[t[s] == e]
            width = cst[e][1] - cst[e][0]
            h = torch.where(width > 0, (h - cst[e][0]) /
                            torch.where(width > 0, width, 1.0), 0.0)
            for l, (W, b) in enumerate(net[e]):
                h = h @ W.T + b
                h = torch.tanh(h) if l < 2 else h
            total = total + h.sum()
        g, = torch.autograd.grad(total, dd)  # dE/d(x_j - x_i)
        ok = J >= 0
        g = torch.where(ok[..., None], g, 0.0)
        f[s] += g.sum(1)
        f.index_add_(0, J[ok], -g[ok])
    return f


def _md64(x, v, t, sysid, Ls, steps, dt, rl, force):
    """Velocity Verlet from the given state, lists rebuilt every EVERY steps;
    mass 1.  Unwrapped positions, velocities and the last force result."""
    x, v, t, Ls = _dev(x).clone(), _dev(v).clone(), _dev(t), _dev(Ls)
    sysid = _dev(sysid)
    L = Ls[sysid]
    i, j = _pairs(x, sysid, Ls, rl)
    got = force(x, t, L, i, j)
    for s in range(1, steps + 1):
        v += 0.5 * dt * got[0]
        x += dt * v
        if s % EVERY == 0:
            i, j = _pairs(x, sysid, Ls, rl)
        got = force(x, t, L, i, j)
        v += 0.5 * dt * got[0]
    return x, v, got


def _lj64(boxes, steps, types=1):
    x, v, t = (np.concatenate([b[k] for b in boxes]) for k in "xvt")
    sysid = np.repeat(np.arange(len(boxes)), [len(b["x"]) for b in boxes])
    return _md64(x, v, t.astype(np.int64), sysid, np.stack([b["L"] for b in boxes]),
                 steps, DT, LJ_CUT + SKIN,
                 lambda *a: _lj_force(*a, types))


def _nnp64(m, box, steps):
    return _md64(box["x"], box["v"], box["t"].astype(np.int64),
                 np.zeros(len(box["x"]), np.int64), box["L"][None], steps,
                 NNP_DT, m["rc"] + SKIN, lambda *a: (_nnp_force(m, *a),))


def exact(case, seed):
    kind = case["kind"]
    if kind == "lj":
        box = _lj_box(case["nx"], case["ny"], case["nz"], case["rho"],
                      case["temp"], case["types"], seed)
        x, v, (f, pe, w) = _lj64([box], case["steps"], case["types"])
        n = len(x)
        mv2 = (v * v).sum()
        thermo = torch.stack([mv2 / (3 * n - 3), pe / n,
                              (pe + 0.5 * mv2) / n, w])
        # a half list's energy weighs pairs across the box by the list's own
        # rule, which has no value here
        return dict(x=x, v=v, f=f, thermo=None if case["half"] else thermo)
    if kind == "modules":
        box = _lj_box(case["nx"], case["ny"], case["nz"], case["rho"], 1.44, 1,
                      seed)
        _, _, (f, pe, w) = _lj64([box], 0)
        half = case["half"]
        return dict(f=f, pe=None if half else pe, w=None if half else w)
    if kind == "nnp":
        per = 1 if case["model"] == "two" else 4
        if per * case["nx"] * case["ny"] * case["nz"] > 25000:
            return None  # over 20 seconds
        m = _model(case["model"])
        box = _nnp_box(case["model"], case["nx"], case["ny"], case["nz"], seed)
        x, v, (f,) = _nnp64(m, box, case["steps"])
        return dict(x=x, v=v, f=f, thermo=None)
    if kind == "batch":
        x, v, (f, _, _) = _lj64(_batch_boxes(case, seed), case["steps"])
        return dict(x=x, v=v, f=f)
    out = {}
    m = _model("two")
    for name, want in (("lj", False), ("nnp", True)):
        got = []
        for nnp, steps, box in _serve_jobs(case, seed):
            if nnp == want:
                got.append(_nnp64(m, box, steps) if nnp
                           else _lj64([box], steps))
        if got:
            out[name + "_x"] = torch.cat([g[0] for g in got])
            out[name + "_v"] = torch.cat([g[1] for g in got])
    return out
