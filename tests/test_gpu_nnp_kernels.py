"""NNP kernels at the sizes where their block and grid mappings can go wrong,
against the FP64 NNP oracle on open clusters (no periodic images in reach).

Bars: FP32 symmetry functions and sums carry 6e-8 relative per operation over
chains of at most a few hundred terms, so 2e-5 of each function's scale and
1e-4 of the energy and force scales leave a factor of ten.
"""
import numpy as np
import pytest

import pyoracle as O
from test_gpu_nnp import _engine_model, _system
from nnp_models import to_oracle

pytestmark = pytest.mark.gpu

BOX = 60.0


def _cluster(n, nelem, seed):
    """n atoms at least 0.9 apart in the middle of the box."""
    rng = np.random.default_rng(seed)
    side = max(2.0, (1.6 * n) ** (1.0 / 3.0))
    x = np.empty((0, 3))
    while len(x) < n:
        p = rng.uniform(0, side, 3)
        if len(x) == 0 or np.min(np.linalg.norm(x - p, axis=1)) >= 0.9:
            x = np.vstack([x, p])
    return x + 0.5 * (BOX - side), rng.integers(0, nelem, n).astype(np.int32)


def _model(nelem, etas, pl, ang_rs=0.0, rc=3.0, hidden=(7, 5), seed=3):
    """Radial functions on any neighbour and the (eta) x (zeta, lambda)
    angular grid for every element, in a shuffled order."""
    rng = np.random.default_rng(seed)
    m = dict(nelem=nelem, hidden=list(hidden), act="ttl", smin=0.0, smax=1.0,
             scale=True, sf=[], gmin=[], gmax=[], W=[], b=[],
             atom_energy=[0.0] * nelem)
    for e in range(nelem):
        sf = [(2, -1, -1, eta, 0.3 * k, 0.0, 0.0, rc)
              for k, eta in enumerate((0.05, 0.4))]
        sf += [(3, -1, -1, eta, ang_rs, lam, z, rc) for eta in etas
               for z, lam in pl]
        sf = [sf[k] for k in rng.permutation(len(sf))]
        n = len(sf)
        sizes = [n] + list(hidden) + [1]
        m["sf"].append(sf)
        m["gmin"].append(rng.uniform(0.0, 0.2, n))
        m["gmax"].append(m["gmin"][-1] + rng.uniform(1.0, 3.0, n))
        m["W"].append([rng.normal(0, 1, (sizes[l + 1], sizes[l])) /
                       np.sqrt(sizes[l]) for l in range(3)])
        m["b"].append([rng.normal(0, 0.1, sizes[l + 1]) for l in range(3)])
    return m


def _check(M, m, x, t, prec):
    nelem = m["nelem"]
    cut = m["sf"][0][0][7] + 0.3
    s, comm, nl = _system(M, x, t, [BOX] * 3, cut, ntypes=nelem)
    # scale every function to the cluster's own range, as a fitted model does
    # (far outside it the layers saturate and 1 - tanh^2 cancels)
    off, idx = nl.get()
    _, _, G0, _, _ = to_oracle(O, m).compute(s.download()[0], t, len(x), off,
                                             idx, ld=96)
    for e in range(nelem):
        if (t == e).any():
            g = G0[t == e][:, :len(m["sf"][e])]
            m["gmin"][e] = g.min(axis=0)
            m["gmax"][e] = np.maximum(g.max(axis=0), g.min(axis=0) + 0.5)
    F = M.ForceNNP(_engine_model(M, m),
                   M.PREC_FP64 if prec == "fp32" else M.PREC_MIXED)
    F.compute(s, nl)
    f = s.download()[2][:len(x)]
    G, _, E = F.atomic(s, 96)
    _, Eo, Go, _, fo = to_oracle(O, m).compute(s.download()[0], t, len(x), off,
                                               idx, ld=96)
    for e in range(nelem):
        k = t == e
        if k.any():
            ns = len(m["sf"][e])
            scale = np.maximum(np.abs(Go[k][:, :ns]).max(axis=0), 1e-3)
            assert (np.abs(G[k][:, :ns] - Go[k][:, :ns]) / scale).max() < 2e-5
    assert np.abs(E - Eo).max() < 1e-4 * max(np.abs(Eo).max(), 1e-3)
    fs = max(np.sqrt((fo[:len(x)] ** 2).sum(1).mean()), 1e-6)
    assert np.sqrt(((f - fo[:len(x)]) ** 2).sum(1)).max() < 1e-4 * fs


PL = [(z, lam) for z in (1.0, 3.0) for lam in (-1.0, 1.0)]


@pytest.mark.parametrize("prec", ["fp32", "bf16"])
@pytest.mark.parametrize("nelem,n", [(1, 1), (1, 16), (1, 65), (2, 63),
                                     (2, 130), (3, 64), (4, 66), (4, 200)])
def test_network_tiles(gpu, nelem, n, prec):
    """The network kernel's blocks of 64 atoms and tiles of 16 atoms of one
    element: part-full tiles and blocks, one to four elements."""
    x, t = _cluster(n, nelem, 10 * n + nelem)
    _check(gpu, _model(nelem, (0.01, 0.2), PL), x, t, prec)


@pytest.mark.parametrize("prec", ["fp32", "bf16"])
@pytest.mark.parametrize("neta", [1, 7, 8])
def test_network_input_widths(gpu, neta, prec):
    """Function counts around the 32-deep blocks of the first product: 10,
    58 and 66 inputs, and hidden layers of 32 and 1 nodes."""
    pl = [(z, lam) for z in (1.0, 2.0, 3.0, 5.0) for lam in (-1.0, 1.0)]
    etas = [0.02 * (k + 1) for k in range(neta)]
    x, t = _cluster(50, 2, neta)
    _check(gpu, _model(2, etas, pl, hidden=(32, 1)), x, t, prec)


POW2 = [(z, lam) for lam in (1.0, -1.0) for z in (16.0, 1.0, 4.0, 2.0)]


@pytest.mark.parametrize("neta", range(1, 9))
def test_power_of_two_grid(gpu, neta):
    """zeta 1, 2, 4, 16 with both lambdas (the squaring kernels), one to
    eight etas, functions in any order; 15 to 20 neighbours per atom."""
    etas = [0.02 * (k + 1) for k in range(neta)]
    x, t = _cluster(60, 2, 100 + neta)
    _check(gpu, _model(2, etas, POW2), x, t, "bf16")


@pytest.mark.parametrize("n", [2, 3, 64, 65, 66, 100, 129])
@pytest.mark.parametrize("pl", ["pow2", "general"])
def test_neighbour_counts(gpu, n, pl):
    """Every atom of the cluster a neighbour of every other: 1, 2, 63, 64, 65
    and 128 neighbours, where the pair walk changes form and the buffer of
    pairs is emptied one or more times."""
    x, t = _cluster(n, 1, n)
    x = BOX / 2 + (x - BOX / 2) * min(1.0, 4.0 / np.ptp(x, axis=0).max())
    m = _model(1, (0.01, 0.05), POW2 if pl == "pow2" else PL, rc=8.0)
    _check(gpu, m, x, t, "fp32")


@pytest.mark.parametrize("neta", [1, 5, 8])
@pytest.mark.parametrize("n", [64, 66, 67, 100, 127])
def test_one_wave_past_64_neighbours(gpu, n, neta):
    """A cluster of n atoms, every one a neighbour of every other, among
    atoms with six at most: too few neighbours on average for four waves on an
    atom, so one wave walks 63 to 126 neighbours, with pair counts of every
    remainder by 4 (the lanes that share a block of matrix products)."""
    x, t = _cluster(n, 1, n)
    x = BOX / 2 + (x - BOX / 2) * min(1.0, 4.0 / np.ptp(x, axis=0).max())
    g = np.arange(9.0, 52.0, 6.0)
    lone = np.array([(a, b, c) for a in g for b in g for c in g])
    lone = lone[np.linalg.norm(lone - BOX / 2, axis=1) > 12.0]
    assert n * (n - 1) + 6 * len(lone) < 32 * (n + len(lone))
    x = np.vstack([x, lone])
    t = np.zeros(len(x), np.int32)
    m = _model(1, [0.01 * (k + 1) for k in range(neta)], POW2, rc=8.0)
    _check(gpu, m, x, t, "fp32")


def test_one_wave_per_atom_at_62_neighbours(gpu):
    """3,375 atoms, past the sizes that put four waves on an atom: the ring
    walk with most lanes in use, forces within 1e-5 of the oracle."""
    from test_gpu_nnp import _fitted_benchmark_model, _run
    M = gpu
    x, t, _ = M.nnp_lattice((15, 15, 15), spacing=2.5, jitter=0.1, seed=5)
    L = [37.5] * 3
    model = _fitted_benchmark_model(M, x, t, L)
    m = model.describe(2)
    m.update(act="ttl", smin=0.0, smax=1.0, scale=True)
    s, comm, nl = _system(M, x, t, L, 6.3)
    r = _run(M, s, comm, nl, M.ForceNNP(model, M.PREC_MIXED), m)
    assert (np.linalg.norm(r["f"] - r["fo"]) <
            1e-5 * np.linalg.norm(r["fo"]))


@pytest.mark.parametrize("cells,spacing", [((11, 11, 12), 2.7), ((11, 12, 12), 2.7),
                                           ((14, 14, 15), 2.5), ((11, 12, 12), 3.5)])
def test_waves_per_atom(gpu, cells, spacing):
    """Around the sizes where an atom gets four waves: 1,452 (four) and 1,584
    atoms (one) of 55 listed neighbours, 2,940 of 75 (four) and 1,584 of 24
    (one): forces within 1e-5 of the oracle."""
    from test_gpu_nnp import _fitted_benchmark_model, _run
    M = gpu
    x, t, _ = M.nnp_lattice(cells, spacing=spacing, jitter=0.1, seed=5)
    L = [spacing * c for c in cells]
    model = _fitted_benchmark_model(M, x, t, L)
    m = model.describe(2)
    m.update(act="ttl", smin=0.0, smax=1.0, scale=True)
    s, comm, nl = _system(M, x, t, L, 6.3)
    r = _run(M, s, comm, nl, M.ForceNNP(model, M.PREC_MIXED), m)
    assert (np.linalg.norm(r["f"] - r["fo"]) <
            1e-5 * np.linalg.norm(r["fo"]))


@pytest.mark.parametrize("batch", [False, True])
def test_joined_kicks_match_separate_ones(gpu, batch):
    """A run whose steps join the final and the next first half kick against
    one with a thermo row (separate kicks) every step, over two rebuilds:
    equal up to the order of the force atomics (1e-16 a step, 45 steps)."""
    M = gpu
    m = _model(2, (0.01, 0.05), POW2, rc=4.0)
    x, t, ids = M.nnp_lattice((6, 6, 7), spacing=2.0, jitter=0.1, seed=3)
    L = [12.0, 12.0, 14.0]
    x = np.mod(x, L)
    v = np.random.default_rng(1).normal(0, 0.5, x.shape)
    out = []
    for thermo in (1, 100):
        p = M.nnp_params(cutoff=4.0, thermo=thermo, dt=0.002)
        if batch:
            B = M.Batch(p, M.PREC_MIXED, nnp_model=_engine_model(M, m))
            h = B.add(x, t, [0, 0, 0], L, v=v, id=ids)
            B.run(45)
            out.append(B.download(h)[:3])
        else:
            md = M.CbnMD(p, M.PREC_MIXED)
            md.set_nnp_model(_engine_model(M, m))
            md.set_initial_state(x, t, [0, 0, 0], L, v=v, id=ids)
            md.init()
            md.run(45)
            n = md.n_local
            a = md.arrays()
            o = np.argsort(a[4][:n])
            out.append([k[:n][o] for k in a[:3]])
    for a, b in zip(*out):
        assert np.abs(a - b).max() < 1e-11 * np.abs(b).max()


@pytest.mark.parametrize("thermo", [3, 100])
@pytest.mark.parametrize("every", [7, 4, 50])
@pytest.mark.parametrize("batch", [False, True])
def test_neighbour_overflow_stops_at_its_step(gpu, batch, every, thermo):
    """A cluster that shrinks evenly (a network of negligible forces) until an
    atom has more than 128 neighbours inside the cutoff, at step 6: the run
    ends with the positions of that step and with no thermo row from it or
    later ones, whether a rebuild, a thermo row or the last step follows."""
    M = gpu
    m = _model(1, (0.01,), POW2, rc=4.0)
    m["W"][0][2] *= 1e-9
    n, dt, rate = 400, 0.01, 0.6
    x, t = _cluster(n, 1, 7)
    c = np.full(3, BOX / 2)

    def most(s):
        d = np.linalg.norm(x[:, None] - x[None], axis=2) * (1 - rate * dt * s)
        return (d < 4.0).sum(1).max() - 1

    # a size from which the limit is passed some steps later
    while most(0) > 120:
        x = c + (x - c) * 1.01
    over = next(s for s in range(1, 100) if most(s) > 128)
    assert over == 6
    v = -rate * (x - c)
    p = M.nnp_params(ntypes=1, cutoff=4.0, skin=2.0, thermo=thermo, dt=dt, every=every,
                     max_neigh_guess=300)
    model = _engine_model(M, m)
    ids = np.arange(1, n + 1, dtype=np.int32)
    if batch:
        B = M.Batch(p, M.PREC_MIXED, nnp_model=model)
        h = B.add(x, t, [0, 0, 0], [BOX] * 3, v=v, id=ids)
        run, rows = B.run, lambda: B.thermo(h)
        state = lambda: B.download(h)[:2]
    else:
        md = M.CbnMD(p, M.PREC_MIXED)
        md.set_nnp_model(model)
        md.set_initial_state(x, t, [0, 0, 0], [BOX] * 3, v=v, id=ids)
        md.init()
        run, rows = md.run, md.thermo

        def state():
            a = md.arrays()
            o = np.argsort(a[4][:n])
            return a[0][:n][o], a[1][:n][o]
    with pytest.raises(RuntimeError, match="more than 128 neighbours"):
        run(60)
    assert rows()[-1, 0] == (over - 1) // thermo * thermo
    xs, vs = state()
    assert np.abs(xs - (x + v * dt * over)).max() < 1e-9
    assert np.abs(vs - v).max() < 1e-9
    if batch:
        assert B.counts()["step"] == over


def test_ghosts_alone_get_zero_forces(gpu):
    """A system of uploaded ghosts and no local atom: force rows cleared."""
    M = gpu
    m = _model(1, (0.01,), POW2)
    x = np.random.default_rng(1).uniform(0, 10, (9, 3))
    s = M.System(1)
    s.create_domain([0, 0, 0], [10.0] * 3, 3.3)
    s.upload(x, None, np.ones_like(x), np.zeros(9, np.int32),
             np.arange(1, 10, dtype=np.int32), n_ghost=9)
    nl = M.NeighborVerlet(3.3, False, 50, lanes=1)
    nl.create(s)
    M.ForceNNP(_engine_model(M, m)).compute(s, nl)
    assert not s.download()[2].any()
