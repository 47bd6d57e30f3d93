"""List builds and layouts at the sizes where their routes change, through the
C ABI: the global build against a search of all pairs, batches on tiled lists
against the FP64 oracle and the global layout, and small boxes over several
rebuilds."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

import pyoracle as O
from test_gpu_batch import SYSTEMS, _add, _min_image, _oracle, _params

pytestmark = pytest.mark.gpu


def _pairs(x, rc, half):
    """Rows of all pairs within rc (accepted in FP64 as the engine does)."""
    d = cKDTree(x).query_pairs(rc * (1 + 1e-9), output_type="ndarray")
    i, j = np.concatenate([d, d[:, ::-1]]).T
    e = x[i] - x[j]
    ok = e[:, 0] ** 2 + e[:, 1] ** 2 + e[:, 2] ** 2 <= rc * rc
    if half:  # j above i in x, then y, then z
        up = [tuple(p) > tuple(q) for p, q in zip(x[j], x[i])]
        ok &= np.array(up, bool)
    i, j = i[ok], j[ok]
    rows = [set() for _ in x]
    for a, b in zip(i, j):
        rows[a].add(b)
    return rows


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("lanes", [1, 8])
@pytest.mark.parametrize("n,side,ghosts", [
    (1, 3.0, 0),       # one atom, one wave
    (5, 4.0, 2),       # waves of four atoms, a part-full one
    (700, 2.0, 60),    # one dense cell: two register passes
    (8191, 22.0, 0),   # the row scan's single block, one below,
    (8192, 22.0, 0),   # at
    (8193, 22.0, 900), # and above its limit
    (140000, 60.0, 0), # sixteen atoms a wave
])
def test_global_list_rows(gpu, n, side, ghosts, lanes, half):
    M = gpu
    if n > 100000 and (half or lanes > 1):
        pytest.skip("one of the large case is enough")
    rc = 1.3
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, side, (n + ghosts, 3))
    x[: n // 3, 0] = np.round(x[: n // 3, 0], 1)  # equal coordinates
    s = M.System(1)
    s.create_domain([0, 0, 0], [side] * 3, rc)
    s.upload(x, np.zeros_like(x), None, np.zeros(len(x), np.int32),
             np.arange(1, len(x) + 1, dtype=np.int32), n_ghost=ghosts)
    nl = M.NeighborVerlet(rc, half, 8, lanes=lanes)
    nl.create(s)
    off, idx = nl.get()
    rows = _pairs(x, rc, half)[:n]
    assert np.array_equal(np.diff(off), [len(r) for r in rows])
    for i in range(n):
        assert set(idx[off[i]:off[i + 1]].tolist()) == rows[i]


@pytest.mark.parametrize("shape", ["2,2,3,0", "4,1,6,0", "8,3,2,0"])
def test_batch_tiles_match_oracle(gpu, monkeypatch, shape):
    """Two rebuilds on tiled lists, as the global layout's own test (the same
    bounds); boxes of 3 to 5 cells, the lattice's atoms on the box faces."""
    M = gpu
    monkeypatch.setenv("CMD_TUNE", shape)
    B = M.Batch(_params(M), M.PREC_FP64, lanes=0)
    hs = [_add(M, B, s) for s in SYSTEMS]
    B.run(50)
    assert B.counts()["lanes"] == int(shape[0])
    for h, spec in zip(hs, SYSTEMS):
        L = np.array(spec[0]) * (4.0 / spec[1]) ** (1.0 / 3.0)
        x, v, f, _, _ = B.download(h)
        xo, vo, fo, tho = _oracle(spec, 50)
        assert np.abs(_min_image(x - xo, L)).max() < 1e-9
        assert np.abs(v - vo).max() < 1e-9
        assert np.abs(f - fo).max() < 1e-7 * np.abs(fo).max()
        for row in B.thermo(h):
            ro = tho[tho[:, 0] == row[0]][0]
            assert np.allclose(row[1:], ro[1:], rtol=1e-10, atol=1e-12), (row, ro)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_batch_tiles_alone_equals_in_mix(gpu, monkeypatch, prec):
    """Members join and leave around a system on tiled lists: bit-identical
    to the same system alone."""
    M = gpu
    monkeypatch.setenv("CMD_TUNE", "2,2,3,0")
    P = M.PREC_FP64 if prec == "fp64" else M.PREC_MIXED
    alone = M.Batch(_params(M), P, lanes=0)
    ha = _add(M, alone, SYSTEMS[1])
    mix = M.Batch(_params(M), P, lanes=0)
    hb = _add(M, mix, SYSTEMS[0])
    hm = _add(M, mix, SYSTEMS[1])
    for k in (20, 20, 7):
        alone.run(k)
        mix.run(k)
        if hb is not None:
            mix.remove(hb)
            _add(M, mix, SYSTEMS[3])
            hb = None
    for a, b in zip(alone.download(ha), mix.download(hm)):
        assert np.array_equal(a, b)
    assert np.array_equal(alone.thermo(ha), mix.thermo(hm))


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("ncells", [(4, 4, 4), (4, 5, 9)])
def test_small_box_rebuilds(gpu, ncells, half):
    """Boxes of two to five cells, every cell beside ghosts: the tiled list
    over five rebuilds against the oracle's loop."""
    M = gpu
    kw = dict(ncells=ncells, nsteps=100, thermo=20, half=half)
    md = M.CbnMD(M.lattice_params(**kw), precision=M.PREC_FP64, lanes=2)
    md.init()
    md.run(100)
    ref = O.MD(O.lj_params(**kw))
    ref.init()
    ref.run(100)
    n = md.n_local
    assert np.allclose(md.thermo()[:, :4], ref.thermo(), rtol=1e-10, atol=1e-13)
    x, v = md.arrays()[:2]
    xo, vo = ref.arrays()[:2]
    o, p = (np.argsort(m.arrays()[4][:n], kind="stable") for m in (md, ref))
    assert np.abs(x[:n][o] - xo[:n][p]).max() < 1e-9
    assert np.abs(v[:n][o] - vo[:n][p]).max() < 1e-9


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("lanes,width", [(2, 1), (2, 2), (8, 2)])
def test_half_list_skips_atoms_at_one_place(gpu, lanes, width, prec):
    """Two atoms at the same coordinates are no pair of a half list (neither
    is above the other), so they exert no force on each other: a list that
    asks for tiles, whose forces walk both sides of each pair, against the
    global layout, whose kernel walks the half rows."""
    M = gpu
    P = M.PREC_FP64 if prec == "fp64" else M.PREC_MIXED
    x, _, _, _, _, hi = M.fcc_system((7, 7, 8), 0.8442, 1.0, 5)
    hi = np.array(hi)
    rng = np.random.default_rng(5)
    x = np.mod(x + rng.normal(0, 0.05, x.shape), hi)
    # copies inside the box, beside a face and beside an edge (their ghosts
    # coincide too), and a triple
    twin = [700, int(np.argmin(x[:, 0])), int(np.argmin(x[:, 1] + x[:, 2])), 300, 300]
    x = np.vstack([x, x[twin]])
    n = len(x)
    out = []
    for kw in (dict(lanes=1), dict(lanes=lanes, tile_width=width)):
        s = M.System(1)
        s.create_domain([0, 0, 0], hi, 2.8)
        s.upload(x, None, None, np.zeros(n, np.int32), np.arange(1, n + 1, dtype=np.int32))
        M.Binning(s).create_binning(2.8, 2.8, 2.8, 1, True, False, True)
        comm = M.Comm(s, 2.8)
        comm.exchange_halo()
        nl = M.NeighborVerlet(2.8, True, 50, **kw)
        nl.create(s)
        F = M.ForceLJ(s, P)
        F.init_coeff([["pair_coeff", "1", "1", "1.0", "1.0", "2.5"]])
        F.compute(s, nl)
        comm.update_force()
        off, idx = nl.get()
        out.append((s.download()[2][:n], off, idx, F.compute_energy(s, nl)))
    (f1, off1, idx1, e1), (f, off, idx, e) = out
    assert np.array_equal(off, off1)
    for i in range(n):
        assert np.array_equal(*(np.sort(k[off[i]:off[i + 1]]) for k in (idx, idx1)))
    assert np.isfinite(f).all()
    tol = 1e-12 if prec == "fp64" else 1e-5
    assert np.abs(f - f1).max() < tol * np.abs(f1).max()
    assert abs(e - e1) < 1e-12 * abs(e1)


@pytest.mark.parametrize("shape", ["2,4,3,0", "2,0,3,0", "1,2,3,0", "3,2,3,0", "2,2,15,0",
                                   "2,2,3,9", "2,2,-1,0"])
@pytest.mark.parametrize("batch", [True, False])
def test_layouts_without_a_kernel_are_refused(gpu, monkeypatch, batch, shape):
    """CMD_TUNE values that no kernel has raise, in a batch and in CbnMD."""
    M = gpu
    monkeypatch.setenv("CMD_TUNE", shape)
    if batch:
        B = M.Batch(_params(M), M.PREC_FP64, lanes=0)
        _add(M, B, SYSTEMS[0])
        with pytest.raises(RuntimeError, match="CMD_TUNE"):
            B.run(1)
    elif shape not in ("2,0,3,0", "1,2,3,0"):  # one system: W 0 is the default
        md = M.CbnMD(M.lattice_params(ncells=(6, 6, 6)), precision=M.PREC_FP64)
        with pytest.raises(RuntimeError, match="CMD_TUNE"):
            md.init()


def test_small_batch_search_rebuilds_nothing(gpu, monkeypatch, capfd):
    """A batch too small for tiles compares lanes on one set of cells: the
    search neither times a rebuild nor makes one."""
    M = gpu
    monkeypatch.setenv("CMD_VERBOSE", "1")
    B = M.Batch(_params(M), M.PREC_FP64, lanes=0)
    for spec in SYSTEMS:
        _add(M, B, spec)
    B.run(1)
    err = capfd.readouterr().err
    assert err.count("# batch lanes=") == 4, err
    assert "# batch rebuild" not in err, err


def _gas_params(M, odd):
    """Atoms of diameter 0.5 (0.2) inside the same cutoff: dense boxes stay
    calm."""
    p = _params(M)
    p.coeff_sigma[0] = 0.2 if odd == "clump" else 0.5
    return p


def _boxed(x, v, hi):
    n = len(x)
    return dict(x=x, type=np.zeros(n, np.int32), lo=[0.0] * 3, hi=list(hi), v=v,
                id=np.arange(1, n + 1, dtype=np.int32))


def _odd_members(M):
    """Systems whose tiles do not fit as the batch's shape has them: one too
    dense for tiles of one cell, one dense in half of its box (fits with
    shorter tiles than its mean density suggests), one whose rows alone are
    too long (a clump around a corner of its cells), one with an atom that
    crosses its box between rebuilds."""
    dense = M.fcc_system((13, 12, 12), 2.9, 0.3, 7)
    half = M.fcc_system((11, 11, 24), 1.9, 0.3, 8)
    keep = half[0][:, 2] < 0.5 * half[5][2]
    x = np.array([[1.0, 1, 1], [5, 1, 1], [1, 5, 1], [5, 5, 1], [1, 4, 4.5]])
    v = np.zeros_like(x)
    v[4, 0] = 300.0
    g = 0.35 * (np.arange(7) - 3.0)
    c = np.array([(5.65 + a, 5.65 + b, 5.0 + e) for a in g for b in g for e in g])
    c = np.vstack([c, c[:49] - [0.35, 0, 0]])
    return dict(dense=_boxed(dense[0], dense[1], dense[5]),
                clump=_boxed(c, np.zeros_like(c), [11.3] * 3),
                half=_boxed(half[0][keep], half[1][keep], half[5]),
                fast=_boxed(x, v, [9.0] * 3))


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("odd", ["dense", "half", "clump", "fast"])
def test_batch_member_off_tiles_changes_no_other(gpu, monkeypatch, capfd, odd, prec):
    """A system that the tiles cannot hold joins a tiled batch: it gets shorter
    tiles or the global layout by itself, the others stay where they are, and
    both trajectories are the bits they are alone."""
    M = gpu
    monkeypatch.setenv("CMD_TUNE", "2,2,3,0")
    monkeypatch.setenv("CMD_VERBOSE", "1")
    P = M.PREC_FP64 if prec == "fp64" else M.PREC_MIXED
    calm = M.fcc_system((9, 9, 10), 1.2, 0.5, 3)
    member = _odd_members(M)[odd]
    alone = M.Batch(_gas_params(M, odd), P, lanes=0)
    ha = alone.add(**_boxed(calm[0], calm[1], calm[5]))
    single = M.Batch(_gas_params(M, odd), P, lanes=0)
    single.add(**_boxed(calm[0], calm[1], calm[5]))  # tunes the batch
    mix = M.Batch(_gas_params(M, odd), P, lanes=0)
    hm = mix.add(**_boxed(calm[0], calm[1], calm[5]))
    for B in (alone, mix, single):
        B.run(20)
    capfd.readouterr()
    ho = mix.add(**member)
    for k in (20, 20, 7):
        alone.run(k)
        mix.run(k)
    err = capfd.readouterr().err
    lowered = [int(l.split()[-1]) for l in err.splitlines() if "tile height" in l]
    for a, b in zip(alone.download(ha), mix.download(hm)):
        assert np.array_equal(a, b)
    assert np.array_equal(alone.thermo(ha), mix.thermo(hm))
    if odd == "half":
        assert lowered in ([2], [2, 1]), err
    else:  # (the mean density gives the uniformly dense box tiles of one cell at once)
        assert lowered == [0], err
    # the odd one against the same system with other company
    extra = M.fcc_system((8, 8, 8), 0.9, 0.5, 5)
    single.add(**_boxed(extra[0], extra[1], extra[5]))
    hs = single.add(**member)
    for k in (20, 20, 7):
        single.run(k)
    for a, b in zip(single.download(hs), mix.download(ho)):
        assert np.array_equal(a, b)
    assert np.array_equal(single.thermo(hs), mix.thermo(ho))
    # and against the global layout
    g = M.Batch(_gas_params(M, odd), P, lanes=4)
    hg = g.add(**member)
    g.run(47)
    x, xg = mix.download(ho)[0], g.download(hg)[0]
    assert np.abs(_min_image(x - xg, np.array(member["hi"]))).max() < 1e-7
    if odd == "fast":
        assert np.abs(_min_image(x[4] - (member["x"][4] + [300 * 0.005 * 47, 0, 0]),
                                 np.array(member["hi"]))).max() < 1e-9


def _two_types(M):
    p = _params(M, thermo=10)
    p.ntypes = 2
    p.mass[1] = 2.0
    p.ncoeff = 3
    for k, (a, b, eps, sig) in enumerate(((1, 1, 1.0, 1.0), (1, 2, 0.8, 1.1),
                                          (2, 2, 1.2, 0.95))):
        p.coeff_i[k], p.coeff_j[k] = a, b
        p.coeff_eps[k], p.coeff_sigma[k], p.coeff_cut[k] = eps, sig, 2.5
    return p


@pytest.mark.parametrize("shape", ["2,2,3,0", "4,1,4,0"])
def test_batch_tiles_two_types(gpu, monkeypatch, shape):
    """Two atom types with their own masses and cross coefficients: forces,
    positions and thermo rows on tiles against the global layout (FP64; the
    same sums in another order over 30 steps)."""
    M = gpu
    out = []
    for lanes in (0, 4):
        monkeypatch.setenv("CMD_TUNE", shape)
        B = M.Batch(_two_types(M), M.PREC_FP64, lanes=lanes)
        hs = []
        for cells, rho, temp, seed in SYSTEMS:
            x, v, t, i, lo, hi = M.fcc_system(cells, rho, temp, seed)
            t = t.copy()
            t[::3] = 1
            hs.append(B.add(x, t, lo, hi, v=v, id=i))
        B.run(30)
        out.append([(*B.download(h)[:3], B.thermo(h)) for h in hs])
    for a, b in zip(*out):
        for u, w in zip(a, b):
            assert np.abs(u - w).max() < 1e-9 * max(np.abs(w).max(), 1.0)


def test_batch_layout_search_with_tiles(gpu, monkeypatch, capfd):
    """A batch above the size from which the search times tiles too (and
    rebuilds on the loser's cells and back): against the fixed global layout,
    FP64, over two rebuilds."""
    M = gpu
    monkeypatch.setenv("CMD_VERBOSE", "1")
    spec = [((9 + k % 4, 10, 11), 0.7 + 0.02 * k, 0.8 + 0.1 * k, 200 + k) for k in range(15)]
    out = []
    for lanes in (0, 4):
        B = M.Batch(_params(M), M.PREC_FP64, lanes=lanes)
        hs = [_add(M, B, s) for s in spec]
        B.run(45)
        assert B.counts()["atoms"] > 65536
        out.append([(*B.download(h)[:3], B.thermo(h)) for h in hs])
    err = capfd.readouterr().err
    assert "tile=2x2x3" in err and "# batch rebuild" in err, err
    for s, a, b in zip(spec, *out):
        L = np.array(s[0]) * (4.0 / s[1]) ** (1.0 / 3.0)
        assert np.abs(_min_image(a[0] - b[0], L)).max() < 1e-9
        for u, w in zip(a[1:], b[1:]):
            assert np.abs(u - w).max() < 1e-8 * np.abs(w).max()


@pytest.mark.parametrize("width", [1, 2])
def test_half_list_ghost_images_in_the_step(gpu, width):
    """A tiled half list's step writes the next step's ghosts as a full
    list's does: 90 steps over four rebuilds equal the separate refresh bit
    for bit, ghost rows included."""
    M = gpu
    out = []
    for fuse in (True, False):
        md = M.CbnMD(M.lattice_params(ncells=(9, 8, 10), thermo=15, half=True),
                     precision=M.PREC_FP64, lanes=2, tile_width=width, fuse_ghosts=fuse)
        md.init()
        for k in (7, 33, 50):
            md.run(k)
        assert md.neighbor.layout()["tiled"]
        out.append((*md.arrays(), md.thermo()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
