"""Kernels at the sizes where their tiles, remainders and dispatch rules change,
against the FP64 oracle.

Bars: lists are the oracle's entry for entry; FP64 energies and forces agree to
1e-12 relative, the repository's bar for sums that differ in order only (n terms
of one sign leave at most n eps, 3e-13 at the 1,026 atoms here; the transforms'
log2(N) rounding steps of 1e-16 lie below that)."""
import ctypes as C

import numpy as np
import pytest

import mdbas_amd as M
import oracle as O
from mdbas_amd import configs
from test_zz_no_alloc import Hip, relerr

pytestmark = pytest.mark.gpu


def water(nw, cut, delr, **kw):
    L = (nw / 0.0334) ** (1 / 3)
    return configs.build(dict(configs.COMMON, name=f"w{nw}", n_waters=nw, L=L, seed=nw,
                              timeStep=0.002, precision="fp64", **dict(
                                  dict(grid=20, cutOff=cut, cutOn=cut - 1.5, delr=delr,
                                       alpha=0.35), **kw)))


# Meshes of the in-LDS convolution (every radix, unequal edges, the largest
# plane) and of the library transforms (odd index 3, a factor 7, a plane above
# the limit); spline orders of the binned spreading and of the general one.
@pytest.mark.parametrize("mesh,order", [
    ((20, 20, 20), 4), ((24, 30, 36), 4), ((45, 27, 32), 4), ((50, 64, 18), 4), ((32, 18, 40), 6),
    ((25, 48, 54), 8), ((80, 80, 80), 4), ((18, 20, 22), 4), ((20, 24, 25), 4), ((28, 20, 20), 4),
    ((18, 96, 90), 4), ((24, 20, 32), 10)])
def test_spme_meshes(mesh, order, monkeypatch):
    wb = water(216, 7.0, 1.0, nbsp=order)
    print("mesh", mesh, order, flush=True)
    o = O.OracleSystem(wb)
    o.p.m1, o.p.m2, o.p.m3 = mesh
    made = M.reference_structs

    def structs(*a):
        s = made(*a)
        s[3].m1max, s[3].m2max, s[3].m3max = mesh
        return s

    monkeypatch.setattr(M, "reference_structs", structs)
    ctx = M.Context(wb)
    # twice on moved positions: the second call finds what the first one left
    for shift in (0.0, 0.3):
        x, y, z = wb.x + shift, wb.y - 2 * shift, wb.z + 3 * shift
        er, fr, st, vr = o.spme(x, y, z)
        eg, fg, sg, vg = ctx.spme_energy(x, y, z)
        assert eg == pytest.approx(er, rel=1e-12)
        assert vg == pytest.approx(vr, rel=1e-10)
        assert np.allclose(sg[[0, 3, 5]], st[[0, 3, 5]], rtol=1e-10)
        # off the diagonal the half spectrum counts a point with one index at
        # m/2 twice with one sign, the full one once with each; those points hold
        # exp(-pi^2 m^2 / (4 a^2 L^2)) of the sum: 7e-9 each way for m = 18, the
        # shortest axis here (4e-7 for 16), with L = 18.6 A and even orders (an
        # odd order's spline transform vanishes there)
        assert np.allclose(sg, st, rtol=1e-10, atol=1e-7 * np.abs(st).max())
        assert relerr(fg, fr) < 1e-12
    ctx.close()


# 33 to 1,026 atoms: below one row group, one past 64 and 128, both sides of
# 1,024 (the offsets' block), lists with one-entry remainders.
@pytest.mark.parametrize("nw", [11, 21, 22, 43, 86, 341, 342])
def test_reference_list_sizes(nw):
    wb = water(nw, 2.6 if nw < 30 else 3.4, 0.4)
    print("atoms", wb.n, flush=True)
    o = O.OracleSystem(wb)
    x, y, z = wb.x.copy(), wb.y.copy(), wb.z.copy()
    nl, np_, no = o.build_list(x, y, z)
    ctx = M.Context(wb)
    gx, gy, gz = wb.x.copy(), wb.y.copy(), wb.z.copy()
    gnl, gnp, gno, _, _ = ctx.makelist(gx, gy, gz)
    assert np.array_equal(gnl, nl) and np.array_equal(gnp, np_) and np.array_equal(gno, no)
    f_o, e_o = o.energy(x, y, z)
    f_g, e_g = ctx.energy(x, y, z, nl, np_, no)
    assert relerr(f_g, f_o) < 1e-12
    # the device-resident path: its own list, cut into chunks by its length
    ctx.upload(x, y, z, wb.vx, wb.vy, wb.vz)
    e_d = ctx.initial_energy()
    terms = sum(abs(e_o[k]) for k in ("eDir", "eRec", "eCorr", "vdw"))
    assert e_d.nInCut == e_o["nInCut"]
    assert abs(e_d.pot - e_o["pot"]) < 1e-12 * terms
    for elec in (2, 3, 4):
        f_n, e_n = o.nonbond_energy(elec, x, y, z)
        f_g, e_g = ctx.nonbond_energy(elec, x, y, z, nl, np_, no)
        assert relerr(f_g, f_n) < 1e-12
    ctrl, param, pbc = ctx.ctrl, ctx.param, ctx.pbc
    ctrl.elecType = 4
    ctx.close()
    # the call that allocates nothing, on the caller's device arrays
    hip = Hip()
    zero = np.zeros(wb.n)
    dev = [hip.put(a) for a in (x, y, z, zero, zero, zero, wb.q, wb.eps, wb.sig, nl, np_, no)]
    en = hip.put(np.zeros(4))
    hip.sync()
    assert M.load().mdg_nonbond_energy_noalloc(C.byref(ctrl), C.byref(param), C.byref(pbc), *dev,
                                               en, None) == 0
    hip.sync()
    f = np.stack([hip.get(p, zero) for p in dev[3:6]])
    hip.free()
    assert relerr(f, f_n) < 1e-12


# Drop-in transfers on both sides of the pinned buffer's limit (1 MiB): an
# integrator stage crosses it between 3,790 and 3,810 molecules (92 bytes an
# atom), the plain energies between 4,150 and 4,170 (84 bytes).
@pytest.mark.parametrize("nw", [3790, 3810, 4150, 4170])
def test_dropin_transfer_sizes(nw):
    wb = water(nw, 4.0, 0.5)
    print("atoms", wb.n, flush=True)
    o = O.OracleSystem(wb)
    x, y, z = wb.x.copy(), wb.y.copy(), wb.z.copy()
    nl, np_, no = o.build_list(x, y, z)
    ctx = M.Context(wb)
    gx, gy, gz = wb.x.copy(), wb.y.copy(), wb.z.copy()
    gnl, gnp, gno, _, _ = ctx.makelist(gx, gy, gz)
    assert np.array_equal(gx, x) and np.array_equal(gnl, nl)
    assert np.array_equal(gnp, np_) and np.array_equal(gno, no)
    f_o, e_o = o.nonbond_energy(4, x, y, z)
    f_g, e_g = ctx.nonbond_energy(4, x, y, z, nl, np_, no)
    assert relerr(f_g, f_o) < 1e-12 and e_g.vdw == pytest.approx(e_o["vdw"], rel=1e-11)
    s_o = [x, y, z, wb.vx.copy(), wb.vy.copy(), wb.vz.copy()]
    s_g = [a.copy() for a in s_o]
    for stage in (1, 2):
        err, *_ = o.vv(stage, *s_o, f_o)
        assert err == 0
        ctx.vv_integrate(stage, *s_g, f_o.copy())
        assert max(np.abs(a - b).max() for a, b in zip(s_o, s_g)) < 1e-12
    ctx.close()


# A drop-in call without one of its arrays is refused, and the context computes
# the same afterwards.
def test_dropin_missing_arrays():
    wb = water(43, 3.4, 0.4)
    ctx = M.Context(wb)
    x, y, z = wb.x.copy(), wb.y.copy(), wb.z.copy()
    lists = ctx.makelist(x, y, z)[:3]
    v = [wb.vx.copy(), wb.vy.copy(), wb.vz.copy()]
    f0 = ctx.energy(x, y, z, *lists)[0]
    g = M.P
    e, s, d = M.MDG_ENERGY(), np.zeros(6), C.c_double(0)
    L, h, by = ctx.L, ctx.h, C.byref
    el, ep = ctx._excl

    def refused(name, fn, head, arrays, tail):
        for k in range(len(arrays)):
            print(name, "without array", k, flush=True)
            got = [g(a.copy()) for a in arrays]
            got[k] = None
            assert fn(h, *head, *got, *tail) != 0, (name, k)

    pos, force = [x, y, z], [np.zeros(wb.n)] * 3
    par, nl = [wb.q, wb.eps, wb.sig], [g(a) for a in lists]
    refused("spme", L.mdg_spme_energy, [by(ctx.param), by(ctx.ewald), by(ctx.pbc)],
            pos + force + [wb.q], [g(s), by(d), by(d)])
    refused("ewald", L.mdg_ewald_energy,
            [by(ctx.ctrl), by(ctx.param), by(e), by(ctx.ewald), by(ctx.pbc)], pos + force,
            [g(a) for a in par] + nl + [el, ep])
    refused("nonbond", L.mdg_nonbond_energy, [by(ctx.ctrl), by(ctx.param), by(e), by(ctx.pbc)],
            pos + force, [g(a) for a in par] + nl)
    head = [by(ctx.ctrl), by(ctx.param), by(e), by(ctx.ewald), by(ctx.pbc), by(ctx.neigh)]
    none = [None] * 5
    tail = [g(a) for a in par] + [None, None, g(wb.frozen)] + nl + [None, el, ep]
    vel = [g(a) for a in v]
    refused("energy positions", L.mdg_energy, head + none, pos,
            vel + [g(a) for a in force] + tail)
    refused("energy forces", L.mdg_energy, head + none + [g(a) for a in pos] + vel, force, tail)
    refused("vv", L.mdg_vv_integrate,
            [by(ctx.ctrl), by(ctx.param), by(e), by(ctx.pbc), None, ctx.cons],
            pos + v + list(f0) + [wb.mass, wb.rmass], [g(wb.nAtConst), 2])
    assert np.allclose(ctx.energy(x, y, z, *lists)[0], f0, rtol=1e-12, atol=1e-9)
    ctx.close()


# Pairs exactly half an edge apart inside the cutoff: 64 equal waters on a 4 A
# lattice along x (edge 16 A, cutoff 9 A), moved along y and z, so that the image
# index is a tie for atoms of one kind two cells apart.
def test_half_edge_images():
    wb = configs.build(dict(configs.COMMON, name="lattice", n_waters=64, L=16.0, seed=3, grid=16,
                            timeStep=0.002, precision="fp64", cutOff=9.0, cutOn=7.5, delr=0.5,
                            alpha=0.35))
    rng = np.random.default_rng(3)
    cell = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(64, 3) * 4.0 - 6.0
    cell[:, 1:] += rng.uniform(-0.4, 0.4, (64, 2))
    mol = np.stack([wb.x[:3], wb.y[:3], wb.z[:3]], 1)
    mol = np.round((mol - mol[0]) * 2**20) / 2**20      # differences along x are exact
    p = (cell[:, None, :] + mol[None]).reshape(-1, 3)
    x, y, z = (np.ascontiguousarray(p[:, k]) for k in range(3))
    ties = np.abs(x[:, None] - x[None]) == 8.0
    assert ties.sum() > 1000
    o = O.OracleSystem(wb)
    nl, np_, no = o.build_list(x, y, z)
    ctx = M.Context(wb)
    ctx.makelist(x.copy(), y.copy(), z.copy())
    for elec in (2, 4):
        f_o, _ = o.nonbond_energy(elec, x, y, z)
        assert relerr(ctx.nonbond_energy(elec, x, y, z, nl, np_, no)[0], f_o) < 1e-12
    f_o, e_o = o.energy(x, y, z)
    assert relerr(ctx.energy(x, y, z, nl, np_, no)[0], f_o) < 1e-12
    ctx.upload(x, y, z, *[np.zeros(wb.n)] * 3)
    e_d = ctx.initial_energy()
    assert e_d.nInCut == e_o["nInCut"]
    assert relerr(np.stack(ctx.download()[6:9]), f_o) < 1e-12
    ctx.close()


def pairset(nl, np_, no, n):
    a, c = np.repeat(no, np_[no]).astype(np.int64), nl.astype(np.int64)
    return np.sort(np.minimum(a, c) * n + np.maximum(a, c))


def device_pairs(ctx):
    pi, pj = ctx.list_pairs()
    return np.sort(pi.astype(np.int64) * ctx.n + pj)


# Cluster search with four wavefronts a cluster at cutoffs where one of them finds
# several hundred entries.
@pytest.mark.parametrize("nw,cut", [(1000, 14.5), (1500, 17.0), (2500, 18.0), (3000, 20.0)])
def test_long_cutoff_lists(nw, cut):
    wb = water(nw, cut, 0.5)
    print("atoms", wb.n, "cutoff", cut, flush=True)
    o = O.OracleSystem(wb)
    x, y, z = wb.x.copy(), wb.y.copy(), wb.z.copy()
    want = pairset(*o.build_list(x, y, z), wb.n)
    ctx = M.Context(wb)
    ctx.upload(x, y, z, wb.vx, wb.vy, wb.vz)
    ctx.initial_energy()
    print(ctx.list_stats(), flush=True)
    assert np.array_equal(device_pairs(ctx), want)
    ctx.close()


# Replicas small enough that a wavefront holds three and more of them, their SHAKE
# sweeps unequal (66 to 600 K), against a single box each.
@pytest.mark.parametrize("spread", [0, 1, 2])
def test_small_replicas(spread):
    boxes = []
    for k, (nw, temp) in enumerate([(30, 66.0), (45, 600.0), (33, 100.0), (52, 300.0), (30, 450.0),
                                    (38, 150.0), (64, 300.0), (31, 500.0)]):
        boxes.append(configs.build(dict(
            configs.COMMON, name=f"r{k}", n_waters=nw, L=(nw / 0.0334) ** (1 / 3), seed=50 + k,
            grid=16, cutOff=4.3, cutOn=2.8, delr=0.3, alpha=0.35, temp=temp, timeStep=0.0005,
            precision="fp64")))
    print("spread", spread, [b.n for b in boxes], flush=True)
    b = M.BatchContext(boxes, precision=M.MDG_FP64)
    b.set_launch(**dict(b.get_launch(), shake_spread=spread))
    b.upload_boxes()
    b.initial_energy()
    rb = M.batch_records(b.run(6), b.R)
    sb = [b.split(a) for a in b.download()[:6]]
    b.close()
    for r, wb in enumerate(boxes):
        c = M.Context(wb)
        c.upload(wb.x, wb.y, wb.z, wb.vx, wb.vy, wb.vz)
        c.initial_energy()
        rs = M.records_to_dict(c.run(6))
        ss = c.download()[:6]
        c.close()
        for k in ("tot", "kin", "virshake"):
            assert np.allclose(rb[k][:, r], rs[k], rtol=1e-10, atol=1e-10 * abs(rs["pot"][0])), k
        assert max(np.abs(sb[k][r] - ss[k]).max() for k in range(6)) < 1e-9


def lists_equal(got, want):
    return all(np.array_equal(a, b) for a, b in zip(got, want))


def frozen_steps(ctx, o, wb, x, y, z, nsteps=3):
    """A few device-resident FP64 steps with frozen atoms (no force and no velocity
    after the energies, utils.c:131-153) against the oracle's stages (1e-9 A over
    the rounding of a few steps, as the batch tests)."""
    s = [x.copy(), y.copy(), z.copy(), wb.vx.copy(), wb.vy.copy(), wb.vz.copy()]
    ctx.upload(*s)
    ctx.initial_energy()
    ctx.run(nsteps)
    g = ctx.download()

    def forces():
        f, _ = o.energy(*s[:3])
        for a in (*s[3:], *f):
            a[wb.frozen != 0] = 0.0
        return f

    f = forces()
    for _ in range(nsteps):
        assert o.vv(1, *s, f)[0] == 0
        f = forces()
        assert o.vv(2, *s, f)[0] == 0
    assert relerr(np.stack(g[6:9]), f) < 1e-9
    assert max(np.abs(a - b).max() for a, b in zip(g[:6], s)) < 1e-9


# Every third molecule frozen, through both list builders (link cells from 136
# molecules on), the device list, a batch, and a step; flags that only makelist is
# given, and their going away.
@pytest.mark.parametrize("nw", [43, 136])
def test_frozen_atoms(nw):
    wb = water(nw, 3.4, 0.4)
    free = M.Context(wb)
    x, y, z = wb.x.copy(), wb.y.copy(), wb.z.copy()
    o_free = O.OracleSystem(wb)
    want_free = [a.copy() for a in o_free.build_list(x, y, z)]
    assert free.key_link == o_free.keyLink == (1 if nw == 136 else 0)
    wb.frozen = np.repeat((np.arange(nw) % 3 == 0).astype(np.int32), 3)
    wb.vx, wb.vy, wb.vz = (np.where(wb.frozen, 0.0, v) for v in (wb.vx, wb.vy, wb.vz))
    o = O.OracleSystem(wb)
    want = [a.copy() for a in o.build_list(x, y, z)]
    assert len(want[0]) < len(want_free[0])
    # the flags come with makelist alone, then without them
    pos = lambda: (x.copy(), y.copy(), z.copy())  # noqa: E731
    assert lists_equal(free.makelist(*pos())[:3], want)
    wb.frozen, flags = np.zeros_like(wb.frozen), wb.frozen
    free.ctrl.newjob = 1
    assert lists_equal(free.makelist(*pos())[:3], want_free)
    free.close()
    wb.frozen = flags
    ctx = M.Context(wb)
    assert lists_equal(ctx.makelist(*pos())[:3], want)
    frozen_steps(ctx, o, wb, x, y, z)
    ctx.upload(x, y, z, wb.vx, wb.vy, wb.vz)
    ctx.initial_energy()
    assert np.array_equal(device_pairs(ctx), pairset(*want, wb.n))
    ctx.close()
    if nw == 43:
        b = M.BatchContext([wb, wb])
        b.upload_boxes()
        b.initial_energy()
        one = pairset(*want, 2 * wb.n)
        assert np.array_equal(device_pairs(b),
                              np.sort(np.concatenate([one, one + wb.n * (2 * wb.n + 1)])))
        b.close()


# Triclinic boxes (the drop-in calls take them): both list builders, the pair loop,
# meshes of the in-LDS convolution and of the library's transforms, and SHAKE.
@pytest.mark.parametrize("nw,grid", [(60, 24), (60, 22), (136, 24)])
def test_triclinic_boxes(nw, grid, monkeypatch):
    wb = water(nw, 3.4, 0.4, grid=grid)
    L = wb.L
    cell = np.array([[L, 0, 0], [0.12 * L, L, 0], [-0.09 * L, 0.07 * L, L]])
    p = np.stack([wb.x, wb.y, wb.z], 1).reshape(-1, 3, 3)
    rel = p - p[:, :1]
    rel -= L * np.round(rel / L)
    p = ((p[:, :1] / L) @ cell + rel).reshape(-1, 3)
    x, y, z = (np.ascontiguousarray(p[:, k]) for k in range(3))
    monkeypatch.setattr(O, "make_box", lambda edge: O.box_from9(cell.ravel(), 3))
    made = M.reference_structs

    def structs(*a):
        s = made(*a)
        s[2].type = 3
        (s[2].a1, s[2].a2, s[2].a3, s[2].b1, s[2].b2, s[2].b3, s[2].c1, s[2].c2,
         s[2].c3) = cell.ravel()
        return s

    monkeypatch.setattr(M, "reference_structs", structs)
    print("triclinic", wb.n, "atoms, mesh", grid, flush=True)
    o = O.OracleSystem(wb)
    ctx = M.Context(wb)
    assert ctx.key_link == o.keyLink == (1 if nw == 136 else 0)
    g = [x.copy(), y.copy(), z.copy()]
    want = [a.copy() for a in o.build_list(x, y, z)]
    assert lists_equal(ctx.makelist(*g)[:3], want)
    assert lists_equal(g, (x, y, z))
    for elec in (2, 4):
        f_o, _ = o.nonbond_energy(elec, x, y, z)
        assert relerr(ctx.nonbond_energy(elec, x, y, z, *want)[0], f_o) < 1e-12
    er, fr, st, vr = o.spme(x, y, z)
    eg, fg, sg, vg = ctx.spme_energy(x, y, z)
    assert eg == pytest.approx(er, rel=1e-12) and relerr(fg, fr) < 1e-11
    f_o, _ = o.energy(x, y, z)
    assert relerr(ctx.energy(x, y, z, *want)[0], f_o) < 1e-12
    s_o = [x, y, z, wb.vx.copy(), wb.vy.copy(), wb.vz.copy()]
    s_g = [a.copy() for a in s_o]
    for stage in (1, 2):
        assert o.vv(stage, *s_o, f_o)[0] == 0
        ctx.vv_integrate(stage, *s_g, f_o.copy())
        assert max(np.abs(a - b).max() for a, b in zip(s_o, s_g)) < 1e-12
    ctx.close()
