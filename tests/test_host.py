"""CPU checks of the host side: the C ABI library loads and exports every
entry point of include/warpmi.h, the product's conductor generation (host
C++ in libwarpmi) equals the oracle's restatement bit for bit, and the
registered-solver plumbing behaves as fieldsolver.py's."""
import os
import re

import numpy as np
import pytest

from oracle import oracle as O
from tests import helpers as H

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header_symbols():
    text = open(os.path.join(ROOT, "include", "warpmi.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(wm_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from warp_amd import _native as N
    L = N.lib()
    syms = _header_symbols()
    assert len(syms) > 20
    missing = [s for s in syms if not hasattr(L, s)]
    assert not missing, missing
    # the ctypes table binds exactly the declared entry points
    assert sorted(N.SIGNATURES) == syms


def test_last_error_is_a_string():
    from warp_amd import _native as N
    assert isinstance(N.lib().wm_last_error(), bytes)


def _product_lists(geoms, n, dom):
    from warp_amd.generateconductors import ConductorData, Grid, installconductor
    nx, ny, nz = n
    g = Grid(nx, ny, nz, *dom)
    cd = ConductorData(nx, ny, nz, g.dx, g.dy, g.dz)
    for c in geoms:
        installconductor(c, g, cd)
    return cd.lists()


def _oracle_lists(geoms, n, dom, crop=None):
    co = O.install_conductors(geoms, *n, *dom, crop=crop)
    d = ((dom[1] - dom[0]) / n[0], (dom[3] - dom[2]) / n[1], (dom[5] - dom[4]) / n[2])
    O.checkconductors(co, *n, *d)
    return co.lists()


@pytest.mark.parametrize("kind,n", [("pipe_annulus", (32, 32, 64)), ("pipe_annulus", (64, 64, 128)),
                                    ("quads", (32, 32, 64)), ("quads", (64, 64, 128))])
def test_product_conductors_equal_oracle(kind, n):
    """conductordelfromintercepts + checkconductors in libwarpmi against the
    oracle: identical interior points, subgrid points, distances and
    voltages on every level."""
    import warp_amd
    from warp_amd import configs
    a = _product_lists(configs.conductors(kind, warp_amd), n, configs.DOMAIN)
    b = _oracle_lists(configs.conductors(kind, O), n, configs.DOMAIN)
    assert a["levels"] == b["levels"]
    np.testing.assert_array_equal(a["int_istart"], b["int_istart"])
    np.testing.assert_array_equal(a["int_indx"], b["int_indx"])
    np.testing.assert_array_equal(a["int_volt"], b["int_volt"])
    for p in (0, 1):
        for k in ("indx", "dels", "volt", "istart"):
            np.testing.assert_array_equal(a["sub%d_%s" % (p, k)], b["sub%d_%s" % (p, k)])
    assert len(a["sub0_dels"]) > 0 and len(a["int_volt"]) > 0


def test_neumann_flag_leaves_intercept_data_unchanged():
    """Assembly(neumann=1): the reference's default intercept generation
    passes the flag to GridIntercepts, which keeps nothing of it
    (generateconductors.py:333-340, 1815-1821), so the installed data equal
    those of neumann=0, and unions inherit the flag of their left part."""
    from warp_amd.generateconductors import ZAnnulus, ZCylinderOut
    from warp_amd import configs
    n = (32, 32, 64)

    def geoms(flag):
        return [ZCylinderOut(0.02, 0.1, voltage=0., zcent=0.05, neumann=flag)
                + ZAnnulus(0.008, 0.012, 0.01, voltage=-1., zcent=0.04, neumann=flag)]

    g1 = geoms(1)
    assert g1[0].neumann == 1 and g1[0].right.neumann == 1
    a = _product_lists(geoms(0), n, configs.DOMAIN)
    b = _product_lists(g1, n, configs.DOMAIN)
    assert a["levels"] == b["levels"]
    for k in a:
        if k != "levels":
            np.testing.assert_array_equal(a[k], b[k])
    assert len(a["sub0_dels"]) > 0


CROPS = [(None, None, None, None, 0.031, 0.05), (-0.005, 0.012, None, 0.0, None, None),
         (None, None, None, None, 0.0326, 0.0329)]


@pytest.mark.parametrize("crop", CROPS)
def test_cropped_conductors_equal_oracle(crop):
    """installconductor(..., xmin..zmax): the data generated only within the
    given region (part of the annulus and of the pipe), identical to the
    oracle's; finest-level points inside the region."""
    import warp_amd
    from warp_amd import configs
    from warp_amd.generateconductors import ConductorData, Grid, installconductor
    n = (64, 64, 128)
    dom = configs.DOMAIN
    nx, ny, nz = n
    g = Grid(nx, ny, nz, *dom, xmin=crop[0], xmax=crop[1], ymin=crop[2], ymax=crop[3],
             zmin=crop[4], zmax=crop[5])
    cd = ConductorData(nx, ny, nz, g.dx, g.dy, g.dz)
    for c in configs.conductors("pipe_annulus", warp_amd):
        installconductor(c, g, cd)
    a = cd.lists()
    b = _oracle_lists(configs.conductors("pipe_annulus", O), n, dom, crop=crop)
    full = _oracle_lists(configs.conductors("pipe_annulus", O), n, dom)
    np.testing.assert_array_equal(a["int_istart"], b["int_istart"])
    np.testing.assert_array_equal(a["int_indx"], b["int_indx"])
    np.testing.assert_array_equal(a["int_volt"], b["int_volt"])
    for p in (0, 1):
        for k in ("indx", "dels", "volt", "istart"):
            np.testing.assert_array_equal(a["sub%d_%s" % (p, k)], b["sub%d_%s" % (p, k)])
    assert 0 < len(a["int_volt"]) < len(full["int_volt"])
    # on the finest level every point lies in the region, widened by the
    # cells getmeshnew adds around the conductor's extent
    e = np.asarray(a["int_istart"])[1] if len(a["int_istart"]) > 1 else len(a["int_volt"])
    ii = np.asarray(a["int_indx"]).reshape(-1, 3)[:e]
    lo = np.array(dom[0::2]); d = (np.array(dom[1::2]) - lo) / np.array(n)
    pos = lo + ii * d
    for ax in range(3):
        if crop[2 * ax] is not None:
            assert (pos[:, ax] >= crop[2 * ax] - 2 * d[ax] - 1e-12).all()
        if crop[2 * ax + 1] is not None:
            assert (pos[:, ax] <= crop[2 * ax + 1] + 2 * d[ax] + 1e-12).all()


def test_solver_records_the_crop():
    """MultiGrid3D.installconductor keeps the region arguments until the
    data is generated (multigrid.py:743-751)."""
    import warp_amd
    from warp_amd import configs
    from warp_amd.multigrid import MultiGrid3D
    s = MultiGrid3D.__new__(MultiGrid3D)
    s.conductordatalist = []
    c = configs.conductors("pipe_annulus", warp_amd)[1]
    MultiGrid3D.installconductor(s, c, zmin=0.031, zmax=0.05, dfill=1.5)
    assert s.conductordatalist == [(c, None, None, None, None, 0.031, 0.05, 1.5)]


def test_product_mglevels_equal_oracle():
    from warp_amd.generateconductors import getmglevels
    for n, d in (((64, 64, 64), (0.04 / 64, 0.04 / 64, 0.08 / 64)),
                 ((256, 256, 512), (0.04 / 256,) * 2 + (0.08 / 512,)),
                 ((24, 22, 18), (2 / 24, 2 / 22, 2 / 18)), ((13, 40, 7), (0.1, 0.02, 0.3))):
        assert getmglevels(*n, *d) == O.getmglevels(*n, *d)


def test_registry():
    """registersolver sets top.fstype = 12 and the *registered calls reach
    every solver in order (fieldsolver.py:173-229)."""
    import warp_amd as W
    calls = []

    class Dummy(W.FieldSolver):
        def __init__(self, tag, **kw):
            W.FieldSolver.__init__(self, kwdict=kw)
            self.tag = tag

        def loadrho(self, *a, **k): calls.append(("loadrho", self.tag))
        def solve(self, iwhich=0): calls.append(("solve", self.tag))
        def fetche(self, *a, **k): calls.append(("fetche", self.tag))
        def fetchphi(self, *a, **k): calls.append(("fetchphi", self.tag))

    a = Dummy("a", nx=8, ny=8, nz=8)
    b = Dummy("b", nx=8, ny=8, nz=8, bounds=[0, 0, 2, 0, 1, 1])
    assert b.bounds == [0, 0, 2, 2, 1, 1]   # periodic applies to both faces
    W.registersolver(a)
    W.registersolver(b)
    try:
        assert W.top.fstype == 12
        assert W.getregisteredsolvers() == [a, b]
        W.loadrhoregistered()
        W.fieldsolregistered()
        W.fetcheregistered()
        assert calls == [("loadrho", "a"), ("loadrho", "b"), ("solve", "a"), ("solve", "b"),
                         ("fetche", "a"), ("fetche", "b")]
        W.top.fstype = 0
        with pytest.raises(RuntimeError):
            W.getregisteredsolvers()
        W.top.fstype = 12
    finally:
        W.unregistersolver(a)
        W.unregistersolver(b)
    assert W.top.fstype == -1


def test_diagnostic_hooks_and_step_order():
    """The diagnostics step3d calls through the registered solvers
    (fieldsolver.py:234-257): rhodia on every step, gtlchg, srhoax, getese,
    sphiax, sezax in that order on special steps (w3d.F:987-1002); a solver
    that defines none of them inherits the reference's no-ops
    (fieldsolver.py:1053-1064)."""
    import warp_amd as W
    from warp_amd import fieldsolver as FS
    from warp_amd import stepper
    calls = []

    class Diag(W.FieldSolver):
        def __init__(self, **kw):
            W.FieldSolver.__init__(self, kwdict=kw)

        def gtlchg(self): calls.append("gtlchg")
        def getese(self): calls.append("getese")
        def rhodia(self): calls.append("rhodia")
        def sezax(self): calls.append("sezax")

    class Plain(W.FieldSolver):
        def __init__(self, **kw):
            W.FieldSolver.__init__(self, kwdict=kw)

    a, b = Diag(nx=8, ny=8, nz=8), Plain(nx=8, ny=8, nz=8)
    for name in ("rhodia", "gtlchg", "srhoax", "getese", "sphiax", "sezax"):
        assert getattr(b, name)() is None
        assert callable(getattr(FS, name + "registered"))
    W.registersolver(a)
    W.registersolver(b)
    try:
        stepper.field_diagnostics(special=False)
        assert calls == ["rhodia"]
        del calls[:]
        stepper.field_diagnostics(special=True)
        assert calls == ["rhodia", "gtlchg", "getese", "sezax"]
    finally:
        W.unregistersolver(a)
        W.unregistersolver(b)


def test_bad_keyword_rejected():
    import warp_amd as W
    with pytest.raises(AssertionError):
        W.MultiGrid3D(nx=8, ny=8, nz=8, mgtoll=1e-6)


def test_unknown_initial_guess_rejected():
    import warp_amd as W
    with pytest.raises(ValueError, match="guess"):
        W.MultiGrid3D(nx=8, ny=8, nz=8, guess="quadratic")


def test_solver_fails_loudly_without_gpu():
    """No CPU fallback: without a HIP device the solver refuses to build."""
    import torch
    import warp_amd as W
    if torch.cuda.is_available():
        pytest.skip("a HIP device is present")
    with pytest.raises(RuntimeError, match="HIP device"):
        W.MultiGrid3D(nx=8, ny=8, nz=8)


def test_beam_weights_follow_current_rule():
    """sw = I * zlen / (v q N) with the peak line charge (w3d.F:7142-7172):
    Gaussian zlen = sqrt(2 pi) sigma_z; KV uniform zlen = zmax - zmin."""
    from warp_amd import configs
    from warp_amd.globals import echarge
    n = 20000
    pg = configs.load_beam(configs.CONFIGS["c0"], device="cpu", npart=n)
    ntot = pg.nps[0]
    assert 0.99 * n < ntot <= n
    want = 1e-3 * np.sqrt(2 * np.pi) * 0.015 / (configs.VZ * echarge * n)
    assert pg.sw[0] == pytest.approx(want, rel=1e-12)
    x = pg.xp[:ntot].numpy()
    assert abs(x.std() - 0.004) < 0.0002
    lo = configs.DOMAIN
    z = pg.zp[:ntot].numpy()
    assert x.min() >= lo[0] and x.max() < lo[1] and z.min() >= lo[4] and z.max() < lo[5]
    # seeded: the same load twice
    pg2 = configs.load_beam(configs.CONFIGS["c0"], device="cpu", npart=n)
    assert np.array_equal(pg2.xp.numpy(), pg.xp.numpy())
    kv = configs.load_beam(configs.CONFIGS["c2"], device="cpu", npart=n)
    m = kv.nps[0]
    r2 = (kv.xp[:m].numpy() / 0.006) ** 2 + (kv.yp[:m].numpy() / 0.006) ** 2
    assert r2.max() <= 1.0
    assert kv.sw[0] == pytest.approx(1e-3 * 0.06 / (configs.VZ * echarge * n), rel=1e-12)


def test_find_mgparam_search_logic():
    """find_mgparam's search on a stand-in solver whose V-cycle count is a
    convex function of mgparam (minimum at 1.6): the search stops at a
    mgparam with the minimal count, and restores mgtol."""
    import torch
    from warp_amd.find_mgparam import find_mgparam

    class Stub:
        def __init__(self):
            self.mgparam, self.downpasses, self.uppasses = 1.2, 1, 1
            self.mgiters, self.mgmaxiters, self.mgtol, self.mgerror = 0, 100, 1e-6, 0.
            self.nx = self.ny = self.nz = 4
            self.bounds = [0] * 6
            self.phi = torch.zeros((7, 7, 7), dtype=torch.float64)
            self.calls = 0

        def solve(self, iwhich=0):
            self.calls += 1
            self.mgiters = 5 + int(round(400 * (self.mgparam - 1.6) ** 2)) + 2 * (self.downpasses - 1)
            time.sleep(1e-3 * self.mgiters * (self.downpasses + self.uppasses))

    import time
    s = Stub()
    find_mgparam(s)
    assert abs(s.mgparam - 1.6) < 0.05
    assert 5 + int(round(400 * (s.mgparam - 1.6) ** 2)) == 5
    assert s.downpasses == 1 and s.uppasses == 1 and s.mgtol == 1e-6


def test_thisstep_control_arrays():
    """dtop.F:764-789: (start, end, increment) then single steps."""
    from warp_amd.stepper import thisstep
    c = [10, 30, 5] + [0] * 47
    assert [i for i in range(1, 40) if thisstep(i, c)] == [10, 15, 20, 25, 30]
    assert thisstep(0, c)  # the zero entries after the triple match step 0
    c = [0, 0, 0, 7, 12] + [0] * 45
    assert [i for i in range(1, 20) if thisstep(i, c)] == [7, 12]
    assert not any(thisstep(i, [0] * 50) for i in range(1, 100))


def test_special_step_cadence():
    """step3d's lspecial (w3d.F:854-880) with the defaults nhist = 5,
    itdump = 500: every 5th step, every 500th, the last step of a call,
    and all steps when allspecl."""
    from warp_amd.globals import top
    from warp_amd.stepper import special_step
    saved = (top.it, top.time, top.allspecl)
    try:
        top.time = 0.
        got = []
        for it in range(1, 13):
            top.it = it
            got.append(special_step(llast=(it == 12))[0])
        assert [i for i, sp in zip(range(1, 13), got) if sp] == [5, 10, 12]
        top.it = 500
        assert special_step(False) == (True, True)
        top.it, top.allspecl = 3, True
        assert special_step(False)[0]
    finally:
        top.it, top.time, top.allspecl = saved


@pytest.mark.parametrize("sort", [False, True])
def test_deposits_in_flight_share_no_workspace(sort, monkeypatch):
    """A deposit that begins while another into the same solver is still
    running (another stream or thread) has a workspace of its own, of the
    same, a smaller or a larger group."""
    import torch
    from warp_amd import _native as N
    from warp_amd.multigrid import MultiGrid3D
    s = MultiGrid3D.__new__(MultiGrid3D)
    s.__dict__.update(device=torch.device("cpu"), sorted_deposit=sort, nx=64, ny=64, nz=64,
                      dx=1., dy=1., dz=1., xmmin=0., ymmin=0., zmmin=0., _rho=torch.zeros(1))
    sizes = [300000, 300000, 262144, 400000]
    live = []

    def call(name, *args):
        base, need = (args[-2], N.lib().wm_setrho3d_sorted_worksize(args[1], 64, 64, 64)) \
            if sort else args[-3:-1]
        assert need > 0
        assert all(base + need <= b or b + n <= base for b, n in live)
        live.append((base, need))
        if len(live) < len(sizes):  # the next one begins before this one ends
            deposit(sizes[len(live)])
        live.pop()

    def deposit(n):
        x = torch.zeros(n, dtype=torch.float64)
        s.setsourcepatposition(x, x, x, 0., 1., 1.)

    monkeypatch.setattr(N, "call", call)
    monkeypatch.setattr(N, "stream_of", lambda device: None)
    deposit(sizes[0])


def test_few_unordered_particles_are_binned():
    """Which deposits take a workspace: unordered ones from the library's
    limit on (0.1M on 64^3, far below 262144), which grows with the mesh's
    tiles; ordered ones of fewer than 262144 only where they are sparse; and
    what a group says of its order."""
    import torch
    from warp_amd import _native as N
    from warp_amd.multigrid import MultiGrid3D
    from warp_amd.particles import ParticleGroup
    f = N.lib().wm_setrho3d_worksize
    for mesh, tiles in (((64, 64, 64), 64), ((128, 128, 256), 1024), ((256, 256, 512), 8192),
                        ((17, 1, 1), 2)):
        assert f(32768 + 16 * tiles, *mesh) > 0 and f(32767 + 16 * tiles, *mesh) == 0
    s = MultiGrid3D.__new__(MultiGrid3D)
    s.nx = s.ny = s.nz = 64
    assert s._binned(32767, True) and not s._binned(32768, True) and s._binned(32768, False)
    assert not s._binned(262143, True) and s._binned(262144, True)
    pg = ParticleGroup("cpu")
    pg.addspecies(1., 1., 1.)
    pg.ordered = True
    v = torch.zeros(3, dtype=torch.float64)
    pg.addparticles(0, *[v] * 6)
    assert not pg.ordered


def test_deposit_workspace_of_the_wrong_kind_is_refused():
    """Too small, or not aligned: an error from the host, before any launch."""
    import ctypes as C
    from warp_amd import _native as N
    mesh = (64, 64, 64)
    need = N.lib().wm_setrho3d_worksize(40000, *mesh)
    assert need > 0
    # (addresses that nothing reads)
    for work, size, what in ((4096, need - 1, "too small"), (4097, need, "not aligned"),
                             (4100, need, "not aligned")):
        rc = N.lib().wm_setrho3d_work(4096, 40000, 4096, 4096, 4096, 0., 1., 1., *mesh, 1., 1., 1.,
                                      0., 0., 0., None, C.c_void_p(work), size, None)
        assert rc != 0 and what in N.lib().wm_last_error().decode()
