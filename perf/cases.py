"""The work that the performance of this framework is measured on.

Six kinds of case, each through the entry points a simulation script calls:

* ``step``: five time steps of the electrostatic PIC loop (gather + push,
  particle boundaries, deposit, multigrid solve; the last of the five is a
  special step with the synchronising kick, the moments and the field
  diagnostics) from a saved moment of a run, as a restart or a scan makes
  them: the particles and phi are put back first.
* ``solve``: one field solve to mgtol for a source that alternates between
  two positions of a bunch one time step apart, from the previous phi: what
  every step of a run asks of the solver.
* ``deposit``: charge of a particle group onto the mesh.
* ``fetch``: E at particle positions into the particles' field arrays.
* ``unet_forward`` / ``unet_train``: the warm-start network's prediction,
  and one training step of it (forward, loss, backward, Adam).

The mesh is always 4 x 4 x 8 cm (warp_amd.configs.DOMAIN), so that the sizes
are resolutions of one problem.
"""
import math

import numpy as np
import torch

import warp_amd
from warp_amd import _native as N
from warp_amd import configs, registersolver, stepper, unregistersolver
from warp_amd import learned
from warp_amd.globals import echarge, eps0, f3d, top
from warp_amd.multigrid import MultiGrid3D
from warp_amd.particles import ParticleGroup, gaussian_weight

DEV = torch.device("cuda", 0)
STEPS = 5          # time steps of one "step" pass: the moment history's interval
SIGMA = (0.004, 0.004, 0.015)   # the bunch of the beam problems (m)
APERTURE = 0.0095  # it is scraped inside the conductors' bores (annulus 12 mm, rods 10 mm)
CURRENT = 1.0e-3


def listed():
    return [
        # the 64^3 free-space problem: the smallest run, launches and latency
        dict(name="step 64x64x64", kind="step", nx=64, ny=64, nz=64, npart=200_000,
             conductors="", zperiodic=False, precision="fp64", guess="previous"),
        # the ordinary run: 128 x 128 x 256 with the pipe and the annulus
        dict(name="step 128x128x256", kind="step", nx=128, ny=128, nz=256, npart=4_000_000,
             conductors="pipe_annulus", zperiodic=False, precision="fp64", guess="previous"),
        # the quadrupole channel, periodic in z, at that resolution
        dict(name="step quads 128x128x256", kind="step", nx=128, ny=128, nz=256,
             npart=4_000_000, conductors="quads", zperiodic=True, precision="fp64",
             guess="previous"),
        # the largest run: the benchmark problem
        dict(name="step 256x256x512", kind="step", nx=256, ny=256, nz=512, npart=32_000_000,
             conductors="pipe_annulus", zperiodic=False, precision="fp64", guess="previous"),
        # the benchmark problem's solve by bf16 V-cycles with FP64 defect correction
        dict(name="solve bf16 256x256x512", kind="solve", nx=256, ny=256, nz=512,
             conductors="pipe_annulus", bounds="000000", precision="bf16"),
        # a ragged mesh: no level halves evenly, mixed Neumann/Dirichlet faces
        dict(name="solve 101x75x190 mixed bounds", kind="solve", nx=101, ny=75, nz=190,
             conductors="", bounds="110001", precision="fp64"),
        # a small box with conductors by fp32 V-cycles: a quick look at a design
        dict(name="solve fp32 48x40x96", kind="solve", nx=48, ny=40, nz=96,
             conductors="pipe_annulus", bounds="000000", precision="fp32"),
        # a freshly loaded beam, in the loader's (random) order
        dict(name="deposit 4M unsorted", kind="deposit", nx=128, ny=128, nz=256,
             npart=4_000_000, ordered=False),
        # fields at the particles of another code: 1M positions, any order
        dict(name="fetch 1M", kind="fetch", nx=128, ny=128, nz=256, npart=1_000_000,
             efetch=1, corrected=False),
        # the network on the half-resolution grid of the 128x128x256 mesh, where
        # it was trained, and on that of the 256x256x512 mesh
        dict(name="unet forward 128x64x64", kind="unet_forward", d=128, h=64, w=64),
        dict(name="unet forward 256x128x128", kind="unet_forward", d=256, h=128, w=128),
        # one training step at the trained size
        dict(name="unet train 128x64x64", kind="unet_train", d=128, h=64, w=64),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "solve", "solve", "solve", "deposit", "fetch",
                       "unet_forward", "unet_train"])
    if kind in ("unet_forward", "unet_train"):
        # the network takes multiples of eight
        m = 16 if kind == "unet_forward" else 8
        return dict(kind=kind, d=8 * _logint(rng, 3, 2 * m), h=8 * _logint(rng, 3, m),
                    w=8 * _logint(rng, 3, m))
    nx, ny, nz = _logint(rng, 24, 256), _logint(rng, 24, 256), _logint(rng, 32, 512)
    cells = nx * ny * nz
    if kind == "step":
        zperiodic = rng.random() < 0.5
        if zperiodic:
            nz += nz % 2  # red and black have to meet again
        return dict(kind=kind, nx=nx, ny=ny, nz=nz,
                    npart=min(_logint(rng, 10_000, 16_000_000), 20 * cells),
                    conductors=rng.choice(["", "pipe_annulus", "quads"]), zperiodic=zperiodic,
                    precision=rng.choice(["fp64", "fp64", "fp64", "fp32", "bf16"]),
                    guess=rng.choice(["previous", "linear"]))
    if kind == "solve":
        bounds = rng.choice(["000000", "000000", "000022", "110001", "000001", "111100"])
        if "2" in bounds:
            nz += nz % 2
        return dict(kind=kind, nx=nx, ny=ny, nz=nz,
                    conductors=rng.choice(["", "pipe_annulus", "quads"]) if bounds in (
                        "000000", "000022") else "",
                    bounds=bounds, precision=rng.choice(["fp64", "fp64", "fp32", "bf16"]))
    npart = _logint(rng, 10_000, 16_000_000)
    if kind == "deposit":
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, npart=npart, ordered=rng.random() < 0.5)
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, npart=npart, efetch=rng.choice([1, 1, 3]),
                corrected=rng.random() < 0.25)


# ----------------------------------------------------------------------
# inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(20261202 + 7919 * seed)


def _randn(n, g):
    return torch.randn(n, generator=g, device=DEV, dtype=torch.float64)


def _spacing(c):
    x0, x1, y0, y1, z0, z1 = configs.DOMAIN
    return (x1 - x0) / c["nx"], (y1 - y0) / c["ny"], (z1 - z0) / c["nz"]


def _bunch(c, seed):
    """Positions and velocities of a Gaussian bunch, scraped transversely;
    in z wrapped into the period or kept within the mesh for a few steps to
    come (what lies outside is folded in)."""
    _, _, _, _, z0, z1 = configs.DOMAIN
    g, n = _gen(seed), c["npart"]
    x, y = SIGMA[0] * _randn(n, g), SIGMA[1] * _randn(n, g)
    k = APERTURE / torch.sqrt(x * x + y * y)
    k = torch.where(k < 1., 0.9 * k * k, 1.)
    x, y = k * x, k * y
    z = SIGMA[2] * _randn(n, g)
    if c.get("zperiodic"):
        z = z0 + torch.remainder(z + 0.04 - z0, z1 - z0)
    else:
        z = 0.035 + torch.where(z.abs() > 0.033, 0.25 * z, z)
    sp = configs.VSPREAD * configs.VZ
    ux, uy, uz = sp * _randn(n, g), sp * _randn(n, g), configs.VZ + sp * _randn(n, g)
    return x, y, z, ux, uy, uz


def _weight(c):
    return gaussian_weight(CURRENT, SIGMA[2], configs.VZ, echarge, c["npart"])


def _group(c, seed):
    pg = ParticleGroup(DEV)
    js = pg.addspecies(echarge, configs.MASS, _weight(c))
    pg.addparticles(js, *_bunch(c, seed))
    return pg


def _nodes(c):
    x0, x1, y0, y1, z0, z1 = configs.DOMAIN
    ax = lambda a, b, n: torch.linspace(a, b, n + 1, dtype=torch.float64, device=DEV)
    return ax(x0, x1, c["nx"]), ax(y0, y1, c["ny"]), ax(z0, z1, c["nz"])


def _sources(c, seed):
    """The charge density of the bunch at two positions one step apart, with
    the noise of a finite number of particles; the same in the last plane
    as in the first where z is periodic."""
    x, y, z = _nodes(c)
    g = _gen(seed)
    lam = CURRENT / configs.VZ
    peak = lam / (2 * math.pi * SIGMA[0] * SIGMA[1])
    r2 = y[:, None] ** 2 + x[None, :] ** 2
    tr = peak * torch.exp(-0.5 * r2 / SIGMA[0] ** 2) * (r2 < APERTURE ** 2)
    out = []
    zc = 0.03 + 0.02 * float(torch.rand(1, generator=g, device=DEV, dtype=torch.float64))
    for shift in (0., configs.VZ * configs.DT):
        gz = torch.exp(-0.5 * ((z - zc - shift) / SIGMA[2]) ** 2)
        r = gz[:, None, None] * tr[None]
        r *= 1. + 0.02 * torch.randn(r.shape, generator=g, device=DEV, dtype=torch.float64)
        if c["bounds"][4] == "2":
            r[-1] = r[0]
        out.append(r)
    return out


def _solver(c, bounds, **kw):
    x0, x1, y0, y1, z0, z1 = configs.DOMAIN
    s = MultiGrid3D(nx=c["nx"], ny=c["ny"], nz=c["nz"], xmmin=x0, xmmax=x1, ymmin=y0, ymmax=y1,
                    zmmin=z0, zmmax=z1, bounds=[int(b) for b in bounds],
                    precision=c.get("precision", "fp64"), device=DEV, mgverbose=-1, **kw)
    for obj in configs.conductors(c.get("conductors") or None, warp_amd):
        s.installconductor(obj)
    return s


class _Run:
    """A simulation of its own among several in one process: the package
    variables that belong to it, its registered solver, and the moment of
    the run that its passes start from."""

    COLUMNS = ("xp", "yp", "zp", "uxp", "uyp", "uzp", "gaminv")

    def __init__(self, solver, pg, zperiodic):
        self.solver, self.pg = solver, pg
        self.zbound = 2 if zperiodic else 0
        self.saved = None

    def save(self):
        self.saved = (self.pg.nps[0], [getattr(self.pg, k).clone() for k in self.COLUMNS],
                      self.solver.phi.clone())

    def __enter__(self):
        top.pgroup, top.dt, top.it, top.time = self.pg, configs.DT, 0, 0.
        top.lspecial, top.nspecial, top.hist, top.moments = True, 0, [], {}
        top.linechg, top.nzzarr, top.zzmin, top.zzmax = None, 0, 0., 0.
        top.particlesortinterval = 25
        top.pboundxy, top.pbound0, top.pboundnz = 0, self.zbound, self.zbound
        registersolver(self.solver)
        if self.saved:
            self.pg.nps[0], columns, phi = self.saved
            for k, v in zip(self.COLUMNS, columns):
                getattr(self.pg, k).copy_(v)
            self.solver.phi = phi
        return self

    def __exit__(self, *a):
        unregistersolver(self.solver)
        top.pgroup = None


def _smooth_phi(c, seed):
    """A potential with its guard cells: the order of a beam's, plus the
    noise of its particles."""
    x0, _, y0, _, z0, _ = configs.DOMAIN
    dx, dy, dz = _spacing(c)
    ax = lambda a, d, n: a + d * torch.arange(-1, n + 2, dtype=torch.float64, device=DEV)
    x, y, z = ax(x0, dx, c["nx"]), ax(y0, dy, c["ny"]), ax(z0, dz, c["nz"])
    p = 40. * (torch.exp(-0.5 * ((z - 0.04) / 0.02) ** 2)[:, None, None] *
               torch.exp(-0.5 * (y / 0.007) ** 2)[None, :, None] *
               torch.exp(-0.5 * (x / 0.007) ** 2)[None, None, :])
    return p + 0.01 * torch.randn(p.shape, generator=_gen(seed), device=DEV, dtype=torch.float64)


def _net_input(c, seed):
    """Second difference of a bunch's density (with noise), the density and
    the conductor fraction, as the warm start feeds them: the first two
    scaled to a largest magnitude of one, the other 13 channels empty."""
    D, H, W = c["d"], c["h"], c["w"]
    g = _gen(seed)
    ax = lambda n, L: (torch.arange(n, dtype=torch.float64, device=DEV) + 0.5) / n * L
    z, y, x = ax(D, 0.08), ax(H, 0.04) - 0.02, ax(W, 0.04) - 0.02
    x0, y0 = [0.003 * (2 * float(torch.rand(1, generator=g, device=DEV)) - 1) for _ in range(2)]
    zc = 0.025 + 0.03 * float(torch.rand(1, generator=g, device=DEV))
    tr = (torch.exp(-0.5 * ((y - y0) / SIGMA[1]) ** 2)[:, None] *
          torch.exp(-0.5 * ((x - x0) / SIGMA[0]) ** 2)[None, :])
    gz = lambda s: torch.exp(-0.5 * ((z - zc - s) / SIGMA[2]) ** 2)[:, None, None] * tr[None]
    r = gz(0.)
    h = 0.001
    d2 = gz(0.) - 2 * gz(-h) + gz(-2 * h)
    d2 = d2 + 0.2 * d2.abs().max() * torch.sqrt(r) * torch.randn(
        r.shape, generator=g, device=DEV, dtype=torch.float64)
    f = torch.zeros(D, H, W, 16, dtype=torch.float64, device=DEV)
    f[..., 0] = d2 / d2.abs().max()
    f[..., 1] = r / r.max()
    f[..., 2] = ((y[:, None] ** 2 + x[None, :] ** 2) > 0.018 ** 2).double()[None]
    # the target of training: smooth, of order one
    t = f[..., 0].float()[None, None]
    for _ in range(3):
        t = torch.nn.functional.avg_pool3d(t, 5, 1, 2)
    t = t[0, 0] / t.abs().max()
    return f.to(torch.bfloat16).reshape(-1), t.reshape(-1).contiguous()


def _step_bounds(c):
    return "000022" if c["zperiodic"] else "000000"


def prepare(c, seed):
    kind = c["kind"]
    if kind == "step":
        s = _solver(c, _step_bounds(c), guess=c["guess"])
        st = _Run(s, _group(c, seed), c["zperiodic"])
        with st:
            s.sortparticles(top.pgroup)
            stepper.generate()
            # the run is well under way: the potential behind the conductors
            # has settled (a first solve stops at mgmaxiters)
            for _ in range(8):
                if s.mgiters <= 10:
                    break
                s.solve()
            st.save()
        return dict(kind=kind, run=st)
    if kind == "solve":
        s = _solver(c, c["bounds"])
        a, b = _sources(c, seed)
        s.finalizesourcep()  # the sources come with their boundary values
        s.rho = b
        for _ in range(8):
            s.solve()
            if s.mgiters <= 10:
                break
        return dict(kind=kind, solver=s, rhos=(a, b), k=0)
    if kind == "deposit":
        s = _solver(c, "000000")
        pg = _group(c, seed)
        if c["ordered"]:
            s.sortparticles(pg)
        return dict(kind=kind, solver=s, pg=pg)
    if kind == "fetch":
        s = _solver(dict(c, conductors="pipe_annulus" if c["corrected"] else ""), "000000")
        s.phi = _smooth_phi(c, seed)
        x, y, z = _bunch(c, seed)[:3]
        return dict(kind=kind, solver=s, at=(x, y, z), e=[torch.zeros_like(x) for _ in range(3)],
                    efetch=c["efetch"], corrected=c["corrected"])
    x, t = _net_input(c, seed)
    net, _, _ = learned.load_weights(learned.default_weights(), DEV)
    st = dict(kind=kind, net=net, x=x.view(torch.int16), target=t, dims=(c["d"], c["h"], c["w"]))
    if kind == "unet_train":
        st["g"] = torch.empty(t.numel() * 16, dtype=torch.int16, device=DEV)
        st["loss"] = torch.zeros(1, dtype=torch.float32, device=DEV)
    return st


def run(st):
    kind = st["kind"]
    if kind == "step":
        r = st["run"]
        with r:
            stepper.step(STEPS)
            pg = top.pgroup
            live = pg.species_slice(0)
            return dict(phi=r.solver.getphi(), rho=r.solver.getrho(), linechg=top.linechg,
                        ese=top.ese, **{k: getattr(pg, k)[live] for k in
                                        ("xp", "yp", "zp", "uxp", "uyp", "uzp")})
    if kind == "solve":
        s = st["solver"]
        s.rho = st["rhos"][st["k"]]
        st["k"] ^= 1
        s.solve()
        return s.getphi()
    if kind == "deposit":
        st["solver"].loadrho(pgroups=[st["pg"]])
        return st["solver"].getrho()
    if kind == "fetch":
        top.efetch, f3d.lcorrectede = st["efetch"], st["corrected"]
        for e in st["e"]:
            e.zero_()
        st["solver"].fetchfieldfrompositions(*st["at"], *st["e"])
        top.efetch, f3d.lcorrectede = 1, False
        return st["e"]
    net = st["net"]
    if kind == "unet_forward":
        return net.forward(st["x"], st["dims"])
    # one step of warp_amd.unet_train.train
    net.zero_grad()
    out = net.forward(st["x"], st["dims"], keep=True)
    st["loss"].zero_()
    N.call("wm_unet_mse", out.data_ptr(), st["target"].data_ptr(), st["target"].numel(),
           st["g"].data_ptr(), st["loss"].data_ptr(), N.stream_of(DEV))
    net.backward(st["g"])
    net.adam_step(3e-4)
    return dict(out=out, loss=st["loss"], gw=[l.gw for l in net.layers()],
                gb=[l.gb for l in net.layers()], w=[l.w for l in net.layers()])


# ----------------------------------------------------------------------
# what a pass cannot do without

VCYCLES = 7  # of a solve that starts from the previous step's phi


def _solve_work(nodes):
    """A V-cycle goes down and up the levels (8/7 of the finest), and each way
    reads phi and rho and writes phi; about 40 operations per node and
    half sweep pair, residual and transfer."""
    return 8 / 7 * nodes * VCYCLES * 2 * 3 * 8, 8 / 7 * nodes * VCYCLES * 100


def _unet_flops(c):
    nv = c["d"] * c["h"] * c["w"]
    ch = (16, 32, 48, 64)
    fwd = [(nv // 8 ** l, a, b) for l in range(4)
           for a, b in (((16, 16) if l == 0 else (ch[l - 1], ch[l])), (ch[l], ch[l]))]
    fwd += [(nv // 8 ** l, a, ch[l]) for l in range(3) for a in (ch[l] + ch[l + 1], ch[l])]
    fwd.append((nv, 16, 16))
    return [2 * 27 * n * a * b for n, a, b in fwd]


def work(c):
    kind = c["kind"]
    if kind in ("unet_forward", "unet_train"):
        nv, f = c["d"] * c["h"] * c["w"], _unet_flops(c)
        if kind == "unet_forward":
            return {"bytes": nv * 16 * (2 + 4), "flops": sum(f)}
        nw = sum(27 * a for a in (16 * 16, 16 * 16, 32 * 16, 32 * 32, 48 * 32, 48 * 48, 64 * 48,
                                  64 * 64, 112 * 48, 48 * 48, 80 * 32, 32 * 32, 48 * 16, 16 * 16,
                                  16 * 16))
        return {"bytes": nv * (16 * 2 + 4) + nw * 4 * 7, "flops": 3 * sum(f) - f[0]}
    nodes = (c["nx"] + 1) * (c["ny"] + 1) * (c["nz"] + 1)
    if kind == "solve":
        b, f = _solve_work(nodes)
        return {"bytes": b, "flops": f}
    n = c["npart"]
    if kind == "deposit":
        return {"bytes": 24 * n + 8 * nodes, "flops": 40 * n}
    if kind == "fetch":
        return {"bytes": 48 * n + 8 * min(nodes, 32 * n), "flops": 130 * n}
    # each step: 7 columns in, 6 out, 3 for the deposit; the synchronising kick once
    b, f = _solve_work(nodes)
    return {"bytes": STEPS * (b + n * (56 + 48 + 24) + 16 * nodes) + n * (48 + 24 + 56),
            "flops": STEPS * (f + 200 * n)}


def tolerance(c):
    kind = c["kind"]
    if kind in ("deposit", "fetch"):
        # FP64 sums in any order: 5e-16 off the 64-bit value as measured
        return {"rel": 1e-13, "max": 1e-11}
    if kind in ("step", "solve"):
        # the solve stops when phi changes by less than mgtol = 1e-6 V, of
        # potentials of tens of volts; FP64 throughout or FP64-corrected
        return {"rel": 1e-7, "max": 4e-6}
    if kind == "unet_forward":
        # bf16 activations through 15 layers: 6e-4 off the 64-bit network
        return {"rel": 2.5e-3, "max": 0.1}
    # the deepest layers' gradients are 8e-3 off in 2-norm, 2e-2 at most
    return {"rel": 1e-2, "max": 0.1}


# ----------------------------------------------------------------------
# the same results in 64 bits, from plain torch

def _axis(n, d, lo, hi):
    """Eigenvalues and the transform pair of the negative second difference
    over the unknown nodes of one axis, and where these nodes start."""
    if lo == 2:
        a = 2 * np.eye(n) - np.eye(n, k=1) - np.eye(n, k=-1)
        a[0, -1] -= 1
        a[-1, 0] -= 1
        w, first, m = np.ones(n), 0, n
    else:
        first, last = (1 if lo == 0 else 0), (n - 1 if hi == 0 else n)
        m = last - first + 1
        a = 2 * np.eye(m) - np.eye(m, k=1) - np.eye(m, k=-1)
        w = np.ones(m)
        if lo == 1:
            a[0, 1] = -2
            w[0] = 0.5
        if hi == 1:
            a[-1, -2] = -2
            w[-1] = 0.5
    r = np.sqrt(w)
    lam, q = np.linalg.eigh(r[:, None] * a / r[None, :] / d ** 2)
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(DEV)
    return t(lam), t(q.T * r[None, :]), t(q / r[:, None]), slice(first, first + m)


def _poisson(c, bounds, rho):
    """The discrete solution of -lap phi = rho/eps0 on the nodes."""
    b = [int(v) for v in bounds]
    dx, dy, dz = _spacing(c)
    X, Y, Z = _axis(c["nx"], dx, *b[:2]), _axis(c["ny"], dy, *b[2:4]), _axis(c["nz"], dz, *b[4:])
    f = rho[Z[3], Y[3], X[3]] / eps0

    def along(m, f, axis):
        return torch.movedim(torch.tensordot(m, f, dims=([1], [axis])), 0, axis)

    for k, A in enumerate((Z, Y, X)):
        f = along(A[1], f, k)
    f = f / (Z[0][:, None, None] + Y[0][None, :, None] + X[0][None, None, :])
    for k, A in enumerate((Z, Y, X)):
        f = along(A[2], f, k)
    phi = torch.zeros_like(rho)
    phi[Z[3], Y[3], X[3]] = f
    for axis, k in ((2, 0), (1, 2), (0, 4)):
        if b[k] == 2:
            phi.transpose(0, axis)[-1] = phi.transpose(0, axis)[0]
    return phi


def _cell(c, x, y, z):
    x0, _, y0, _, z0, _ = configs.DOMAIN
    dx, dy, dz = _spacing(c)
    out = []
    for p, a, d in ((x, x0, dx), (y, y0, dy), (z, z0, dz)):
        s = (p - a) * (1. / d)
        i = s.long()
        out.append((i, s - i))
    return out


def _corners(cell):
    (i, u), (j, v), (k, w) = cell
    for a in (0, 1):
        for b in (0, 1):
            for e in (0, 1):
                wt = ((u if a else 1 - u) * (v if b else 1 - v)) * (w if e else 1 - w)
                yield i + a, j + b, k + e, wt


def _rho(c, x, y, z, periodic):
    dx, dy, dz = _spacing(c)
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    rho = torch.zeros((nz + 1) * (ny + 1) * (nx + 1), dtype=torch.float64, device=DEV)
    q = echarge * _weight(c) / (dx * dy * dz)
    for i, j, k, wt in _corners(_cell(c, x, y, z)):
        rho.index_add_(0, i + (nx + 1) * (j + (ny + 1) * k), wt * q)
    rho = rho.reshape(nz + 1, ny + 1, nx + 1)
    if periodic:
        rho[0] += rho[-1]
        rho[-1] = rho[0]
    return rho


def _field(c, p, x, y, z):
    """-grad p by centred differences (p with one guard cell), interpolated."""
    d = _spacing(c)
    C = slice(1, -1)
    nx, ny = c["nx"], c["ny"]
    cell = _cell(c, x, y, z)
    out = []
    for axis, h in ((2, d[0]), (1, d[1]), (0, d[2])):
        lo, hi = [C, C, C], [C, C, C]
        lo[axis], hi[axis] = slice(0, -2), slice(2, None)
        e = ((p[tuple(lo)] - p[tuple(hi)]) / (2 * h)).reshape(-1)
        out.append(sum(wt * e[i + (nx + 1) * (j + (ny + 1) * k)]
                       for i, j, k, wt in _corners(cell)))
    return out


def _guarded(phi, zperiodic):
    """phi = 0 on the faces (extrapolated beyond), or periodic in z."""
    p = torch.nn.functional.pad(phi, (1, 1, 1, 1, 1, 1))
    p[:, :, 0], p[:, :, -1] = -p[:, :, 2], -p[:, :, -3]
    p[:, 0], p[:, -1] = -p[:, 2], -p[:, -3]
    p[0], p[-1] = (p[-3], p[2]) if zperiodic else (-p[2], -p[-3])
    return p


def _exact_step(c, seed):
    if c["conductors"]:
        return None
    _, _, _, _, z0, z1 = configs.DOMAIN
    x, y, z, ux, uy, uz = _bunch(c, seed)
    (i, _), (j, _), (k, _) = _cell(c, x, y, z)
    order = torch.argsort(i + (c["nx"] + 1) * (j + (c["ny"] + 1) * k), stable=True)
    x, y, z, ux, uy, uz = [t[order] for t in (x, y, z, ux, uy, uz)]
    kick = echarge / configs.MASS * 0.5 * configs.DT
    fields = lambda phi: _field(c, _guarded(phi, c["zperiodic"]), x, y, z)
    rho = _rho(c, x, y, z, c["zperiodic"])
    phi = _poisson(c, _step_bounds(c), rho)
    for n in range(STEPS):
        ex, ey, ez = fields(phi)
        h = kick if n == 0 else 2 * kick
        ux, uy, uz = ux + h * ex, uy + h * ey, uz + h * ez
        x, y, z = x + ux * configs.DT, y + uy * configs.DT, z + uz * configs.DT
        if c["zperiodic"]:
            z = z0 + torch.remainder(z - z0, z1 - z0)
        rho = _rho(c, x, y, z, c["zperiodic"])
        phi = _poisson(c, _step_bounds(c), rho)
    ex, ey, ez = fields(phi)
    return dict(phi=phi, rho=rho, linechg=None, ese=None, xp=x, yp=y, zp=z, uxp=ux + kick * ex,
                uyp=uy + kick * ey, uzp=uz + kick * ez)


class _Conv3(torch.autograd.Function):
    """3x3x3 convolution with zero padding over (D, H, W, C), in 64 bits."""

    @staticmethod
    def forward(ctx, x, w, b):
        ctx.save_for_backward(x, w)
        p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        y = b.expand(*x.shape[:3], len(b)).clone()
        for t, v in enumerate(_shifts(p, x.shape)):
            y += v @ w[:, :, t].t()
        return y

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        gf = g.reshape(-1, g.shape[-1])
        gw = torch.stack([gf.t() @ v.reshape(-1, x.shape[-1]) for v in _shifts(p, x.shape)], 2)
        q = torch.nn.functional.pad(g, (0, 0, 1, 1, 1, 1, 1, 1))
        gx = torch.zeros_like(x)
        for t, v in enumerate(_shifts(q, x.shape)):
            gx += v @ w[:, :, 26 - t]
        return gx, gw, gf.sum(0)


def _shifts(p, shape):
    for t in range(27):
        a, b, e = t // 9, t // 3 % 3, t % 3
        yield p[a:a + shape[0], b:b + shape[1], e:e + shape[2]]


def _exact_unet(c, seed):
    x, tgt = _net_input(c, seed)
    D, H, W = c["d"], c["h"], c["w"]
    with np.load(learned.default_weights(), allow_pickle=False) as f:
        master = [torch.from_numpy(f["w%02d" % i]).to(DEV) for i in range(15)]
        bias = [torch.from_numpy(f["b%02d" % i]).to(DEV).double() for i in range(15)]
        slope = float(f["slope"])
    train = c["kind"] == "unet_train"
    # the network multiplies by its weights' bf16 values
    ws = [m.to(torch.bfloat16).double().requires_grad_(train) for m in master]
    bs = [b.requires_grad_(train) for b in bias]
    k = [0]

    def conv(h, act=True):
        i = k[0]
        k[0] += 1
        y = _Conv3.apply(h, ws[i], bs[i])
        return torch.where(y > 0, y, slope * y) if act else y

    def pool(h):
        return h.reshape(h.shape[0] // 2, 2, h.shape[1] // 2, 2, h.shape[2] // 2, 2, -1).mean(
            (1, 3, 5))

    def up(h):
        for a in (0, 1, 2):
            h = h.repeat_interleave(2, a)
        return h

    with torch.set_grad_enabled(train):
        h = x.double().reshape(D, H, W, 16)
        skips = []
        for l in range(4):
            h = conv(conv(pool(h) if l else h))
            skips.append(h)
        for l in range(3):
            h = conv(conv(torch.cat([up(h), skips[2 - l]], 3)))
        out = conv(h, act=False)
        if not train:
            return out.reshape(-1)
        loss = ((out[..., 0].reshape(-1) - tgt.double()) ** 2).mean()
        loss.backward()
    # Adam's first step from zero moments: the rate times the gradient's sign
    new = [m.double() - 3e-4 * w.grad / (w.grad.abs() + 1e-8) for m, w in zip(master, ws)]
    return dict(out=out.detach().reshape(-1), loss=loss.detach().reshape(1),
                gw=[w.grad for w in ws], gb=[b.grad for b in bs], w=new)


def exact(c, seed):
    kind = c["kind"]
    if kind == "step":
        return _exact_step(c, seed)
    if kind == "solve":
        return None if c["conductors"] else _poisson(c, c["bounds"], _sources(c, seed)[0])
    if kind == "deposit":
        x, y, z = _bunch(c, seed)[:3]
        return _rho(c, x, y, z, False)
    if kind == "fetch":
        if c["corrected"]:
            return None
        return _field(c, _smooth_phi(c, seed), *_bunch(c, seed)[:3])
    return _exact_unet(c, seed)
