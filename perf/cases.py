"""Performance cases of the package: the calls a kernel computation makes, timed through
the public entry points (MCKernel, run_job, the autograd stage).

The set-ups are the package's own synthetic workloads (mc_kernel_amd.synth): databases,
receivers, filters and kernels are fixed per set-up, as a program opens them once per
process; a case's seed draws the points, elements or traces of one call.  The library
holds one set-up per process, so the handle of the current set-up is kept here and
replaced when a case needs another one.

`exact` restates the path in FP64 torch from its definitions (location, strain at the GLL
nodes, FFTs, base kernels, window integrals, Monte Carlo sums), as a reference for the
outputs; it shares no code with the library.
"""
import ctypes as C
import math

import numpy as np
import torch

import mc_kernel_amd as mk
from mc_kernel_amd import autograd as ad
from mc_kernel_amd import job, results, synth

# ---------------------------------------------------------------------------------------
# set-ups
# ---------------------------------------------------------------------------------------

#: a general moment tensor (N m; rr, tt, pp, rt, rp, tp)
GENERAL = [0.3e20, 1.0e20, -1.3e20, 0.5e20, -0.4e20, 0.7e20]


def _setups():
    two = synth._kernels(2, 2, ["CC", "AM"], ["vp", "vs"])
    three = synth._kernels(3, 4, ["CC"], ["vp", "vs"])
    return {
        # trace-only kernels, one receiver, nt 1024
        "c0": ("c0", {}),
        # 160 kernels of 10 receivers, explosion and Z receivers, nt 2048 (61 GB resident)
        "c1": ("c1", {}),
        # 1,200 kernels of 50 receivers on the same databases
        "c2": ("c2", {}),
        # 1,600 kernels of 200 stations, a real event's moment tensor, nt 4096
        "c4": ("c4", dict(nelem_target=4000)),
        # general moment tensor and R receivers (six components each way) at a trace length
        # that is no power of two
        "mt": ("c1", dict(nelem_target=2000, nt=1000, receivers_deg=[25.0, 40.0, 55.0], kernels=three,
                          mij=GENERAL, component="R")),
        # the kernel set of c1 on a small mesh, for the differentiable stage
        "ad": ("c1", dict(nelem_target=450)),
        # two receivers, eight kernels, nt 256
        "tiny": ("tiny", dict(kernels=two)),
    }


def _problem(setup):
    name, over = _setups()[setup]
    return synth.make_problem(name, **dict(over, ntet=1, fill=False))


class _Handle:
    """The process's current set-up: problem, device databases, library handle."""

    def __init__(self):
        self.setup = self.problem = self.kernel = self.dbs = self.dbkey = None

    def get(self, setup):
        if self.setup == setup:
            return self
        if self.kernel is not None:
            self.kernel.close()
            self.kernel = None
        self.setup = None
        p = _problem(setup)
        key = (p.mesh.nelem, p.nt, p.dt, p.seed)
        if key != self.dbkey:
            if self.dbs is not None:
                self.dbs.free()
            self.dbs, self.dbkey = synth.DeviceDatabases(p), key
        else:
            self.dbs.p = p
            self.dbs.attach()
        self.kernel = mk.MCKernel(p.setup)
        if setup == "tiny":
            self.kernel.set_hetero(*_cloud())
        self.problem, self.setup = p, setup
        return self


_handle = _Handle()

# ---------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------


def listed():
    return [
        # strain traces of a few points: one location launch, one gather (latency)
        {"name": "strain-64", "kind": "strain", "setup": "c0", "points": 64, "frame": 0},
        # base kernels of one Monte Carlo step's points, trace-only set
        {"name": "base-c0-96", "kind": "base", "setup": "c0", "points": 96},
        # base kernels of points spread over the mantle, 10 receivers (few pairs per element)
        {"name": "base-c1-400", "kind": "base", "setup": "c1", "points": 400},
        # an odd number of points, six components each way, nt 1000
        {"name": "base-mt-37", "kind": "base", "setup": "mt", "points": 37},
        # the differentiable stage and its adjoint
        {"name": "ad-300", "kind": "ad", "setup": "ad", "points": 300},
        # the model and heterogeneity integrals of a task on the tetrahedra's vertices
        {"name": "integrals-4000", "kind": "integrals", "setup": "tiny", "elements": 4000, "nbasis": 4},
        # the whole small job: 500 tetrahedra in one task
        {"name": "job-c0-500", "kind": "job", "setup": "c0", "elements": 500, "per_task": 500, "nbasis": 1},
        # tasks of the reference's default size
        {"name": "job-c1-3x100", "kind": "job", "setup": "c1", "elements": 300, "per_task": 100, "nbasis": 1},
        # one task of a GPU slave, basis functions on the vertices
        {"name": "job-c1-1000v", "kind": "job", "setup": "c1", "elements": 1000, "per_task": 1000, "nbasis": 4},
        # a large task
        {"name": "job-c1-12000", "kind": "job", "setup": "c1", "elements": 12000, "per_task": 12000, "nbasis": 1},
        # many kernels per receiver (72 window spectra and base kernels), 50 receivers
        {"name": "job-c2-100", "kind": "job", "setup": "c2", "elements": 100, "per_task": 100, "nbasis": 1},
        # voxels, 200 stations, long traces, six forward components
        {"name": "job-c4-40", "kind": "job", "setup": "c4", "elements": 40, "per_task": 40, "nbasis": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["strain", "base", "base", "ad", "integrals", "job", "job", "job"])
    if kind == "strain":
        return {"kind": kind, "setup": rng.choice(["c0", "mt"]), "points": _log(rng, 16, 3000),
                "frame": rng.randrange(2)}
    if kind == "base":
        setup = rng.choice(["c0", "c1", "mt"])
        return {"kind": kind, "setup": setup, "points": _log(rng, 16, 1500)}
    if kind == "ad":
        return {"kind": kind, "setup": "ad", "points": _log(rng, 16, 600)}
    if kind == "integrals":
        return {"kind": kind, "setup": "tiny", "elements": _log(rng, 300, 4000), "nbasis": rng.choice([1, 4])}
    setup = rng.choice(["c0", "c1", "c1", "c2", "c4"])
    n = _log(rng, *{"c0": (50, 3000), "c1": (100, 12000), "c2": (20, 100), "c4": (10, 40)}[setup])
    per = rng.choice([n, max(1, n // 2)]) if n < 3000 else n
    return {"kind": kind, "setup": setup, "elements": n, "per_task": per,
            "nbasis": 1 if setup in ("c2", "c4") else rng.choice([1, 4])}


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------


def _points(n, seed):
    """n points uniform in the mantle (radius from the core to 50 km depth)."""
    rng = np.random.default_rng(seed)
    r = np.cbrt(rng.uniform((synth.R_CMB + 20e3) ** 3, (synth.R_EARTH - 50e3) ** 3, n))
    v = rng.normal(size=(n, 3))
    return np.ascontiguousarray(v / np.linalg.norm(v, axis=1)[:, None] * r[:, None])


def _elements(p, setup, n, seed):
    """(vertices, connectivity) of a task: n consecutive tetrahedra of a Morton-ordered mesh
    of 50,000, around a point between the source and one of the receivers (elsewhere the
    travel-time masks leave nothing to do); or (c4) n voxels between the source and the
    first receiver."""
    if setup == "c4":
        return p.voxels(n, seed=seed, dlat=1.25, dlon=1.25, dr=96e3)
    total = 50000
    rng = np.random.default_rng(seed + 1)
    verts, conn = synth.random_tets(total, 400e3 if setup == "c0" else 300e3, seed)
    verts = verts.reshape(total, 4, 3)
    r = int(rng.integers(0, (p.nrec + 1) // 2))
    a = synth.geo_xyz(p.src_lat, p.src_lon, synth.R_EARTH - p.src_depth * 1e3)
    b = synth.geo_xyz(p.rec_lat[r], p.rec_lon[r], synth.R_EARTH)
    x = a + rng.uniform(0.2, 0.8) * (b - a)
    near = int(np.argmin(((verts.mean(1) - x) ** 2).sum(1)))
    first = min(max(0, near - n // 2), total - n)
    v = np.ascontiguousarray(verts[first:first + n].reshape(-1, 3))
    return v, np.arange(1, 4 * n + 1, dtype=np.int32).reshape(n, 4)


def _cloud(n=20000):
    """The heterogeneity model: points uniform in the mantle (km, degrees), 2 % anomalies."""
    rng = np.random.default_rng(3)
    r = np.cbrt(rng.uniform(synth.R_CMB ** 3, synth.R_EARTH ** 3, n)) / 1e3
    lat = np.degrees(np.arcsin(rng.uniform(-1, 1, n)))
    rtp = np.stack([r, lat, rng.uniform(-180, 180, n)], 1)
    return np.ascontiguousarray(rtp), (rng.standard_normal((n, 3)) * 0.02).astype(np.float32)


def _traces(gen, shape, nt, dt, scale, device):
    """Strain traces: per trace two wave packets of periods 25 .. 80 s at random arrival
    times, float32."""
    n = int(np.prod(shape))
    t = torch.arange(nt, device=device, dtype=torch.float32) * dt
    out = torch.empty((n, nt), device=device, dtype=torch.float32)
    u = torch.rand((n, 6), generator=gen, device=device)
    for a in range(0, n, 4096):
        x = u[a:a + 4096]
        o = torch.zeros((x.shape[0], nt), device=device)
        for j in range(2):
            t0 = (100.0 + 700.0 * x[:, 3 * j])[:, None]
            per = (25.0 + 55.0 * x[:, 3 * j + 1])[:, None]
            s = (t[None] - t0) / per
            o += (x[:, 3 * j + 2] - 0.5)[:, None] * torch.exp(-s * s) * torch.cos(2 * math.pi * s)
        out[a:a + 4096] = o * scale
    return out.reshape(*shape, nt)


def _ad_inputs(p, nd, nfilter, points, seed, device):
    gen = torch.Generator(device=device).manual_seed(seed)
    fw = _traces(gen, (points, nd), p.nt, p.dt, 1e-9, device)
    bw = _traces(gen, (points, p.nrec, nd), p.nt, p.dt, 1e-27, device)
    gbase = torch.randn((points, p.nkernel, 6), generator=gen, device=device, dtype=torch.float64)
    return fw, bw, gbase


def prepare(case, seed):
    h = _handle.get(case["setup"])
    p, kind = h.problem, case["kind"]
    if kind in ("strain", "base"):
        return dict(case=case, x=_points(case["points"], seed))
    if kind == "ad":
        tf = ad.transfer_functions("cuda")
        fw, bw, gbase = _ad_inputs(p, h.kernel.nd, len(p.filters), case["points"], seed, "cuda")
        return dict(case=case, tf=tf.requires_grad_(), fw=fw.requires_grad_(), bw=bw.requires_grad_(), gbase=gbase)
    verts, conn = _elements(p, case["setup"], case["elements"], seed)
    return dict(case=case, verts=verts, conn=conn)


def run(state):
    case = state["case"]
    h = _handle.get(case["setup"])
    k, kind = h.kernel, case["kind"]
    if kind == "strain":
        return {"traces": k.load_strain(case["frame"], state["x"])}
    if kind == "base":
        return {"base": k.base_kernels(state["x"])}
    if kind == "ad":
        base = ad.filter_convolve_window(state["tf"], state["fw"], state["bw"])
        gtf, gfw, gbw = torch.autograd.grad(base, (state["tf"], state["fw"], state["bw"]), state["gbase"])
        return {"base": base.detach(), "gtf": gtf, "gfw": gfw, "gbw": gbw}
    k.halton_step = 0
    if kind == "integrals":
        model, ns = k.integrate_model(state["verts"], state["conn"], nbasis=case["nbasis"])
        het, nsh = k.integrate_hetero(state["verts"], state["conn"], nbasis=case["nbasis"])
        return {"model": model, "nsteps": ns, "hetero": het, "nsteps_hetero": nsh}
    # a whole job: the kernels as finalize exports them, and their standard errors (the
    # variances themselves, of order 1e60, are beyond single precision)
    res = job.run_job(k, state["verts"], state["conn"], nbasis=case["nbasis"], nelems_per_task=case["per_task"])
    acc = res.get()
    return {"kernel": res.export(results.MCK_RES_KERNEL), "error": _error(acc["variance"]),
            "niterations": acc["niterations"]}


def _error(variance):
    return np.sqrt(np.maximum(variance, 0.0)).astype(np.float32)


# ---------------------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------------------


def _sizes(setup):
    """nt, receivers, kernels, window spectra x base kernels per receiver, carried components
    and variables of each field, database elements, active receivers per point of a job, MC
    steps of a job, points per step."""
    return {"c0": (1024, 1, 2, 2, 1, 1, 4, 2, 2000, 0.5, 8, 32),
            "c1": (2048, 10, 160, 16, 4, 4, 4, 2, 20064, 5.0, 32, 16),
            "c2": (2048, 50, 1200, 24, 4, 4, 4, 2, 20064, 40.0, 128, 16),
            "c4": (4096, 200, 1600, 8, 6, 4, 10, 2, 4000, 78.0, 32, 16),
            "mt": (1000, 3, 24, 8, 6, 6, 10, 3, 2000, 3.0, 32, 16),
            "ad": (2048, 10, 160, 16, 6, 6, 0, 0, 450, 10.0, 0, 0),
            "tiny": (256, 2, 16, 8, 4, 4, 4, 2, 450, 2.0, 3, 8)}[setup]


def work(case):
    """Blocks of the distinct elements once, outputs once; per point (and active receiver)
    the strain at its samples, the FFTs of its components, the base kernels per bin and the
    window sums."""
    nt, R, nk, slots, ndf, ndb, nvf, nvb, nel, act, steps, P = _sizes(case["setup"])
    N = 2 * 2 ** math.ceil(math.log2(nt))
    nw, fft = N // 2 + 1, 2.5 * N * math.log2(N)
    kind = case["kind"]
    if kind == "integrals":
        n = case["elements"]
        return {"bytes": n * (96 + case["nbasis"] * 15 * 8), "flops": n * (100 * 150 + 40 * 200)}
    if kind == "ad":
        n = case["points"]
        tr = n * (ndf + R * ndb)
        return {"bytes": 2 * 4 * tr * nt + 2 * 48 * n * nk,
                "flops": 2 * tr * fft + n * R * nw * (8 * (slots + 8) + 24 * slots + 100)}
    blk = 25 * nt * 4
    fwd = 2 * 25 * nvf * ndf * nt + ndf * fft
    if kind == "strain":
        n = case["points"]
        nd = 1 if case["setup"] == "c0" else 6
        nv = nvf if case["frame"] == 0 else nvb
        return {"bytes": min(n, nel) * nv * blk + 4 * n * nd * nt, "flops": 2 * 25 * nv * nd * nt * n}
    pair = 2 * 25 * nvb * ndb * nt + ndb * fft + nw * (8 * ndf * ndb + 4 * slots)
    if kind == "base":
        n = case["points"]
        return {"bytes": min(n, nel) * nvf * blk + R * min(n, nel) * nvb * blk + 48 * n * nk,
                "flops": n * (fwd + R * pair)}
    n = case["elements"] * steps * P
    touched = min(nel, case["elements"] * 4)
    return {"bytes": touched * nvf * blk + min(nel, touched * act) * nvb * blk + 20 * case["elements"] * nk,
            "flops": n * (fwd + act * pair)}


# ---------------------------------------------------------------------------------------
# the path in FP64
# ---------------------------------------------------------------------------------------

PI = 3.1415926535898          # the path's own truncated pi
DEG = PI / 180.0


class _Memory:
    """A device array of floats at an address, for torch.as_tensor."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (ptr, False), "version": 3}


def _jacobi(n, a, b):
    """zeros of the Jacobi polynomial P_n^(a, b) (Golub and Welsch 1969)."""
    k = np.arange(n)
    with np.errstate(invalid="ignore", divide="ignore"):
        d = np.where(2 * k + a + b == 0, (b - a) / (a + b + 2.0),
                     (b * b - a * a) / ((2 * k + a + b) * (2 * k + a + b + 2.0)))
    k = np.arange(1, n)
    e = 2.0 / (2 * k + a + b) * np.sqrt(k * (k + a) * (k + b) * (k + a + b) / ((2 * k + a + b) ** 2 - 1.0))
    z = np.linalg.eigvalsh(np.diag(d) + np.diag(e, 1) + np.diag(e, -1))
    for _ in range(3):                                        # polish on the monic polynomial's factors
        c = np.polynomial.polynomial.polyfromroots(z)
        z = z - np.polynomial.polynomial.polyval(z, c) / np.polynomial.polynomial.polyval(
            z, np.polynomial.polynomial.polyder(c))
    return z


def _lobatto(a, b):
    return np.concatenate([[-1.0], _jacobi(3, a + 1, b + 1), [1.0]])


def _derivatives(x):
    """G[j, i] = l_i'(x_j) of the Lagrange polynomials on the nodes x."""
    n = len(x)
    G = np.zeros((n, n))
    for i in range(n):
        o = [m for m in range(n) if m != i]
        c = np.polynomial.polynomial.polyfromroots(x[o]) / np.prod(x[i] - x[o])
        G[:, i] = np.polynomial.polynomial.polyval(x, np.polynomial.polynomial.polyder(c))
    return G


def _lagrange(x, at):
    """l_i(at) for node rows x [n][5] and abscissae at [n]."""
    out = torch.ones_like(x)
    for i in range(5):
        for m in range(5):
            if m != i:
                out[:, i] *= (at - x[:, m]) / (x[:, i] - x[:, m])
    return out


def _frame_angles(p, frame):
    lat, lon = (p.src_lat, p.src_lon) if frame == 0 else (float(p.rec_lat[frame - 1]), float(p.rec_lon[frame - 1]))
    return lon * DEG, (90.0 - lat) * DEG


def _xyz(lat, lon, r):
    la, lo = lat * DEG, lon * DEG
    return np.array([math.cos(la) * math.cos(lo), math.cos(la) * math.sin(lo), math.sin(la)]) * r


class Reference:
    """The path of one problem in FP64.  u: the two databases [nelem][nvar][25][nt]
    (node = ipol + 5 jpol), float32 tensors on the device the work is done on."""

    def __init__(self, p, u_fwd, u_bwd, tf=None):
        self.p, self.u = p, (u_fwd, u_bwd)
        self.dev = dev = u_fwd.device
        m = p.mesh
        T = lambda a: torch.as_tensor(np.asarray(a), device=dev)  # noqa: E731
        self.mp = T(np.stack([m.mp_s, m.mp_z], 1))
        self.cs, self.cz = T(m.mesh_s[m.fem].astype(np.float64)), T(m.mesh_z[m.fem].astype(np.float64))
        self.type, self.axis = T(m.eltype), T(m.axis) != 0
        self.gll, self.glj = _lobatto(0, 0), _lobatto(0, 1)
        self.G2, self.G1 = T(_derivatives(self.gll)), T(_derivatives(self.glj))
        # the curved edge of semi-spheroidal elements: the ellipse through its corners, as
        # (a, b, mid angle, angle range)
        def ellipse(i, j):
            s1, z1, s2, z2 = self.cs[:, i], self.cz[:, i], self.cs[:, j], self.cz[:, j]
            det = s2 ** 2 * z1 ** 2 - z2 ** 2 * s1 ** 2
            a = torch.sqrt(torch.abs(det / (z1 ** 2 - z2 ** 2)))
            b = torch.sqrt(torch.abs(det / (s2 ** 2 - s1 ** 2)))
            t1, t2 = torch.atan2(z1 * a, s1 * b), torch.atan2(z2 * a, s2 * b)
            return torch.stack([a, b, (t1 + t2) / 2, t2 - t1], 1)
        top, bot = ellipse(3, 2), ellipse(0, 1)
        self.arc = torch.where((self.type == 2)[:, None], top, bot)
        self.r = torch.sqrt(self.cs ** 2 + self.cz ** 2)
        self.th = torch.where(self.r > 0, torch.acos(self.cz / self.r.clamp_min(1e-300)), torch.zeros_like(self.r))
        params = set(int(q) for q in p.kernel_param)
        self.full = bool(params - {0, 1})                     # lambda and vp kernels read the trace alone
        self.nd = 6 if self.full else 1
        self._kernels(tf)

    # ---- location ---------------------------------------------------------------------
    def _map(self, e, xi, eta):
        """(s, z) and its derivatives (s_xi, s_eta, z_xi, z_eta) at (xi, eta) of elements e."""
        cs, cz, th, r, arc, ty = self.cs[e], self.cz[e], self.th[e], self.r[e], self.arc[e], self.type[e]
        am, ap, bm, bp = 1 - xi, 1 + xi, 1 - eta, 1 + eta
        # spheroidal: concentric arcs
        tt, tb = (am * th[:, 3] + ap * th[:, 2]) / 2, (am * th[:, 0] + ap * th[:, 1]) / 2
        dt, db = (th[:, 2] - th[:, 3]) / 2, (th[:, 1] - th[:, 0]) / 2
        R3, R0 = r[:, 3], r[:, 0]
        sph = [bp * R3 / 2 * torch.sin(tt) + bm * R0 / 2 * torch.sin(tb),
               bp * R3 / 2 * torch.cos(tt) + bm * R0 / 2 * torch.cos(tb),
               bp * R3 / 2 * torch.cos(tt) * dt + bm * R0 / 2 * torch.cos(tb) * db,
               (R3 * torch.sin(tt) - R0 * torch.sin(tb)) / 2,
               -bp * R3 / 2 * torch.sin(tt) * dt - bm * R0 / 2 * torch.sin(tb) * db,
               (R3 * torch.cos(tt) - R0 * torch.cos(tb)) / 2]
        # straight bottom and top edges, one of them replaced by an elliptic arc
        sb, zb = (am * cs[:, 0] + ap * cs[:, 1]) / 2, (am * cz[:, 0] + ap * cz[:, 1]) / 2
        st, zt = (am * cs[:, 3] + ap * cs[:, 2]) / 2, (am * cz[:, 3] + ap * cz[:, 2]) / 2
        dsb, dzb = (cs[:, 1] - cs[:, 0]) / 2, (cz[:, 1] - cz[:, 0]) / 2
        dst, dzt = (cs[:, 2] - cs[:, 3]) / 2, (cz[:, 2] - cz[:, 3]) / 2
        w = arc[:, 2] + xi * arc[:, 3] / 2
        sc, zc = arc[:, 0] * torch.cos(w), arc[:, 1] * torch.sin(w)
        dsc, dzc = -arc[:, 0] * torch.sin(w) * arc[:, 3] / 2, arc[:, 1] * torch.cos(w) * arc[:, 3] / 2
        t2, t3 = ty == 2, ty == 3
        st, zt, dst, dzt = (torch.where(t2, c, o) for c, o in ((sc, st), (zc, zt), (dsc, dst), (dzc, dzt)))
        sb, zb, dsb, dzb = (torch.where(t3, c, o) for c, o in ((sc, sb), (zc, zb), (dsc, dsb), (dzc, dzb)))
        lin = [(bm * sb + bp * st) / 2, (bm * zb + bp * zt) / 2, (bm * dsb + bp * dst) / 2, (st - sb) / 2,
               (bm * dzb + bp * dzt) / 2, (zt - zb) / 2]
        return [torch.where(ty == 0, a, b) for a, b in zip(sph, lin)]

    def locate(self, frame, xyz):
        """Element, (xi, eta) and azimuth of points xyz [n][3] in a frame: the first of the
        12 nearest midpoints' elements (single-precision distances) that holds the point."""
        lon, col = _frame_angles(self.p, frame)
        x, y, z = xyz.unbind(1)
        xc, yc = x * math.cos(lon) + y * math.sin(lon), -x * math.sin(lon) + y * math.cos(lon)
        xp, zp = xc * math.cos(col) - z * math.sin(col), xc * math.sin(col) + z * math.cos(col)
        s, phi = torch.sqrt(xp ** 2 + yc ** 2), torch.atan2(yc, xp)
        phi = torch.where(phi < 0, phi + 2 * PI, phi)
        d = torch.sqrt(s * s + zp * zp)
        f = torch.where(d > self.p.mesh.R, self.p.mesh.R / d, torch.ones_like(d))
        s, z = s * f, zp * f
        elem = torch.full((len(s),), -1, dtype=torch.long, device=self.dev)
        XI, ETA = torch.zeros_like(s), torch.zeros_like(s)
        for a in range(0, len(s), 4096):
            sa, za = s[a:a + 4096], z[a:a + 4096]
            ds, dz = self.mp[None, :, 0] - sa.float()[:, None], self.mp[None, :, 1] - za.float()[:, None]
            near = torch.topk(ds * ds + dz * dz, 12, dim=1, largest=False, sorted=True).indices
            found = torch.zeros(len(sa), dtype=torch.bool, device=self.dev)
            for c in range(12):
                if found.all():
                    break
                e = near[:, c]
                xi, eta = torch.zeros_like(sa), torch.zeros_like(sa)
                for _ in range(10):
                    ms, mz, sx, se, zx, ze = self._map(e, xi, eta)
                    rs, rz, det = sa - ms, za - mz, sx * ze - se * zx
                    near_enough = (rs ** 2 + rz ** 2) / (sa ** 2 + za ** 2) < 1e-14   # the path stops here
                    xi = torch.where(near_enough, xi, xi + (ze * rs - se * rz) / det)
                    eta = torch.where(near_enough, eta, eta + (sx * rz - zx * rs) / det)
                ok = ~found & (xi.abs() <= 1.001) & (eta.abs() <= 1.001)
                at = torch.nonzero(ok).squeeze(1)
                elem[a + at], XI[a + at], ETA[a + at] = e[at], xi[at], eta[at]
                found |= ok
        assert bool((elem >= 0).all()), "point outside the mesh"
        return elem, XI, ETA, phi

    # ---- strain -----------------------------------------------------------------------
    def _operators(self, e, xi, eta):
        """[n][3][25] weights of d/ds, d/dz and 1/s at (xi, eta): evaluated at the GLL nodes
        of the elements and interpolated (on the axis 1/s is the s derivative)."""
        n, ax = len(e), self.axis[e]
        gll = torch.as_tensor(self.gll, device=self.dev)
        glj = torch.as_tensor(self.glj, device=self.dev)
        nx = torch.where(ax[:, None], glj[None], gll[None])
        li, lj = _lagrange(nx, xi), _lagrange(gll[None].expand(n, 5).contiguous(), eta)
        Gx = torch.where(ax[:, None, None], self.G1[None], self.G2[None])
        W = torch.zeros((n, 3, 5, 5), dtype=torch.float64, device=self.dev)       # [op][j][i]
        for i in range(5):
            for j in range(5):
                s, _, sx, se, zx, ze = self._map(e, nx[:, i], gll[j].expand(n))
                det, l = sx * ze - se * zx, li[:, i] * lj[:, j]
                xs, es, xz, ez = ze / det, -zx / det, -se / det, sx / det
                # nodal d/ds = xs d/dxi + es d/deta, d/dz = xz d/dxi + ez d/deta
                W[:, 0, j, :] += (l * xs)[:, None] * Gx[:, i, :]
                W[:, 0, :, i] += (l * es)[:, None] * self.G2[None, j, :]
                W[:, 1, j, :] += (l * xz)[:, None] * Gx[:, i, :]
                W[:, 1, :, i] += (l * ez)[:, None] * self.G2[None, j, :]
                if i == 0:
                    W[:, 2, j, :] += torch.where(ax, l * xs, torch.zeros_like(l))[:, None] * Gx[:, i, :]
                    W[:, 2, :, i] += torch.where(ax, l * es, torch.zeros_like(l))[:, None] * self.G2[None, j, :]
                    W[:, 2, j, i] += torch.where(ax, torch.zeros_like(l), l / s)
                else:
                    W[:, 2, j, i] += l / s
        return W.reshape(n, 3, 25)

    @staticmethod
    def _strain(g, pole):
        """Voigt strain (ss, pp, zz, zp, sz, sp; components 4 and 6 negated as the merged
        databases are read) from g[variable][operator] = [n][nt]."""
        z = torch.zeros_like(g[0][0])
        if pole == 0:
            a, b = g
            return [a[0], a[2], b[1], z, (a[1] + b[0]) / 2, z]
        a, b, c = g
        return [a[0], a[2] - pole * b[2], c[1], (pole * c[2] + b[1]) / 2, (a[1] + c[0]) / 2,
                (pole * a[2] - b[2] + b[0]) / 2]

    def traces(self, frame, xyz, loc=None):
        """Earth-frame strain (or trace) [n][nd][nt] of one frame, before cumsum."""
        p, which = self.p, 0 if frame == 0 else 1
        e, xi, eta, phi = loc if loc is not None else self.locate(frame, xyz)
        W = self._operators(e, xi, eta)
        c1, s1, c2, s2 = torch.cos(phi), torch.sin(phi), torch.cos(2 * phi), torch.sin(2 * phi)
        one, nil = torch.ones_like(phi), torch.zeros_like(phi)
        M = p.mij
        if which == 0:       # (variables, pole, radiation factors of the even and odd components)
            sims = [(0, 0, M[0] * one, nil), (2, 0, 0.5 * (M[1] + M[2]) * one, nil),
                    (4, 1, M[3] * c1 + M[4] * s1, -M[3] * s1 + M[4] * c1),
                    (7, 2, 0.5 * (M[1] - M[2]) * c2 + M[5] * s2, -0.5 * (M[1] - M[2]) * s2 + M[5] * c2)]
            sims = [s for s in sims if float(s[2].abs().max()) > 0 or float(s[3].abs().max()) > 0]
        elif p.component == "Z":
            sims = [(0, 0, one, one)]
        else:
            fr, ft = (1.0, 0.0) if p.component == "R" else (0.0, 1.0)
            sims = [(2, 1, fr * c1 + ft * s1, -fr * s1 + ft * c1)]
        amp = (p.setup.fwd if which == 0 else p.setup.bwd).amplitude
        out = [0.0] * self.nd
        for v0, pole, even, odd in sims:
            nv = 2 if pole == 0 else 3
            u = self.u[which][e, v0:v0 + nv].double()                     # [n][nv][25][nt]
            g = [[t for t in torch.matmul(W, u[:, v]).unbind(1)] for v in range(nv)]
            E = self._strain(g, pole)
            if not self.full:
                out[0] = out[0] + (E[0] + E[1] + E[2]) * (even / amp)[:, None]
                continue
            two = 2.0 if which == 1 and p.component != "Z" else 1.0
            fac = [even, even, even, odd, two * even, two * odd]
            for c in range(6):
                out[c] = out[c] + E[c] * (fac[c] / amp)[:, None]
        if not self.full:
            return torch.stack(out, 1)
        # strain tensor in (s, phi, z) -> xyz of the frame -> xyz of the earth
        lon, col = _frame_angles(p, frame)
        n = len(phi)
        A = torch.zeros((n, 3, 3), dtype=torch.float64, device=self.dev)
        A[:, 0, 0], A[:, 0, 1], A[:, 1, 0], A[:, 1, 1], A[:, 2, 2] = c1, -s1, s1, c1, 1.0
        cl, sl, ct, st = math.cos(lon), math.sin(lon), math.cos(col), math.sin(col)
        Q = torch.tensor([[cl * ct, -sl, cl * st], [sl * ct, cl, sl * st], [-st, 0.0, ct]], dtype=torch.float64,
                         device=self.dev)
        A = torch.matmul(Q[None].expand(n, 3, 3).contiguous(), A)
        S = torch.stack([torch.stack([out[i] for i in r], 1) for r in ((0, 5, 4), (5, 1, 3), (4, 3, 2))], 1)
        idx = [(0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1)]
        res = torch.zeros((n, 6, out[0].shape[1]), dtype=torch.float64, device=self.dev)
        for c, (a, b) in enumerate(idx):
            for i in range(3):
                for j in range(3):
                    res[:, c] += (A[:, a, i] * A[:, b, j])[:, None] * S[:, i, j]
        return res

    # ---- kernels ----------------------------------------------------------------------
    def _window(self, n, ntaper, end_only=False):
        """The Gaussian taper of ntaper samples (single-precision values) at the ends."""
        i = np.arange(1, ntaper + 1, dtype=np.float32)
        w = np.exp(-(np.float32(3.3) * i / np.float32(ntaper)) ** 2).astype(np.float64)
        t = np.ones(n)
        t[n - ntaper:] = w
        if not end_only:
            t[:ntaper] = w[::-1]
        return torch.as_tensor(t, device=self.dev)

    def rfft(self, x):
        return torch.fft.rfft(x * self.taper, n=self.N) * self.p.dt

    def _butterworth(self, f, period, n, low):
        k = np.arange(1, n + 1)
        s = np.exp(1j * (2 * k + n - 1) * PI / (2 * n))
        w = 1j * f * period
        with np.errstate(divide="ignore", invalid="ignore"):
            q = w if low else 1 / w
            H = 1 / np.prod(q[:, None] - s[None], axis=1)
        if not low:
            H[0] = 0
        return H

    def _kernels(self, tf):
        p = self.p
        nt, dt = p.nt, p.dt
        N = 2 * 2 ** math.ceil(math.log2(nt))
        nw, df = N // 2 + 1, 1.0 / (dt * N)
        self.N, self.nw, self.df = N, nw, df
        self.taper = self._window(nt, 10)
        f = df * np.arange(nw)
        G = []
        for flt in p.filters:
            fr = list(flt.frequencies)
            if flt.filterclass == 1:
                with np.errstate(divide="ignore"):
                    G.append(np.where(f > 0, np.exp(-np.log(f * fr[0]) ** 2 / (2 * math.log(fr[1]) ** 2)), 0.0)
                             * np.exp(-2j * PI * f * fr[2]))
            else:
                G.append(self._butterworth(f, fr[0], int(fr[2]), False)
                         * self._butterworth(f, fr[1], int(fr[2]), True))
        # STF deconvolution: divide by the database's source spectrum, the earthquake's a
        # unit impulse, a squared low pass of order 12 at 3/4 of the highest frequency
        stf = torch.as_tensor(p.stf, device=self.dev) * self._window(nt, 2)
        Fs = (torch.fft.rfft(stf, n=N) * dt).cpu().numpy()
        lp = np.abs(self._butterworth(f, 1.0 / (0.75 * f[-1]), 12, True)) ** 2
        back = p.setup.fwd.amplitude / Fs * lp
        fore = back * dt
        self.tf0 = np.stack(G)
        T = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev)  # noqa: E731
        tff, rest = T(np.stack([g * fore for g in G])), T(fore * back)
        self.G = T(self.tf0)
        seis = T(p.seis)
        cum = torch.zeros_like(seis)
        x = seis.clone()
        x[:, 2:] += seis[:, 1:-1]
        cum = torch.cumsum(x, 1) * (dt * 0.5)
        spec = {0: torch.fft.rfft(seis, n=N) * dt, 1: torch.fft.rfft(cum, n=N) * dt}
        t = np.arange(N) * dt
        self.win, self.slot = [], []         # window spectra; kernel -> (window, filter)
        c = torch.full((nw,), 2.0, dtype=torch.float64, device=self.dev)
        c[0] = c[-1] = 1.0
        seen = {}
        for k in range(p.nkernel):
            r, fi, mf = int(p.kernel_receiver[k]), int(p.kernel_filter[k]), int(p.kernel_misfit[k])
            key = (r, fi, mf) + tuple(p.kernel_window[k])
            if key not in seen:
                xs = torch.fft.irfft(spec[mf][r] * tff[fi], n=N) * (N * df)
                at = np.nonzero((t >= p.kernel_window[k][0]) & (t <= p.kernel_window[k][1]))[0]
                w = torch.zeros(N, dtype=torch.float64, device=self.dev)
                w[at] = xs[at]
                norm = dt * float((w * w).sum())
                # -(1 / norm) sum_t x_t w_t dt as a sum over the bins of X
                S = torch.conj(torch.fft.rfft(w)) * (c * (-df * dt / norm if norm > 1e-100 else 0.0))
                seen[key] = len(self.win)
                self.win.append(S * rest)
            self.slot.append((seen[key], fi))
        self.win = torch.stack(self.win)
        self.klist = [np.nonzero(p.kernel_receiver == r)[0] for r in range(p.nrec)]

    def fwd_spectra(self, tr):
        x = tr.clone()
        x[..., 2:] += tr[..., 1:-1]
        return self.rfft(torch.cumsum(x, -1) * (self.p.dt * 0.5))

    def contract(self, r, F, B, G=None):
        """Base kernels lambda, mu of receiver r's kernels: [n][kernels of r][6]."""
        p, ks = self.p, self.klist[r]
        G = self.G if G is None else G
        if self.full:
            lam = -F[:, :3].sum(1) * B[:, :3].sum(1)
            mu = -2.0 * (F * B).sum(1)
        else:
            lam, mu = -(F * B).sum(1), None
        H = torch.stack([self.win[self.slot[k][0]] * G[self.slot[k][1]] ** 2 for k in ks])
        L = torch.matmul(lam, H.t().contiguous()).real
        zero = torch.zeros_like(L)
        vp = torch.as_tensor(np.isin(p.kernel_param[ks], (0, 1, 2)), device=self.dev)
        out = [torch.where(vp[None], L, zero)]
        if mu is not None:
            needs = torch.as_tensor(np.isin(p.kernel_param[ks], (2, 3)), device=self.dev)
            out.append(torch.where(needs[None], torch.matmul(mu, H.t().contiguous()).real, zero))
        else:
            out.append(zero)
        return torch.stack(out + [zero] * 4, 2)

    def base(self, xyz, chunk=128):
        out = torch.zeros((len(xyz), self.p.nkernel, 6), dtype=torch.float64, device=self.dev)
        for a in range(0, len(xyz), chunk):
            x = xyz[a:a + chunk]
            F = self.fwd_spectra(self.traces(0, x))
            for r in range(self.p.nrec):
                out[a:a + chunk, self.klist[r]] = self.contract(r, F, self.rfft(self.traces(1 + r, x)))
        return out

    def stage(self, tf, fw, bw):
        """The differentiable stage: tf [nfilter][nw], fw [n][nd][nt], bw [n][R][nd][nt]."""
        F = self.fwd_spectra(fw)
        return torch.cat([self.contract(r, F, self.rfft(bw[:, r]), tf) for r in range(self.p.nrec)], 1)

    # ---- Monte Carlo ------------------------------------------------------------------
    @staticmethod
    def halton(idx):
        """Halton points (bases 2, 3, 5, seed 20, leap 2) at stream positions idx."""
        out = np.zeros((len(idx), 3))
        for d, b in enumerate((2, 3, 5)):
            s, w = 20 + 2 * idx.astype(np.int64), float(b)
            while s.any():
                out[:, d] += (s % b) / w
                s, w = s // b, w * b
        return out

    @classmethod
    def tet_points(cls, V, idx):
        """Points of tetrahedra V [n][4][3] at positions idx [n][P] (Rocchini and Cignoni 2001)."""
        c = cls.halton(idx.ravel()).reshape(idx.shape + (3,))
        a, b, g = c[..., 0], c[..., 1], c[..., 2]
        f = a + b > 1.0
        a, b = np.where(f, 1.0 - a, a), np.where(f, 1.0 - b, b)
        f1, f2 = b + g > 1.0, (a + b + g > 1.0) & ~(b + g > 1.0)
        a, b, g = (np.where(f2, 1.0 - b - g, a), np.where(f1, 1.0 - g, b),
                   np.where(f1, 1.0 - a - b, np.where(f2, a + b + g - 1.0, g)))
        w = np.stack([a, b, g, 1.0 - (a + b + g)], -1)
        return np.einsum("npk,nki->npi", w, V), w

    def model_at(self, x):
        r = np.sqrt((x * x).sum(-1))
        return np.clip((r / 100.0 + 1).astype(np.int64), 1, self.p.model.shape[1]) - 1

    def job(self, verts, conn, nbasis):
        """slave_work of all elements (tetrahedra): values, variances [ne][nbasis][nk] and
        niterations [ne][nk]; element e draws from position e (max_iter + 1) P."""
        p = self.p
        ne, nk, P = len(conn), p.nkernel, p.npoints_per_step
        V = np.asarray(verts).reshape(-1, 3)[np.asarray(conn) - 1]
        vol = np.abs(np.linalg.det(V[:, 1:] - V[:, :1])) / 6.0
        src = _xyz(p.src_lat, p.src_lon, p.mesh.R - p.src_depth * 1e3)
        centre = V.mean(1)
        ab = np.concatenate([(V - V[:, :1]).transpose(0, 2, 1), np.ones((ne, 1, 4))], 1)
        inv = np.linalg.inv(ab)
        masked = np.zeros((ne, p.nrec), bool)
        for r in range(p.nrec):
            d = np.linalg.norm(centre - src, axis=1) + np.linalg.norm(
                centre - _xyz(p.rec_lat[r], p.rec_lon[r], p.mesh.R), axis=1)
            ks = self.klist[r]
            isp = np.isin(p.kernel_param[ks], (0, 1))
            tp = p.kernel_window[ks][isp, 1].max(initial=0.0)
            ts = p.kernel_window[ks][~isp, 1].max(initial=0.0)
            masked[:, r] = (d / p.setup.vp_max > tp) & (d / p.setup.vs_max > ts)
        kmask = masked[:, p.kernel_receiver]
        nbk = np.where(p.kernel_param == 2, 2, 1)
        fs, f2 = np.zeros((ne, nbasis, nk)), np.zeros((ne, nbasis, nk))
        integral, var = np.zeros((ne, nbasis, nk)), np.zeros((ne, nbasis, nk))
        conv = np.zeros((ne, nbasis, nk), bool)
        niter, drawn = np.zeros((ne, nk), np.int32), 0
        vp, vs, rho = (p.model[i] for i in range(3))
        while True:
            live = ~conv.all((1, 2)) & ~(niter == p.max_iter).any(1)
            at = np.nonzero(live)[0]
            if not len(at):
                return integral, var, niter
            idx = at[:, None] * (p.max_iter + 1) * P + drawn * P + np.arange(P)[None]
            drawn += 1
            x, _ = self.tet_points(V[at], idx)
            dx = x - V[at][:, :1]
            bw = (np.einsum("nbk,npk->npb", inv[at], np.concatenate([dx, np.ones(x.shape[:2] + (1,))], 2))
                  if nbasis > 1 else np.ones(x.shape[:2] + (1,)))
            done = conv[at].all(1)
            active = ~masked[at] & np.stack([~done[:, ks].all(1) for ks in self.klist], 1)
            xt = torch.as_tensor(x.reshape(-1, 3), device=self.dev)
            phys = np.zeros((len(at) * P, nk))
            step = max(1, 1024 // P)
            for a in range(0, len(at), step):
                lo, hi = a * P, min(len(at), a + step) * P
                if not active[a:a + step].any():
                    continue
                F = self.fwd_spectra(self.traces(0, xt[lo:hi]))
                for r in range(p.nrec):
                    use = np.nonzero(np.repeat(active[a:a + step, r], P))[0]
                    if not len(use):
                        continue
                    u = torch.as_tensor(use, device=self.dev)
                    b = self.contract(r, F[u], self.rfft(self.traces(1 + r, xt[lo:hi][u]))).cpu().numpy()
                    m = self.model_at(x.reshape(-1, 3)[lo + use])
                    cp, cv = (2.0 * rho[m].astype(float) * (v[m] * v[m]).astype(float) for v in (vp, vs))
                    ks = self.klist[r]
                    isvs = p.kernel_param[ks] == 2
                    phys[(lo + use)[:, None], ks[None]] = np.where(isvs[None], cv[:, None] * (b[..., 1] - 2 * b[..., 0]),
                                                                   cp[:, None] * b[..., 0])
            phys = phys.reshape(len(at), P, nk)
            km = kmask[at]
            ran = active[:, p.kernel_receiver] & ~done & ~km
            niter[at] += km.astype(np.int32) + np.where(ran, nbk[None], 0).astype(np.int32)
            n = drawn * P
            for b in range(nbasis):
                y = phys * bw[:, :, b][:, :, None]
                go = ~conv[at, b]
                fs[at, b] += np.where(go, y.sum(1), 0)
                f2[at, b] += np.where(go, (y * y).sum(1), 0)
                Vv = vol[at][:, None]
                I = fs[at, b] * Vv / n
                S = Vv * Vv / (n - 1) * (f2[at, b] / n - (fs[at, b] / n) ** 2)
                integral[at, b], var[at, b] = np.where(go, I, integral[at, b]), np.where(go, S, var[at, b])
                aerr = (p.allowed_error * Vv) ** 2
                conv[at, b] |= go & ((S < aerr) | (np.sqrt(np.maximum(S, 0)) < p.allowed_relative_error * np.abs(I)))

    def integrals(self, verts, conn, nbasis, values, npts, rel, start=0):
        """The Monte Carlo integrals (volume 1, errors 1e-2 and rel, npts points per step) of
        values(x) [n][P][m] times the basis functions: [ne][nbasis][m], steps [ne].  start:
        stream position of the first element, each reserving 9999 steps."""
        V = np.asarray(verts).reshape(-1, 3)[np.asarray(conn) - 1]
        ne = len(V)
        inv = np.linalg.inv(np.concatenate([(V - V[:, :1]).transpose(0, 2, 1), np.ones((ne, 1, 4))], 1))
        out = fs = f2 = conv = None
        steps = np.zeros(ne, np.int32)
        for it in range(9999):
            at = np.arange(ne) if conv is None else np.nonzero(~conv.all((1, 2)))[0]
            if not len(at):
                break
            x, _ = self.tet_points(V[at], start + (at[:, None] * 9999 + it) * npts + np.arange(npts)[None])
            bw = (np.einsum("nbk,npk->npb", inv[at], np.concatenate([x - V[at][:, :1], np.ones(x.shape[:2] + (1,))], 2))
                  if nbasis > 1 else np.ones(x.shape[:2] + (1,)))
            v = values(x)
            if conv is None:
                out, fs, f2 = (np.zeros((ne, nbasis, v.shape[2])) for _ in range(3))
                conv = np.zeros(out.shape, bool)
            y = v[:, :, None, :] * bw[..., None]
            go, n = ~conv[at], (it + 1) * npts
            fs[at] += np.where(go, y.sum(1), 0)
            f2[at] += np.where(go, (y * y).sum(1), 0)
            I, S = fs[at] / n, (f2[at] / n - (fs[at] / n) ** 2) / (n - 1)
            out[at] = np.where(go, I, out[at])
            conv[at] |= go & ((S < 1e-4) | (np.sqrt(np.maximum(S, 0)) < rel * np.abs(I)))
            steps[at] += 1
        return out, steps

    def background(self, x):
        vp, vs, rho, phi, xi, eta = (self.p.model[i][self.model_at(x)] for i in range(6))
        lam, mu = rho * (vp * vp - 2 * (vs * vs)), rho * (vs * vs)
        return np.stack([vp, vs, rho, vp, vp * np.sqrt(phi), vs, vs / np.sqrt(xi), eta, phi, xi, lam, mu],
                        -1).astype(np.float64)


def _nearest(cloud, x, device):
    """Index of the cloud's point nearest to each x, by single-precision distances."""
    rtp, _ = cloud
    la, lo = (rtp[:, 1] * DEG), (rtp[:, 2] * DEG)
    c = (rtp[:, 0] * 1e3)[:, None] * np.stack([np.cos(la) * np.cos(lo), np.cos(la) * np.sin(lo), np.sin(la)], 1)
    c = torch.as_tensor(c.astype(np.float32), device=device)
    q = torch.as_tensor(x.reshape(-1, 3).astype(np.float32), device=device)
    out = []
    for a in range(0, len(q), 8192):
        d = q[a:a + 8192, None, 0] - c[None, :, 0]
        d = d * d
        for i in (1, 2):
            e = q[a:a + 8192, None, i] - c[None, :, i]
            d += e * e
        out.append(d.argmin(1))
    return torch.cat(out).cpu().numpy().reshape(x.shape[:-1])


def _reference(h):
    p, m = h.problem, h.problem.mesh
    u = [torch.as_tensor(_Memory(d.value, (m.nelem, nv, 25, p.nt)), device="cuda")
         for d, nv in zip(h.dbs.ptrs, (10, 5))]
    return Reference(p, *u)


#: (point, receiver) pairs of a job above which its FP64 restatement takes over 20 s
EXACT_PAIRS = 100000


def exact(case, seed):
    setup, kind = case["setup"], case["kind"]
    if kind == "job":
        s = _sizes(setup)
        if setup in ("c2", "c4") or case["elements"] * s[10] * s[11] * s[9] > EXACT_PAIRS:
            return None
    h = _handle.get(setup)
    ref, p = _reference(h), h.problem
    if kind in ("strain", "base"):
        x = torch.as_tensor(_points(case["points"], seed), device="cuda")
        if kind == "base":
            return {"base": ref.base(x)}
        return {"traces": torch.cat([ref.traces(case["frame"], x[a:a + 64]) for a in range(0, len(x), 64)])}
    if kind == "ad":
        fw, bw, gbase = _ad_inputs(p, ref.nd, len(p.filters), case["points"], seed, "cuda")
        tf = ref.G.to(torch.complex64).to(torch.complex128).requires_grad_()
        base, gfw, gbw, gtf = [], [], [], torch.zeros_like(tf)
        for a in range(0, len(fw), 32):
            f, b = (t[a:a + 32].double().requires_grad_() for t in (fw, bw))
            o = ref.stage(tf, f, b)
            g = torch.autograd.grad(o, (tf, f, b), gbase[a:a + 32])
            gtf += g[0]
            base.append(o.detach())
            gfw.append(g[1])
            gbw.append(g[2])
        return {"base": torch.cat(base), "gtf": gtf.detach(), "gfw": torch.cat(gfw), "gbw": torch.cat(gbw)}
    verts, conn = _elements(p, setup, case["elements"], seed)
    if kind == "integrals":
        model, ns = ref.integrals(verts, conn, case["nbasis"], ref.background, 100, 1e-2)
        cloud = _cloud()
        dln = cloud[1].astype(np.float64)
        # drawn after the stream range of the model integrals
        het, nsh = ref.integrals(verts, conn, case["nbasis"], lambda x: dln[_nearest(cloud, x, "cuda")], 10, 1e-1,
                                 start=len(conn) * 9999 * 100)
        return {"model": model, "nsteps": ns, "hetero": het, "nsteps_hetero": nsh}
    val, var, nit = ref.job(verts, conn, case["nbasis"])
    if case["nbasis"] > 1:           # vertices belong to one element each: basis function b -> vertex 4 e + b
        val, var = val.reshape(-1, p.nkernel), var.reshape(-1, p.nkernel)
    else:
        val, var = val[:, 0], var[:, 0]
    return {"kernel": np.ascontiguousarray(val.T), "error": np.sqrt(np.maximum(var, 0.0)), "niterations": nit}
