"""What a user of this framework has it do, as timed cases.

A case is a whole call sequence through the public entry points:

  run       a short simulation: upload an initial condition, initialize, a few
            time steps, and the snapshot and energy sums that such a program
            writes at its output time (steps = 0: one evaluation of the
            density, pressure and forces of a given configuration)
  rollout   the differentiable rollout: forward through torch.autograd and
            the gradient of sum m |v|^2 with respect to the initial state
  timestep  the time-step criterion over the caller's own device arrays

Snapshots of mixed-precision runs are kept in FP32, those of FP64 runs in
FP64.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from sphcode_amd import DISPH, FP64, GSPH, MIXED, SSPH, CUBIC_SPLINE, WENDLAND, GPUEngine, ics, library
from sphcode_amd.autograd import rollout

TYPES = {"ssph": SSPH, "disph": DISPH, "gsph": GSPH}
SNAPSHOT = ("pos", "vel", "dens", "ene")
FORCES = ("acc", "dene", "dens", "pres", "sml", "neighbor")


def listed():
    return [
        # the smallest call: the time-step criterion of a small state on the
        # caller's stream (two launches, nothing allocated)
        dict(name="timestep-4k", do="timestep", n=4096, dim=3),
        # the reference's own shock tube: 1D, FP64; latency of a step
        dict(name="sod-1d-fp64", do="run", ic="sod", size=1600, type="ssph", precision="fp64", steps=20),
        # one evaluation of a small 2D state, odd sizes
        dict(name="eval-2d-fp64", do="run", ic="khi", size=91, type="ssph", precision="fp64", steps=0),
        # a small self-gravitating run, odd size
        dict(name="evrard-20k-mixed", do="run", ic="evrard", size=20011, type="disph", precision="mixed", steps=16),
        # one GPU's share of the collapse on eight, in FP64
        dict(name="evrard-131k-fp64", do="run", ic="evrard", size=131072, type="disph", precision="fp64", steps=12),
        # the benchmark's collapse
        dict(name="evrard-1m-mixed", do="run", ic="evrard", size=1 << 20, type="disph", precision="mixed", steps=20),
        # the Kelvin-Helmholtz workload, 393,160 particles in 2D
        dict(name="khi-393k-mixed", do="run", ic="khi", size=512, type="disph", precision="mixed", steps=20),
        # forces of a given 3D periodic configuration in FP64
        dict(name="eval-110k-fp64", do="run", ic="box", size=48, type="ssph", precision="fp64", steps=0),
        # a blast wave, GSPH second order, 2,097,152 particles
        dict(name="blast-2m-mixed", do="run", ic="blast", size=128, type="gsph", precision="mixed", steps=4),
        # gradient of the rollout workload (262,144 particles, 16 steps); the
        # Balsara switch, whose kink no gradient passes smoothly, is off
        dict(name="rollout-262k-mixed", do="rollout", size=64, dim=3, precision="mixed", steps=16, balsara=False),
        # the same in FP64 with the switch, smaller and odd
        dict(name="rollout-30k-fp64", do="rollout", size=31, dim=3, precision="fp64", steps=8, balsara=True),
        # a 2D gradient: the small training step
        dict(name="rollout-2d-fp64", do="rollout", size=48, dim=2, precision="fp64", steps=4, balsara=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["timestep", "sod", "khi", "evrard", "evrard", "box", "blast", "rollout", "rollout"])
    precision = rng.choice(["fp64", "mixed"])
    if what == "timestep":
        return dict(do="timestep", n=_log_int(rng, 1000, 1 << 24), dim=rng.choice([1, 2, 3]))
    if what == "rollout":
        dim = rng.choice([2, 3, 3])
        size = _log_int(rng, 32, 256) if dim == 2 else _log_int(rng, 12, 56)
        return dict(do="rollout", size=size, dim=dim, precision=precision, steps=rng.randint(2, 12),
                    balsara=precision == "fp64" and rng.random() < 0.5)
    c = dict(do="run", ic=what, precision=precision)
    if what == "sod":
        # an FP64 workload (in 1D a small state's rounding decides its course)
        c.update(precision="fp64", size=8 * _log_int(rng, 60, 10000), type=rng.choice(["ssph", "disph"]), steps=rng.randint(0, 24))
    elif what == "khi":
        c.update(size=_log_int(rng, 40, 500), type=rng.choice(["ssph", "disph", "gsph"]), steps=rng.randint(0, 20))
    elif what == "evrard":
        big = (1 << 20) if precision == "mixed" else 400000
        c.update(size=_log_int(rng, 1500, big), type=rng.choice(["ssph", "disph", "disph"]), steps=rng.randint(0, 14))
    elif what == "box":
        c.update(size=_log_int(rng, 12, 100), type=rng.choice(["ssph", "disph", "gsph"]), steps=rng.randint(0, 6))
    else:
        c.update(size=_log_int(rng, 16, 110), type="gsph", steps=rng.randint(0, 4))
    return c


def _initial(case, seed):
    """Parameters and fields of a run's or rollout's initial condition."""
    precision = FP64 if case["precision"] == "fp64" else MIXED
    size = case["size"]
    rng = np.random.default_rng(seed)
    if case["do"] == "rollout":
        p, f = ics.rollout(size, seed=seed, precision=precision, dim=case["dim"])
        p.av_use_balsara_switch = 1 if case["balsara"] else 0
        return p, f
    ic = case["ic"]
    kind = TYPES[case["type"]]
    if ic == "sod":
        # the lattice of the shock tube, with the seed in a small velocity noise
        p, f = ics.sod(size, size // 8, precision=precision)
        f["vel"] = rng.normal(0.0, 1e-3, f["vel"].shape)
    elif ic == "khi":
        p, f = ics.khi(n_low=size, n_high=int(round(size * math.sqrt(2.0))), jitter=0.02, seed=seed, precision=precision)
    elif ic == "evrard":
        p, f = ics.evrard(size, seed=seed, precision=precision)
        f["vel"] = rng.normal(0.0, 0.02, f["vel"].shape)
    elif ic == "box":
        p, f = ics.rollout(size, seed=seed, precision=precision)
    else:
        # the blast of the Sedov workload at an energy whose contrast to the
        # background the second-order scheme follows from the first step on
        u0, hot = 1e-2, 64
        p, f = ics.sedov(size, seed=seed, n_hot=hot, energy=2e3 * u0 * hot / size ** 3, precision=precision, u_background=u0)
        f["vel"] = rng.normal(0.0, 1e-2, f["vel"].shape)
    p.sph_type = kind
    return p, f


def _timestep_call():
    lib, _ = library()
    fn = lib.sphgpu_timestep_noalloc
    fn.restype = C.c_int
    fn.argtypes = [C.c_int, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                   C.c_double, C.c_double, C.c_void_p, C.c_void_p]
    return fn


def _timestep_arrays(case, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    n = case["n"]
    sml = 0.01 * (0.5 + torch.rand(n, generator=g, dtype=torch.float64))
    acc = torch.randn(case["dim"], n, generator=g, dtype=torch.float64) * 3.0
    hvs = 1e-3 * (1.0 + torch.rand(1, generator=g, dtype=torch.float64)) * 50.0
    return sml, acc, hvs


def prepare(case, seed):
    if case["do"] == "timestep":
        sml, acc, hvs = (a.cuda() for a in _timestep_arrays(case, seed))
        return dict(case=case, fn=_timestep_call(), sml=sml, acc=acc, hvs=hvs)
    p, f = _initial(case, seed)
    state = dict(case=case, params=p, fields=f, engine=GPUEngine(p, stats=False))
    if case["do"] == "rollout":
        dtype = torch.float64 if case["precision"] == "fp64" else torch.float32
        state.update({k: torch.from_numpy(f[k]).to("cuda", dtype) for k in ("pos", "vel", "ene", "mass")})
    return state


ROLLOUT_DT = 1e-3


def run(state):
    case = state["case"]
    if case["do"] == "timestep":
        acc, dim = state["acc"], case["dim"]
        out = torch.empty(1, dtype=torch.float64, device="cuda")
        ptr = [acc[k].data_ptr() if k < dim else None for k in range(3)]
        rc = state["fn"](dim, case["n"], state["sml"].data_ptr(), ptr[0], ptr[1], ptr[2], state["hvs"].data_ptr(),
                         0.3, 0.125, out.data_ptr(), torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise RuntimeError("sphgpu_timestep_noalloc: status %d" % rc)
        return out
    engine = state["engine"]
    if case["do"] == "rollout":
        x, v, u = (state[k].detach().requires_grad_(True) for k in ("pos", "vel", "ene"))
        xk, vk, uk = rollout(engine, state["fields"], x, v, u, case["steps"], ROLLOUT_DT)
        loss = (state["mass"][:, None] * vk * vk).sum()
        loss.backward()
        return dict(pos=xk.detach(), vel=vk.detach(), ene=uk.detach(), g_pos=x.grad, g_vel=v.grad, g_ene=u.grad)
    engine.upload(state["fields"])
    engine.initialize()
    for _ in range(case["steps"]):
        engine.integrate()
    out = engine.download(SNAPSHOT if case["steps"] else FORCES)
    if case["precision"] == "mixed":
        out = {k: a.astype(np.float32) if a.dtype == np.float64 else a for k, a in out.items()}
        if not case["steps"]:
            # FP32 pair sums: a pair at the edge of the support, where it
            # contributes nothing, may be counted or not
            del out["neighbor"]
    if case["steps"]:
        out["time"] = np.array(engine.time()[0], dtype=np.float64 if case["precision"] == "fp64" else np.float32)
        e = engine.energy()
        out["energy"] = e[:4] if case["precision"] == "fp64" else e[:4].astype(np.float32)
    return out


def work(case):
    if case["do"] == "timestep":
        return {"bytes": 8.0 * case["n"] * (case["dim"] + 1) + 16, "flops": 6.0 * case["n"]}
    if case["do"] == "rollout":
        dim, n = case["dim"], case["size"] ** case["dim"]
        pairs = {2: 24, 3: 50}[dim]
        evals = case["steps"] + 1
        # forward evaluation, and its adjoint (which needs the evaluation's
        # sums again); the state in and out once a step and way
        return {"bytes": evals * n * 8.0 * (4 * (2 * dim + 1) + 10), "flops": evals * n * pairs * (33.0 + 53 + 105 + 33 + 53 + 300)}
    ic, size = case["ic"], case["size"]
    dim = {"sod": 1, "khi": 2}.get(ic, 3)
    n = {"sod": size + size // 8, "khi": int(1.5 * size * size), "evrard": size}.get(ic, size ** 3)
    pairs = {"sod": 4, "khi": 64, "evrard": 64, "blast": 64}.get(ic, 50)
    evals = case["steps"] + 1
    per_pair = 33 + 53 + 48 + {"ssph": 105, "disph": 115, "gsph": 255}[case["type"]]
    flops = evals * n * float(pairs * per_pair)
    if ic == "evrard":
        # Barnes-Hut at theta 0.5: particle pairs and accepted cells
        flops += evals * n * (71.0 * 340 + 33.0 * 60 * max(1.0, math.log2(n) - 5))
    state_bytes = 8.0 * (3 * dim + 8)  # x, v, a, and eight scalars
    out_bytes = 8.0 * (2 * dim + 2)
    return {"bytes": n * (evals * 2 * state_bytes + out_bytes + 8.0 * (2 * dim + 4)), "flops": flops}


# ------------------------------------------------------------- 64-bit values
# The same sums in plain FP64 torch over explicit pair lists.  Self-gravity
# is left out (None): its value is that of one particular Barnes-Hut tree.

PAIR_CHUNK = 1 << 25


def _pairs(x, radius, lo, length):
    """Index pairs (i, j), j = i left out, with |x_i - x_j| < max(radius_i,
    radius_j), in the periodic box [lo, lo + length) or, length None, open."""
    n, dim = x.shape
    dev = x.device
    r2 = radius * radius
    per = length is not None

    def close(i, j):
        d = x[i] - x[j]
        if per:
            d = d - length * torch.round(d / length)
        keep = (d.square().sum(1) < torch.maximum(r2[i], r2[j])) & (i != j)
        return i[keep], j[keep]

    if not per:
        lo = x.min(0).values
        extent = (x.max(0).values - lo).clamp_min(1e-300) * (1 + 1e-9)
    else:
        extent = length
    nc = (extent / radius.max()).floor().clamp(1, 512).to(torch.int64)
    if per:
        nc = torch.where(nc < 3, torch.ones_like(nc), nc)
    cell = ((x - lo) / extent * nc).floor().to(torch.int64)
    cell = torch.minimum(cell.clamp_min(0), nc - 1)
    stride = torch.ones(dim, dtype=torch.int64, device=dev)
    for k in range(1, dim):
        stride[k] = stride[k - 1] * nc[k - 1]
    flat, order = (cell * stride).sum(1).sort()
    total = int(nc.prod())
    begin = torch.searchsorted(flat, torch.arange(total + 1, device=dev))
    shifts = [[0] if per and int(nc[k]) == 1 else [-1, 0, 1] for k in range(dim)]
    grids = torch.meshgrid(*[torch.tensor(s, device=dev) for s in shifts], indexing="ij")
    got_i, got_j = [], []
    for off in torch.stack([g.reshape(-1) for g in grids], 1):
        other = cell + off
        ok = torch.ones(n, dtype=torch.bool, device=dev)
        if per:
            other = torch.remainder(other, nc)
        else:
            ok = ((other >= 0) & (other < nc)).all(1)
        f = torch.where(ok, (other * stride).sum(1), torch.zeros_like(flat))
        count = torch.where(ok, begin[f + 1] - begin[f], torch.zeros_like(f))
        ends = count.cumsum(0)
        at = 0
        while at < n:  # particles at .. to - 1: up to PAIR_CHUNK candidates
            done = int(ends[at - 1]) if at else 0
            to = max(at + 1, int(torch.searchsorted(ends, done + PAIR_CHUNK)))
            c = count[at:to]
            i = torch.repeat_interleave(torch.arange(at, to, device=dev), c)
            first = torch.repeat_interleave(begin[f[at:to]] - (c.cumsum(0) - c), c)
            i, j = close(i, order[first + torch.arange(i.numel(), device=dev)])
            got_i.append(i)
            got_j.append(j)
            at = to
    return torch.cat(got_i), torch.cat(got_j)


class _Kernel:
    """W, dW/dr / r and dW/dh of the two SPH kernels (support h)."""

    def __init__(self, kernel, dim):
        self.wendland, self.dim = kernel == WENDLAND, dim
        if self.wendland:
            self.sigma = {2: 9 / math.pi, 3: 495 / (32 * math.pi)}[dim]
        else:
            self.sigma = {1: 2 / 3, 2: 10 / (7 * math.pi), 3: 1 / math.pi}[dim]

    def phi(self, q):
        """The profile and its derivative: W = sigma h^-D phi(r / h)."""
        if self.wendland:
            t = (1 - q).clamp_min(0)
            return t ** 6 * (1 + 6 * q + 35 / 3 * q * q), -56 / 3 * q * t ** 5 * (1 + 5 * q)
        s = 2 * q
        a, b = (2 - s).clamp_min(0), (1 - s).clamp_min(0)
        f = 2.0 ** self.dim
        return f * (0.25 * a ** 3 - b ** 3), 2 * f * (-0.75 * a * a + 3 * b * b)

    def w(self, r, h):
        return self.sigma / h ** self.dim * self.phi(r / h)[0]

    def dw(self, r, h):
        return self.sigma / h ** (self.dim + 1) * self.phi(r / h)[1] / r

    def dh(self, r, h):
        p, dp = self.phi(r / h)
        return -self.sigma / h ** (self.dim + 1) * (self.dim * p + r / h * dp)


class _Sph:
    """One state and its evaluation."""

    def __init__(self, p, f, dev):
        t = lambda k: torch.as_tensor(f[k], dtype=torch.float64, device=dev)  # noqa: E731
        self.p, self.dim = p, int(p.dim)
        self.x, self.v, self.m, self.u, self.rho = t("pos"), t("vel"), t("mass"), t("ene"), t("dens")
        self.kern = _Kernel(p.kernel, self.dim)
        self.lo = self.len = None
        if p.periodic_is_valid:
            lo, hi = ([a[k] for k in range(self.dim)] for a in (p.range_min, p.range_max))
            self.lo = torch.tensor(lo, dtype=torch.float64, device=dev)
            self.len = torch.tensor(hi, dtype=torch.float64, device=dev) - self.lo
        self.unit = {1: 2.0, 2: math.pi, 3: 4 * math.pi / 3}[self.dim]
        self.alpha = torch.full_like(self.m, p.av_alpha)
        self.bal = torch.ones_like(self.m)
        self.dt = 0.0

    def sep(self, i, j):
        d = self.x[i] - self.x[j]
        if self.len is not None:
            d = d - (self.len * torch.round(d / self.len)).detach()
        return d, d.square().sum(1).sqrt()

    def guess(self):
        return (self.p.neighbor_number * self.m / (self.rho * self.unit)) ** (1 / self.dim)

    def sound(self):
        g = self.p.gamma
        return (g * (g - 1) * self.u).sqrt()

    def smooth(self):
        """The one-off initial smoothing."""
        h = self.guess()
        i, j = _pairs(self.x, h, self.lo, self.len)
        r = self.sep(i, j)[1]
        k = r < h[i]
        i, j, r = i[k], j[k], r[k]
        rho = self.m * self.kern.w(torch.zeros_like(h), h)
        self.rho = rho.index_add(0, i, self.m[j] * self.kern.w(r, h[i]))

    def lists(self):
        """The search radius and the pairs within it of either particle."""
        with torch.no_grad():
            self.radius = self.guess() * (1.2 if self.p.iterative_sml else 1.0)
            i, j = _pairs(self.x, self.radius, self.lo, self.len)
            self.ij = (i, j)

    def chunks(self):
        i, j = self.ij
        if torch.is_grad_enabled():
            yield i, j
            return
        for a in range(0, i.numel(), PAIR_CHUNK):
            yield i[a:a + PAIR_CHUNK], j[a:a + PAIR_CHUNK]

    def gather(self, h, term, width):
        """sum_j term(i, j, d, r) over r < min(h_i, radius_i), per particle."""
        out = [torch.zeros_like(self.m) for _ in range(width)]
        for i, j in self.chunks():
            d, r = self.sep(i, j)
            k = (r < h[i]) & (r < self.radius[i])
            i, j, d, r = i[k], j[k], d[k], r[k]
            out = [o.index_add(0, i, t) for o, t in zip(out, term(i, j, d, r))]
        return out

    def solve_h(self):
        p, dim, kern = self.p, self.dim, self.kern
        number = p.sph_type == DISPH
        wt = torch.ones_like(self.m) if number else self.m
        b = p.neighbor_number / self.unit * wt
        zero = torch.zeros_like(self.m)

        def sums(h):
            s, ds = self.gather(h, lambda i, j, d, r: (wt[j] * kern.w(r, h[i]), wt[j] * kern.dh(r, h[i])), 2)
            return s + wt * kern.w(zero, h), ds + wt * kern.dh(zero, h)

        with torch.no_grad():
            guess = self.radius / (1.2 if p.iterative_sml else 1.0)
            h = guess.clone()
            if not p.iterative_sml:
                return h
            done = torch.zeros_like(h, dtype=torch.bool)
            for _ in range(10):
                s, ds = sums(h)
                step = (s * h ** dim - b) / (ds * h ** dim + dim * s * h ** (dim - 1))
                new = torch.where(done, h, h - step)
                done = done | ((new - h).abs() < (new + h) * 1e-4)
                h = new
                if bool(done.all()):
                    break
            h = torch.where(done, h, guess)
        if torch.is_grad_enabled():
            # the derivative of h through the equation that it solves
            s, ds = sums(h)
            g = s * h ** dim - b
            h = h - (g - g.detach()) / (ds * h ** dim + dim * s * h ** (dim - 1)).detach()
        return h

    def evaluate(self):
        p, dim, kern, m, v, u = self.p, self.dim, self.kern, self.m, self.v, self.u
        gm1 = p.gamma - 1
        disph, gsph = p.sph_type == DISPH, p.sph_type == GSPH
        c = self.sound()
        h = self.solve_h()
        zero = torch.zeros_like(m)
        w0, dh0 = kern.w(zero, h), kern.dh(zero, h)
        wt = m * u if disph else m

        def dot(a, b):
            return (a * b).sum(1)

        def first(i, j, d, r):
            w, dh = kern.w(r, h[i]), kern.dh(r, h[i])
            return m[j] * w, wt[j] * w, wt[j] * dh, w, dh

        rho, s, ds, num, dnum = self.gather(h, first, 5)
        rho, s, ds, num, dnum = rho + m * w0, s + wt * w0, ds + wt * dh0, num + w0, dnum + dh0
        one = torch.ones_like(m)
        self.count = self.gather(h, lambda i, j, d, r: (one[j],), 1)[0] + 1
        pres = gm1 * s if disph else gm1 * rho * u
        x = h / (dim * num)
        gradh = x * ds / (1 + x * dnum) if disph else 1 / (1 + h / (dim * rho) * ds)
        vsig = 2 * c.detach()
        for i, j in self.chunks():
            d, r = (t.detach() for t in self.sep(i, j))
            k = (r < h[i]) & (r < self.radius[i])
            i, j, d, r = i[k], j[k], d[k], r[k]
            vs = (c[i] + c[j] - 3 * dot(d, v[i] - v[j]) / r).detach()
            vsig = vsig.scatter_reduce(0, i, vs, "amax")
        self.hvs = float((h.detach() / vsig).min())
        grads = None
        if gsph and p.gsph_is_2nd_order:
            def slopes(i, j, d, r):
                g = d * (kern.dw(r, h[i]) * m[j])[:, None]
                du, dv = u[j] - u[i], v[j] - v[i]
                return ([g[:, k] for k in range(dim)] + [g[:, k] * du for k in range(dim)] +
                        [g[:, k] * dv[:, a] for a in range(dim) for k in range(dim)])
            q = torch.stack(self.gather(h, slopes, 2 * dim + dim * dim), 1)
            gd, gu = q[:, :dim], q[:, dim:2 * dim]
            grads = gd, (gd * u[:, None] + gu) * gm1, (q[:, 2 * dim:] / rho[:, None]).reshape(-1, dim, dim)
        elif not gsph and (p.av_use_balsara_switch or p.av_use_time_dependent):
            def shear(i, j, d, r):
                dv = v[i] - v[j]
                g = d * (kern.dw(r, h[i]) * wt[j])[:, None]
                cr = []
                if dim == 3:
                    cr = list(torch.linalg.cross(dv, g, dim=1).unbind(1))
                elif dim == 2:
                    cr = [dv[:, 0] * g[:, 1] - dv[:, 1] * g[:, 0]]
                return [-dot(dv, g)] + cr
            q = self.gather(h, shear, {1: 1, 2: 2, 3: 4}[dim])
            norm = gm1 / pres if disph else 1 / rho
            div = q[0] * norm
            if p.av_use_balsara_switch and dim > 1:
                rot2 = sum(t * t for t in q[1:])
                rot = torch.where(rot2 > 0, rot2.clamp_min(1e-300), torch.ones_like(rot2)).sqrt() * (rot2 > 0) * norm.abs()
                self.bal = div.abs() / (div.abs() + rot + 1e-4 * c / h)
            if p.av_use_time_dependent:
                tau, src = p.av_epsilon * c / h, (-div).clamp_min(0)
                if p.av_use_balsara_switch and dim > 1:
                    self.alpha = self.alpha + (-(self.alpha - p.av_alpha_min) * tau + src * (p.av_alpha_max - self.alpha)) * self.dt
                else:
                    self.alpha = ((self.alpha + self.dt * tau * p.av_alpha_min + src * self.dt * p.av_alpha_max) /
                                  (1 + self.dt * tau + src * self.dt))
        self.h, self.rho, self.pres = h, rho, pres
        acc, du = [zero] * dim, zero
        for i, j in self.chunks():
            d, r = self.sep(i, j)
            k = r < torch.maximum(h[i], h[j])
            i, j, d, r = i[k], j[k], d[k], r[k]
            dwi, dwj = d * kern.dw(r, h[i])[:, None], d * kern.dw(r, h[j])[:, None]
            dv = v[i] - v[j]
            if gsph:
                e = d / r[:, None]
                vi, vj = dot(v[i], e), dot(v[j], e)
                if grads is not None:
                    fi, fj = (0.5 * (1 - c[t] * self.dt / r) for t in (i, j))

                    def limited(a, b):
                        return torch.where(a * b > 0, 2 * a * b / torch.where(a * b > 0, a + b, torch.ones_like(a)), torch.zeros_like(a))

                    gd, gp, gv = grads

                    def sides(qi, qj, si, sj):
                        return qi - limited(qi - qj, si * r) * fi, qj + limited(qi - qj, sj * r) * fj

                    ri, rj = sides(rho[i], rho[j], dot(gd[i], e), dot(gd[j], e))
                    pi, pj = sides(pres[i], pres[j], dot(gp[i], e), dot(gp[j], e))
                    vi, vj = sides(vi, vj, *(dot((gv[t] * e[:, None, :]).sum(2), e) for t in (i, j)))
                    ci, cj = (p.gamma * pi / ri).sqrt(), (p.gamma * pj / rj).sqrt()
                else:
                    ri, rj, pi, pj, ci, cj = rho[i], rho[j], pres[i], pres[j], c[i], c[j]
                sl, sr = rj.sqrt(), ri.sqrt()
                ut, ct = (sl * vj + sr * vi) / (sl + sr), (sl * cj + sr * ci) / (sl + sr)
                left, right = torch.minimum(vj - cj, ut - ct), torch.maximum(vi + ci, ut + ct)
                c1, c2 = rj * (left - vj), ri * (right - vi)
                c4, c5 = pj - vj * c1, pi - vi * c2
                vstar, pstar = (c5 - c4) / (c1 - c2), (c1 * c5 - c2 * c4) / (c1 - c2)
                f = dwi * (m[j] * pstar / rho[i] ** 2)[:, None] + dwj * (m[j] * pstar / rho[j] ** 2)[:, None]
                de = -dot(f, e * vstar[:, None] - v[i])
            else:
                vr = dot(dv, d)
                w = vr / r
                visc = torch.where(vr < 0, -0.5 * (self.bal[i] + self.bal[j]) / 2 * (self.alpha[i] + self.alpha[j]) / 2 *
                                   (c[i] + c[j] - 3 * w) * w * 2 / (rho[i] + rho[j]), torch.zeros_like(w))
                if disph:
                    ai = gm1 * gm1 * u[i] * u[j] / pres[i] * (1 - gradh[i] / (m[j] * u[j]))
                    aj = gm1 * gm1 * u[i] * u[j] / pres[j] * (1 - gradh[j] / (m[i] * u[i]))
                else:
                    ai, aj = pres[i] / rho[i] ** 2 * gradh[i], pres[j] / rho[j] ** 2 * gradh[j]
                f = dwi * (m[j] * (ai + 0.5 * visc))[:, None] + dwj * (m[j] * (aj + 0.5 * visc))[:, None]
                de = m[j] * ai * dot(dv, dwi) + 0.5 * m[j] * visc * dot(dv, 0.5 * (dwi + dwj))
            acc = [a.index_add(0, i, -f[:, k]) for k, a in enumerate(acc)]
            du = du.index_add(0, i, de)
        self.acc, self.du = torch.stack(acc, 1), du

    def step(self, dt=None):
        p = self.p
        if dt is None:
            a = self.acc.square().sum(1).sqrt()
            dt = min(p.cfl_sound * self.hvs, p.cfl_force * float((self.h / a)[a > 0].sqrt().min()))
        self.dt = dt
        vp, up = self.v + 0.5 * dt * self.acc, self.u + 0.5 * dt * self.du
        self.x = self.x + vp * dt
        if self.lo is not None:
            self.x = self.x + self.len * ((self.x < self.lo).double() - (self.x > self.lo + self.len).double())
        self.v, self.u = self.v + self.acc * dt, self.u + self.du * dt
        self.lists()
        self.evaluate()
        self.v, self.u = vp + 0.5 * dt * self.acc, up + 0.5 * dt * self.du
        return dt


def _exact_rollout(case, p, f):
    from torch.utils.checkpoint import checkpoint
    dev = torch.device("cuda")
    # what the call is given: the state in the tensors' own type
    if case["precision"] == "mixed":
        f = dict(f, **{k: f[k].astype(np.float32).astype(np.float64) for k in ("pos", "vel", "ene")})
    s = _Sph(p, f, dev)
    mass = s.m.to(torch.float32).double() if case["precision"] == "mixed" else s.m
    start = [t.clone().requires_grad_(True) for t in (s.x, s.v, s.u)]
    s.x, s.v, s.u = start
    with torch.no_grad():
        s.smooth()
    names = ("x", "v", "u", "acc", "du")

    def begin(x, v, u):
        s.x, s.v, s.u = x, v, u
        s.lists()
        s.evaluate()
        return s.acc, s.du

    def one(x, v, u, acc, du, rho):
        s.x, s.v, s.u, s.acc, s.du, s.rho = x, v, u, acc, du, rho
        s.step(ROLLOUT_DT)
        return s.x, s.v, s.u, s.acc, s.du, s.rho

    rho0 = s.rho
    first = lambda x, v, u: (setattr(s, "rho", rho0), begin(x, v, u))[1]  # noqa: E731
    acc, du = checkpoint(first, *start, use_reentrant=False)
    state = (*start, acc, du)
    rho = s.rho.detach()
    for _ in range(case["steps"]):
        *state, rho = checkpoint(one, *state, rho, use_reentrant=False)
        rho = rho.detach()
    x, v, u = state[:3]
    (mass[:, None] * v * v).sum().backward()
    return dict(pos=x.detach(), vel=v.detach(), ene=u.detach(), g_pos=start[0].grad, g_vel=start[1].grad, g_ene=start[2].grad)


def exact(case, seed):
    if case["do"] == "timestep":
        sml, acc, hvs = _timestep_arrays(case, seed)
        a = acc.square().sum(0).sqrt()
        return torch.minimum(0.3 * hvs, 0.125 * (sml / a)[a > 0].sqrt().min().reshape(1))
    if case.get("ic") == "evrard":
        return None
    p, f = _initial(case, seed)
    if case["do"] == "rollout":
        return _exact_rollout(case, p, f)
    with torch.no_grad():
        s = _Sph(p, f, torch.device("cuda"))
        s.smooth()
        s.lists()
        s.evaluate()
        time = 0.0
        for _ in range(case["steps"]):
            time += s.step()
        if not case["steps"]:
            out = dict(acc=s.acc, dene=s.du, dens=s.rho, pres=s.pres, sml=s.h, neighbor=s.count.to(torch.int32))
            if case["precision"] == "mixed":
                del out["neighbor"]
            return out
        kin, therm = float((0.5 * s.m * s.v.square().sum(1)).sum()), float((s.m * s.u).sum())
        return dict(pos=s.x, vel=s.v, dens=s.rho, ene=s.u, time=np.array(time), energy=np.array([kin, therm, 0.0, kin + therm]))
