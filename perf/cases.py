"""The work that a user of this framework has it do, as cases to be measured.

A user's program builds a scene (mphimplicit_amd.scenes or a *.grid file), hands it to
Scene or Batch, advances it and reads the fields back.  The cases are that, over the
range of the repository's own scenes, tests and benchmark: from the smallest pool (a
few hundred particles, where launches count) to the million-particle slab of
bench.py; 2D and 3D; both operator forms and the mixed-precision solve; one scene, a
batch, and one request of the serving loop from creation to result; the particle
matrix applied on its own.  Pools fill their tank's width and come to rest, so that a
scene that is stepped on and on keeps doing the same work.
"""
import functools
import math

import numpy as np
import torch

from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Batch, Scene, lib

L0 = 0.01
FORMS = {"assembled": abi.OPERATOR_ASSEMBLED, "factored": abi.OPERATOR_FACTORED}
PRECISIONS = {"fp64": abi.PRECISION_FP64, "mixed": abi.PRECISION_MIXED}


def _case(name, kind, layout, dim, nx, ny, nz=0, form="factored", precision="fp64", tol=1e-16, mu=0.1, steps=1,
          members=0, multigrid=1):
    return {"name": name, "kind": kind, "layout": layout, "dim": dim, "nx": nx, "ny": ny, "nz": nz, "form": form,
            "precision": precision, "tol": tol, "mu": mu, "steps": steps, "members": members,
            "multigrid": multigrid}


def listed():
    return [
        # the smallest 3D scene of the tests as a pool: every launch and wait counts
        _case("pool 3d 6x6x6", "step", "pool", 3, 6, 6, 6, tol=1e-12, steps=4),
        # the 2D configuration (box of 100 x 60 cells) at the library's default form and
        # stop rule, an interactive 2D run
        _case("pool 2d 100x41 assembled", "step", "pool", 2, 100, 41, form="assembled", tol=1e-12, steps=4),
        # one request of the serving loop near its lower size: scene in, three steps,
        # fields out; creation and release are part of what the user waits for
        _case("request 3d 17x17x17", "request", "pool", 3, 17, 17, 17, mu=0.5, steps=3),
        # an output step of a run with surface tension and two fluids: the step, the
        # pressures and virial stresses, every field of a *.vtk file read back
        _case("frame 3d 21x19x23", "frame", "pool", 3, 21, 19, 23, form="assembled", tol=1e-12, mu=0.01),
        # the batched workload: 12 scenes of 2k to 20k fluid particles, 2D and 3D
        _case("batch of 12", "batch", "sweep", 3, 2000, 20000, members=12),
        # the 64,000-particle drop (118,016 wall particles) in the factored form, in the
        # bit-exact assembled form (the library's default) and in mixed precision
        _case("drop 3d 64k factored", "step", "drop", 3, 40, 80, 16, steps=2),
        _case("drop 3d 64k assembled", "step", "drop", 3, 40, 80, 16, form="assembled", tol=1e-12, steps=2),
        _case("drop 3d 64k mixed", "step", "drop", 3, 40, 80, 16, precision="mixed", steps=2),
        # the largest 2D scene of the tests
        _case("pool 2d 400x400", "step", "pool", 2, 400, 400, steps=2),
        # the particle matrix alone on device arrays, for a caller's own Krylov solver
        _case("product 3d 63x61x59", "product", "pool", 3, 63, 61, 59, mu=1.0),
        # a ragged slab in the assembled form: the largest that solves on stored blocks
        _case("pool 3d 57x71x49 assembled", "step", "pool", 3, 57, 71, 49, form="assembled", mu=1.0),
        # the benchmark's scene: 1,000,000 fluid particles in a closed box, to 1e-8
        _case("slab 3d 1M", "step", "slab", 3, 100, 140, mu=1.0, steps=3),
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    kind = rng.choice(["step", "step", "step", "step", "product", "request", "batch"])
    dim = rng.choice([2, 3, 3])
    mu = float("%.3g" % log(0.01, 10.0))
    if kind == "batch":
        lo = int(log(500, 4000))
        return _drawn("batch", "sweep", 3, lo, int(lo * log(2, 10)), mu=mu, members=rng.randint(2, 12),
                      form=rng.choice(["factored", "factored", "assembled"]))
    form = rng.choice(["factored", "factored", "assembled"])
    precision = rng.choice(["fp64", "fp64", "fp64", "mixed"])
    nf = log(400, 20000 if kind == "request" else 250000)
    side = nf ** (1.0 / dim)
    nx, ny = max(5, round(side * log(0.7, 1.4))), max(5, round(side * log(0.7, 1.4)))
    nz = max(5, round(nf / (nx * ny))) if dim == 3 else 0
    if dim == 2:
        ny = max(5, round(nf / nx))
    tol = rng.choice([1e-12, 1e-16])
    multigrid = 0 if kind == "step" and nf < 5000 and rng.random() < 0.15 else 1
    return _drawn(kind, "pool", dim, nx, ny, nz, form, precision, tol, mu, rng.randint(1, 3), 0, multigrid)


def _drawn(*args, **kw):
    c = _case("", *args, **kw)
    del c["name"]
    return c


# ---- scenes -----------------------------------------------------------------


@functools.lru_cache(maxsize=4)
def _lattice(layout, dim, nx, ny, nz):
    """A pool's fluid and wall lattice and its domain: the fluid fills the floor of an
    open tank of 4 wall layers with 6 cells of freeboard."""
    n = [nx, ny, nz][:dim]
    inner = list(n)
    inner[dim - 1] += 6
    fluid = scenes.lattice([0] * 3, n + [0] * (3 - dim), L0, dim)
    walls = scenes.box_walls([0] * dim, inner, 4, L0, dim, open_top=True)
    lo = [-9 * L0] * dim + [-0.05] * (3 - dim)
    hi = [(m + 9) * L0 for m in inner] + [0.05] * (3 - dim)
    for d in range(dim):  # a width of whole cells may round to a search over two (box_scene)
        w = hi[d] - lo[d]
        r = 3.5 * L0
        if math.ceil(r / (w / math.floor(w / r))) > 1:
            hi[d] += 0.5 * L0
    return fluid, walls, lo, hi


def _params(case, p):
    p.operator_form = FORMS[case["form"]]
    p.precision = PRECISIONS[case["precision"]]
    p.cr_tolerance = case["tol"]
    p.multigrid = case["multigrid"]
    p.end_time = 1.0e9
    return p


def _scene(case, seed):
    """(params, grid) of a case's scene; the seed moves the fluid's jitter."""
    dim, nx, ny, nz = case["dim"], case["nx"], case["ny"], case["nz"]
    if case["layout"] == "drop":
        p, g = scenes.config_3d_drop(n=nx, box=ny, lift=nz, seed=seed, mu=case["mu"])
    elif case["layout"] == "slab":
        p, g = scenes.config_3d_slab(n=nx, inner=ny, seed=seed, mu=case["mu"])
    else:
        fluid, walls, lo, hi = _lattice("pool", dim, nx, ny, nz)
        p = scenes.base_params(dim, case["mu"], (0.0, -9.8, 0.0) if dim == 2 else (0.0, 0.0, -9.8), 5.0e-4, 2)
        g = scenes.assemble(fluid, walls, 0.0, L0, lo, hi, seed, dim)
    if case["kind"] == "frame":
        half = g.pos[:, 0] < 0.5 * nx * L0
        g.type[(g.type == 0) & half] = 1
        for t in (0, 1):
            p.surface_tension[t] = 0.07
        p.density[1] = 500.0
        p.interaction_ratio[0][1] = p.interaction_ratio[1][0] = 0.5
        p.vtk_output_interval = p.dt
    return _params(case, p), g


def _sweep(case, seed):
    """The members of a batch: the batched workload's scenes with fluid counts spread
    over nx..ny."""
    for s in range(case["members"]):
        p, g = scenes.batch_sweep_member(s, seed0=1000, nf_range=(case["nx"], case["ny"]))
        fluid = g.type < 2
        d = 2 if p.dim == 2 else 3
        u = scenes.splitmix64_uniform(seed + 31 * s, int(fluid.sum()) * d).reshape(-1, d)
        g.pos[fluid, :d] += (2.0 * u - 1.0) * (0.01 * L0)
        yield _params(case, p), g


# ---- one pass ---------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        members = [Scene(p, g) for p, g in _sweep(case, seed)]
        b = Batch()
        for s in members:
            b.add(s)
        return {"kind": kind, "batch": b, "members": members}
    p, g = _scene(case, seed)
    if kind == "request":
        return {"kind": kind, "params": p, "grid": g, "steps": case["steps"]}
    s = Scene(p, g)
    if kind == "product":
        for phase in range(abi.PHASE_KINEMATICS, abi.PHASE_MULTIPLY_C + 1):
            s.run_phase(phase)
        return {"kind": kind, "scene": s, "x": _vector(case, seed, int(s.scalar("FluidCount"))),
                "y": torch.empty(3 * int(s.scalar("FluidCount")), dtype=torch.float64, device="cuda"),
                "precision": PRECISIONS[case["precision"]]}
    return {"kind": kind, "scene": s, "steps": case["steps"]}


def _vector(case, seed, nf):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(3 * nf, dtype=torch.float64, device="cuda", generator=gen)


def _fields(s, names=("Velocity", "Position", "ParticleIndex")):
    return {n: s.read(n) for n in names}


def run(state):
    kind = state["kind"]
    if kind == "step":
        state["scene"].step(state["steps"])
        return _fields(state["scene"])
    if kind == "frame":
        state["scene"].step(1)
        return _fields(state["scene"], ("Velocity", "Position", "Force", "VolStrainP", "DivergenceP", "PressureP",
                                        "VirialPressureAtParticle", "Property", "NeighborCount"))
    if kind == "product":
        rc = lib().mph_scene_apply_matrix_noalloc(state["scene"].h, state["precision"], state["x"].data_ptr(),
                                                  state["y"].data_ptr())
        if rc:
            raise RuntimeError(lib().mph_last_error().decode())
        return state["y"]
    if kind == "request":
        with Scene(state["params"], state["grid"]) as s:
            s.step(state["steps"])
            return _fields(s)
    state["batch"].step()
    return [_fields(s, ("Velocity", "Position")) for s in state["members"]]


def _counts(case):
    """(fluid, all particles, neighbours per fluid particle, CR iterations) of each scene."""
    if case["kind"] == "batch":
        for s in range(case["members"]):
            u = scenes.splitmix64_uniform(1000 + s + 0x5EED, 6)
            nf = math.exp(math.log(case["nx"]) + u[1] * math.log(case["ny"] / case["nx"]))
            dim = 2 if u[0] < 0.5 else 3
            f, n = scenes.box_scene_counts(dim, int(nf))
            yield f, n, 38 if dim == 2 else 180, 30
        return
    dim, nx, ny, nz = case["dim"], case["nx"], case["ny"], case["nz"]
    iters = 60 if case["tol"] < 1e-14 else 40
    if case["layout"] == "drop":
        yield nx ** 3, nx ** 3 + ny ** 3 - (ny - 8) ** 2 * (ny - 4), 180, iters
    elif case["layout"] == "slab":
        yield nx ** 3, nx ** 3 + (ny + 8) ** 3 - ny ** 3, 180, iters
    elif dim == 2:
        yield nx * ny, nx * ny + (nx + 8) * (ny + 10) - nx * (ny + 6), 38, iters
    else:
        yield nx * ny * nz, nx * ny * nz + (nx + 8) * (ny + 8) * (nz + 10) - nx * ny * (nz + 6), 180, iters


def work(case):
    """What a pass cannot do without.  Per step: the state read and written (position,
    velocity, type, index) and, for each of a typical number of CR iterations, the six
    solver vectors read and written once; for a product: positions, x and y.  Flops: a
    pair's displacement, weight and 3x3 term once per step (40) and its share of every
    product (16)."""
    b = f = 0.0
    for nf, n, neigh, iters in _counts(case):
        if case["kind"] == "product":
            b += 24 * n + 48 * nf
            f += 16 * nf * neigh
        else:
            steps = max(1, case["steps"])
            b += steps * (112 * n + iters * 6 * 48 * nf)
            f += steps * (40 * nf * neigh + iters * 16 * nf * neigh)
    return {"bytes": b, "flops": f}


# ---- the same in plain torch and numpy, 64 bits ------------------------------
# The discretisation as published with the reference: for particles i, j at distance d
# the weights w_p (radius P), w_v (radius V), both K (1 - d/h)^2; the matrix
#   A = m/(V dt) + viscous blocks + C lambda C^T,   b = m/(V dt) v + ... - C P.
# Walls at rest, no surface tension.  Fields come in the order that the reference's
# bitonic network leaves the particles in.


def exact(case, seed):
    if case["kind"] in ("frame", "batch"):
        return None
    nf = next(iter(_counts(case)))[0]
    if nf > 70000 and case["kind"] != "product" or case["steps"] > 4 or nf > 260000:
        return None
    p, g = _scene(case, seed)
    m = _Exact(p, g)
    if case["kind"] == "product":
        m.move()
        m.assemble()
        return m.apply(_vector(case, seed, m.nf).reshape(-1, 3).to(m.dev)).reshape(-1)
    for _ in range(case["steps"]):
        m.move()
        m.assemble()
        m.solve()
    return {"Velocity": m.vel.reshape(-1), "Position": m.pos.reshape(-1), "ParticleIndex": None}


class _Exact:
    def __init__(self, p, g):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.dim, self.dt, l = p.dim, p.dt, g.spacing
        dim = self.dim
        self.V = l ** dim
        self.hP, self.hV = p.radius_ratio_p * l, p.radius_ratio_v * l
        self.h = max(p.radius_ratio_a * l, 2.0 * self.hP, self.hV)
        sw = (0.5 / 3.0 if dim == 2 else 2.0 / 15.0) * math.pi / l ** dim
        self.KP, self.KV = 1.0 / (sw * self.hP ** dim), 1.0 / (sw * self.hV ** dim)
        r = np.arange(-4, 5) * l
        q = np.sqrt(sum(a * a for a in np.meshgrid(*([r] * dim))))
        q = q[(q > 0) & (q * q <= self.hP * self.hP)]
        self.N0 = float((self.KP * (1.0 - q / self.hP) ** 2).sum())
        self.lo = np.array(g.domain_min, dtype=np.float64)
        self.W = np.array(g.domain_max, dtype=np.float64) - self.lo
        self.C = np.floor(self.W / self.h).astype(np.int64)
        if dim == 2:
            self.C[2] = 1
        self.type = np.array(g.type)
        self.pos, self.vel = np.array(g.pos, dtype=np.float64), np.array(g.vel, dtype=np.float64)
        self.p, self.nf = p, int((self.type < 2).sum())
        self._sort()

    def _sort(self):
        n, c = len(self.type), self.C
        k = np.floor((self.pos - self.lo) / (self.W / c)).astype(np.int64) % c
        key = (k[:, 0] * c[1] + k[:, 1]) * c[2] + k[:, 2]
        size = 1 << n.bit_length()
        keys = np.full(size, 2 * c.prod(), dtype=np.int64)
        keys[:n] = key + np.where(self.type >= 2, c.prod(), 0)
        t = torch.from_numpy(np.stack([keys, np.arange(size)], axis=1)).to(self.dev)
        for main in range(size.bit_length() - 1):
            for dist in (1 << b for b in range(main, -1, -1)):
                v = t.view(-1, 2, dist, 2)
                a, b = v[:, 0], v[:, 1]
                first = torch.arange(len(v), device=t.device) * 2 * dist
                up = (((first >> main) & 2) == 0)[:, None]
                swap = ((a[..., 0] > b[..., 0]) == up)[..., None]
                t = torch.stack([torch.where(swap, b, a), torch.where(swap, a, b)], dim=1).view(-1, 2)
        t = t[:n].cpu().numpy()
        self.cell, o = t[:, 0] % c.prod(), t[:, 1]
        self.type, self.pos, self.vel = self.type[o], self.pos[o], self.vel[o]

    def move(self):
        x = self.pos - self.lo
        x[: self.nf] = self.pos[: self.nf] + self.vel[: self.nf] * self.dt - self.lo
        self.pos = x - self.W * np.floor(x / self.W) + self.lo
        self._sort()

    def _pairs(self, pos):
        """Ordered pairs i (fluid) and j != i within the largest radius: i, j, r, d^2."""
        n, c, dev = len(self.type), torch.tensor(self.C, device=self.dev), self.dev
        cell = torch.from_numpy(self.cell).to(dev)
        order = torch.argsort(cell, stable=True)
        total = int(self.C.prod())
        start = torch.searchsorted(cell[order].contiguous(), torch.arange(total + 1, device=dev))
        fl = torch.arange(self.nf, device=dev)
        x = torch.stack([cell // (c[1] * c[2]), cell // c[2] % c[1], cell % c[2]], dim=1)[: self.nf]
        W = torch.tensor(self.W, device=dev)
        ii, jj, rr, dd = [], [], [], []
        for o in np.ndindex(3, 3, 3 if self.dim == 3 else 1):
            o = torch.tensor([o[0] - 1, o[1] - 1, o[2] - 1 if self.dim == 3 else 0], device=dev)
            y = (x + o) % c
            k = (y[:, 0] * c[1] + y[:, 1]) * c[2] + y[:, 2]
            cnt = start[k + 1] - start[k]
            i = torch.repeat_interleave(fl, cnt)
            at = torch.arange(len(i), device=dev) - torch.repeat_interleave(cnt.cumsum(0) - cnt, cnt)
            j = order[start[k][i] + at]
            r = pos[j] - pos[i]
            r = r - W * torch.round(r / W)
            d2 = (r * r).sum(1)
            keep = (d2 <= self.h * self.h) & (i != j)
            ii.append(i[keep]), jj.append(j[keep]), rr.append(r[keep]), dd.append(d2[keep])
        return torch.cat(ii), torch.cat(jj), torch.cat(rr), torch.cat(dd)

    def assemble(self):
        p, nf, n, dev = self.p, self.nf, len(self.type), self.dev
        pos = torch.from_numpy(self.pos).to(dev)
        typ = torch.from_numpy(self.type.astype(np.int64)).to(dev)
        i, j, r, d2 = self._pairs(pos)
        d = d2.sqrt()
        mu = torch.tensor(list(p.shear_viscosity), dtype=torch.float64, device=dev)[typ]
        self.lam = torch.tensor(list(p.bulk_viscosity), dtype=torch.float64, device=dev)[typ]
        # viscous: alpha r r^T, alpha = c mu_ij (-w_v')/d^3
        v = d < self.hV
        iv, jv, rv, dv = i[v], j[v], r[v], d[v]
        m = 2.0 * mu[iv] * mu[jv] / (mu[iv] + mu[jv])
        al = (8.0 if self.dim == 2 else 10.0) * m * self.KV * 2.0 / self.hV * (1.0 - dv / self.hV) / dv ** 3
        rho = torch.tensor(list(p.density), dtype=torch.float64, device=dev)[typ[:nf]]
        D = torch.zeros(nf, 9, dtype=torch.float64, device=dev)
        D.index_add_(0, iv, (al[:, None, None] * rv[:, :, None] * rv[:, None, :]).reshape(-1, 9))
        self.D = D.view(nf, 3, 3) + (rho / self.dt)[:, None, None] * torch.eye(3, dtype=torch.float64, device=dev)
        f = jv < nf
        self.visc = (iv[f], jv[f], rv[f], al[f])
        # pressure: C_ik = beta r_ik, C_ii = sum of them
        q = d < self.hP
        ip, jp, rp, dp = i[q], j[q], r[q], d[q]
        cp = rp * (self.KP * 2.0 / self.hP * (1.0 - dp / self.hP) / dp)[:, None]
        own = torch.zeros(nf, 3, dtype=torch.float64, device=dev).index_add_(0, ip, cp)
        self.C_ = (torch.cat([ip, torch.arange(nf, device=dev)]), torch.cat([jp, torch.arange(nf, device=dev)]),
                   torch.cat([cp, own]))
        w = self.KP * (1.0 - dp / self.hP) ** 2
        dens = torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, ip, w)
        wall = jp >= nf  # a wall's density: its fluid neighbours here, its walls below
        dens.index_add_(0, jp[wall], w[wall])
        dens[nf:] += self._wall_density(pos)
        s = dens - self.N0
        self.P = torch.where(s > 0, torch.tensor(list(p.bulk_modulus), dtype=torch.float64, device=dev)[typ] * s,
                             torch.zeros_like(s))
        self.rho = rho

    def _wall_density(self, pos):
        """Sum of w_p over the wall neighbours of each wall particle."""
        w = pos[self.nf :]
        out = torch.zeros(len(w), dtype=torch.float64, device=pos.device)
        W = torch.tensor(self.W, device=pos.device)
        for k in range(0, len(w), 256):
            # walls near this stretch only, by a slab along x
            a = w[k : k + 256]
            near = w[(w[:, 0] >= a[:, 0].min() - self.hP) & (w[:, 0] <= a[:, 0].max() + self.hP)]
            r = near[None] - a[:, None]
            r = r - W * torch.round(r / W)
            d = (r * r).sum(2).sqrt()
            out[k : k + 256] = torch.where((d > 0) & (d <= self.hP), self.KP * (1.0 - d / self.hP) ** 2,
                                           torch.zeros_like(d)).sum(1)
        return out

    def apply(self, x):
        i, j, r, al = self.visc
        y = (self.D @ x[:, :, None])[:, :, 0]
        y.index_add_(0, i, -(al * (r * x[j]).sum(1))[:, None] * r)
        i, k, c = self.C_
        t = torch.zeros(len(self.type), dtype=torch.float64, device=x.device).index_add_(0, k, (c * x[i]).sum(1))
        t = t * self.lam
        return y.index_add_(0, i, c * t[k][:, None])

    def solve(self):
        nf = self.nf
        g = np.array(list(self.p.gravity))
        v = self.vel[:nf] + g * self.dt
        x = torch.from_numpy(v).to(self.dev)
        b = (self.rho / self.dt)[:, None] * x
        i, k, c = self.C_
        b = b.index_add(0, i, -c * self.P[k][:, None])
        # conjugate gradients with the diagonal as preconditioner, to rounding
        diag = torch.diagonal(self.D, dim1=1, dim2=2).clone()
        diag.index_add_(0, i, c * c * self.lam[k][:, None])
        r = b - self.apply(x)
        z = r / diag
        q, rz = z.clone(), (r * z).sum()
        stop = 1e-13 * float(b.norm())
        for it in range(20000):
            aq = self.apply(q)
            a = rz / (q * aq).sum()
            x = x + a * q
            r = r - a * aq
            if it % 20 == 0 and float(r.norm()) < stop:
                break
            z = r / diag
            new = (r * z).sum()
            q, rz = z + (new / rz) * q, new
        self.vel[:nf] = x.cpu().numpy()
