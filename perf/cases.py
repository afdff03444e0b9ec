"""The work whose speed counts: what programs have this framework do, through
its Python entry points (lbm_amd.capi, lbm_amd.autograd).

A case is one of four kinds:
  flow     one domain: `steps` time steps, then the moments of every cell,
           as the driver's loop runs between two outputs;
  adjoint  the inverse problem: forward run and gradient with respect to the
           Brinkman porosity, on device tensors through torch.autograd;
  batch    many lid-driven cavities of uneven sizes stepped together, then
           the moments of each and the divergence flags;
  batchadj their kinetic energies and lid-velocity gradients.

`exact` restates the same physics in plain torch, in 64 bits.
"""
import math

import numpy as np
import torch

from lbm_amd import autograd, capi

SIZEOF = {"f64": 8, "f64s": 8, "f32": 4, "f16": 2, "bf16": 2}
LID = 0.05       # lid velocity of the cavities along x
INFLOW = 0.04    # inflow velocity of the channels along x
FORCE = 1e-5     # body acceleration of the inverse problem along x


def _flow(name, geom, q, storage, size, tau, steps, layout="ab"):
    return {"name": name, "kind": "flow", "geom": geom, "q": q, "storage": storage, "layout": layout,
            "xl": size[0], "yl": size[1], "zl": size[2], "tau": tau, "steps": steps}


def listed():
    return [
        # A small interactive run: few cells, output every ten steps; launches
        # and calls count more than bytes.
        _flow("cavity-16-f32", "cavity", 19, "f32", (16, 16, 16), 0.6, 10),
        # The reference's own use: its cavity scenario in fp64 (the default
        # storage, reference operation order) at 64^3, fields every 100 steps.
        _flow("cavity-64-f64", "cavity", 19, "f64", (64, 64, 64), 0.6, 100),
        # A production cavity in the fast storage.
        _flow("cavity-192-f32", "cavity", 19, "f32", (192, 192, 192), 0.6, 200),
        # The benchmark's decaying vortex, 256^3, fp32 and fp16 storage.
        _flow("box-256-f32", "box", 19, "f32", (256, 256, 256), 0.8, 600),
        _flow("box-256-f16", "box", 19, "f16", (256, 256, 256), 0.8, 600),
        # A ragged periodic box in the third storage format.
        _flow("box-ragged-bf16", "box", 19, "bf16", (131, 70, 97), 0.8, 100),
        # A vortex in the in-place layout, which halves the memory of a run.
        _flow("box-aa-f32", "box", 19, "f32", (200, 150, 170), 0.8, 200, layout="aa"),
        # Flow around obstacles with inflow and outflow, the finest lattice.
        _flow("channel-q27-f32", "spheres", 27, "f32", (192, 96, 96), 0.55, 100),
        # A pipe flow (250 x 54 x 54, the size of the reference's pipe) in
        # half the memory.
        _flow("pipe-q19-f16", "pipe", 19, "f16", (250, 54, 54), 0.6, 100),
        # One gradient of the 128^3 porosity inverse problem.
        {"name": "adjoint-128-f32", "kind": "adjoint", "q": 19, "storage": "f32", "n": 128, "nc": 32, "tau": 0.8,
         "steps": 100},
        # A parameter study: uneven cavities (16 to 96 cells a side) stepped
        # together, and their sensitivities to the lid.
        {"name": "batch-30-f32", "kind": "batch", "storage": "f32", "n": 30, "lmin": 16, "lmax": 96, "steps": 200},
        {"name": "batchadj-64-f32", "kind": "batchadj", "storage": "f32", "n": 64, "lmin": 16, "lmax": 96,
         "steps": 50},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow", "flow", "flow", "flow", "flow", "flow", "adjoint", "batch", "batchadj"])
    if kind == "flow":
        geom = rng.choice(["box", "box", "cavity", "cavity", "spheres", "pipe"])
        q = rng.choice([15, 19, 19, 19, 27])
        storage = rng.choice(["f64", "f32", "f32", "f32", "f16", "bf16"])
        layout = "aa" if rng.random() < 0.15 else "ab"
        lo = 12 if geom in ("box", "cavity") else 32
        size = [_log_int(rng, lo, 208) for _ in range(3)]
        if geom in ("spheres", "pipe"):
            size = [max(size), min(size[1], 112), min(size[2], 112)]
        steps = _log_int(rng, 5, 200)
        return {"kind": "flow", "geom": geom, "q": q, "storage": storage, "layout": layout, "xl": size[0],
                "yl": size[1], "zl": size[2], "tau": round(rng.uniform(0.56, 1.0), 3), "steps": steps}
    if kind == "adjoint":
        nc = rng.randint(8, 32)
        return {"kind": "adjoint", "q": rng.choice([15, 19, 19]), "storage": "f32", "n": 4 * nc + rng.randint(-3, 0),
                "nc": nc, "tau": round(rng.uniform(0.6, 1.0), 3), "steps": _log_int(rng, 10, 100)}
    if kind == "batch":
        return {"kind": "batch", "storage": rng.choice(["f32", "f32", "f16"]), "n": rng.randint(4, 31), "lmin": 16,
                "lmax": rng.randint(32, 96), "steps": _log_int(rng, 10, 200)}
    return {"kind": "batchadj", "storage": "f32", "n": rng.randint(4, 64), "lmin": 16, "lmax": rng.randint(32, 96),
            "steps": _log_int(rng, 10, 50)}


# ---------------------------------------------------------------------------
# Inputs, the same for the framework and for `exact`.

NOSLIP, MOVINGWALL, OUTFLOW, INFLOWBC = capi.NOSLIP, capi.MOVINGWALL, capi.OUTFLOW, capi.INFLOW
REST = (0.0, 0.0, 0.0, 1.0)


def _faces(xl, yl, zl):
    return {"x0": (0, 0, 0, yl + 1, 0, zl + 1), "xmax": (xl + 1, xl + 1, 0, yl + 1, 0, zl + 1),
            "y0": (0, xl + 1, 0, 0, 0, zl + 1), "ymax": (0, xl + 1, yl + 1, yl + 1, 0, zl + 1),
            "z0": (0, xl + 1, 0, yl + 1, 0, 0), "zmax": (0, xl + 1, 0, yl + 1, zl + 1, zl + 1)}


def _boundaries(geom, size):
    """(kind, params, box) in the order they are set; later boxes win."""
    f = _faces(*size)
    if geom == "box":
        return []
    if geom == "cavity":
        return [(NOSLIP, REST, f["z0"]), (MOVINGWALL, (LID, 0.0, 0.0, 1.0), f["zmax"])] + [
            (NOSLIP, REST, f[k]) for k in ("x0", "xmax", "y0", "ymax")]
    return [(NOSLIP, REST, f[k]) for k in ("z0", "zmax", "y0", "ymax")] + [
        (INFLOWBC, (INFLOW, 0.0, 0.0, 1.0), f["x0"]), (OUTFLOW, REST, f["xmax"])]


def _fluid_mask(case, seed):
    """(zl, yl, xl) bytes, 1 = fluid; None where all cells are."""
    xl, yl, zl = case["xl"], case["yl"], case["zl"]
    if case["geom"] == "pipe":
        y, z = np.arange(yl) - 0.5 * (yl - 1), np.arange(zl) - 0.5 * (zl - 1)
        r2 = (y[None, :] / (0.5 * yl)) ** 2 + (z[:, None] / (0.5 * zl)) ** 2
        return np.ascontiguousarray(np.broadcast_to((r2 <= 1.0)[:, :, None], (zl, yl, xl)).astype(np.uint8))
    if case["geom"] != "spheres":
        return None
    # spheres with radii of 6 to 12 cells until a fifth of the box is solid,
    # their centres clear of the inflow and outflow faces
    rng = np.random.default_rng(seed)
    solid = np.zeros((zl, yl, xl), dtype=bool)
    while solid.sum() < 0.2 * solid.size:
        cx, cy, cz, r = rng.uniform(14, xl - 14), rng.uniform(0, yl), rng.uniform(0, zl), rng.uniform(6, 12)
        lo = [max(0, int(c - r)) for c in (cz, cy, cx)]
        hi = [min(n, int(c + r) + 2) for c, n in ((cz, zl), (cy, yl), (cx, xl))]
        z, y, x = np.ogrid[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]]
        solid[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]] |= (x - cx) ** 2 + (y - cy) ** 2 + (z - cz) ** 2 <= r * r
    return (~solid).astype(np.uint8)


def _start_fields(geom, size, seed):
    """Density and velocity at the start, fp64 on the GPU: a Taylor-Green
    vortex in the periodic box, rest elsewhere, with density noise."""
    xl, yl, zl = size
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rho = torch.randn((zl, yl, xl), generator=gen, device="cuda", dtype=torch.float64).mul_(1e-4).add_(1.0)
    u = torch.zeros((zl, yl, xl, 3), device="cuda", dtype=torch.float64)
    if geom == "box":
        kx, ky = 2 * math.pi / xl, 2 * math.pi / yl
        x = torch.arange(xl, device="cuda", dtype=torch.float64)[None, None, :] * kx
        y = torch.arange(yl, device="cuda", dtype=torch.float64)[None, :, None] * ky
        top = 0.02 / max(kx, ky)
        u[..., 0] = top * ky * torch.sin(x) * torch.cos(y)
        u[..., 1] = -top * kx * torch.cos(x) * torch.sin(y)
    return rho, u


def _cavities(case):
    """(xl, yl, zl, tau) of the set: edges log-uniform, Reynolds numbers up to
    200 (the stable part of the range at these sizes)."""
    rng = np.random.default_rng(12345)
    lo, hi = math.log(case["lmin"]), math.log(case["lmax"])
    out = []
    for _ in range(case["n"]):
        size = [int(round(math.exp(rng.uniform(lo, hi)))) for _ in range(3)]
        out.append((*size, 3.0 * LID * size[0] / rng.uniform(10.0, 200.0) + 0.52))
    return out


def _porosity(case, seed):
    """(fine porosity on the GPU, target velocities of the middle plane)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n, nc = case["n"], case["nc"]
    coarse = torch.rand((nc, nc, nc), generator=gen, device="cuda", dtype=torch.float64)
    alpha = autograd.upsample_periodic(coarse, (n, n, n)).contiguous()
    target = torch.rand((n, n, 3), generator=gen, device="cuda", dtype=torch.float64) * 1e-4
    return alpha, target


def _domain(geom, q, storage, size, tau, layout="ab", mask=None):
    d = capi.Domain(*size, tau, q=q, storage=storage, periodic=(geom == "box",) * 3, layout=layout)
    if mask is not None:
        d.set_solid_mask(mask)
    for kind, params, box in _boundaries(geom, size):
        d.set_boundary_box(kind, params, *box)
    d.finalize()
    return d


# ---------------------------------------------------------------------------


def prepare(case, seed):
    if case["kind"] == "flow":
        size = (case["xl"], case["yl"], case["zl"])
        d = _domain(case["geom"], case["q"], case["storage"], size, case["tau"], case["layout"],
                    _fluid_mask(case, seed))
        rho, u = _start_fields(case["geom"], size, seed)
        d.init_equilibrium(rho.cpu().numpy(), u.cpu().numpy())
        return {"kind": "flow", "domain": d, "steps": case["steps"]}
    if case["kind"] == "adjoint":
        n = case["n"]
        alpha, target = _porosity(case, seed)
        d = capi.Domain(n, n, n, case["tau"], q=case["q"], storage=case["storage"], periodic=(True, True, True))
        d.set_brinkman(alpha.cpu().numpy(), (FORCE, 0.0, 0.0))
        d.finalize()
        tape = capi.Tape(d, case["steps"], capi.OBJ_PLANE_VELOCITY_MISFIT, plane_x=n // 2,
                         target_u=target.cpu().numpy())
        return {"kind": "adjoint", "alpha": alpha, "tape": tape, "objective": autograd.make_objective_function()}
    doms = []
    for i, (xl, yl, zl, tau) in enumerate(_cavities(case)):
        d = _domain("cavity", 19, case["storage"], (xl, yl, zl), tau)
        rho, u = _start_fields("cavity", (xl, yl, zl), seed + i)
        d.init_equilibrium(rho.cpu().numpy(), u.cpu().numpy())
        doms.append(d)
    batch = capi.Batch(doms)
    if case["kind"] == "batch":
        return {"kind": "batch", "domains": doms, "batch": batch, "steps": case["steps"]}
    return {"kind": "batchadj", "domains": doms, "batch": batch, "tape": capi.BatchTape(batch, case["steps"])}


def run(state):
    if state["kind"] == "flow":
        state["domain"].step(state["steps"])
        rho, u = state["domain"].moments()
        return {"rho": rho, "u": u}
    if state["kind"] == "adjoint":
        alpha = state["alpha"].detach().requires_grad_(True)
        j = state["objective"].apply(alpha, state["tape"])
        j.backward()
        return {"j": j.detach(), "grad": alpha.grad}
    if state["kind"] == "batch":
        state["batch"].step(state["steps"])
        state["batch"].sync()
        return {"moments": [d.moments() for d in state["domains"]], "diverged": state["batch"].status()}
    return {"j": state["tape"].forward(), "grad": state["tape"].backward()}


def work(case):
    """Each population read and written once per step, in its storage format;
    about 12 operations per population and 40 per cell of a collision."""
    if case["kind"] in ("flow", "adjoint"):
        q = case["q"]
        n = case["n"] ** 3 if case["kind"] == "adjoint" else case["xl"] * case["yl"] * case["zl"]
        if case.get("geom") == "spheres":
            n = int(0.8 * n)
        elif case.get("geom") == "pipe":
            n = int(math.pi / 4 * n)
    else:
        q, n = 19, sum(c[0] * c[1] * c[2] for c in _cavities(case))
    s, t = SIZEOF[case["storage"]], case["steps"]
    step_bytes, step_flops = 2 * q * s * n, (12 * q + 40) * n
    if case["kind"] in ("flow", "batch"):
        return {"bytes": step_bytes * t + 32 * n, "flops": step_flops * t}
    # forward, recompute, and an adjoint step that reads g and mu and writes mu
    return {"bytes": int(3.5 * step_bytes * t), "flops": 4 * step_flops * t}


# ---------------------------------------------------------------------------
# The same in plain torch, 64 bits.


def _lattice(q):
    c = [(x, y, z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
    w27 = {0: 8 / 27, 1: 2 / 27, 2: 1 / 54, 3: 1 / 216}
    w19 = {0: 1 / 3, 1: 1 / 18, 2: 1 / 36}
    w15 = {0: 2 / 9, 1: 1 / 9, 3: 1 / 72}
    w = {15: w15, 19: w19, 27: w27}[q]
    c = [v for v in c if sum(map(abs, v)) in w]
    return c, [w[sum(map(abs, v))] for v in c]


class _Reference:
    """One domain on the ghosted box, populations (Q, zl + 2, yl + 2, xl + 2)."""

    def __init__(self, geom, q, size, tau, cs2, mask=None):
        xl, yl, zl = size
        self.size, self.tau, self.cs2, self.periodic = size, tau, cs2, geom == "box"
        self.cl, self.wl = _lattice(q)
        self.q, dev = q, "cuda"
        self.c = torch.tensor(self.cl, dtype=torch.float64, device=dev)
        self.w = torch.tensor(self.wl, dtype=torch.float64, device=dev)
        owner = np.zeros((zl + 2, yl + 2, xl + 2), dtype=np.int64)
        bounds = _boundaries(geom, size)
        if mask is not None:
            owner[1:-1, 1:-1, 1:-1][mask == 0] = len(bounds) + 1
        for i, (_, _, (x0, x1, y0, y1, z0, z1)) in enumerate(bounds):
            owner[z0:z1 + 1, y0:y1 + 1, x0:x1 + 1] = i + 1
        bounds = bounds + [(NOSLIP, REST, None)]
        inner = np.zeros(owner.shape, dtype=bool)
        inner[1:-1, 1:-1, 1:-1] = owner[1:-1, 1:-1, 1:-1] == 0
        self.fluid = torch.from_numpy(inner[1:-1, 1:-1, 1:-1].copy()).to(dev)
        # links (b, q): b not fluid, x = b + c_q an interior fluid cell
        n = owner.size
        self.links = []  # kind, params, flat index of (q, b), of (qbar, x), of x, q
        fx = np.flatnonzero(inner)
        flat_owner = owner.reshape(-1)
        for kind in (NOSLIP, MOVINGWALL, INFLOWBC, OUTFLOW):
            ids = [i + 1 for i, b in enumerate(bounds) if b[0] == kind]
            if not ids or self.periodic:
                continue
            dst, src, cell, qs = [], [], [], []
            for k, v in enumerate(self.cl):
                b = fx - (v[0] + owner.shape[2] * (v[1] + owner.shape[1] * v[2]))
                hit = np.isin(flat_owner[b], ids)
                kb = self.cl.index((-v[0], -v[1], -v[2]))
                dst.append(b[hit] + k * n)
                src.append(fx[hit] + kb * n)
                cell.append(fx[hit])
                qs.append(np.full(int(hit.sum()), k))
            to = [torch.from_numpy(np.concatenate(a)).to(dev) for a in (dst, src, cell, qs)]
            self.links.append((kind, bounds[ids[0] - 1][1], *to))

    def rest(self):
        xl, yl, zl = self.size
        return self.w[:, None, None, None].expand(self.q, zl + 2, yl + 2, xl + 2).contiguous()

    def equilibrium(self, rho, u):
        cu = torch.tensordot(self.c, u, dims=([1], [-1])) / self.cs2
        uu = (u * u).sum(-1) / (2 * self.cs2)
        w = self.w.reshape((-1,) + (1,) * rho.dim())
        return w * rho * (1 + cu + 0.5 * cu * cu - uu)

    def start(self, rho, u):
        f = self.rest()
        i = f[:, 1:-1, 1:-1, 1:-1]
        i[:] = torch.where(self.fluid, self.equilibrium(rho, u), i)
        return f

    def moments(self, f):
        i = f[:, 1:-1, 1:-1, 1:-1]
        rho = i.sum(0)
        return rho, torch.tensordot(i, self.c, dims=([0], [0])) / rho[..., None]

    def step(self, f, lid=None, alpha=None, g=None):
        xl, yl, zl = self.size
        if self.periodic:
            f = f[:, 1:-1, 1:-1, 1:-1]
            h = torch.stack([torch.roll(f[k], (v[2], v[1], v[0]), (0, 1, 2)) for k, v in enumerate(self.cl)])
        else:
            h = torch.stack([f[k, 1 - v[2]:zl + 1 - v[2], 1 - v[1]:yl + 1 - v[1], 1 - v[0]:xl + 1 - v[0]]
                             for k, v in enumerate(self.cl)])
        rho = h.sum(0)
        u = torch.tensordot(h, self.c, dims=([0], [0])) / rho[..., None]
        if alpha is not None:
            u = (1 - alpha)[..., None] * (u + self.tau * g)
        h = h - (h - self.equilibrium(rho, u)) / self.tau
        if self.periodic:
            return torch.nn.functional.pad(h, (1, 1, 1, 1, 1, 1))
        i = torch.where(self.fluid, h, f[:, 1:-1, 1:-1, 1:-1])
        pad = torch.nn.functional.pad
        edge = f.clone()
        edge[:, 1:-1, 1:-1, 1:-1] = 0
        f = pad(i, (1, 1, 1, 1, 1, 1)) + edge
        flat, n = f.reshape(-1), f[0].numel()
        dst, val = [], []
        for kind, p, d, s, cell, qs in self.links:
            back = flat[s]
            if kind == NOSLIP:
                v = back
            elif kind == MOVINGWALL:
                ul = self.c.new_tensor(p[:3]) if lid is None else lid
                v = back + 2 * self.w[qs] * f.reshape(self.q, n).sum(0)[cell] * (self.c[qs] @ ul) / self.cs2
            elif kind == INFLOWBC:
                ui = self.c.new_tensor(p[:3])
                v = self.equilibrium(self.c.new_ones(1), ui[None])[:, 0][qs]
            else:  # outflow: the two opposite equilibria at the reference density, minus the outgoing value
                ux = (self.c.t() @ f.reshape(self.q, n))[:, cell]
                cu, uu = (self.c[qs] * ux.t()).sum(1) / self.cs2, (ux * ux).sum(0) / (2 * self.cs2)
                v = 2 * self.w[qs] * (1 + 0.5 * cu * cu - uu) - back
            dst.append(d)
            val.append(v)
        return flat.index_put((torch.cat(dst),), torch.cat(val)).reshape(f.shape)


def _cs2(storage):
    # fp64 storage keeps the reference's literal of the speed of sound
    return float.fromhex("0x1.279a745904047p-1") ** 2 if storage == "f64" else 1.0 / 3.0


def _vjp_chain(states, step, lam, params):
    """Gradients of lam . (last state) with respect to params through
    state_{t+1} = step(state_t)."""
    grads = [torch.zeros_like(p) for p in params]
    for f in reversed(states):
        f = f.detach().requires_grad_(True)
        with torch.enable_grad():
            out = step(f)
        got = torch.autograd.grad(out, [f, *params], lam, allow_unused=True)
        lam = got[0]
        grads = [a if b is None else a + b for a, b in zip(grads, got[1:])]
    return grads


@torch.no_grad()
def exact(case, seed):
    cs2 = _cs2(case["storage"])
    if case["kind"] == "flow":
        size = (case["xl"], case["yl"], case["zl"])
        if size[0] * size[1] * size[2] * case["steps"] * case["q"] > 2e11:
            return None
        r = _Reference(case["geom"], case["q"], size, case["tau"], cs2, _fluid_mask(case, seed))
        f = r.start(*_start_fields(case["geom"], size, seed))
        for _ in range(case["steps"]):
            f = r.step(f)
        rho, u = r.moments(f)
        return {"rho": rho, "u": u}
    if case["kind"] == "adjoint":
        n = case["n"]
        alpha, target = _porosity(case, seed)
        r = _Reference("box", case["q"], (n, n, n), case["tau"], cs2)
        g = alpha.new_tensor([FORCE, 0.0, 0.0])
        states, f = [], r.rest()
        for _ in range(case["steps"]):
            states.append(f)
            f = r.step(f, alpha=alpha, g=g)
        f = f.detach().requires_grad_(True)
        a = alpha.requires_grad_(True)
        with torch.enable_grad():
            j = ((r.moments(f)[1][:, :, n // 2 - 1] - target) ** 2).sum()
        lam = torch.autograd.grad(j, f)[0]
        return {"j": j.detach(), "grad": _vjp_chain(states, lambda s: r.step(s, alpha=a, g=g), lam, [a])[0]}
    doms = _cavities(case)
    if sum(x * y * z for x, y, z, _ in doms) * case["steps"] > 1.5e9 or case["n"] * case["steps"] > 7000:
        return None
    moments, js, grads = [], [], []
    for i, (xl, yl, zl, tau) in enumerate(doms):
        r = _Reference("cavity", 19, (xl, yl, zl), tau, cs2)
        f = r.start(*_start_fields("cavity", (xl, yl, zl), seed + i))
        lid = f.new_tensor([LID, 0.0, 0.0])
        states = []
        for _ in range(case["steps"]):
            if case["kind"] == "batchadj":
                states.append(f)
            f = r.step(f, lid=lid)
        if case["kind"] == "batch":
            moments.append(r.moments(f))
            continue
        f = f.detach().requires_grad_(True)
        lid = lid.requires_grad_(True)
        with torch.enable_grad():
            j = 0.5 * (r.moments(f)[1] ** 2).sum()
        lam = torch.autograd.grad(j, f)[0]
        js.append(j.detach())
        grads.append(_vjp_chain(states, lambda s: r.step(s, lid=lid), lam, [lid])[0])
    if case["kind"] == "batch":
        return {"moments": moments, "diverged": None}
    return {"j": torch.stack(js), "grad": torch.stack(grads)}
