"""The work a program of this framework has it do, as cases that can be timed and compared.

Every case goes through the package's public entry points (the C ABI behind `rhs_box`, `Level`, `Amr`,
`Batch`), on inputs made from a seed on the GPU, with the handles a program keeps (the level, its
Phase-Field set-up, the hierarchy, the batch) made once in `prepare`. All states are FP64.

Kinds of case (`case["kind"]`):

  box      one right-hand side of one box whose ghost cells are filled (`rhs_box`): the call that a
           host code makes per box in place of its own compute_dUdt_FV. The smallest call there is.
  level    `steps` time steps of one level (`Level.advance`: device ComputeDt, the RK3 step replayed
           from a graph and, with `pf`, the Phase-Field step after each), for the advected interface,
           a shock and a bubble (2D), a shock and a droplet (3D, water and air), a smooth state, or
           three-phase converging rings on uneven boxes.
  gradq    the interface regularisation's gradient on the faces of one level
           (`Level.PhaseField_GradQPF`), CAC with the implicit solve.
  amr      `steps` steps of a hierarchy with refined levels made from the GPU's tags (`Amr.advance`),
           flow only or with the CAC Phase-Field step.
  batch    one tick of the served stream: `Batch.step` over the admitted cases and, with `pf`,
           `Batch.pf_step`.
"""
import math

import numpy as np
import torch

import compas_amd
from compas_amd import Amr, Batch, Layout, Level, make_geometry, make_params, make_pf_params, regrid, rhs_box, roofline, split_domain

DEV = "cuda"
F64 = torch.float64


# ---- the cases ---------------------------------------------------------------------------------------

def listed():
    return [
        # the drop-in call on the smallest box a regrid makes: launch latency
        dict(name="box-2d-16", kind="box", dim=2, nx=16, ny=16, nz=1, scheme="WENO5", thinc=0),
        # the same call on one 3D box of the water-air droplet
        dict(name="box-3d-32-thinc", kind="box", dim=3, nx=32, ny=32, nz=32, scheme="WENO5", thinc=1),
        # the advected interface at its quoted size: one box, too few tiles to fill the card
        dict(name="interface-2d-256", kind="level", flow="interface", nx=256, ny=256, nz=1, grid=256, scheme="WENO5",
             thinc=0, pf="", steps=10),
        # the shock-bubble configuration's base grid with the bounded reconstruction
        dict(name="bubble-2d-weno5b", kind="level", flow="bubble", nx=1024, ny=256, nz=1, grid=64, scheme="WENO5B",
             thinc=0, pf="", steps=5),
        # a 3D level of odd extents and ragged boxes, periodic, no THINC
        dict(name="smooth-3d-ragged", kind="level", flow="smooth", nx=75, ny=61, nz=50, grid=21, scheme="WENO5",
             thinc=0, pf="", steps=4),
        # the largest: the 3D water-air droplet with THINC and the ACDI Phase-Field step
        dict(name="droplet-3d-256", kind="level", flow="droplet", nx=256, ny=256, nz=256, grid=32, scheme="WENO5",
             thinc=1, pf="ACDI", steps=2),
        # the AMR configuration's base level: three phases on boxes of 8 to 64 cells a side
        dict(name="rings-level-512", kind="level", flow="rings", nx=512, ny=512, nz=1, grid=0, scheme="WENO5", thinc=0,
             pf="", steps=5),
        # the implicit regularisation alone on one level
        dict(name="gradq-2d-cac", kind="gradq", nx=512, ny=256, grid=64),
        # the AMR configuration's flow: the rings' base level and three refined ones
        dict(name="rings-amr-4", kind="amr", flow="rings", n=512, levels=4, pf="", steps=4),
        # the shock-bubble configuration: two levels, flow and CAC Phase-Field step
        dict(name="bubble-amr-cac", kind="amr", flow="bubble", n=256, levels=2, pf="CAC-Adv", steps=2),
        # the served stream's flow tick over a mix of grids
        dict(name="served-24", kind="batch", cases=24, pf=""),
        # the served stream's whole tick, Phase-Field step included
        dict(name="served-8-cac", kind="batch", cases=8, pf="CAC-Adv"),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["box", "level", "level", "level", "gradq", "amr", "batch"])
    if kind == "box":
        dim = rng.choice([2, 3])
        n = [_size(rng, 8, 64) for _ in range(2)] + [_size(rng, 8, 40)]
        thinc = rng.choice([0, 1])
        scheme = rng.choice(["WENO5", "WENO5", "WENO5B", "MUSCL"]) if not thinc else "WENO5"
        return dict(kind="box", dim=dim, nx=n[0], ny=n[1], nz=n[2] if dim == 3 else 1, scheme=scheme, thinc=thinc)
    if kind == "level":
        flow = rng.choice(["interface", "bubble", "smooth", "droplet", "rings"])
        steps = rng.randint(2, 6)
        if flow == "interface":
            n, scheme = _size(rng, 64, 1024), rng.choice(["WENO5", "WENO5", "MUSCL"])
            return dict(kind="level", flow=flow, nx=n, ny=n, nz=1, grid=rng.choice([n, 64, 50, 128]), scheme=scheme,
                        thinc=rng.choice([0, 0, 1]) if scheme == "WENO5" else 0, pf="", steps=steps)
        if flow == "bubble":
            n = _size(rng, 64, 400)
            pf = rng.choice(["", "", "CAC-Adv", "ACDI"])
            return dict(kind="level", flow=flow, nx=n * rng.choice([1, 2, 4]), ny=n, nz=1, grid=rng.choice([32, 48, 64]),
                        scheme=rng.choice(["WENO5", "WENO5B"]), thinc=0, pf=pf, steps=2 if pf else steps)
        if flow == "rings":
            n = 8 * _size(rng, 16, 80)
            return dict(kind="level", flow=flow, nx=n, ny=n, nz=1, grid=0, scheme="WENO5", thinc=0, pf="", steps=steps)
        if flow == "smooth":
            n = [_size(rng, 24, 128) for _ in range(3)]
            return dict(kind="level", flow=flow, nx=n[0], ny=n[1], nz=n[2], grid=rng.choice([16, 21, 32, 40, 64]),
                        scheme=rng.choice(["WENO5", "WENO5", "WENO5B"]), thinc=0, pf="", steps=steps)
        n = 2 * _size(rng, 20, 100)
        return dict(kind="level", flow=flow, nx=n, ny=n, nz=n, grid=rng.choice([16, 32, 64]), scheme="WENO5",
                    thinc=rng.choice([0, 1, 1]), pf=rng.choice(["", "ACDI"]), steps=2)
    if kind == "gradq":
        n = _size(rng, 64, 512)
        return dict(kind="gradq", nx=n * rng.choice([1, 2]), ny=n, grid=rng.choice([32, 40, 64]))
    if kind == "amr":
        if rng.random() < 0.5:
            return dict(kind="amr", flow="rings", n=64 * rng.randint(2, 8), levels=rng.randint(2, 4), pf="",
                        steps=rng.randint(2, 4))
        return dict(kind="amr", flow="bubble", n=32 * rng.randint(3, 8), levels=2, pf=rng.choice(["", "CAC-Adv"]),
                    steps=2)
    pf = rng.choice(["", "", "CAC-Adv"])
    return dict(kind="batch", cases=rng.randint(1, 8 if pf else 48), pf=pf)


# ---- initial states (on the GPU) -----------------------------------------------------------------------

def _centres(shape, dx):
    """Cell-centre coordinates x, y(, z) of a grid with extents shape = (nx, ny(, nz))."""
    ax = [(torch.arange(n, dtype=F64, device=DEV) + 0.5) * h for n, h in zip(shape, dx)]
    g = torch.meshgrid(*reversed(ax), indexing="ij")
    return list(reversed(g))


def _tanh01(d, w):
    return 0.5 * (1.0 + torch.tanh(d / w))


def _post_shock(gamma, p1, rho1, mach):
    """Rankine-Hugoniot state behind a shock of Mach number mach running into gas at rest."""
    m2 = mach * mach
    p2 = p1 * (1.0 + 2.0 * gamma / (gamma + 1.0) * (m2 - 1.0))
    rho2 = rho1 * (gamma + 1.0) * m2 / ((gamma - 1.0) * m2 + 2.0)
    return p2, rho2, mach * math.sqrt(gamma * p1 / rho1) * (1.0 - rho1 / rho2)


def _modes(X, rng, length):
    """A few random Fourier modes, periodic over `length`."""
    f = torch.zeros_like(X[0])
    for _ in range(3):
        t = torch.ones_like(f) * rng.uniform(-1, 1)
        for x, n in zip(X, length):
            t = t * torch.sin(2 * math.pi * int(rng.integers(1, 3)) * x / n + rng.uniform(0, 2 * math.pi))
        f = f + t
    return f / 3.0


class _Flow:
    """A flow's parameters, geometry, boxes and initial state (a global array [N, (k,) j, i] on the GPU)."""

    def __init__(self, case, seed, level=0):
        rng = np.random.default_rng(seed)
        # a hierarchy's boxes follow its interfaces: those are the case's own, the gases the seed's
        shape, var = (np.random.default_rng(1), rng.uniform(0.95, 1.05)) if case["kind"] == "amr" else (rng, 1.0)
        flow = case["flow"]
        r = 2 ** level
        if case["kind"] == "amr":
            nx, ny, nz = (case["n"] * r, case["n"] * r, 1) if flow == "rings" else (4 * case["n"] * r, case["n"] * r, 1)
        else:
            nx, ny, nz = case["nx"], case["ny"], case["nz"]
        scheme, thinc = case.get("scheme", "WENO5"), case.get("thinc", 0)
        self.periodic, self.nphase, self.cfl = 0, 0, 0.4
        if flow == "interface":
            n, length, self.periodic, self.cfl = (nx, ny), (1.0, 1.0), 1, 0.5
            X = _centres(n, (1.0 / nx, 1.0 / ny))
            c = [0.5 + rng.uniform(-0.05, 0.05) for _ in range(2)]
            d = torch.sqrt((X[0] - c[0]) ** 2 + (X[1] - c[1]) ** 2)
            a = _tanh01(rng.uniform(0.22, 0.28) - d, 2.0 / nx).clamp(1e-8, 1 - 1e-8)
            one = torch.ones_like(a)
            self.gamma, self.pinf = (1.4, 1.6), (0.0, 0.0)
            W = [a, (1 - a) * 10.0, one, one, one, a]
        elif flow == "bubble":
            n, length = (nx, ny), (nx / ny, 1.0)
            X = _centres(n, (1.0 / ny, 1.0 / ny))
            if case["kind"] == "batch":
                mach, ratio, rad = rng.uniform(1.1, 3.0), math.exp(rng.uniform(math.log(0.1), math.log(10.0))), rng.uniform(0.1, 0.3)
                self.gamma = (rng.uniform(1.1, 1.7), rng.uniform(1.1, 1.7))
            else:
                mach, ratio, rad = 1.22, 0.138 * var, 0.25 + shape.uniform(-0.02, 0.02)
                self.gamma = (1.648, 1.4)
                if case["kind"] == "amr":
                    scheme = "WENO5B"
            self.pinf = (0.0, 0.0)
            xb = max(rad + 0.25, 0.45 * length[0]) + shape.uniform(0, 0.05)
            yb = 0.5 + shape.uniform(-0.03, 0.03)
            d = torch.sqrt((X[0] - xb) ** 2 + (X[1] - yb) ** 2)
            a = _tanh01(rad - d, 2.0 / ny).clamp(1e-8, 1 - 1e-8)
            p2, rho2, u2 = _post_shock(self.gamma[1], 1.0, 1.0, mach)
            post = X[0] < max(xb - rad - 0.1, 0.05)
            z = torch.zeros_like(a)
            W = [a * ratio, (1 - a) * torch.where(post, z + rho2, z + 1.0), torch.where(post, z + u2, z), z,
                 torch.where(post, z + p2, z + 1.0), a]
        elif flow == "droplet":
            n, length = (nx, ny, nz), (1.0, ny / nx, nz / nx)
            X = _centres(n, (1.0 / nx,) * 3)
            c = [0.5 * v + rng.uniform(-0.01, 0.01) for v in length]
            d = torch.sqrt(sum((x - q) ** 2 for x, q in zip(X, c)))
            a = _tanh01(0.1 + rng.uniform(-0.01, 0.01) - d, 2.0 / nx).clamp(1e-8, 1 - 1e-8)
            self.gamma, self.pinf = (4.4, 1.4), (6.0e8, 0.0)
            p2, rho2, u2 = _post_shock(1.4, 1.0e5, 1.2, 2.4)
            post = X[0] < 0.25 + rng.uniform(0, 0.02)
            z = torch.zeros_like(a)
            W = [a * 1000.0, (1 - a) * torch.where(post, z + rho2, z + 1.2), torch.where(post, z + u2, z), z, z,
                 torch.where(post, z + p2, z + 1.0e5), a]
        elif flow == "smooth":
            n = (nx, ny) if nz == 1 else (nx, ny, nz)
            h = 1.0 / max(n)
            length = tuple(v * h for v in n)
            self.periodic = 1
            X = _centres(n, (h,) * len(n))
            a = _tanh01(torch.sin(2 * math.pi * (X[0] / length[0] + 0.05 * _modes(X, rng, length))), 20.0 * h).clamp(1e-8, 1 - 1e-8)
            self.gamma, self.pinf = (1.4, 1.6), (0.0, 0.0)
            W = [a * (1.0 + 0.1 * _modes(X, rng, length)), (1 - a) * (5.0 + 0.5 * _modes(X, rng, length))]
            W += [0.5 + 0.1 * _modes(X, rng, length) for _ in n] + [1.0 + 0.1 * _modes(X, rng, length), a]
        else:
            n, length, self.nphase = (nx, ny), (1.0, 1.0), 3
            X = _centres(n, (1.0 / nx, 1.0 / ny))
            d = torch.sqrt((X[0] - 0.5) ** 2 + (X[1] - 0.5) ** 2)
            th = torch.atan2(X[1] - 0.5, X[0] - 0.5)

            def ring(r0):
                s = torch.zeros_like(th)
                for m in range(1, 9):
                    s = s + shape.uniform(-1, 1) * torch.cos(m * th + shape.uniform(0, 2 * math.pi))
                return r0 + 0.005 * s / 8.0

            w = 2.0 / nx
            h1, h2 = _tanh01(ring(0.30) - d, w), _tanh01(ring(0.35) - d, w)
            al = [h1.clamp(1e-8, 1.0), (h2 - h1).clamp(1e-8, 1.0), (1.0 - h2).clamp(1e-8, 1.0)]
            tot = al[0] + al[1] + al[2]
            al = [v / tot for v in al]
            self.gamma, self.pinf = (1.4, 1.67, 1.09), (0.0, 0.0, 0.0)
            p2, rho2, u2 = _post_shock(1.09, 1.0, 5.0, 1.5)
            post = d > 0.45
            z = torch.zeros_like(d)
            ur = torch.where(post, z - u2, z)
            W = [al[0], al[1] * 0.14 * var, al[2] * torch.where(post, z + rho2, z + 5.0), ur * torch.cos(th), ur * torch.sin(th),
                 torch.where(post, z + p2, z + 1.0)] + al
        self.scheme, self.thinc, self.n, self.dim = scheme, thinc, n, len(n)
        self.P = make_params(self.dim, gamma=self.gamma, pinf=self.pinf, scheme=scheme, thinc=thinc, nphase=self.nphase)
        bc = dict(lo_bc=[2] * self.dim, hi_bc=[2] * self.dim)
        self.G = make_geometry(n, (0.0,) * self.dim, length, (self.periodic,) * self.dim, **bc)
        self.dx = [length[q] / n[q] for q in range(self.dim)]
        self.ref = _Ref(self)
        if case["kind"] == "amr":
            W = self._ambient(W, X, rng)
        self.U = self.ref.to_cons(torch.stack(W))
        grid = case.get("grid", 64)
        self.boxes = _uneven(n, case["nx"] if grid == 0 else 1) if grid == 0 or (case["kind"] == "amr" and flow == "rings") else split_domain(n, grid)

    def _ambient(self, W, X, rng):
        """A hierarchy's gases move a little everywhere: smooth waves of 1e-5 on every primitive (half of the
        1e-8 that a phase leaves outside its region). In a gas at exact rest the slopes that the refined levels'
        ghost cells are interpolated with are rounding alone, and one slope factor serves all components."""
        r = self.ref
        wave = lambda: torch.sin(2 * math.pi * X[0] / 0.9 + rng.uniform(0, 6)) * torch.cos(2 * math.pi * X[1] / 0.7 + rng.uniform(0, 6))  # noqa: E731
        al = r.alphas(torch.stack(W))
        new = [a + 0.5e-8 * wave() for a in al[:-1]] + [al[-1] + 0.5e-8 * wave()]
        tot = sum(new)
        new = [a / tot for a in new]
        out = list(W)
        for k in range(r.nm):
            out[k] = W[k] / al[k] * new[k] * (1.0 + 1e-5 * wave())
        for m in range(r.nm, r.E):
            out[m] = W[m] + 1e-5 * wave()
        out[r.E] = W[r.E] * (1.0 + 1e-5 * wave())
        for k in range(r.N - r.alpha0):
            out[r.alpha0 + k] = new[k]
        return out

    def layout(self, boxes=None):
        return Layout(self.dim, boxes or self.boxes, 3, self.P.nstate)


def _uneven(n, seed):
    """A split of the domain into boxes of 8 to 64 cells a side at multiples of 8, as regrids make them."""
    rng = np.random.default_rng(seed)
    out, stack = [], [([0, 0], [v - 1 for v in n])]
    while stack:
        lo, hi = stack.pop()
        ext = [h - l + 1 for l, h in zip(lo, hi)]
        d = int(np.argmax(ext))
        if max(ext) <= 64 and (rng.uniform() < 0.5 or ext[d] < 16):
            out.append((list(lo), list(hi)))
            continue
        cut = lo[d] + 8 * int(rng.integers(1, -(-ext[d] // 8)))
        a, b = list(hi), list(lo)
        a[d], b[d] = cut - 1, cut
        stack += [(list(lo), a), (b, list(hi))]
    return out


def _pack(lay, U):
    """Global valid field -> level buffer (ghost cells zero), both on the GPU."""
    buf = torch.zeros(lay.total, dtype=F64, device=DEV)
    for b, (lo, hi) in enumerate(lay.boxes):
        sh = lay.fab_shape(b)
        off = lay.cboxes[b].offset
        dst = buf[off:off + math.prod(sh)].view(sh)
        dst[(slice(None),) + tuple(slice(3, s - 3) for s in sh[1:])] = U[
            (slice(None),) + tuple(slice(lo[d], hi[d] + 1) for d in reversed(range(lay.dim)))]
    return buf


def _valid(lay):
    """How the valid cells of a level buffer are taken out: a view where all boxes have one shape,
    else the cells' indices (box by box, [n, (k,) j, i])."""
    shapes = {tuple(lay.fab_shape(b)) for b in range(lay.nbox)}
    if len(shapes) == 1:
        sh = shapes.pop()
        cut = (slice(None), slice(None)) + tuple(slice(3, s - 3) for s in sh[1:])
        return lambda buf: buf.view((lay.nbox,) + sh)[cut]
    idx = []
    for b in range(lay.nbox):
        sh = lay.fab_shape(b)
        off = lay.cboxes[b].offset
        q = np.arange(off, off + math.prod(sh), dtype=np.int64).reshape(sh)
        idx.append(q[(slice(None),) + tuple(slice(3, s - 3) for s in sh[1:])].reshape(-1))
    idx = torch.from_numpy(np.concatenate(idx)).to(DEV)
    return lambda buf: torch.index_select(buf, 0, idx)


# ---- prepare / run -------------------------------------------------------------------------------------

class _Kept(dict):
    """What a program keeps between calls; closes its handles in order when it goes."""

    def __del__(self):
        for h in self.get("close", ()):
            h.close()


def _pf(mechanism):
    """The Phase-Field set-ups that the benchmark runs: ACDI with the explicit, CAC with the implicit
    regularisation, CFL 0.3, eta half a cell."""
    return make_pf_params(mechanism=mechanism, explicit_rc=1 if mechanism == "ACDI" else 0, cfl=0.3, eta_multiplier=0.5)


def _scalars(n=1):
    return torch.zeros(1, dtype=F64, device=DEV), torch.zeros(n, dtype=F64, device=DEV)


def _box_input(case, seed):
    """One box's fab with its ghost cells: the cut of a larger level that a host's fill leaves there."""
    n = [case["nx"] + 6, case["ny"] + 6] + ([case["nz"] + 6] if case["dim"] == 3 else [])
    c = dict(kind="level", flow="smooth", nx=n[0], ny=n[1], nz=n[2] if case["dim"] == 3 else 1, scheme=case["scheme"],
             thinc=case["thinc"], grid=64)
    return _Flow(c, seed)


def _served(case, seed):
    grids = [(128, 128), (256, 256), (512, 128), (512, 512), (1024, 256)]
    out = []
    for q in range(case["cases"]):
        nx, ny = grids[q % len(grids)]
        out.append(_Flow(dict(kind="batch", flow="bubble", nx=nx, ny=ny, nz=1, grid=64), seed * 1009 + q))
    return out


def _hierarchy(case, seed):
    """The levels of a hierarchy, coarsest first: (flow, layout, Level, state). Every refined level comes
    from the GPU's tags on the level below, clustered, nested and refined, as a program's first regrid
    makes it. The tags are those of seed 0, so that the boxes are the case's own."""
    if seed:
        out = []
        for l, (f0, lay, lev, U) in enumerate(_hierarchy(case, 0)):
            f = _Flow(case, seed, level=l)
            U.copy_(_pack(lay, f.U))
            out.append((f, lay, lev, U))
        for l in range(len(out) - 1, 0, -1):
            out[l][2].AverageDownTo(out[l][3], out[l - 1][2], out[l - 1][3], 2)
        return out
    out = []
    f = _Flow(case, seed)
    grads = [(6, "grad", 0.1), (7, "grad", 0.1), (8, "grad", 0.1)] if f.nphase else [(5, "grad", 0.1)]
    crit = grads + [("P", "grad", 0.1)]
    lay = f.layout()
    out.append((f, lay, Level(f.P, f.G, lay), _pack(lay, f.U)))
    for l in range(1, case["levels"]):
        fc, lc, lev, U = out[-1]
        lev.FillPatch(U) if l == 1 else lev.FillPatchTwoLevels(U, out[-2][2], out[-2][3], 2)
        shape = tuple(reversed(fc.n))
        boxes, _ = regrid.regrid(lev, U, crit, shape, ratio=1, blocking_factor=4, max_grid_size=32)
        if l > 1:
            boxes = regrid.nest(boxes, lc.boxes, shape, blocking_factor=4, margin=4)
        f = _Flow(case, seed, level=l)
        lay = f.layout(regrid.refine(boxes, 2))
        out.append((f, lay, Level(f.P, f.G, lay), _pack(lay, f.U)))
    for l in range(len(out) - 1, 0, -1):
        out[l][2].AverageDownTo(out[l][3], out[l - 1][2], out[l - 1][3], 2)
    return out


class _Foreign:
    """A device array of another owner, for torch.as_tensor; the tensor keeps the owner alive."""

    def __init__(self, ptr, n, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(ptr, False), version=3)


def prepare(case, seed):
    kind = case["kind"]
    s = _Kept(kind=kind, case=dict(case))
    if kind == "box":
        f = _box_input(case, seed)
        n = f.n
        s.update(flow=f, box=([0] * f.dim, [v - 7 for v in n]), U=f.U.contiguous(), cmax=_scalars()[1],
                 dU=torch.zeros((f.P.nstate,) + tuple(v - 6 for v in reversed(n)), dtype=F64, device=DEV))
        f.U = None
        torch.cuda.synchronize()
        return s
    s["stream"] = torch.cuda.Stream()
    if kind in ("level", "gradq"):
        c = dict(case, flow="bubble", nz=1, scheme="WENO5", thinc=0) if kind == "gradq" else case
        f = _Flow(c, seed)
        lay = f.layout()
        lev = Level(f.P, f.G, lay)
        Un = _pack(lay, f.U)
        f.U = None
        if kind == "gradq":
            lev.pf_setup(_pf("CAC-Adv"))
            dt, cm = _scalars()
            lev.CalculateInitialcmax(Un, cm)
            lev.ComputeDt(cm, dt, 0.4)
            s.update(lev=lev, U=Un, dt=float(dt.item()), gq=torch.zeros(lev.faces.total, dtype=F64, device=DEV), close=[lev])
        else:
            if case["pf"]:
                lev.pf_setup(_pf(case["pf"]))
            dt, cm = _scalars()
            U1, U2 = torch.zeros_like(Un), torch.zeros_like(Un)
            lev.advance(Un, U1, U2, 0, f.cfl, dt, cm)
            s.update(lev=lev, U=(Un, U1, U2), dt=dt, cmax=cm, cfl=f.cfl, take=_valid(lay), close=[lev])
    elif kind == "amr":
        h = _hierarchy(case, seed)
        levels = [q[2] for q in h]
        amr = Amr(levels, 2)
        if case["pf"]:
            amr.pf_setup(_pf(case["pf"]))
        U = [[q[3] for q in h], [torch.zeros_like(q[3]) for q in h], [torch.zeros_like(q[3]) for q in h]]
        dt, cm = _scalars(len(h))
        s.update(amr=amr, U=U, dt=dt, cmax=cm, take=[_valid(q[1]) for q in h], close=[amr] + levels)
    else:
        flows = _served(case, seed)
        lays = [f.layout() for f in flows]
        batch = Batch(flows[0].P, sum(l.total + 64 for l in lays), len(flows))
        if case["pf"]:
            batch.pf_setup(_pf(case["pf"]))
        ids = [batch.admit(f.P, f.G, l, _pack(l, f.U).cpu().numpy(), f.cfl) for f, l in zip(flows, lays)]
        views = []
        for q, l in zip(ids, lays):
            p, n = compas_amd.ctypes.c_void_p(), compas_amd.ctypes.c_longlong()
            compas_amd.check(batch.lib.cmp_batch_case_state(batch.h, q, compas_amd.ctypes.byref(p), compas_amd.ctypes.byref(n),
                                                            None, None, None), "cmp_batch_case_state")
            views.append(_valid(l)(torch.as_tensor(_Foreign(p.value, n.value, batch), device=DEV)))
        # (closed by its own end: the views that run() returns hold it)
        s.update(batch=batch, views=views)
    torch.cuda.synchronize()
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "box":
        f = s["flow"]
        rhs_box(f.P, f.G, s["box"], 3, s["U"], s["dU"], s["cmax"])
        return {"dUdt": s["dU"], "cmax": s["cmax"]}
    st = s["stream"]
    if kind == "batch":
        s["batch"].step(stream=st)
        if case["pf"]:
            s["batch"].pf_step(stream=st)
        return s["views"]
    with torch.cuda.stream(st):
        if kind == "gradq":
            gmax, _ = s["lev"].PhaseField_GradQPF(s["U"], s["dt"], s["gq"], stream=st)
            return {"gradq": s["gq"], "max": gmax}
        if kind == "level":
            Un, U1, U2 = s["U"]
            s["lev"].advance(Un, U1, U2, case["steps"], s["cfl"], s["dt"], s["cmax"], resume=True, stream=st)
            return {"U": s["take"](Un), "dt": s["dt"]}
        Un, U1, U2 = s["U"]
        s["amr"].advance(Un, U1, U2, case["steps"], 0.4, s["dt"], s["cmax"], stream=st)
        return {"U": [t(u) for t, u in zip(s["take"], Un)], "dt": s["dt"]}


# ---- what a pass cannot do without -----------------------------------------------------------------------

def _levels_cells(case):
    """Cells of each level of a hierarchy, about: the refined share that the tags of these flows give."""
    if case["flow"] == "rings":
        n = case["n"]
        return [n * n] + [int(2 * math.pi * 0.6 * 14.0 * n * 2 ** l) for l in range(1, case["levels"])]
    n = case["n"]
    return [4 * n * n, int(0.25 * 16 * n * n)]


def work(case):
    """Bytes: the state read once and written once per step (per call for a right-hand side). Operations:
    the minimal fused algorithm's (compas_amd/roofline.py), three stages a step; the Phase-Field step's
    own are left out: they are few away from interfaces."""
    kind = case["kind"]
    if kind == "box":
        P = make_params(case["dim"], scheme=case["scheme"])
        ext = [case["nx"], case["ny"], case["nz"]][:case["dim"]]
        ghost = math.prod(v + 6 for v in ext)
        return {"bytes": 8.0 * P.nstate * (ghost + math.prod(ext)), "flops": float(roofline.flops_per_cell_stage(P) * math.prod(ext))}
    if kind == "gradq":
        # alpha in, one value a face out; the solve's traffic is the method's own
        return {"bytes": 8.0 * case["nx"] * case["ny"] * 3, "flops": 0.0}
    if kind == "batch":
        P, cells, steps = make_params(2), int(case["cases"] * 134000), 1
    elif kind == "amr":
        P = make_params(2, gamma=(1.4,) * 3, nphase=3) if case["flow"] == "rings" else make_params(2)
        cells, steps = sum(_levels_cells(case)), case["steps"]
    else:
        dim = 2 if case["nz"] == 1 else 3
        P = make_params(2, gamma=(1.4,) * 3, nphase=3) if case["flow"] == "rings" else make_params(dim, scheme=case["scheme"])
        cells, steps = case["nx"] * case["ny"] * case["nz"], case["steps"]
    return {"bytes": 16.0 * P.nstate * cells * steps, "flops": 3.0 * roofline.flops_per_cell_stage(P) * cells * steps}


def tolerance(case):
    """About four times and more what run() was seen to differ from exact() by, over the listed cases and 30
    drawn ones: a right-hand side 4e-13 (differences of fluxes that nearly cancel), a level's or a batch's
    steps 7e-16 to 1.5e-15, the implicit gradient 1e-10 (the solve's floor), steps with that solve 2e-14 in the
    state. The steps of a hierarchy 2.7e-7 (1.8e-4 in one cell): one slope factor serves all components of a ghost
    cell interpolated from the coarser level, and it jumps where a slope passes through zero; the plain form
    moves as much when its own input moves in the last bit. A step over THINC's or the bounded
    reconstruction's switches can turn rounding into more in a few cells."""
    kind, pf = case["kind"], case.get("pf")
    if kind == "box":
        return {"rel": 2e-12, "max": 1e-10}
    if kind == "gradq":
        return {"rel": 5e-10, "max": 2e-8}
    if kind == "amr":
        return {"rel": 1e-6, "max": 8e-4}
    if pf == "CAC-Adv":
        return {"rel": 1e-11, "max": 1e-9}
    if case.get("thinc") or case.get("scheme") == "WENO5B" or pf:
        return {"rel": 1e-11, "max": 1e-8}
    return {"rel": 1e-13, "max": 1e-11}


# ---- the same results in plain torch --------------------------------------------------------------------

class _Ref:
    """The five-equation model on a global array [N, (k,) j, i], in the formulas' own order."""

    def __init__(self, f):
        self.f, self.dim, self.np = f, f.dim, f.nphase
        self.A = [1.0 / (g - 1.0) for g in f.gamma]
        self.B = [g * p / (g - 1.0) for g, p in zip(f.gamma, f.pinf)]
        self.nm = self.np or 2
        self.E = self.nm + self.dim
        self.alpha0 = self.E + 1
        self.N = 2 * self.np + self.dim + 1 if self.np else 4 + self.dim

    # -- equation of state
    def alphas(self, V):
        if self.np:
            return [V[self.alpha0 + k] for k in range(self.np)]
        return [V[self.alpha0], 1.0 - V[self.alpha0]]

    def mix(self, V):
        al = self.alphas(V)
        return sum(a * c for a, c in zip(al, self.A)), sum(a * c for a, c in zip(al, self.B))

    def to_cons(self, W):
        U = W.clone()
        rho = W[:self.nm].sum(0)
        AP, BP = self.mix(W)
        U[self.nm:self.E] = rho * W[self.nm:self.E]
        U[self.E] = AP * W[self.E] + BP + 0.5 * rho * (W[self.nm:self.E] ** 2).sum(0)
        return U

    def to_prim(self, U):
        W = U.clone()
        rho = U[:self.nm].sum(0)
        AP, BP = self.mix(U)
        W[self.nm:self.E] = U[self.nm:self.E] / rho
        W[self.E] = (U[self.E] - 0.5 * rho * (W[self.nm:self.E] ** 2).sum(0) - BP) / AP
        return W

    def sound(self, W):
        rho = W[:self.nm].sum(0)
        al = self.alphas(W)
        AP, _ = self.mix(W)
        return torch.sqrt(sum(a * ((c + 1.0) * W[self.E] + b) for a, c, b in zip(al, self.A, self.B)) / (AP * rho))

    # -- ghost cells
    def axis(self, d):
        return -1 - d

    def pad(self, V, d, g):
        n = V.shape[self.axis(d)]
        i = torch.arange(-g, n + g, device=V.device)
        i = i % n if self.f.periodic else i.clamp(0, n - 1)
        return V.index_select(V.dim() - 1 - d, i)

    def cut(self, V, d, lo, n):
        return V.narrow(V.dim() - 1 - d, lo, n)

    # -- reconstructions
    @staticmethod
    def weno_parts(v, face):
        mm, m, c, p, pp = v
        if face > 0:
            fs = [c + (2 / 3) * (p - c) - (1 / 6) * (pp - p), c + (1 / 6) * (c - m) + (1 / 3) * (p - c),
                  c - (1 / 3) * (m - mm) + (5 / 6) * (c - m)]
        else:
            fs = [c - (5 / 6) * (p - c) + (1 / 3) * (pp - p), c - (1 / 3) * (c - m) - (1 / 6) * (p - c),
                  c + (1 / 6) * (m - mm) - (2 / 3) * (c - m)]
        a, b, k, e = p - c, pp - p, c - m, m - mm
        IS = [(10 / 3) * a * a - (11 / 3) * a * b + (4 / 3) * b * b, -(5 / 3) * k * a + (4 / 3) * k * k + (4 / 3) * a * a,
              (10 / 3) * k * k - (11 / 3) * e * k + (4 / 3) * e * e]
        return fs, IS

    @staticmethod
    def weno_weights(IS, face):
        d = [0.3, 0.6, 0.1] if face > 0 else [0.1, 0.6, 0.3]
        one = torch.ones_like(IS[0])
        r01, r02, r12 = (torch.where(torch.isnan(q), one, q) for q in (IS[0] / IS[1], IS[0] / IS[2], IS[1] / IS[2]))
        r10, r20, r21 = 1 / r01, 1 / r02, 1 / r12
        return [d[0] / (d[0] + r01 * r01 * d[1] + r02 * r02 * d[2]), d[1] / (r10 * r10 * d[0] + d[1] + r12 * r12 * d[2]),
                d[2] / (r20 * r20 * d[0] + r21 * r21 * d[1] + d[2])]

    def weno(self, v, face):
        fs, IS = self.weno_parts(v, face)
        return sum(w * x for w, x in zip(self.weno_weights(IS, face), fs))

    @staticmethod
    def minmod(m, c, p, face):
        a, b, z = c - m, p - c, torch.zeros_like(c)
        s = torch.minimum(torch.maximum(a, z), torch.maximum(b, z)) + torch.maximum(torch.minimum(a, z), torch.minimum(b, z))
        return c + face * 0.5 * s

    def bounded(self, st, face):
        """WENO5B: phase masses and volume fractions of one face of the middle cell of st (5 cells)."""
        ar = [[w[k] for w in st] for k in range(2)]
        al = [[w[self.alpha0] for w in st], [1.0 - w[self.alpha0] for w in st]]
        Wq = 1.0 / 12.0

        def theta(c, l, r):
            mn = torch.minimum(torch.minimum((c - Wq * l - Wq * r) / (1 - 2 * Wq), l), r)
            return torch.clamp(c.clamp(min=0) / (c - mn).clamp(min=0), max=1.0)

        out = {}
        for k in range(2):
            for q in (1, -1):
                fs, IS = self.weno_parts(ar[k], q)
                w = self.weno_weights(IS, q)
                fa, _ = self.weno_parts(al[k], q)
                out[k, q] = [sum(x * y for x, y in zip(w, fs)), sum(x * y for x, y in zip(w, fa))]
            c = (ar[k][2], al[k][2])
            t = torch.fmin(theta(c[0], out[k, 1][0], out[k, -1][0]), theta(c[1], out[k, 1][1], out[k, -1][1]))
            for q in (1, -1):
                out[k, q] = [c[m] + t * (out[k, q][m] - c[m]) for m in range(2)]
        tot = {q: out[0, q][1] + out[1, q][1] for q in (1, -1)}
        t = torch.ones_like(tot[1])
        for k in range(2):
            for q in (1, -1):
                out[k, q] = [v / tot[q] for v in out[k, q]]
            for m, c in enumerate((ar[k][2], al[k][2])):
                t = torch.fmin(t, theta(c, out[k, 1][m], out[k, -1][m]))
        return [ar[0][2] + t * (out[0, face][0] - ar[0][2]), ar[1][2] + t * (out[1, face][0] - ar[1][2]),
                al[0][2] + t * (out[0, face][1] - al[0][2])]

    def consistent(self, Wf, Wc, face, dx):
        """The N-phase model's consistent limiter of a reconstructed side."""
        h = face * 0.5 * dx
        sa = (Wf[self.alpha0:] - Wc[self.alpha0:]) / h
        S = sa.sum(0)
        mx, im = sa.abs().max(0)
        sm = sa.gather(0, im[None])[0]
        off = (sm.abs() < 1e-10) | (S.abs() < 1e-10)
        one = torch.ones_like(S)
        th = torch.where(off, one, (sm / (sm - S)).clamp(0, 1))[None].repeat(self.np, *([1] * S.dim()))
        th.scatter_(0, im[None], torch.where(off, one, ((sm - S) / sm).clamp(0, 1))[None])
        out = Wf.clone()
        out[:self.np] = Wc[:self.np] + th * (Wf[:self.np] - Wc[:self.np])
        out[self.alpha0:] = Wc[self.alpha0:] + th * (Wf[self.alpha0:] - Wc[self.alpha0:])
        return out

    def sides(self, Wp, d, g, alpha=None):
        """Primitive states on both sides of every face along d (Wp padded by g >= 3 along d)."""
        n = Wp.shape[Wp.dim() - 1 - d] - 2 * g
        st = [self.cut(Wp, d, g - 3 + t, n + 1) for t in range(6)]
        sch = self.f.scheme
        if sch.startswith("WENO5"):
            L = torch.stack([self.weno([w[q] for w in st[:5]], 1) for q in range(self.N)])
            R = torch.stack([self.weno([w[q] for w in st[1:]], -1) for q in range(self.N)])
            if sch == "WENO5B":
                for side, cells, face in ((L, st[:5], 1), (R, st[1:], -1)):
                    side[0], side[1], side[self.alpha0] = self.bounded(cells, face)
        else:
            L, R = self.minmod(st[1], st[2], st[3], 1), self.minmod(st[2], st[3], st[4], -1)
        if self.np:
            L, R = self.consistent(L, st[2], 1, self.f.dx[d]), self.consistent(R, st[3], -1, self.f.dx[d])
        if self.f.thinc and alpha is not None:
            L, R = self.thinc(st, L, R, d, alpha)
        return L, R

    def thinc(self, st, L, R, d, alpha):
        """THINC on the volume fraction of interface faces; alpha: the fraction padded by 1 on every side
        (faces along d lie between its cells)."""
        amm, am, ac, ap = (w[self.alpha0] for w in st[1:5])
        dim, n = self.dim, [alpha.shape[alpha.dim() - 1 - q] - 2 for q in range(self.dim)]

        def at(shift):
            v = alpha
            for q in range(dim):
                v = self.cut(v, q, 1 + shift[q] if q != d else shift[q], n[q] + (1 if q == d else 0))
            return v

        grads = []
        for q in range(dim):
            sh = [0] * dim
            if q == d:
                hi = [0] * dim
                hi[d] = 1
                grads.append((at(hi) - at(sh)) / self.f.dx[d])
                continue
            edge = []
            for s in (-1, 1):
                v = 0.0
                for o in (0, 1):
                    for t in (0, s):
                        z = [0] * dim
                        z[d], z[q] = o, t
                        v = v + 0.25 * at(z)
                edge.append(v)
            grads.append((edge[1] - edge[0]) / self.f.dx[q])
        norm = torch.sqrt(sum(g * g for g in grads))
        nd = torch.where(norm == 0, torch.zeros_like(norm), grads[d] / norm).abs()
        gL, gR = (ac - am) * (am - amm) > 0, (ap - ac) * (ac - am) > 0
        sym = (amm == ap) & (am == ac) & (am != amm)
        eps, gate = 1e-4, nd > 0.25
        cL = (am > eps) & (am < 1 - eps) & (gL | sym) & gate
        cR = (ac > eps) & (ac < 1 - eps) & (gR | sym) & gate
        beta = 2.3 * nd + 0.01

        def face(sigma, abar, hi):
            e = torch.exp(2 * beta * abar)
            c = 0.5 / beta * torch.log((e - 1) / (torch.exp(2 * beta) - e))
            a, b = (0.0, 1.0) if hi else (1.0, -1.0)
            return (0.5 * (1 + torch.tanh(beta * (a + 0.5 * b * (sigma + 1) + c)))).clamp(0, 1)

        both = cL | cR
        base = (self.minmod(st[1], st[2], st[3], 1), self.minmod(st[2], st[3], st[4], -1))
        out = []
        for W, b, use, sig, abar, hi in ((L, base[0], cL, ac - amm, am, True), (R, base[1], cR, ap - am, ac, False)):
            V = torch.where(both, b, W)
            an = face(torch.where(sig > 0, 1.0, -1.0).to(F64), abar, hi)
            T = V.clone()
            T[0], T[1], T[self.alpha0] = an * V[0] / V[self.alpha0], (1 - an) * V[1] / (1 - V[self.alpha0]), an
            out.append(torch.where(use, T, V))
        return out

    # -- Riemann solver and right-hand side
    def hllc(self, L, R, d):
        m, E = self.nm, self.E
        UL, UR = self.to_cons(L), self.to_cons(R)
        cL, cR = self.sound(L), self.sound(R)
        rL, rR = L[:m].sum(0), R[:m].sum(0)
        vL, vR, pL, pR = L[m + d], R[m + d], L[E], R[E]
        SL = torch.minimum(0.5 * (vL + vR) - 0.5 * (cL + cR), vL - cL)
        SR = torch.maximum(0.5 * (vL + vR) + 0.5 * (cL + cR), vR + cR)
        S = (pR - pL + rL * vL * (SL - vL) - rR * vR * (SR - vR)) / (rL * (SL - vL) - rR * (SR - vR))

        def half(W, U, rho, v, p, Sk, Sb):
            F = U * v
            F[m + d] += p
            F[E] += p * v
            q = (Sk - v) / (Sk - S)
            C = q * U
            C[m + d] += q * rho * (S - v)
            C[E] += q * (S - v) * (rho * S + p / (Sk - v))
            return F + Sb * (C - U), v + Sb * (q - 1)

        z = torch.zeros_like(SL)
        FL, uL = half(L, UL, rL, vL, pL, SL, torch.minimum(z, SL))
        FR, uR = half(R, UR, rR, vR, pR, SR, torch.maximum(z, SR))
        w = 0.5 * (1 + torch.sign(S))
        F = torch.where(w == 1, FL, torch.where(w == 0, FR, 0.5 * FL + 0.5 * FR))
        u = torch.where(w == 1, uL, torch.where(w == 0, uR, 0.5 * uL + 0.5 * uR))
        c = torch.maximum(cL + torch.sqrt((L[m:E] ** 2).sum(0)), cR + torch.sqrt((R[m:E] ** 2).sum(0)))
        return F, u, c

    def alpha_padded(self, U):
        a = U[self.alpha0]
        for q in range(self.dim):
            a = self.pad(a, q, 1)
        return a

    def faces(self, U, d, Wp=None, alpha=None):
        if Wp is None:
            Wp = self.to_prim(self.pad(U, d, 3))
            alpha = self.alpha_padded(U) if self.f.thinc else None
        L, R = self.sides(Wp, d, 3, alpha)
        return self.hllc(L, R, d)

    def diff(self, F, d):
        n = F.shape[F.dim() - 1 - d] - 1
        return (self.cut(F, d, 1, n) - self.cut(F, d, 0, n)) / self.f.dx[d]

    def finish(self, U, div, divu):
        dU = -div
        dU[self.alpha0:] += U[self.alpha0:] * divu
        return dU

    def rhs(self, U):
        div, divu, cm = 0.0, 0.0, 0.0
        for d in range(self.dim):
            F, u, c = self.faces(U, d)
            div, divu = div + self.diff(F, d), divu + self.diff(u, d)
            cm = max(cm, float(self.cut(c, d, 0, c.shape[c.dim() - 1 - d] - 1).max()))
        return self.finish(U, div, divu), cm

    def rk3(self, U, dt, rhs):
        k, c0 = rhs(U)
        U1 = U + dt * k
        k, c1 = rhs(U1)
        U2 = 0.25 * U1 + 0.75 * U + 0.25 * dt * k
        k, c2 = rhs(U2)
        return (2 / 3) * U2 + (1 / 3) * U + (2 / 3) * dt * k, max(c0, c1, c2)

    def next_dt(self, cm, prev, cfl):
        dt = min(cfl * h / cm for h in self.f.dx)
        return min(dt, 1.1 * prev) if prev > 0 else dt

    # -- the Phase-Field step (two phases)
    @staticmethod
    def back(phi, eta):
        return math.sqrt(2.0) * eta * torch.atanh(2.0 * phi.clamp(1e-12, 1 - 1e-12) - 1.0)

    @staticmethod
    def sharp(phi, eta, factor=2.0):
        return 0.5 + 0.5 * torch.tanh(_Ref.back(phi, eta) / (math.sqrt(2.0) * factor * eta))

    def two(self, V, d):
        """The low and high cells of every face along d."""
        p = self.pad(V, d, 1)
        n = V.shape[V.dim() - 1 - d]
        return self.cut(p, d, 0, n + 1), self.cut(p, d, 1, n + 1)

    def inner(self, F, d):
        """Faces with the domain's own cleared (Neumann sides)."""
        if not self.f.periodic:
            F = F.clone()
            F.select(F.dim() - 1 - d, 0).zero_()
            F.select(F.dim() - 1 - d, -1).zero_()
        return F

    def mechanism(self, a, dt, mob, eta, cac):
        """(alpha after the mechanism's sub-steps, its accumulated flux per direction over dt)."""
        dx = self.f.dx
        step = 0.9 / (2 * mob) / (sum(1 / h / h for h in dx) + 1 / eta / eta)
        H, t = [0.0] * self.dim, 0.0
        while t < dt:
            step = min(step, dt - t) if t + step > dt else step
            psi = a if cac else self.back(a, eta)
            g = []
            for d in range(self.dim):
                n = a.shape[a.dim() - 1 - d]
                p = self.pad(psi, d, 1)
                g.append((self.cut(p, d, 2, n) - self.cut(p, d, 0, n)) / (2 * dx[d]))
            s = torch.sqrt(sum(q * q for q in g))
            nrm = [torch.where(s == 0, torch.zeros_like(s), q / s) for q in g]
            if cac:
                lap, divn, ag = 0.0, 0.0, 0.0
                for d in range(self.dim):
                    lo, hi = self.two(a, d)
                    fg = (hi - lo) / dx[d]
                    lap = lap + self.diff(fg, d)
                    nl, nh = self.two(nrm[d], d)
                    divn = divn + self.diff(0.5 * nl + 0.5 * nh, d)
                    k = fg.shape[fg.dim() - 1 - d] - 1
                    ag = ag + (0.5 * self.cut(fg, d, 0, k) + 0.5 * self.cut(fg, d, 1, k)) ** 2
                mu = 2 * a * (1 - a) * (1 - 2 * a) / eta / eta - lap + torch.sqrt(ag) * divn
                W = a * (1 - a)
                a = a + step * (-mob * mu + W * (mob * mu).sum() / W.sum())
            else:
                div = 0.0
                for d in range(self.dim):
                    lo, hi = self.two(a, d)
                    nl, nh = self.two(nrm[d], d)
                    x = (0.5 * self.back(lo, eta) + 0.5 * self.back(hi, eta)) / (math.sqrt(2.0) * eta)
                    J = mob * ((hi - lo) / dx[d] - 0.5 / (math.sqrt(2.0) * eta) / torch.cosh(x) ** 2 * (0.5 * nl + 0.5 * nh))
                    H[d] = H[d] + step * J
                    div = div + self.diff(J, d)
                a = a + step * div
            t += step
        return a, [h / dt for h in H] if not cac else None

    def gradq(self, U, dt, mech):
        cac, a = mech != "ACDI", U[self.alpha0]
        eta = 0.5 * max(self.f.dx)
        rho = U[:2].sum(0)
        mob = 0.5 * eta * float(torch.sqrt(((U[2:self.E] / rho) ** 2).sum(0)).max())
        new, H = self.mechanism(a, dt, mob, eta, cac)
        sh = self.sharp(a, eta)
        mid = []
        for d in range(self.dim):
            lo, hi = self.two(sh, d)
            mid.append(0.5 * lo + 0.5 * hi)
        if not cac:
            return [torch.where((p < 1e-3) | (p > 1 - 1e-3), torch.zeros_like(p), h) / (p * (1 - p) + 1e-3) for p, h in zip(mid, H)]
        b = [p * (1 - p) + 1e-3 for p in mid]
        return self.solve(b, (new - a) / dt)

    def solve(self, b, rhs):
        """grad Q of div(b grad Q) = rhs - mean(rhs), Neumann or periodic: conjugate gradients with the
        diagonal, down to the rounding floor."""
        dx = self.f.dx
        bi = [self.inner(q, d) for d, q in enumerate(b)]

        def grad(Q):
            out = []
            for d in range(self.dim):
                lo, hi = self.two(Q, d)
                out.append(self.inner((hi - lo) / dx[d], d))
            return out

        def apply(Q):
            return -sum(self.diff(q * g, d) for d, (q, g) in enumerate(zip(bi, grad(Q))))

        diag = 0.0
        for d in range(self.dim):
            n = bi[d].shape[bi[d].dim() - 1 - d] - 1
            diag = diag + (self.cut(bi[d], d, 0, n) + self.cut(bi[d], d, 1, n)) / dx[d] ** 2
        r = -(rhs - rhs.mean())
        x, z = torch.zeros_like(r), r / diag
        p, rz = z.clone(), (r * z).sum()
        first = float((r * r).sum())
        best, kept, since = first, x.clone(), 0
        for it in range(20000):
            ap = apply(p)
            al = rz / (p * ap).sum()
            x += al * p
            r -= al * ap
            z = r / diag
            new = (r * z).sum()
            p = z + (new / rz) * p
            rz = new
            if it % 20 == 19:
                rr = float((r * r).sum())
                since += 1
                if rr < best:
                    best, kept, since = rr, x.clone(), 0
                if best <= 1e-28 * first or since >= 20 or not math.isfinite(rr):
                    break
        return grad(kept)

    def pf_rhs(self, U, gq):
        out = 0.0
        for d in range(self.dim):
            L, R = self.sides(self.to_prim(self.pad(U, d, 3)), d, 3)
            g = gq[d]

            def down(a, b, v):
                return torch.where(v > 0, b, torch.where(v < 0, a, 0.5 * (a + b)))

            ia, E = self.alpha0, self.E
            J1w = down(1 - R[ia], 1 - L[ia], g) * g
            J2w = -down(R[ia], L[ia], -g) * g
            J1r, J2r = down(L[0], R[0], g) * J1w, down(L[1], R[1], -g) * J2w
            J1, J2 = down(L[ia], R[ia], g) * J1w, down(1 - L[ia], 1 - R[ia], -g) * J2w
            M = J1r + J2r
            u = torch.stack([down(L[2 + m], R[2 + m], M) for m in range(self.dim)])
            F = torch.zeros_like(L)
            F[0], F[1], F[ia] = J1r, J2r, J1
            F[2:E] = M * u
            F[E] = (0.5 * (u * u).sum(0) * M + self.A[0] * J1 * down(L[E], R[E], J1) + self.B[0] * J1
                    + self.A[1] * J2 * down(L[E], R[E], J2) + self.B[1] * J2)
            out = out + self.diff(F, d)
        return out, 0.0

    def pf_step(self, U, dt, mech):
        gq = self.gradq(U, dt, mech)
        top = max(float(g.abs().max()) for g in gq)
        t, prev = 0.0, 0.0
        while t < dt:
            h = 0.3 * min(self.f.dx) / (top + 1e-14)
            prev = h if t == 0.0 else prev
            h = min(h, 1.1 * prev)
            if t + h > dt - 1e-3 * h:
                h = dt - t
            prev = h
            U, _ = self.rk3(U, h, lambda V: self.pf_rhs(V, gq))
            t += h
            if t >= dt - 1e-6 * dt:
                break
        return U

    def advance(self, U, steps, cfl, pf=""):
        _, cm = self.rhs(U)
        dt = 0.0
        for _ in range(steps):
            dt = self.next_dt(cm, dt, cfl)
            U, cm = self.rk3(U, dt, self.rhs)
            if pf:
                U = self.pf_step(U, dt, pf)
        return U, dt


def _boxed(U, boxes, dim):
    """The valid cells of a global array in the order and shape run() returns them."""
    cuts = [U[(slice(None),) + tuple(slice(lo[d], hi[d] + 1) for d in reversed(range(dim)))] for lo, hi in boxes]
    if len({tuple(c.shape) for c in cuts}) == 1:
        return torch.stack(cuts)
    return torch.cat([c.reshape(-1) for c in cuts])


class _Levels:
    """The stage-coupled flow step of a 2D hierarchy with open sides: every level as an array over the
    whole domain, valid where its mask says so."""

    def __init__(self, h):
        self.refs = [q[0].ref for q in h]
        self.U = [q[0].U for q in h]
        self.mask = []
        for f, lay, _, _ in h:
            m = torch.zeros(tuple(reversed(f.n)), dtype=torch.bool, device=DEV)
            for lo, hi in lay.boxes:
                m[lo[1]:hi[1] + 1, lo[0]:hi[0] + 1] = True
            self.mask.append(m)
        self.down(self.U)

    @staticmethod
    def mean4(F):
        n, j, i = F.shape
        return F.reshape(n, j // 2, 2, i // 2, 2).sum((2, 4)) * 0.25

    def down(self, U):
        for l in range(len(U) - 1, 0, -1):
            cover = self.mask[l][::2, ::2]
            U[l - 1] = torch.where(cover, self.mean4(U[l]), U[l - 1])

    def interp(self, C, ref):
        """Conservative linear interpolation with one slope factor for all components."""
        parts = []
        for d in range(2):
            p = ref.pad(C, d, 1)
            n = C.shape[C.dim() - 1 - d]
            lo, hi = ref.cut(p, d, 0, n), ref.cut(p, d, 2, n)
            dc, df, db = 0.5 * (hi - lo), 2 * (hi - C), 2 * (C - lo)
            z = torch.zeros_like(dc)
            s = torch.where(df * db >= 0, torch.minimum(df.abs(), db.abs()), z)
            s = torch.copysign(torch.ones_like(dc), dc) * torch.minimum(s, dc.abs())
            f = torch.where(dc != 0, s / dc, torch.ones_like(dc)).amin(0).clamp(max=1.0)
            parts.append(dc * f)
        up = lambda V: V.repeat_interleave(2, -1).repeat_interleave(2, -2)  # noqa: E731
        out = up(C)
        for d, s in enumerate(parts):
            off = torch.tensor([-0.25, 0.25], dtype=F64, device=C.device).repeat(C.shape[-1 - d])
            out = out + up(s) * (off if d == 0 else off[:, None])
        return out

    def rhs(self, U):
        """(dU/dt per level, c_max per level) of the filled hierarchy."""
        full = [U[0]]
        for l in range(1, len(U)):
            full.append(torch.where(self.mask[l], U[l], self.interp(U[l - 1], self.refs[l - 1])))
        F, cm = [], []
        for l, r in enumerate(self.refs):
            row, top = [], 0.0
            for d in range(2):
                f, u, c = r.faces(full[l], d)
                row.append(torch.cat([f, u[None]]))
                low = r.cut(c, d, 0, c.shape[1 - d] - 1)
                top = max(top, float(torch.where(self.mask[l], low, torch.zeros_like(low)).max()))
            F.append(row)
            cm.append(top)
        for l in range(len(U) - 1, 0, -1):
            for d in range(2):
                fine = F[l][d][:, :, ::2] if d == 0 else F[l][d][:, ::2, :]
                n, j, i = fine.shape
                mean = fine.reshape(n, j // 2, 2, i).sum(2) * 0.5 if d == 0 else fine.reshape(n, j, i // 2, 2).sum(3) * 0.5
                cover = self.mask[l][::2, ::2]
                z = torch.zeros_like(cover.narrow(1 - d, 0, 1))
                use = torch.cat([cover, z], 1 - d) | torch.cat([z, cover], 1 - d)
                F[l - 1][d] = torch.where(use, mean, F[l - 1][d])
        out = []
        for l, r in enumerate(self.refs):
            D = r.diff(F[l][0], 0) + r.diff(F[l][1], 1)
            out.append(r.finish(full[l], D[:-1], D[-1]))
        return out, cm

    def advance(self, steps, cfl):
        U = self.U
        _, cm = self.rhs(U)
        dt = 0.0
        for _ in range(steps):
            dt = min(r.next_dt(c, dt, cfl) for r, c in zip(self.refs, cm))
            new, tops = U, []
            for a, b, w in ((1.0, 0.0, 1.0), (0.25, 0.75, 0.25), (2 / 3, 1 / 3, 2 / 3)):
                k, c = self.rhs(new)
                tops.append(c)
                new = [a * v + b * u + w * dt * q for v, u, q in zip(new, U, k)]
                new = [torch.where(m, v, u) for m, v, u in zip(self.mask, new, U)]
                self.down(new)
            cm = [max(c) for c in zip(*tops)]
            U = new
        return U, dt


def exact(case, seed):
    """run()'s outputs in plain torch on the same inputs. None for the hierarchy's Phase-Field step, whose
    composite solve over the levels has no plain form of its own here (its parts, the flow step of a
    hierarchy and the Phase-Field step of a level, have)."""
    kind = case["kind"]
    if kind == "box":
        f = _box_input(case, seed)
        r, n = f.ref, [v - 6 for v in f.n]
        div, divu, cm = 0.0, 0.0, 0.0
        for d in range(f.dim):
            V, al = f.U, f.U[r.alpha0]
            for q in range(f.dim):
                V = r.cut(V, q, 3, n[q]) if q != d else V
                al = r.cut(al, q, 2, n[q] + 2)
            F, u, c = r.faces(None, d, r.to_prim(V), al)
            div, divu = div + r.diff(F, d), divu + r.diff(u, d)
            cm = max(cm, float(r.cut(c, d, 0, n[d]).max()))
        U = f.U
        for q in range(f.dim):
            U = r.cut(U, q, 3, n[q])
        return {"dUdt": r.finish(U, div, divu), "cmax": torch.tensor([cm], dtype=F64)}
    if kind == "gradq":
        f = _Flow(dict(case, flow="bubble", nz=1, scheme="WENO5", thinc=0), seed)
        gq = f.ref.gradq(f.U, f.ref.next_dt(f.ref.rhs(f.U)[1], 0.0, 0.4), "CAC-Adv")
        parts = []
        for lo, hi in f.boxes:
            parts += [gq[d][lo[1]:hi[1] + 1 + (d == 1), lo[0]:hi[0] + 1 + (d == 0)].reshape(-1) for d in range(2)]
        return {"gradq": torch.cat(parts), "max": float(max(g.abs().max() for g in gq))}
    if kind == "level":
        f = _Flow(case, seed)
        U, dt = f.ref.advance(f.U, case["steps"], f.cfl, case["pf"])
        return {"U": _boxed(U, f.boxes, f.dim), "dt": torch.tensor([dt], dtype=F64)}
    if kind == "amr":
        if case["pf"]:
            return None
        h = _hierarchy(case, seed)
        boxes = [q[1].boxes for q in h]
        U, dt = _Levels(h).advance(case["steps"], 0.4)
        for q in h:
            q[2].close()
        return {"U": [_boxed(u, b, 2) for u, b in zip(U, boxes)], "dt": torch.tensor([dt], dtype=F64)}
    out = []
    for f in _served(case, seed):
        out.append(_boxed(f.ref.advance(f.U, 1, f.cfl, case["pf"])[0], f.boxes, 2))
    return out
