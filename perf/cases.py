"""The work a docking program has this library do, as measurable cases.

Each case is one call of a public entry point (a Context method, or a Batch
replay) on seeded bodies, grids and poses of the workload generator: receptor
density of 1000 beads per 25 A sphere, ligand 300 per 15 A sphere, 12 bead
types, 20 % of the beads charged, translations on the docking shell.  Sizes
are those of the benchmark and test configurations and odd ones between them.

kind      entry point (host: buffers in host memory, else resident in HBM)
rigid     Context.score_rigid / score_rigid_dev      energy, force, torque
modes     Context.score_modes / score_modes_dev      the same, flexible bodies
adjoint   Context.adjoint_dev                        exact gradients [, parameters]
noalloc   Context.adjoint_dev_noalloc                the same inside captured loops
batch     Batch.run                                  many uneven pairs, graph replay
minimize  Context.minimize_dev                       VA13 from every pose
grid      Context.generate_grid                      potential grids of a new body
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG_DIR = os.path.join(ROOT, "gpuattract_2.0_amd")
CHARGED = 0.2     # share of charged beads
PLATEAU = 10.0
NEIGHBOURS = 10.8
TYPES = 12


def _package():
    """The package (its directory name is not an identifier)."""
    if "gpuattract_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "gpuattract_amd", os.path.join(PKG_DIR, "__init__.py"),
            submodule_search_locations=[PKG_DIR])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["gpuattract_amd"] = mod
        spec.loader.exec_module(mod)
    from gpuattract_amd import hip, workload
    return hip, workload


def listed():
    return [
        # a single pose from an interactive program or an outside minimizer:
        # nothing but latency
        dict(name="one_pose", kind="rigid", host=True, rec=300, lig=80, mr=0, ml=0, n=1),
        # the reference's work item: 100 poses, buffers in host memory
        dict(name="item_rigid", kind="rigid", host=True, rec=1000, lig=300, mr=0, ml=0, n=100),
        dict(name="item_modes", kind="modes", host=True, rec=3000, lig=800, mr=5, ml=5, n=100),
        # a docking scan: many poses resident in HBM
        dict(name="scan_rigid", kind="rigid", host=False, rec=1000, lig=300, mr=0, ml=0, n=100000),
        dict(name="scan_modes", kind="modes", host=False, rec=3000, lig=800, mr=5, ml=5, n=20011),
        # exact gradients for a gradient-based search
        dict(name="grad_rigid", kind="adjoint", rec=1000, lig=300, mr=0, ml=0, n=30001, w=False,
             pgrad=False),
        # the same with every mode slot in use, odd counts, and upstream weights
        dict(name="grad_modes_10", kind="adjoint", rec=3989, lig=997, mr=10, ml=10, n=10007, w=True,
             pgrad=False),
        # one step of fitting the pair table: energies, all gradients and the
        # 12 x 12 parameter gradient (the benchmark's headline step)
        dict(name="fit_params", kind="adjoint", rec=3000, lig=800, mr=5, ml=5, n=100000, w=False,
             pgrad=True),
        # a small fitting step inside a captured loop
        dict(name="fit_small", kind="noalloc", rec=613, lig=167, mr=3, ml=2, n=64, w=True,
             pgrad=True),
        # uneven pairs of a screening run scored in one replay
        dict(name="batch_pairs", kind="batch", pairs=8, rec=1800, lig=500, mr=7, ml=7, n=3000),
        # docking: minimization from many starts on the device
        dict(name="minimize", kind="minimize", rec=1000, lig=300, mr=3, ml=3, n=4000, evals=60),
        # potential grids of a new receptor
        dict(name="grid_new", kind="grid", rec=500, shape=8),
    ]


def draw(rng):
    def logu(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["rigid", "rigid", "modes", "modes", "adjoint", "adjoint", "adjoint", "noalloc",
                       "batch", "minimize", "grid"])
    rec, lig = logu(300, 4000), logu(80, 1000)
    mr, ml = rng.randint(0, 10), rng.randint(0, 10)
    if kind == "grid":
        return dict(kind="grid", rec=logu(200, 1200), shape=rng.choice([8, 12]))
    if kind == "batch":
        return dict(kind="batch", pairs=rng.randint(3, 8), rec=min(rec, 2500), lig=min(lig, 600),
                    mr=mr, ml=ml, n=logu(200, 3000))
    if kind == "minimize":
        return dict(kind="minimize", rec=min(rec, 1500), lig=min(lig, 400), mr=mr, ml=ml,
                    n=logu(50, 3000), evals=rng.randint(10, 60))
    if kind == "rigid":
        host = rng.random() < 0.4
        n = logu(1, 1000) if host else logu(100, 60000)
        return dict(kind="rigid", host=host, rec=rec, lig=lig, mr=0, ml=0, n=n)
    if kind == "modes":
        host = rng.random() < 0.4
        n = logu(1, 1000) if host else logu(100, 15000)
        return dict(kind="modes", host=host, rec=rec, lig=lig, mr=max(mr, 1), ml=max(ml, 1), n=n)
    if kind == "noalloc":
        return dict(kind="noalloc", rec=min(rec, 1500), lig=lig, mr=mr, ml=ml, n=logu(1, 2000),
                    w=rng.random() < 0.5, pgrad=rng.random() < 0.7)
    return dict(kind="adjoint", rec=rec, lig=lig, mr=mr, ml=ml, n=logu(64, 30000),
                w=rng.random() < 0.5, pgrad=rng.random() < 0.4)


# ------------------------------------------------------------------- inputs

class _Inputs:
    """One pair and its poses on the host, made from the seed alone."""

    def __init__(self, case, seed, shell=True):
        _, W = _package()
        self.W = W
        n_rec, n_lig, mr, ml = case["rec"], case["lig"], case["mr"], case["ml"]
        R_rec = W.scaled_radius(n_rec, W.DENSITY_REF)
        R_lig = W.scaled_radius(n_lig, W.LIG_REF)
        self.rec = W.add_modes(W.make_body(seed, 0, n_rec, R_rec, TYPES, CHARGED), seed, 50, mr)
        self.lig = W.add_modes(W.make_body(seed, 1, n_lig, R_lig, TYPES, CHARGED), seed, 60, ml)
        self.params = W.make_params(seed, TYPES)
        r_lo, r_hi = 0.75 * (R_rec + R_lig), R_rec + R_lig
        self.inner = W.inner_geom(self.rec)
        self.outer = W.cube_geom((0.0, 0.0, 0.0), r_hi + R_lig + 2.0, 2.6)
        self.lig_inner, self.lig_outer = W.lig_grid_geoms(self.lig, R_rec, r_hi)
        n = case["n"]
        d6 = W.make_poses(seed, n, r_lo, r_hi)
        self.flexible = case["kind"] == "modes" or mr > 0 or ml > 0
        if self.flexible:
            self.dofs = np.zeros((n, 26), np.float32)
            self.dofs[:, :6] = d6
            self.dofs[:, 6:6 + mr] = W.make_amplitudes(seed, n, mr, entity=5)
            self.dofs[:, 16:16 + ml] = W.make_amplitudes(seed, n, ml, entity=6)
        else:
            self.dofs = d6
        self.weights = np.random.default_rng(seed).uniform(0.25, 1.75, n).astype(np.float32)

    def basis(self, geom):
        """The receptor's per-type sums of 1/r'^8 and 1/r'^6, r' = max(r, plateau)."""
        dev = "cuda"
        rec = torch.from_numpy(self.rec.xyz.reshape(3, -1)).to(dev)
        onehot = torch.zeros(self.rec.n, TYPES, device=dev)
        onehot[torch.arange(self.rec.n), torch.from_numpy(self.rec.type.astype(np.int64)) - 1] = 1.0
        ax = [torch.arange(m, device=dev) * geom.spacing + o
              for m, o in ((geom.nx, geom.ox), (geom.ny, geom.oy), (geom.nz, geom.oz))]
        z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
        pts = torch.stack([x.reshape(-1), y.reshape(-1), z.reshape(-1)], 1).float()
        out = torch.empty(2 * TYPES, pts.shape[0], device=dev)
        for a in range(0, pts.shape[0], 16384):
            p = pts[a:a + 16384]
            r2 = sum((p[:, k:k + 1] - rec[k]) ** 2 for k in range(3))
            i2 = 1.0 / torch.clamp(r2, min=PLATEAU * PLATEAU)
            i6 = i2 * i2 * i2
            out[0::2, a:a + 16384] = ((i6 * i2) @ onehot).T
            out[1::2, a:a + 16384] = (i6 @ onehot).T
        return out.reshape(-1).cpu().numpy()


class _State:
    pass


def _upload(ctx, inp, lig_grid):
    hs = dict(rec=ctx.upload_protein(inp.rec), lig=ctx.upload_protein(inp.lig),
              grid=ctx.build_grid(inp.rec, inp.params, inp.inner, inp.outer, PLATEAU, NEIGHBOURS),
              params=ctx.upload_params(inp.params))
    if lig_grid:
        hs["lig_grid"] = ctx.build_grid(inp.lig, inp.params, inp.lig_inner, inp.lig_outer, PLATEAU,
                                        0.0, src_is_ligand=True)
    return hs


def _pair_cases(case):
    """The pairs of a batch: sizes and pose counts spread below the case's."""
    rng = np.random.default_rng([case["pairs"], case["rec"], case["lig"], case["n"]])
    out = []
    for k in range(case["pairs"]):
        out.append(dict(kind="batch", rec=int(case["rec"] * rng.uniform(0.3, 1.0)),
                        lig=max(40, int(case["lig"] * rng.uniform(0.25, 1.0))),
                        mr=int(rng.integers(0, case["mr"] + 1)), ml=int(rng.integers(0, case["ml"] + 1)),
                        n=max(1, int(case["n"] * rng.uniform(0.2, 1.0)))))
    return out


def _inputs(case, seed):
    if case["kind"] == "batch":
        return [_Inputs(c, seed + 1000 * (k + 1)) for k, c in enumerate(_pair_cases(case))]
    return _Inputs(case, seed)


def _grid_inputs(case, seed):
    _, W = _package()
    R = W.scaled_radius(case["rec"], W.DENSITY_REF)
    body = W.make_body(seed, 0, case["rec"], R, TYPES, CHARGED)
    geom = W.cube_geom((0.0, 0.0, 0.0), R + 10.0, 0.875)
    return body, W.make_params(seed, TYPES, shape=case["shape"]), geom


def prepare(case, seed):
    hip, _ = _package()
    s = _State()
    s.case, s.kind = case, case["kind"]
    s.ctx = ctx = hip.Context(0)
    dev = "cuda"
    if s.kind == "grid":
        s.body, s.params, s.geom = _grid_inputs(case, seed)
        return s
    if s.kind == "batch":
        s.dofs, s.outs, pairs = [], [], []
        for inp in _inputs(case, seed):
            hs = _upload(ctx, inp, False)
            s.dofs.append(torch.from_numpy(inp.dofs).to(dev))
            s.outs.append(torch.zeros(inp.dofs.shape[0], 27 if inp.flexible else 7, device=dev))
            pairs.append(dict(hs=hs, d_dofs=s.dofs[-1].data_ptr(), d_out=s.outs[-1].data_ptr(),
                              n=inp.dofs.shape[0], modes=inp.flexible))
        torch.cuda.synchronize()  # the batch sorts the poses when it is made
        s.batch = ctx.batch(pairs)
        s.batch.tune()
        return s
    inp = _inputs(case, seed)
    s.hs = _upload(ctx, inp, s.kind == "modes")
    s.n, s.flexible = case["n"], inp.flexible
    if case.get("host"):
        s.dofs = inp.dofs
        return s
    width = 27 if inp.flexible else 7
    s.dofs = torch.from_numpy(inp.dofs).to(dev)
    s.out = torch.zeros(s.n, width, device=dev)
    if s.kind == "minimize":
        s.out = torch.zeros_like(s.dofs)
        s.energy, s.best = torch.zeros(s.n, device=dev), torch.zeros(s.n, device=dev)
        s.nfun = torch.zeros(s.n, dtype=torch.int32, device=dev)
    if s.kind in ("adjoint", "noalloc"):
        s.w = torch.from_numpy(inp.weights).to(dev) if case["w"] else None
        s.pgrad = None
        if case["pgrad"]:
            s.pgrad = torch.zeros(TYPES * TYPES, 3, device=dev)
            inp.rec_inner_basis, inp.rec_outer_basis = inp.basis(inp.inner), inp.basis(inp.outer)
            ctx.upload_basis(s.hs["grid"], inp)
    torch.cuda.synchronize()
    return s


def run(s):
    c, ctx = s.case, s.ctx
    if s.kind == "grid":
        return ctx.generate_grid(s.body, s.params, s.geom, PLATEAU)
    if s.kind == "batch":
        s.batch.run()
        return s.outs
    if s.kind == "minimize":
        ctx.minimize_dev(s.hs, s.dofs.data_ptr(), s.flexible, s.n, c["evals"], s.out.data_ptr(),
                         s.energy.data_ptr(), s.best.data_ptr(), s.nfun.data_ptr())
        return [s.out, s.energy, s.best, s.nfun]
    if s.kind in ("adjoint", "noalloc"):
        call = ctx.adjoint_dev if s.kind == "adjoint" else ctx.adjoint_dev_noalloc
        call(s.hs, s.dofs.data_ptr(), s.flexible, s.n, None if s.w is None else s.w.data_ptr(),
             s.out.data_ptr(), None if s.pgrad is None else s.pgrad.data_ptr())
        return [s.out] if s.pgrad is None else [s.out, s.pgrad]
    if s.kind == "rigid":
        if c["host"]:
            return ctx.score_rigid(s.hs, s.dofs)
        ctx.score_rigid_dev(s.hs, s.dofs.data_ptr(), s.n, s.out.data_ptr())
        return s.out
    if c["host"]:
        out = ctx.score_modes(s.hs, s.dofs)
    else:
        ctx.score_modes_dev(s.hs, s.dofs.data_ptr(), s.n, s.out.data_ptr())
        out = s.out
    # the mode gradients apart: their fourth power dwarfs (and overflows) all else
    return [out[:, :7], out[:, 7:]]


# ---------------------------------------------------------------- least work

def _radius(n, ref):
    return ref[1] * (n / ref[0]) ** (1.0 / 3.0)


def work(case):
    """Inputs read once and outputs written once; the grid values counted at
    most once each (few poses touch fewer: 8 corners per lookup), lists
    likewise; floating-point operations of the transform, the interpolation
    and the listed pairs (about 6 per ligand bead on these shells)."""
    if case["kind"] == "grid":
        side = (2 * _radius(case["rec"], (1000, 25.0)) + 20.0) / 0.875 + 2
        pts = side ** 3
        return dict(bytes=pts * (TYPES + 1) * 16 + 20 * case["rec"],
                    flops=pts * (case["rec"] * 30.0 + TYPES * TYPES * 20.0))
    if case["kind"] == "batch":
        parts = [work(dict(c, kind="adjoint", w=False, pgrad=False)) for c in _pair_cases(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    rec, lig, mr, ml, n = case["rec"], case["lig"], case["mr"], case["ml"], case["n"]
    flexible = case["kind"] == "modes" or mr > 0 or ml > 0
    if case["kind"] == "minimize":
        n = n * case["evals"]
    forward = case["kind"] in ("rigid", "modes")
    R = _radius(rec, (1000, 25.0))
    side = (2 * R + 20.0) / 0.875 + 2
    channels = 4 if forward else 1
    bodies = (20 + 12 * mr) * rec + (20 + 12 * ml) * lig
    io = (212 if flexible else 52) * case["n"] + (4 * n if case.get("w") else 0)
    grid = min(side ** 3 * (TYPES + 1) * 4 * channels, n * lig * (1 + CHARGED) * 32 * channels)
    lists = min(side ** 3 * 8 + 40 * 4 * side ** 3, n * lig * (8 + 6 * 4))
    look = (1 + CHARGED) * (25 + 16 * channels)
    flops = n * (lig * (18 + 6 * ml + look + 30) + 6.0 * lig * (60 + 12 * mr))
    if case["kind"] == "modes":  # the receptor on the ligand's grids
        grid += min(2e7, n * rec * (1 + CHARGED) * 128)
        flops += n * rec * (33 + 12 * mr + look)
    if case.get("pgrad"):
        grid += min(side ** 3 * 2 * TYPES * 4, n * lig * 2 * TYPES * 32)
        flops += n * lig * 24 + min(side ** 3 * TYPES, n * lig) * 2 * TYPES * 16
    return dict(bytes=float(bodies + io + grid + lists), flops=float(flops))


# ------------------------------------------------- the same results in 64 bits

def _rot(ang):
    phi, ssi, rot = ang[:, 0], ang[:, 1], ang[:, 2]
    cs, cp, ss, sp, cr, sr = ssi.cos(), phi.cos(), ssi.sin(), phi.sin(), rot.cos(), rot.sin()
    rows = [cr * cs * cp + sr * sp, sr * cs * cp - cr * sp, ss * cp,
            cr * cs * sp - sr * cp, sr * cs * sp + cr * cp, ss * sp, -cr * ss, -sr * ss, cs]
    return torch.stack(rows, 1).reshape(-1, 3, 3)


class _Grid64:
    """An inner and an outer potential grid, as 64-bit interpolants."""

    def __init__(self, parts, per_point):
        self.parts = [(g, torch.from_numpy(v).to("cuda").reshape(-1, g.nz, g.ny, g.nx, per_point))
                      for g, v in parts]

    @staticmethod
    def inside(g, p):
        lo = torch.tensor([g.ox, g.oy, g.oz], device=p.device, dtype=p.dtype)
        n = torch.tensor([g.nx, g.ny, g.nz], device=p.device, dtype=p.dtype)
        return ((p >= lo) & (p <= lo + (n - 1) * g.spacing)).all(-1)

    @staticmethod
    def cell(g, p):
        lo = torch.tensor([g.ox, g.oy, g.oz], device=p.device, dtype=p.dtype)
        top = torch.tensor([g.nx - 2, g.ny - 2, g.nz - 2], device=p.device)
        u = (p - lo) / g.spacing
        i = torch.minimum(u.detach().floor().long().clamp(min=0), top)
        return i, u - i

    def at(self, p, grid, channels):
        """Values (m, channels) at points (m, 3) of grids (m,); 0 outside both."""
        out = torch.zeros(p.shape[0], channels, device=p.device, dtype=p.dtype)
        free = torch.ones(p.shape[0], dtype=torch.bool, device=p.device)
        for g, v in self.parts:
            use = (free & self.inside(g, p.detach())).nonzero()[:, 0]
            free[use] = False
            i, f = self.cell(g, p[use])
            val = 0.0
            for dz in (0, 1):
                for dy in (0, 1):
                    for dx in (0, 1):
                        w = (f[:, 0] if dx else 1 - f[:, 0]) * (f[:, 1] if dy else 1 - f[:, 1]) \
                            * (f[:, 2] if dz else 1 - f[:, 2])
                        c = v[grid[use], i[:, 2] + dz, i[:, 1] + dy, i[:, 0] + dx, -channels:]
                        val = val + w[:, None] * c.double()
            out = out.index_add(0, use, val) if use.numel() else out
        return out

    def weights(self, p, typ, types):
        """Per grid: flat index over (type, z, y, x) and weight of the 8 corners."""
        free = torch.ones(p.shape[0], dtype=torch.bool, device=p.device)
        for g, v in self.parts:
            use = (free & self.inside(g, p)).nonzero()[:, 0]
            free[use] = False
            i, f = self.cell(g, p[use])
            for k in range(8):
                d = [(k >> b) & 1 for b in range(3)]
                w = 1.0
                for a in range(3):
                    w = w * (f[:, a] if d[a] else 1 - f[:, a])
                yield g, v, use, ((i[:, 2] + d[2]) * g.ny + i[:, 1] + d[1]) * g.nx + i[:, 0] + d[0], w


class _Pair64:
    """Scoring of one pair in 64 bits with torch."""

    def __init__(self, ctx, inp, lig_grid=False, basis=False):
        dev = "cuda"
        gen = lambda body, g, lig: ctx.generate_grid(body, inp.params, g, PLATEAU, lig)  # noqa: E731
        self.grid = _Grid64([(g, gen(inp.rec, g, False)) for g in (inp.inner, inp.outer)], 4)
        if lig_grid:
            self.lig_grid = _Grid64([(g, gen(inp.lig, g, True)) for g in (inp.lig_inner, inp.lig_outer)], 4)
        if basis:
            self.basis = _Grid64([(g, inp.basis(g)) for g in (inp.inner, inp.outer)], 1)
        desc, lst = ctx.generate_nl(inp.rec, inp.inner, NEIGHBOURS)
        self.nl = inp.inner
        self.desc = torch.from_numpy(desc.astype(np.int64).reshape(-1, 2)).to(dev)
        self.list = torch.from_numpy(lst.astype(np.int64)).to(dev)
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).double()  # noqa: E731
        self.x, self.y = t(inp.lig.xyz.reshape(3, -1).T), t(inp.rec.xyz.reshape(3, -1).T)
        self.ml = t(inp.lig.modes.reshape(3, inp.lig.n, inp.lig.M).transpose(2, 1, 0))  # (M, n, 3)
        self.mr = t(inp.rec.modes.reshape(3, inp.rec.n, inp.rec.M).transpose(2, 1, 0))
        self.kl, self.kr = t(inp.lig.mode_force), t(inp.rec.mode_force)
        self.ql, self.qr = t(inp.lig.charge), t(inp.rec.charge)
        self.tl = torch.from_numpy(inp.lig.type.astype(np.int64)).to(dev)
        self.tr = torch.from_numpy(inp.rec.type.astype(np.int64)).to(dev)
        p = inp.params
        self.tab = {k: t(getattr(p, k)) for k in ("rc", "ac", "rmin2", "emin")}
        self.tab["ipon"] = t(p.ipon.astype(np.float32))
        self.fe, self.flexible = float(p.ffelec), inp.flexible

    def lj(self, r2, k, tab):
        i2 = 1.0 / r2
        i6 = i2 ** 3
        rep = tab["rc"][k] * i2
        v = (rep - tab["ac"][k]) * i6
        s = 6.0 * v + 2.0 * rep * i6
        near, ip = (r2 < tab["rmin2"][k]).double(), tab["ipon"][k]
        return near * (v + (ip - 1) * tab["emin"][k]) + (1 - near) * ip * v, (near + (1 - near) * ip) * s

    def place(self, d):
        """(R, receptor (n,N,3), ligand coordinates before and after the motion)."""
        R = _rot(d[:, 3:6])
        xt, y = self.x.expand(d.shape[0], -1, -1), self.y.expand(d.shape[0], -1, -1)
        if self.flexible:
            if len(self.ml):
                xt = xt + torch.einsum("pm,mic->pic", d[:, 16:16 + len(self.ml)], self.ml)
            if len(self.mr):
                y = y + torch.einsum("pm,mic->pic", d[:, 6:6 + len(self.mr)], self.mr)
        return R, y, xt, xt @ R.transpose(1, 2) + d[:, None, :3]

    def field(self, grid, p, typ, q, channels):
        n, m = p.shape[:2]
        flat, t = p.reshape(-1, 3), typ.expand(n, m).reshape(-1)
        v = grid.at(flat, t, channels)
        c = (q.abs() > 0.001).expand(n, m).reshape(-1).nonzero()[:, 0]
        el = grid.at(flat[c], torch.zeros_like(t[c]), channels) * q.expand(n, m).reshape(-1)[c][:, None]
        return v.index_add(0, c, el).reshape(n, m, channels)

    def pairs(self, p, y):
        """Listed pairs inside the plateau: (pose * m + bead, pose, receptor bead, difference)."""
        n, m = p.shape[:2]
        flat = p.detach().reshape(-1, 3)
        g = self.nl
        b = _Grid64.inside(g, flat).nonzero()[:, 0]
        lo = torch.tensor([g.ox, g.oy, g.oz], device=p.device, dtype=p.dtype)
        i = ((flat[b] - lo) / g.spacing + 0.5).floor().long()
        d = self.desc[(i[:, 2] * g.ny + i[:, 1]) * g.nx + i[:, 0]]
        cnt = d[:, 0]
        own = torch.repeat_interleave(torch.arange(len(b), device=p.device), cnt)
        at = torch.arange(len(own), device=p.device) - (cnt.cumsum(0) - cnt)[own] + d[own, 1]
        j, b = self.list[at], b[own]
        pose = b // m
        diff = p.reshape(-1, 3)[b] - y[pose, j]
        keep = ((diff.detach() ** 2).sum(1) <= PLATEAU ** 2).nonzero()[:, 0]
        return b[keep], pose[keep], j[keep], diff[keep]

    def pair_terms(self, b, j, diff, m, tab):
        """Per pair: energy above the plateau's, force, and their pieces."""
        l = b % m  # noqa: E741
        k = TYPES * (self.tr[j] - 1) + self.tl[l] - 1
        r2 = (diff ** 2).sum(1)
        P2 = torch.full_like(r2, PLATEAU ** 2)
        e, fb = self.lj(r2, k, tab)
        eP, fbP = self.lj(P2, k, tab)
        q = self.ql[l] * self.qr[j] * self.fe
        e = e - eP + q * (1.0 / r2 - 1.0 / P2)
        ratio = torch.sqrt(((r2.detach() * 10000).floor() + 0.5) / 10000 / PLATEAU ** 2)
        mag = fb / r2 + 2 * q / r2 ** 2 - ratio / r2 * (fbP + 2 * q / P2)
        return k, e, mag[:, None] * diff

    def forward(self, d):
        """The reference's energy, force, torque and mode gradients."""
        ang = d[:, 3:6].clone().requires_grad_(True)
        R, y, xt, p = self.place(d)
        n, m = p.shape[:2]
        f = self.field(self.grid, p, self.tl, self.ql, 4)
        b, pose, j, diff = self.pairs(p, y)
        _, e, pf = self.pair_terms(b, j, diff, m, self.tab)
        f = f.reshape(-1, 4).index_add(0, b, torch.cat([pf, e[:, None]], 1)).reshape(n, m, 4)
        F = f[..., :3].sum(1)
        for _ in range(3):
            F = torch.where((F * F).sum(1, keepdim=True) > 1e18, F * 0.01, F)
        T = torch.einsum("pik,il->pkl", f[..., :3], self.x)
        ga, = torch.autograd.grad((_rot(ang) * T).sum(), ang)
        out = [f[..., 3].sum(1, keepdim=True), F, ga]
        if self.flexible:
            inv = y @ _rot(-d[:, 3:6]).transpose(1, 2) - (d[:, None, :3] @ R)
            r = self.field(self.lig_grid, inv, self.tr, self.qr, 4)[..., :3] @ R.transpose(1, 2)
            r = r.reshape(-1, 3).index_add(0, pose * len(self.y) + j, -pf).reshape(n, -1, 3)
            for modes, k, g in ((self.mr, self.kr, r), (self.ml, self.kl, f[..., :3] @ R)):
                v = -torch.einsum("pic,mic->pm", g, modes)
                v = v + 4 * k * v ** 4
                out.append(torch.cat([v, torch.zeros(n, 10 - len(modes), device=d.device)], 1))
        return torch.cat(out, 1)

    def adjoint(self, d, w, pgrad):
        """Energy, its weighted gradient, and the weighted parameter gradient."""
        d = d.clone().requires_grad_(True)
        tab = self.tab
        if pgrad:
            tab = {k: v.clone().requires_grad_(k in ("rc", "ac", "emin")) for k, v in tab.items()}
        _, y, _, p = self.place(d)
        n, m = p.shape[:2]
        e = self.field(self.grid, p, self.tl, self.ql, 1).sum((1, 2))
        b, pose, j, diff = self.pairs(p, y)
        _, ep, _ = self.pair_terms(b, j, diff, m, tab)
        e = e.index_add(0, pose, ep)
        leaves = [d] + ([tab[k] for k in ("rc", "ac", "emin")] if pgrad else [])
        g = torch.autograd.grad((e * w).sum(), leaves)
        out = torch.cat([e.detach()[:, None], g[0] if self.flexible else g[0][:, :6]], 1)
        if not pgrad:
            return out, None
        pg = torch.stack(g[1:], 1)
        flat, tl = p.detach().reshape(-1, 3), self.tl.expand(n, m).reshape(-1)
        wt = w[:, None].expand(n, m).reshape(-1)
        ip = self.tab["ipon"].reshape(TYPES, TYPES)
        for g, v, use, at, cw in self.basis.weights(flat, tl, TYPES):
            npts = g.nx * g.ny * g.nz
            D = torch.zeros(TYPES * npts, device=d.device, dtype=torch.float64)
            D.index_add_(0, (tl[use] - 1) * npts + at, cw * wt[use])
            D = D.reshape(TYPES, npts)
            v = v.reshape(2 * TYPES, npts)
            for a in range(2 * TYPES):
                s = D @ v[a].double()
                pg.view(TYPES, TYPES, 3)[a // 2, :, a % 2] += ip[a // 2] * s * (1 if a % 2 == 0 else -1)
        return out, pg


def _chunks(n, cost):
    step = max(1, int(4e5 / cost))
    return [(a, min(n, a + step)) for a in range(0, n, step)]


def _exact_grid(case, seed):
    body, params, g = _grid_inputs(case, seed)
    dev = "cuda"
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).double()  # noqa: E731
    ax = [torch.arange(m, device=dev).double() * float(np.float32(g.spacing)) + float(np.float32(o))
          for m, o in ((g.nx, g.ox), (g.ny, g.oy), (g.nz, g.oz))]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    pts = torch.stack([x.reshape(-1), y.reshape(-1), z.reshape(-1)], 1)
    src, q = f(body.xyz.reshape(3, -1).T), f(body.charge) * float(np.float32(params.ffelec))
    one = torch.zeros(body.n, TYPES, device=dev, dtype=torch.float64)
    one[torch.arange(body.n), torch.from_numpy(body.type.astype(np.int64)) - 1] = 1.0
    ip = f(params.ipon.astype(np.float32)).reshape(TYPES, TYPES)
    rc, ac = f(params.rc).reshape(TYPES, TYPES) * ip, f(params.ac).reshape(TYPES, TYPES) * ip
    power = params.shape // 2
    out = torch.empty(TYPES + 1, pts.shape[0], 4, device=dev, dtype=torch.float64)
    for a in range(0, pts.shape[0], 16384):
        diff = pts[a:a + 16384, None] - src[None]
        r2 = (diff ** 2).sum(2)
        rp2 = r2.clamp(min=PLATEAU ** 2)
        u = diff / (r2.clamp(min=1e-300) * rp2).sqrt()[..., None] * (r2 > 0)[..., None]
        i6, js = rp2 ** -3, rp2 ** -power
        sl = slice(a, a + len(r2))
        out[1:, sl, 3] = ((js @ one) @ rc - (i6 @ one) @ ac).T
        dd = (1 / rp2 - 1 / 2500.0).clamp(min=0)
        out[0, sl, 3] = dd @ q
        fq = 2 / rp2 * (dd > 0) * q
        for c in range(3):
            s, t = (js * u[..., c]) @ one, (i6 * u[..., c]) @ one
            out[1:, sl, c] = (params.shape * (s @ rc) - 6.0 * (t @ ac)).T
            out[0, sl, c] = (fq * u[..., c]).sum(1)
    return out.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "minimize":
        return None  # a trajectory of rounded evaluations has no 64-bit value
    hip, _ = _package()
    if kind == "grid":
        return _exact_grid(case, seed).cpu().numpy()
    ctx = hip.Context(0)
    forward = kind in ("rigid", "modes")
    many = kind == "batch"
    outs = []
    for inp in _inputs(case, seed) if many else [_inputs(case, seed)]:
        P = _Pair64(ctx, inp, lig_grid=kind == "modes", basis=bool(case.get("pgrad")))
        n = inp.dofs.shape[0]
        d = torch.from_numpy(inp.dofs).to("cuda").double()
        w = torch.ones(n, device="cuda", dtype=torch.float64)
        if case.get("w"):
            w = torch.from_numpy(inp.weights).to("cuda").double()
        rows, pg = [], None
        for a, b in _chunks(n, inp.lig.n + (inp.rec.n if inp.flexible else 0)):
            if forward:
                rows.append(P.forward(d[a:b]))
            else:
                o, g = P.adjoint(d[a:b], w[a:b], bool(case.get("pgrad")))
                rows.append(o)
                pg = g if pg is None or g is None else pg + g
        outs.append(torch.cat(rows))
    if kind == "modes":
        return [outs[0][:, :7], outs[0][:, 7:].float().double()]  # overflows as the results do
    if forward:
        return outs[0]
    return outs if many or not case["pgrad"] else [outs[0], pg]
