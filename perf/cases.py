"""The work a program that uses this framework has it do, as timed cases.

A pass advances one simulation, or an ensemble of them in shared launches, a
number of steps through the public entry points (`Session`, its scene and
backend, `time_integrate`) and takes the state back to the host.  The scenes
are the repository's own configurations over the range of sizes its tests, its
benchmark and its served job stream use: a few hundred particles to 1.4
million, one scene to 64 together, 2D and 3D, both precisions, leapfrog and
RK4, fluid, elasto-plastic and visco-plastic material, walls of boundary
particles and ghost mirrors.

`exact` integrates the same scenes in 64-bit torch from the same initial
arrays, by its own pair search and its own formulas.

A session in "f32" mode sums FP32 pair terms over FP64 positions: its program
keeps positions in double and the fields in single precision.  A session in
"f64" mode keeps all of them in double.
"""
import math

import numpy as np
import torch

import __graft_entry__

G = __graft_entry__.package()
A = G._abi

# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
# scene     : configuration builder (and `size`, its parameters)
# precision : arithmetic of the pair sums
# steps     : steps of a pass
# restart   : the pass starts from the saved state, uploaded again (a restart,
#             or one run of a parameter study); otherwise it goes on from where
#             the last pass ended, as a long run does between two saves
# entry     : "step_many" (the session's backend with graph replay, as the
#             benchmark and the server drive it) or "time_integrate" (the whole
#             call with its defaults)


def listed():
    return [
        # the smallest scene of the test-suite: launches and latency count
        _case("dambreak2d-tiny", "dambreak_2d", dx=0.05, steps=20, restart=True),
        # the 2D dam break of the configurations, through the whole call
        _case("dambreak2d-whole-call", "dambreak_2d", dx=0.01, steps=100, restart=True,
              entry="time_integrate"),
        # double precision at a ragged size (no extent is a multiple of dx)
        _case("dambreak2d-f64", "dambreak_2d", dx=0.0137, steps=50, precision="f64", restart=True),
        _case("dambreak3d-f64", "dambreak_3d", dx=0.0213, steps=40, precision="f64", restart=True),
        # a 3D dam break of ordinary size, and the benchmark's 1.4 million
        _case("dambreak3d-medium", "dambreak_3d", dx=0.012, steps=50, restart=True),
        _case("dambreak3d-full", "dambreak_3d", dx=0.006, steps=100),
        # one elasto-plastic column with ghost walls (two stages a step)
        _case("column2d", "ep_column_2d", dx=0.0025, width=0.4, height=0.2, steps=50, restart=True),
        _case("column2d-f64", "ep_column_2d", dx=0.0025, width=0.1575, height=0.0925, steps=25,
              precision="f64", restart=True),
        # a parameter study: 64 columns advanced in shared launches
        _case("columns2d-64", "ensemble_columns", dx=0.0025, sims=64, steps=100),
        # 3D visco-plastic columns as the served stream has them
        _case("column3d-small", "granular_column_3d", dx=0.005, width=0.2, depth=0.05, height=0.1,
              steps=25, restart=True),
        _case("column3d-served", "granular_column_3d", dx=0.005, width=0.4, depth=0.15, height=0.3,
              steps=25),
        # two phases, RK4 with XSPH, eight ghost mirrors
        _case("bubble2d-rk4", "bubble_2d", dx=0.05, variant="bubble3", steps=10, restart=True),
    ]


def _case(name, scene, steps, precision="f32", restart=False, entry="step_many", **size):
    return {"name": name, "scene": scene, "precision": precision, "steps": steps,
            "restart": restart, "entry": entry, **size}


def draw(rng):
    def log(a, b):
        return math.exp(rng.uniform(math.log(a), math.log(b)))

    scene = rng.choice(["dambreak_2d", "dambreak_3d", "ep_column_2d", "ensemble_columns",
                        "granular_column_3d", "bubble_2d"])
    precision = "f64" if rng.random() < 0.25 else "f32"
    size = {}
    if scene == "dambreak_2d":
        size, steps = {"dx": log(0.006, 0.06)}, rng.randint(20, 100)
    elif scene == "dambreak_3d":
        size, steps = {"dx": log(0.0075, 0.05)}, rng.randint(20, 60)
    elif scene == "ep_column_2d":
        size = {"dx": log(0.0015, 0.006), "width": rng.uniform(0.1, 0.4)}
        size["height"] = size["width"] * rng.uniform(0.3, 1.5)
        steps = rng.randint(20, 60)
    elif scene == "ensemble_columns":
        size, steps = {"dx": 0.0025, "sims": rng.randint(2, 40)}, rng.randint(20, 50)
    elif scene == "granular_column_3d":
        size = {"dx": log(0.004, 0.01), "width": rng.uniform(0.1, 0.35),
                "depth": rng.uniform(0.04, 0.15), "height": rng.uniform(0.06, 0.25)}
        steps = rng.randint(20, 50)
    else:
        size = {"dx": log(0.03, 0.12), "variant": rng.choice(["bubble", "bubble3"])}
        steps = rng.randint(5, 20)
    one = scene != "ensemble_columns"
    c = _case("", scene, steps, precision=precision, restart=one,
              entry="time_integrate" if one and rng.random() < 0.2 else "step_many",
              **{k: round(v, 5) if isinstance(v, float) else v for k, v in size.items()})
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Scenes
# ---------------------------------------------------------------------------
_OWN = ("name", "scene", "precision", "steps", "restart", "entry", "sims")


def _build(case):
    kw = {k: v for k, v in case.items() if k not in _OWN}
    if case["scene"] == "ensemble_columns":
        return G.configs.ensemble_columns(n_sims=case["sims"], **kw)
    return [getattr(G.configs, case["scene"])(**kw)]


def _moving(cfg):
    """The systems that move (boundary particles rest)."""
    return [ps for ps in cfg["integrator"].systems if ps.source_v.any()]


def _scene(case, seed):
    """The configuration with its particles off the lattice and in motion, as
    they are some time into a run: positions scattered by up to 5 % of the
    spacing, a smooth velocity field of a fraction of sqrt(g·height), densities
    and stresses scattered by a little."""
    cfgs = _build(case)
    for k, cfg in enumerate(cfgs):
        rng = np.random.default_rng([seed, k])
        for ps in _moving(cfg):
            lo, ext = ps.x.min(0), np.ptp(ps.x, axis=0)
            amp = 0.15 * math.sqrt(9.81 * ext[-1])
            dx = (ps.mass / ps.rho[0]) ** (1.0 / ps.ndims)
            s = (ps.x - lo) / np.maximum(ext, dx)
            for d in range(ps.ndims):
                w = rng.uniform(-1.0, 1.0, (3, ps.ndims)) * math.pi
                ph = rng.uniform(0.0, 2.0 * math.pi, 3)
                ps.v[:, d] = amp / 3.0 * np.sin(s @ w.T + ph).sum(1)
            ps.x += rng.uniform(-0.05, 0.05, ps.x.shape) * dx
            ps.rho *= 1.0 + rng.uniform(-1e-4, 1e-4, ps.n)
            if ps.kind >= A.GR_SYS_STRESS:
                ps.stress *= 1.0 + rng.uniform(-0.01, 0.01, ps.stress.shape)
    return cfgs


def _fields(ps):
    """The updated state of a system a program keeps."""
    return ["x", "v", "rho"] + (["stress"] if ps.kind >= A.GR_SYS_STRESS else ["p"])


def _kept(case, name, a):
    return a if name == "x" or case["precision"] == "f64" else a.astype(np.float32)


def prepare(case, seed):
    cfgs = _scene(case, seed)
    ndims = cfgs[0]["integrator"].ndims
    s = G.Session(ndims, case["precision"])
    moving = [ps for cfg in cfgs for ps in _moving(cfg)]
    st = {"case": case, "session": s, "cfgs": cfgs, "moving": moving}
    if case["entry"] == "time_integrate":
        st["saved"] = [(ps, [(f, getattr(ps, f).copy()) for f in ps.field_names() + ["id"]])
                       for ps in moving]
        return st
    s.backend.set_graph_mode(True)
    st["handles"] = []
    for cfg in cfgs:
        h = s.scene.integrator(cfg["integrator"])
        s.scene.upload_all(cfg["integrator"])
        s.backend.integrator_set_dt(h, s.backend.integrator_dt(h, cfg["cfl"]))
        st["handles"].append(h)
    return st


def run(st):
    case, moving = st["case"], st["moving"]
    be, sc = st["session"].backend, st["session"].scene
    if case["entry"] == "time_integrate":
        for ps, saved in st["saved"]:
            for f, a in saved:
                getattr(ps, f)[...] = a
        cfg = st["cfgs"][0]
        G.time_integrate(cfg["integrator"], case["steps"], 0, 0, cfg["cfl"], None,
                         print_timer=False, session=st["session"])
        got = [{**{f: getattr(ps, f) for f in _fields(ps)}, "id": ps.id} for ps in moving]
    else:
        if case["restart"]:
            for ps in moving:
                sc.upload(ps)
        be.step_many(st["handles"], case["steps"])
        got = []
        for ps in moving:
            h = sc.system(ps)
            out = {f: be.system_download(h, A.FIELD_IDS[f], getattr(ps, f).size)
                   .reshape(getattr(ps, f).shape) for f in _fields(ps)}
            out["id"] = be.system_download_index(h, A.GR_I_ID, ps.n)
            got.append(out)
    return _outputs(case, got)


def _outputs(case, got):
    """{field: values}, an ensemble's systems one after another."""
    if case["scene"] == "ensemble_columns":
        got = [{f: np.concatenate([g[f] for g in got]) for f in got[0]}]
    return [{f: _kept(case, f, a) for f, a in g.items()} for g in got]


def work(case):
    """A step reads and writes the moving particles' state once, reads the
    resting ones' positions, and evaluates each particle's partners; a pass
    takes the saved state in (restart) and the kept fields out."""
    nbytes = flops = 0.0
    for cfg in _build(case):
        lf = cfg["integrator"]
        D, two = lf.ndims, len(lf.interactions[0].pfns)
        kern = lf.interactions[0].kernel
        r = 8 if case["precision"] == "f64" else 4
        passes = 4 if lf.scheme == A.GR_SCHEME_RK4 else 1
        for ps in lf.systems:
            if ps not in _moving(cfg):
                nbytes += case["steps"] * ps.n * 8 * D
                continue
            state = ps.n * 8.0 * sum(getattr(ps, f).size // ps.n for f in ps.field_names()
                                     if f not in ("dvdt", "drhodt", "v_adjustment", "p",
                                                  "strain_rate", "vorticity"))
            dx = (ps.mass / ps.rho[0]) ** (1.0 / D)
            q = 2.0 * kern.h / dx
            partners = (math.pi * q * q if D == 2 else 4.0 / 3.0 * math.pi * q ** 3) - 1.0
            per_pair = (45 + 80) if two == 2 else 59
            nbytes += case["steps"] * 2.0 * state + ps.n * 8.0
            nbytes += ps.n * sum(getattr(ps, f).size // ps.n * (8 if f == "x" else r)
                                 for f in _fields(ps))
            nbytes += state if case["restart"] else 0.0
            flops += case["steps"] * passes * ps.n * partners * per_pair
    return {"bytes": float(nbytes), "flops": float(flops)}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------


def exact(case, seed):
    cfgs = _scene(case, seed)
    # about 20 s: pair evaluations (about 40 tensor operations each) and the
    # overhead of the operations themselves
    pairs = work(case)["flops"] / 59
    if pairs > 1.5e10 or (not torch.cuda.is_available() and pairs > 1e8) or len(cfgs) > 8:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    got = []
    for cfg in cfgs:
        lf = cfg["integrator"]
        sim = _Exact(lf, cfg["cfl"], dev)
        for _ in range(case["steps"]):
            sim.step()
        for ps in _moving(cfg):
            s = sim.sys[id(ps)]
            got.append({f: s[f][s["perm"]].cpu().numpy().reshape(getattr(ps, f).shape)
                        for f in _fields(ps)} | {"id": ps.id[s["perm"].cpu().numpy()]})
    if case["scene"] == "ensemble_columns":
        got = [{f: np.concatenate([g[f] for g in got]) for f in got[0]}]
    return got


def _near(xa, xb, cut):
    """Index pairs (a, b) with |xa - xb| < cut."""
    D = xa.shape[1]
    lo = torch.minimum(xa.min(0).values, xb.min(0).values) - 1.5 * cut
    hi = torch.maximum(xa.max(0).values, xb.max(0).values) + 1.5 * cut
    ng = ((hi - lo) / cut).floor().long() + 1
    stride = torch.ones_like(ng)
    for d in range(D - 2, -1, -1):
        stride[d] = stride[d + 1] * ng[d + 1]
    ca = ((xa - lo) / cut).floor().long()
    kb = (((xb - lo) / cut).floor().long() * stride).sum(1)
    kb, order = torch.sort(kb)
    found_i, found_j = [], []
    for o in range(3 ** (D - 1)):
        off = [o // 3 - 1, o % 3 - 1][-(D - 1):]
        base = sum((ca[:, d] + off[d]) * stride[d] for d in range(D - 1)) + ca[:, D - 1]
        first = torch.searchsorted(kb, base - 1)
        n = torch.searchsorted(kb, base + 1, right=True) - first
        i = torch.repeat_interleave(torch.arange(len(xa), device=xa.device), n)
        start = torch.cumsum(n, 0) - n
        j = order[first[i] + torch.arange(len(i), device=xa.device) - start[i]]
        keep = ((xa[i] - xb[j]) ** 2).sum(1) < cut * cut
        found_i.append(i[keep])
        found_j.append(j[keep])
    return torch.cat(found_i), torch.cat(found_j)


def _scalar(a, b):
    return (a * b).sum(1, keepdim=True)


class _Exact:
    """Leapfrog or RK4 steps of one simulation.  Particles keep their initial
    order; `perm` is the order the cell sorts have brought them into."""

    def __init__(self, lf, cfl, dev):
        self.lf, self.dev, self.D = lf, dev, lf.ndims
        self.dt = cfl * lf.h / lf.c
        self.sys, self.lists = {}, {}
        for ps in lf.systems:
            s = {f: self.t(getattr(ps, f)) for f in ps.field_names()}
            for f in ("rho", "drhodt", "p", "vorticity"):
                if f in s and s[f].dim() == 1:
                    s[f] = s[f][:, None]
            s["perm"] = torch.arange(ps.n, device=dev)
            self.sys[id(ps)] = s

    def t(self, a):
        return torch.tensor(np.asarray(a, dtype=np.float64), device=self.dev)

    # ---- one step ------------------------------------------------------------
    def order(self, x, perm):
        """`perm` sorted stably by the cells of its particles, first
        coordinate slowest."""
        c = torch.floor(x[perm] / (2.0 * self.lf.h)).long()
        c -= c.min(0).values
        key = torch.zeros(len(perm), dtype=torch.long, device=self.dev)
        for d in range(self.D):
            key = key * (c[:, d].max() + 1) + c[:, d]
        return perm[torch.sort(key, stable=True).indices]

    def step(self):
        lf, dt = self.lf, self.dt
        for ps in lf.systems:
            s = self.sys[id(ps)]
            s["perm"] = self.order(s["x"], s["perm"])
        self.make_ghosts()
        self.pairs = [self.find(si) for si in lf.interactions]
        real = [(ps, self.sys[id(ps)]) for ps in lf.systems]
        if lf.scheme == A.GR_SCHEME_RK4:
            for _, s in real:
                s["acc"] = [torch.zeros_like(s["v"]), torch.zeros_like(s["rho"])]
            for adv, w in ((0.0, 1 / 6), (0.5, 1 / 3), (0.5, 1 / 3), (1.0, 1 / 6)):
                self.sweep_stages(adv)
                for _, s in real:
                    s["acc"] = [s["acc"][0] + w * s["dvdt"], s["acc"][1] + w * s["drhodt"]]
            for _, s in real:
                s["v"] = s["v"] + dt * s["acc"][0]
                s["rho"] = s["rho"] + dt * s["acc"][1]
        else:
            self.sweep_stages(0.5)
            for ps, s in real:
                s["v"] = s["v"] + dt * s["dvdt"]
                s["rho"] = s["rho"] + dt * s["drhodt"]
        if any(si.vadjust_pfn is not None for si in lf.interactions):
            self.xsph()
        for _, s in real:
            s["x"] = s["x"] + dt * s["v"]

    def sweep_stages(self, adv):
        """Rates of the state q0 + adv·dt·dq/dt."""
        lf = self.lf
        for ps in lf.systems:
            s = self.sys[id(ps)]
            s["vh"] = s["v"] + adv * self.dt * s["dvdt"]
            s["rh"] = s["rho"] + adv * self.dt * s["drhodt"]
            s["dvdt"] = self.t(ps.source_v).expand(ps.n, -1).clone()
            s["drhodt"] = torch.full_like(s["rho"], float(ps.source_rho))
        for ge in lf.ghosts:
            g, src = self.sys[id(ge.ghost)], self.sys[id(ge.ghost.source)]
            v = src["vh"][g["of"]]
            g["vh"] = v - 2.0 * _scalar(v, g["n"]) * g["n"]
            g["rh"] = src["rh"][g["of"]]
        nst = len(lf.interactions[0].pfns)
        for k in range(nst):
            for ps in lf.systems:
                if len(ps.state_updater) == nst:
                    ups = ps.state_updater[k]
                    for u in ups if isinstance(ups, tuple) else (ups,):
                        if u is not None:
                            self.update(ps, self.sys[id(ps)], u)
            for ge in lf.ghosts:
                cop = ge.ghost.updaters[k] if k < len(ge.ghost.updaters) else None
                if cop is not None:
                    self.copy_to_ghost(ge, cop)
            for si, pr in zip(lf.interactions, self.pairs):
                if si.pfns[k] is not None:
                    self.sweep(si, si.pfns[k], pr)

    # ---- ghosts --------------------------------------------------------------
    def make_ghosts(self):
        for ge in self.lf.ghosts:
            src = self.sys[id(ge.ghost.source)]
            xs, of, nrm = [], [], []
            for n, p in zip(ge.normals, ge.points):
                n, p = self.t(n)[None], self.t(p)[None]
                x = src["x"][src["perm"]]
                da = _scalar(x - p, n)
                hit = ((da.abs() <= ge.cutoff) & (da > 0.0))[:, 0]
                xs.append((x - 2.0 * da * n)[hit])
                of.append(src["perm"][hit])
                nrm.append(n.expand(int(hit.sum()), -1))
            xs, of, nrm = torch.cat(xs), torch.cat(of), torch.cat(nrm)
            o = (self.order(xs, torch.arange(len(xs), device=self.dev)) if len(xs)
                 else torch.arange(0, device=self.dev))
            g = self.sys.setdefault(id(ge.ghost), {})
            # the sort moves positions and sources; slot k keeps its normal
            g.update(x=xs[o], of=of[o], n=nrm, p=torch.zeros(len(xs), 1, device=self.dev,
                                                             dtype=torch.float64))

    def copy_to_ghost(self, ge, cop):
        g, src = self.sys[id(ge.ghost)], self.sys[id(ge.ghost.source)]
        for f, mode in zip(cop.fields, cop.modes):
            val = src[f][g["of"]]
            if mode == A.GR_COPY_HOUSEHOLDER:
                n = torch.zeros(len(val), 3, dtype=torch.float64, device=self.dev)
                n[:, :self.D] = g["n"]
                hm = torch.eye(3, dtype=torch.float64, device=self.dev) \
                    - 2.0 * n[:, :, None] * n[:, None, :]
                t = self.tensor(val)
                val = self.voigt(hm @ t @ hm, val.shape[1])
            g[f] = val

    _AT = {3: [(0, 0), (1, 1), (0, 1)], 4: [(0, 0), (1, 1), (2, 2), (0, 1)],
           6: [(0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2)]}

    def tensor(self, s):
        t = torch.zeros(len(s), 3, 3, dtype=torch.float64, device=self.dev)
        for k, (a, b) in enumerate(self._AT[s.shape[1]]):
            t[:, a, b] = s[:, k]
            t[:, b, a] = s[:, k]
        return t

    def voigt(self, t, ns):
        return torch.stack([t[:, a, b] for a, b in self._AT[ns]], 1)

    # ---- pairs ---------------------------------------------------------------
    def other(self, si):
        b = si.system_b
        return b if b is None else getattr(b, "inner", b)

    def find(self, si):
        """(i, j) of an interaction's pairs within 2h; candidates are kept
        while no particle has moved far (not for ghosts)."""
        a = self.sys[id(si.system_a)]
        b = self.other(si)
        sb = a if b is None else self.sys[id(b)]
        cut = 2.0 * si.kernel.h
        none = torch.zeros(0, dtype=torch.long, device=self.dev)
        if len(sb["x"]) == 0:
            return none, none
        skin = 0.0 if "of" in sb else 0.1 * cut
        at = self.lists.get(id(si))
        if at is None or not skin or max(float((a["x"] - at[2]).abs().max()),
                                         float((sb["x"] - at[3]).abs().max())) > 0.02 * cut:
            i, j = _near(a["x"], sb["x"], cut + skin)
            if b is None:
                keep = i != j
                i, j = i[keep], j[keep]
            at = self.lists[id(si)] = (i, j, a["x"], sb["x"])
        i, j = at[0], at[1]
        keep = ((a["x"][i] - sb["x"][j]) ** 2).sum(1) < cut * cut
        return i[keep], j[keep]

    def gradient(self, kern, dx):
        r = torch.sqrt(_scalar(dx, dx))
        q = r / kern.h
        C = kern.norm_coeff
        if kern.kind == A.GR_KERNEL_CUBIC:
            dw = -3.0 * C * (0.25 * (2.0 - q).clamp(min=0) ** 2 - (1.0 - q).clamp(min=0) ** 2)
            w = C * (0.25 * (2.0 - q).clamp(min=0) ** 3 - (1.0 - q).clamp(min=0) ** 3)
        else:
            t = (2.0 - q).clamp(min=0)
            dw = -10.0 * C * q * t ** 3
            w = C * t ** 4 * (2.0 * q + 1.0)
        return dw / (r * kern.h) * dx, _scalar(dx, dx), w

    def sweep(self, si, fn, pr):
        i, j = pr
        if len(i) == 0:
            return
        ps, b = si.system_a, self.other(si)
        sa = self.sys[id(ps)]
        sb = sa if b is None else self.sys[id(b)]
        ghost = b is not None and "of" in sb
        dyn = isinstance(si.system_b, G.DynamicBoundarySystem)
        dx = sa["x"][i] - sb["x"][j]
        g, r2, _ = self.gradient(si.kernel, dx)
        vi, ri = sa["vh"][i], sa["rh"][i]
        if dyn:
            n, p = self.t(si.system_b.boundary_normal), self.t(si.system_b.boundary_point)
            da = ((sa["x"][i] - p) * n).sum(1, keepdim=True)
            db = ((sb["x"][j] - p) * n).sum(1, keepdim=True)
            vj = -torch.clamp((db / da).abs(), max=si.system_b.boundary_beta) * vi
            rj = ri
        else:
            vj, rj = sb["vh"][j], sb["rh"][j]
        m_j = ps.mass if (b is None or dyn or ghost) else b.mass
        if isinstance(fn, (G.StrainRatePfn, G.StrainRateVorticityPfn)):
            dv = vj - vi
            lg = dv[:, :, None] * g[:, None, :] * (m_j / rj)[:, :, None]
            full = torch.zeros(len(i), 3, 3, dtype=torch.float64, device=self.dev)
            full[:, :self.D, :self.D] = 0.5 * (lg + lg.transpose(1, 2))
            sa["strain_rate"] = sa["strain_rate"].index_add(0, i, self.voigt(full, ps.ns))
            if isinstance(fn, G.StrainRateVorticityPfn):
                at = [(0, 1)] if self.D == 2 else [(0, 1), (0, 2), (1, 2)]
                w = torch.stack([0.5 * (lg[:, p, q] - lg[:, q, p]) for p, q in at], 1)
                sa["vorticity"] = sa["vorticity"].index_add(0, i, w)
            return
        two = b is not None and not dyn and not ghost
        c = 0.5 * (ps.c + (b.c if two else ps.c))
        dv = vi - vj
        mu = fn.h * _scalar(dx, dv).clamp(max=0.0) / (r2 + 0.01 * fn.h * fn.h)
        visc = (fn.art_visc_beta * mu - fn.art_visc_alpha * c) * mu / (0.5 * ri * rj)
        dr = _scalar(dv, g)
        if isinstance(fn, G.CauchyFluidPfn):
            D = self.D
            ti = self.tensor(sa["stress"])[i][:, :D, :D]
            tj = ti if dyn else self.tensor(sb["stress"])[j][:, :D, :D]
            acc = ((ti / (ri * ri)[:, :, None] + tj / (rj * rj)[:, :, None]) @ g[:, :, None])[:, :, 0]
            acc = acc - visc * g
            sa["dvdt"] = sa["dvdt"].index_add(0, i, m_j * acc)
            sa["drhodt"] = sa["drhodt"].index_add(0, i, m_j * dr)
            return
        pi = sa["p"][i]
        pj = pi if dyn else sb["p"][j]
        if fn.sigma == 1:
            t = -(pi + pj) / (ri * rj)
        else:
            t = -(pi / (ri * ri) + pj / (rj * rj))
        if fn.epsilon is not None and two:
            t = t - fn.epsilon * (pi.abs() + pj.abs()) / (ri * rj)
        t = (t - visc) * g
        sa["dvdt"] = sa["dvdt"].index_add(0, i, m_j * t)
        sa["drhodt"] = sa["drhodt"].index_add(0, i, m_j * dr * (ri / rj if fn.sigma == 1 else 1.0))
        if two:
            sb["dvdt"] = sb["dvdt"].index_add(0, j, -ps.mass * t)
            sb["drhodt"] = sb["drhodt"].index_add(
                0, j, ps.mass * dr * (rj / ri if fn.sigma == 1 else 1.0))

    def xsph(self):
        """v gets the velocity adjustment of each pair (the last step's taken
        out first); a ghost's share goes to its source's particle of the same
        place in the sorted order."""
        for ps in self.lf.systems:
            s = self.sys[id(ps)]
            s["v"] = s["v"] - s["v_adjustment"]
            s["v_adjustment"] = torch.zeros_like(s["v"])
        for si, (i, j) in zip(self.lf.interactions, self.pairs):
            if si.vadjust_pfn is None or len(i) == 0:
                continue
            sa, b = self.sys[id(si.system_a)], self.other(si)
            sb = sa if b is None else self.sys[id(b)]
            ghost = "of" in sb
            _, _, w = self.gradient(si.kernel, sa["x"][i] - sb["x"][j])
            vb, rb = (sb["vh"], sb["rh"]) if ghost else (sb["v"], sb["rho"])
            du = -si.vadjust_pfn.epsilon * (sa["v"][i] - vb[j]) * w / (sa["rho"][i] + rb[j])
            m = si.system_a.mass
            sa["v_adjustment"] = sa["v_adjustment"].index_add(0, i, du * (m if ghost or b is None
                                                                          else b.mass))
            if ghost:
                sa["v_adjustment"] = sa["v_adjustment"].index_add(0, sa["perm"][j], -du * m)
            elif b is not None:
                sb["v_adjustment"] = sb["v_adjustment"].index_add(0, j, -du * m)
        for ps in self.lf.systems:
            s = self.sys[id(ps)]
            s["v"] = s["v"] + s["v_adjustment"]

    # ---- state updaters --------------------------------------------------------
    def pressure(self, u, rho, c):
        if isinstance(u, G.TaitEOSUpdater):
            return u.rho0 * c * c / u.gamma * ((rho / u.rho0) ** u.gamma - 1.0)
        return c * c * (rho - u.rho0)

    def update(self, ps, s, u):
        if isinstance(u, G.ZeroFieldUpdater):
            for f in u.fields:
                s[f] = torch.zeros_like(s[f])
        elif isinstance(u, (G.TaitEOSUpdater, G.LinearEOSUpdater)):
            s["p"] = self.pressure(u, s["rh"], ps.c)
        elif isinstance(u, G.ViscoPlasticMCStressUpdater):
            p = s["p"] = self.pressure(u.eos, s["rh"], ps.c)
            e = self.tensor(s["strain_rate"])
            mag = torch.sqrt((e * e).sum((1, 2)))[:, None].clamp(min=2.220446049250313e-16)
            t = 2.0 * (u.cohesion + p * math.tan(u.friction_angle)) / mag * s["strain_rate"]
            t[:, :3] -= p
            s["stress"] = torch.where(t[:, :3].sum(1, keepdim=True) > 0.0, torch.zeros_like(t), t)
        else:
            self.drucker_prager(s, u)

    def drucker_prager(self, s, u):
        dt, eye = self.dt, torch.eye(3, dtype=torch.float64, device=self.dev)
        q = math.sqrt(3.0) * (3.0 - math.sin(u.phi))
        a, k = 2.0 * math.sin(u.phi) / q, 6.0 * u.cohesion * math.cos(u.phi) / q
        a_psi = 2.0 * math.sin(u.psi) / (math.sqrt(3.0) * (3.0 - math.sin(u.psi)))
        shear = u.E / (2.0 * (1.0 + u.nu))
        lam = u.E * u.nu / ((1.0 + u.nu) * (1.0 - 2.0 * u.nu))

        def trace(t):
            return (t * eye).sum((1, 2))[:, None, None]

        def elastic(e):
            return lam * trace(e) * eye + 2.0 * shear * e

        t0 = self.tensor(s["stress"])
        e = dt * self.tensor(s["strain_rate"])
        w = dt * s["vorticity"][:, 0]
        inc = elastic(e)
        inc[:, 0, 0] -= 2.0 * t0[:, 0, 1] * w
        inc[:, 1, 1] += 2.0 * t0[:, 0, 1] * w
        turn = (t0[:, 0, 0] - t0[:, 1, 1]) * w
        inc[:, 0, 1] += turn
        inc[:, 1, 0] += turn
        t = t0 + inc
        dev = t - trace(t) / 3.0 * eye
        j2 = torch.sqrt(0.5 * (dev * dev).sum((1, 2)))[:, None, None]
        f = a * trace(t) + j2 - k
        df, dg = a * eye + dev / (2.0 * j2), a_psi * eye + dev / (2.0 * j2)
        lam_p = f / (df * elastic(dg)).sum((1, 2))[:, None, None]
        plastic = torch.where(f > 0.0, lam_p * dg, torch.zeros_like(dg))
        t = t - torch.where(f > 0.0, elastic(lam_p * dg), torch.zeros_like(dg))
        t = torch.where(trace(t) > k / a, k / a / 3.0 * eye, t)
        s["stress"] = self.voigt(t, 4)
        s["strain"] = s["strain"] + self.voigt(e, 4)
        s["strain_p"] = s["strain_p"] + self.voigt(plastic, 4)
