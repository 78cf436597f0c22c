"""The work that a user of this solver has it do, as cases that can be timed and compared.

Every kind of case but ``dec`` is the time loop of a simulation: a context holds all blocks of a
run on the GPU, and one pass advances it by ``steps`` explicit steps through the public entry
points (``Mercury.graph_launch`` where the program replays a captured step, ``Mercury.step``
where it reads dt back after every step or where the implicit resistive correction makes the
step data dependent).  A pass returns the whole conserved state, the face field and the derived
cell fields, as views of the context's own device arrays.  The ``dec`` kind applies the discrete
exterior derivatives to arrays of the caller.

Sizes, boundary types, physics and forms are those of the package's own configurations
(``mpcns_mercury_amd.cases``): the periodic cube, the six-sector shell, the same shell cut into
glued blocks, the cubed sphere, the resistive shell and the batched ensemble.
"""
import ctypes
import math
import random

import numpy as np
import torch

from mpcns_mercury_amd import cases as sim
from mpcns_mercury_amd import hip

G = 4  # ghost layers of every configuration

# ---------------------------------------------------------------------------------------------
# what is measured
# ---------------------------------------------------------------------------------------------


def listed():
    return [
        # a debugging-size periodic block: launches and latency are all there is
        {"name": "cube_tiny", "kind": "cube", "ni": 12, "nj": 10, "nk": 8, "form": 1, "rk2": False, "hall": False, "eager": False, "steps": 10},
        # the single-fluid configuration: 48^3 periodic curvilinear block, two-stage Runge-Kutta
        {"name": "cube_48_rk2", "kind": "cube", "ni": 48, "nj": 48, "nk": 48, "form": 1, "rk2": True, "hall": False, "eager": False, "steps": 4},
        # a ragged periodic Hall block driven step by step: the driver prints dt after every step
        {"name": "cube_ragged_eager", "kind": "cube", "ni": 61, "nj": 50, "nk": 67, "form": 1, "rk2": False, "hall": True, "eager": True, "steps": 4},
        # a coarse six-sector shell (a first look at a set-up), mixed precision
        {"name": "shell_coarse_mixed", "kind": "shell", "scale": 0.4, "form": 2, "rk2": False, "steps": 4},
        # the production shell: six uneven sectors, 2.5 M cells, two-fluid Hall MHD in double precision
        {"name": "shell", "kind": "shell", "scale": 1.0, "form": 1, "rk2": False, "steps": 2},
        # the same in mixed precision
        {"name": "shell_mixed", "kind": "shell", "scale": 1.0, "form": 2, "rk2": False, "steps": 2},
        # the shell cut into 24 blocks glued by interfaces: ghost copies between blocks in every sync
        {"name": "cut_shell", "kind": "cut", "scale": 0.6, "form": 1, "rk2": False, "steps": 2},
        # a whole cubed sphere: rotated patch connections and singular corner edges
        {"name": "cubed_sphere", "kind": "sphere", "n": 30, "nr": 30, "rule": 0, "form": 1, "steps": 2},
        # three ion species with the implicit resistive correction on every edge (mixed explicit stages)
        {"name": "resistive_shell_mixed", "kind": "resistive", "scale": 0.4, "form": 2, "steps": 1},
        # the two-fluid shell with the resistive window near the surface, double precision
        {"name": "shell_resist_window", "kind": "window", "scale": 0.5, "form": 1, "steps": 1},
        # a batch of independent runs of uneven size in one context, mixed precision
        {"name": "ensemble_mixed", "kind": "ensemble", "runs": 16, "scale": 0.5, "form": 2, "steps": 2},
        # the discrete exterior derivatives on the caller's own arrays
        {"name": "dec_operators", "kind": "dec", "ni": 160, "nj": 121, "nk": 144},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng: random.Random):
    kind = rng.choice(["cube", "cube", "shell", "shell", "cut", "sphere", "resistive", "window", "ensemble", "dec"])
    if kind == "cube":
        n = _log(rng, 8, 80)
        d = [max(6, int(round(n * rng.uniform(0.7, 1.2)))) for _ in range(3)]
        eager = rng.random() < 0.3
        return {"kind": kind, "ni": d[0], "nj": d[1], "nk": d[2], "form": rng.choice([1, 1, 2]), "rk2": rng.random() < 0.4,
                "hall": rng.random() < 0.6, "eager": eager, "steps": rng.choice([1, 2])}
    if kind == "shell":
        rk2 = rng.random() < 0.3
        return {"kind": kind, "scale": round(_log(rng, 0.12, 0.95), 3), "form": rng.choice([1, 2]), "rk2": rk2,
                "steps": 1 if rk2 else rng.choice([1, 2])}
    if kind == "cut":
        return {"kind": kind, "scale": round(_log(rng, 0.2, 0.7), 3), "form": rng.choice([1, 2]), "rk2": rng.random() < 0.3, "steps": 2}
    if kind == "sphere":
        return {"kind": kind, "n": rng.randint(8, 32), "nr": rng.randint(8, 40), "rule": rng.choice([0, 1]), "form": rng.choice([1, 2]), "steps": 2}
    if kind == "resistive":
        return {"kind": kind, "scale": round(_log(rng, 0.08, 0.4), 3), "form": rng.choice([1, 2]), "steps": 1}
    if kind == "window":
        return {"kind": kind, "scale": round(_log(rng, 0.15, 0.5), 3), "form": rng.choice([1, 2]), "steps": 1}
    if kind == "ensemble":
        return {"kind": kind, "runs": rng.randint(2, 16), "scale": round(rng.uniform(0.2, 0.5), 3), "form": rng.choice([1, 2]), "steps": 2}
    n = _log(rng, 12, 150)
    d = [max(4, int(round(n * rng.uniform(0.6, 1.2)))) for _ in range(3)]
    return {"kind": "dec", "ni": d[0], "nj": d[1], "nk": d[2]}


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------


def _problem(case, seed):
    """The simulation's grid, physics and initial state."""
    kind = case["kind"]
    if kind == "cube":
        return sim.make_periodic_cube((case["ni"], case["nj"], case["nk"]), g=G, seed=seed, hall=case["hall"], integrator=int(case["rk2"]))
    if kind == "shell":
        return sim.make_shell(scale=case["scale"], g=G, seed=seed)
    if kind == "cut":
        return sim.make_cut_shell(scale=case["scale"], g=G, seed=seed)
    if kind == "sphere":
        return sim.make_cubed_sphere(case["n"], case["nr"], g=G, rule=case["rule"], seed=seed)
    if kind == "window":
        return sim.make_shell(scale=case["scale"], g=G, seed=seed, resist=0.05)
    # the remaining configurations fix their seeds: the density noise of this run comes on top of them
    if kind == "resistive":
        p = sim.make_resistive_shell(scale=case["scale"], g=G)
    else:
        p = sim.concat_runs([sim.make_ensemble_run(r, scale=case["scale"], g=G) for r in range(case["runs"])])
    for b, fl in enumerate(p.fields):
        fl["U_H"] = fl["U_H"] * (1.0 + np.random.default_rng([seed, b]).uniform(-1e-3, 1e-3, fl["U_H"].shape[1:]))
    return p


class _Memory:
    """A device array of a context, as torch.as_tensor takes it; the tensor holds this object, and with it the context."""

    def __init__(self, ctx, ptr, shape, strides):
        self.ctx = ctx
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "strides": tuple(8 * s for s in strides),
                                         "typestr": "<f8", "version": 2}


def _view(ctx, names, block):
    """The components of one field (or of a triplet of one-component fields) on a block: the owned part of the box."""
    box = ctx.case.box(block)
    at = [ctx.field_device(n, block, c) for n in names for c in range(hip.field_info(n)[1])]
    step = (at[1] - at[0]) // 8
    if any(b - a != 8 * step for a, b in zip(at, at[1:])):
        raise RuntimeError("the components are not evenly spaced")
    strides = (step, box[1] * box[2], box[2], 1)
    t = torch.as_tensor(_Memory(ctx, at[0], (len(at),) + tuple(box), strides), device="cuda")
    return t[(slice(None),) + tuple(slice(G, G + m) for m in ctx.case.blocks[block].dims)]


def _spans(ctx, names):
    """The components of a field on all blocks of a many-block run, block after block with their ghosts."""
    vol = [int(np.prod(ctx.case.box(b))) for b in range(ctx.case.nb)]
    out = []
    for n in names:
        for c in range(hip.field_info(n)[1]):
            at = [ctx.field_device(n, b, c) for b in range(ctx.case.nb)]
            if any(at[b + 1] - at[b] != 8 * vol[b] for b in range(len(vol) - 1)):
                raise RuntimeError("the blocks are not adjacent")
            out.append(torch.as_tensor(_Memory(ctx, at[0], (sum(vol),), (1,)), device="cuda"))
    return out


class _Run:
    """What a simulation program holds between passes."""

    def __init__(self, case, seed):
        problem = _problem(case, seed)
        self.steps, self.rk2 = case["steps"], int(bool(case.get("rk2")))
        self.eager = bool(case.get("eager")) or case["kind"] in ("resistive", "window")
        self.ctx = hip.Mercury(problem)
        self.ctx.set_form(case["form"])
        self.ctx.prepare()
        if not self.eager:
            self.ctx.graph_capture(self.rk2)
        species = ["U_H", "U_Na"] + (["U_He"] if problem.phys.n_species >= 3 else [])
        faces = ["B_xi", "B_eta", "B_zeta"]
        self.out = {}
        if problem.nb > 6:
            for key, names in [(n, [n]) for n in species] + [("B", faces), ("B_cell", ["B_cell"]), ("J_cell", ["J_cell"])]:
                self.out[key] = _spans(self.ctx, names)
            return
        for b in range(problem.nb):
            for key, names in [(n, [n]) for n in species] + [("B", faces), ("B_cell", ["B_cell"]), ("J_cell", ["J_cell"])]:
                self.out["%s.%d" % (key, b)] = _view(self.ctx, names, b)


class _Forms:
    """Discrete forms on one block, in the caller's arrays."""

    def __init__(self, case, seed):
        m = (case["ni"], case["nj"], case["nk"])
        n = tuple(x + 1 + 2 * G for x in m)
        gen = torch.Generator(device="cuda").manual_seed(seed)
        new = lambda: torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)  # noqa: E731
        self.m = m
        self.node = new()
        self.A = [new() for _ in range(3)]  # edge 1-form
        self.grad = [torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(3)]
        self.flux = [torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(3)]
        self.div = torch.zeros(n, device="cuda", dtype=torch.float64)
        self.B0 = [new() for _ in range(3)]  # face 2-form before the update
        self.B = [torch.empty_like(b) for b in self.B0]
        self.worst = torch.zeros(1, device="cuda", dtype=torch.float64)
        self.dims = (ctypes.c_int * 3)(*m)
        p = lambda ts: (ctypes.c_void_p * 3)(*[t.data_ptr() for t in ts])  # noqa: E731
        self.pA, self.pgrad, self.pflux, self.pB = p(self.A), p(self.grad), p(self.flux), p(self.B)


def prepare(case, seed):
    return _Forms(case, seed) if case["kind"] == "dec" else _Run(case, seed)


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------

_DT = 0.25  # time step of the Faraday update of the caller's 2-form


def _check(rc):
    if rc != 0:
        raise hip.MercuryError(hip.load().mercury_last_error().decode())


def run(state):
    if isinstance(state, _Forms):
        L, s = hip.load(), state
        st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        for b, b0 in zip(s.B, s.B0):
            b.copy_(b0)
        _check(L.mercury_dec_d0(s.dims, G, s.node.data_ptr(), s.pgrad, st))
        _check(L.mercury_dec_d1(s.dims, G, s.pA, s.pflux, st))
        _check(L.mercury_dec_d2(s.dims, G, s.pflux, s.div.data_ptr(), st))
        _check(L.mercury_dec_faraday_update(s.dims, G, s.pA, s.pB, _DT, st))
        _check(L.mercury_dec_max_abs_div_curl(s.dims, G, s.pA, s.worst.data_ptr(), st))
        return {"grad": s.grad, "curl": s.flux, "div": s.div, "B": s.B, "worst": s.worst}
    if state.eager:
        dt = state.ctx.step(state.steps, state.rk2)
        return {"dt": dt, **state.out}
    state.ctx.graph_launch(state.steps)
    return state.out


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------


def _cells(case):
    kind = case["kind"]
    if kind in ("cube", "dec"):
        return case["ni"] * case["nj"] * case["nk"]
    if kind in ("shell", "window"):
        return sum(int(np.prod([max(4, int(round(d * case["scale"]))) for d in b])) for b in sim.C2_BLOCKS)
    if kind == "cut":
        return sum(int(np.prod([max(2 * G, int(round(d * case["scale"]))) for d in b])) for b in sim.C2_BLOCKS)
    if kind == "sphere":
        return 6 * case["n"] ** 2 * case["nr"]
    if kind == "resistive":
        d = [max(2 * G, 2 * int(round(x * case["scale"] / 2))) for x in sim.C5_DIMS]
        return max(G, int(round(sim.C5_DIMS[0] * case["scale"]))) * d[1] * d[2]
    return int(case["runs"] * 1.3 * 2.5 * (64 * case["scale"]) ** 3)  # the mean member: 2.5 blocks of 64^3 at scale 1


def work(case):
    n = _cells(case)
    if case["kind"] == "dec":
        # d0: 1 in, 3 out; d1: 3 in, 3 out; d2: 3 in, 1 out; the Faraday update: 3 + 3 in, 3 out, and the copy before it; the diagnostic: 3 in
        return {"bytes": 8 * n * (4 + 6 + 4 + 9 + 6 + 3), "flops": n * (3 + 9 + 5 + 15 + 14)}
    ns = 3 if case["kind"] == "resistive" else 2
    # one stage, perfectly fused: the state and the face field in and out; dipole-free background, metric (10), the edge,
    # face and cell statics (60 + 2), the photo rate and centre, the face field's weights (18)
    static = 10 + 60 + 2 + 3 + 18
    words = 2 * (5 * ns + 3) + static
    size = 8 * words if case["form"] != 2 else 8 * (2 * (5 * ns + 3) + 10 + 2 + 3) + 4 * (60 + 18)
    stages = case["steps"] * (2 if case.get("rk2") else 1)
    out = {"bytes": size * n * stages, "flops": 2500 * n * stages}
    if case["kind"] in ("resistive", "window"):
        edges = 3 * n if case["kind"] == "resistive" else 0.27 * n
        its = 8 if case["kind"] == "resistive" else 12
        # a conjugate-gradient iteration: x, r and p in and out, A p out, and eta, the diagonal, the weights, alpha and beta
        out["bytes"] += case["steps"] * its * edges * 8 * 13
        out["flops"] += case["steps"] * its * edges * 40
    return out


def tolerance(case):
    if case["kind"] == "dec":
        return "exact"
    if case["kind"] in ("resistive", "window"):
        # the linear solve stops at a relative residual of 1e-10 (double precision stages), or sits on mixed stages
        return {"rel": 1e-9, "max": 1e-6} if case["form"] == 1 else {"rel": 1.2e-5, "max": 5e-4}
    # double precision: the step is a fixed sequence of rounded operations and reproduces bit for bit; mixed: single
    # precision fluxes, EMFs and Hall terms, 3.7e-6 from 64 bits in the face field of the shell after two steps
    return "exact" if case["form"] == 1 else {"rel": 1.2e-5, "max": 5e-4}


# ---------------------------------------------------------------------------------------------
# the same pass in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------


def _at(x, a, n):
    """x at index + n along axis a of its last three axes (the wrapped ends are never used)."""
    return torch.roll(x, -n, a - 3)


class _Block:
    """One block of the plain step: state, face field and the static geometry, each over the block's box.

    The geometry (areas, edge lengths, reconstruction weights) is an input of the step, read from a context."""

    def __init__(self, ctx, problem, b):
        self.bc, self.m, self.P = problem.blocks[b].bc, problem.blocks[b].dims, problem.phys
        cuda = lambda v: torch.tensor(v, dtype=torch.float64, device="cuda")  # noqa: E731
        get = lambda n: cuda(ctx.get(n, b))  # noqa: E731
        self.U = [cuda(problem.fields[b][n]) for n in ("U_H", "U_Na")]
        three = lambda n: [get("%s_%s" % (n, a)) for a in ("xi", "eta", "zeta")]  # noqa: E731
        self.Bf, self.Badd = [x[0] for x in three("B")], [x[0] for x in three("Badd")]
        self.JD = [get(n) for n in ("JDxi", "JDet", "JDze")]
        self.area, self.beta, self.dl, self.alpha, self.taper, self.leta = (
            [x[0] for x in three(n)] for n in ("Area", "beta", "dl", "alpha", "taper", "eta_local"))
        self.dr = three("dr")
        self.jac, self.photo, self.centre = get("Jac")[0], get("Photo_rate")[0], get("cell_center")
        self.wb, self.wj = get("Bcell_from_Bface_w"), get("Jcell_from_Jedge_w")
        self.box = tuple(self.jac.shape)
        self.zero = torch.zeros(self.box, dtype=torch.float64, device="cuda")
        self.Bc, self.Bi, self.Jc = (self.zero.expand(3, *self.box).clone() for _ in range(3))

    # --- index ranges -------------------------------------------------------------------------
    def hi(self, d):
        """Owned extents of a location that lies between nodes along the axes where d is 1."""
        return [self.m[a] + 1 - d[a] for a in range(3)]

    def inside(self, lo, hi):
        return tuple(slice(G + l, G + h) for l, h in zip(lo, hi))

    def owned(self, new, old, d):
        """old with the owned part of new."""
        s = (Ellipsis,) + self.inside((0, 0, 0), self.hi(d))
        out = old.clone()
        out[s] = new[s]
        return out

    # --- ghosts -------------------------------------------------------------------------------
    def _slab(self, d, face, ghost):
        a, up, hi = face // 2, face & 1, self.hi(d)
        lo, h = [0, 0, 0], list(hi)
        if ghost:
            lo[a], h[a] = (hi[a], hi[a] + G) if up else (-G, 0)
        else:
            lo[a], h[a] = (hi[a] - 1, hi[a]) if up else (0, 1)
        return (Ellipsis,) + self.inside(lo, h)

    def extend(self, x, d, face):
        x[self._slab(d, face, True)] = x[self._slab(d, face, False)]

    def corners(self, x, d):
        """Ghosts outside two or three physical faces take the value of the nearest owned point."""
        hi = self.hi(d)
        at = [torch.arange(-G, self.m[a] + G + 1, device="cuda") for a in range(3)]
        out = [((t < 0) | (t >= h)) & (t < h + G) for t, h in zip(at, hi)]
        near = [t.clamp(0, h - 1) + G for t, h in zip(at, hi)]
        n = [o.long().view([-1 if c == a else 1 for c in range(3)]) for a, o in enumerate(out)]
        v = x[..., near[0][:, None, None], near[1][None, :, None], near[2][None, None, :]]
        return torch.where((n[0] + n[1] + n[2]) >= 2, v, x)

    def periodic(self, x, d, level):
        """Wrapped ghosts outside at most ``level`` axes, and shared planes equal to their owners."""
        hi = self.hi(d)
        at = [torch.arange(-G, self.m[a] + G + 1, device="cuda") for a in range(3)]
        out = [((t < 0) | (t >= h)) & (t < h + G) for t, h in zip(at, hi)]
        src = [torch.where(o, torch.remainder(t, m), t.clamp(max=h + G - 1)) + G for t, o, m, h in zip(at, out, self.m, hi)]
        n = [o.long().view([-1 if c == a else 1 for c in range(3)]) for a, o in enumerate(out)]
        n = n[0] + n[1] + n[2]
        v = x[..., src[0][:, None, None], src[1][None, :, None], src[2][None, None, :]]
        x = torch.where((n >= 1) & (n <= level), v, x)
        for a in range(3):
            if not d[a]:  # the upper shared plane is the lower one
                lo, up = [slice(None)] * 3, [slice(None)] * 3
                lo[a], up[a] = slice(G, G + 1), slice(G + self.m[a], G + self.m[a] + 1)
                x[(Ellipsis,) + tuple(up)] = x[(Ellipsis,) + tuple(lo)]
        return x

    @property
    def wraps(self):
        return self.bc[0] == sim.BC_PERIODIC

    def sync(self, x, d, level=3, copy=False, fill=None, wall_copy=False):
        """The ghosts of one field: far field extended (copy) or filled, walls extended or left, corners, wraps."""
        if self.wraps:
            return self.periodic(x, d, level)
        for f in range(6):
            if self.bc[f] == sim.BC_FARFIELD:
                if fill is not None:
                    s = self._slab(d, f, True)
                    x[s] = fill.view(-1, 1, 1, 1).expand_as(x[s])
                elif copy:
                    self.extend(x, d, f)
        if wall_copy:
            for f in range(6):
                if self.bc[f] == sim.BC_WALL:
                    self.extend(x, d, f)
        return self.corners(x, d)

    def vector(self, v):
        return torch.tensor(list(v), dtype=torch.float64, device="cuda")

    def sync_state(self):
        P = self.P
        for s, (far, floor) in enumerate(((P.qinf, P.wall_rho_floor_H), (P.qinfs, P.wall_rho_floor_Na))):
            x = self.U[s]
            if self.wraps:
                self.U[s] = self.periodic(x, (1, 1, 1), 1)
                continue
            for f in range(6):
                if self.bc[f] == sim.BC_FARFIELD:
                    w = self._slab((1, 1, 1), f, True)
                    x[w] = self.vector(far).view(-1, 1, 1, 1).expand_as(x[w])
            own = [slice(G, G + m) for m in self.m]
            for f in range(6):
                if self.bc[f] != sim.BC_WALL:
                    continue
                a, up = f // 2, f & 1

                def layer(n):
                    w = list(own)
                    i = G + (self.m[a] - 1 + n if up else -n)
                    w[a] = slice(i, i + 1)
                    return (slice(None),) + tuple(w)

                def at_rest(v):
                    rho = torch.clamp(v[0], min=floor)
                    e = (v[4] - 0.5 * (v[1] ** 2 + v[2] ** 2 + v[3] ** 2) / rho).clamp(min=0.0)
                    p = ((P.gamma - 1.0) * e).clamp(min=P.wall_p_floor)
                    z = torch.zeros_like(rho)
                    return torch.stack([rho, z, z, z, p / (P.gamma - 1.0)])

                if s == 1:  # the heavy ions: a floor state behind the wall
                    for n in range(1, G + 1):
                        v = torch.zeros_like(x[layer(n)])
                        v[0], v[4] = floor, P.wall_p_floor / (P.gamma - 1.0)
                        x[layer(n)] = v
                else:
                    x[layer(0)] = at_rest(x[layer(-1)])
                    for n in range(1, G + 1):
                        x[layer(n)] = at_rest(x[layer(0)])
            self.U[s] = self.corners(x, (1, 1, 1))

    def sync_faces(self, F, copy=False):
        for a in range(3):
            d = [1, 1, 1]
            d[a] = 0
            F[a] = self.sync(F[a], d, copy=copy)

    def shared_mean(self, E):
        """Edges shared across the wrap: the mean of their copies."""
        if not self.wraps:
            return
        for a in range(3):
            for c in range(3):
                if c == a:
                    continue
                x = E[a].movedim(c, 0)
                mean = 0.5 * (x[G] + x[G + self.m[c]])
                x[G] = mean
                x[G + self.m[c]] = mean

    # --- derived fields -----------------------------------------------------------------------
    def limiter(self, rho):
        P = self.P
        n = [torch.clamp(r, min=0.0) / M * P.M_ref for r, M in zip(rho, (P.M_H, P.M_Na))]
        ne = n[0] + n[1]
        eff = torch.sqrt(ne * ne + P.ne_floor ** 2)
        return n, eff, [x / ne for x in n], [x / eff for x in n]

    def derive(self):
        P, one = self.P, (1, 1, 1)
        tot = [b + c for b, c in zip(self.Bf, self.Badd)]
        ends = lambda f: torch.stack([s * _at(f[a], a, n) for a in range(3) for s, n in ((-1.0, 0), (1.0, 1))])  # noqa: E731
        for name, f, far in (("Bc", tot, self.vector(P.B_imf)), ("Bi", self.Bf, self.vector((0, 0, 0)))):
            new = torch.stack([(self.wb[6 * c:6 * c + 6] * ends(f)).sum(0) for c in range(3)])
            setattr(self, name, self.sync(self.owned(new, getattr(self, name), one), one, fill=far))
        h = [b * f for b, f in zip(self.beta, self.Bf)]
        J = []
        for a in range(3):
            c, e = (a + 1) % 3, (a + 2) % 3
            curl = (h[e] - _at(h[e], c, -1)) - (h[c] - _at(h[c], e, -1))
            d = [0, 0, 0]
            d[a] = 1
            J.append(self.owned(curl * self.alpha[a], self.zero, d))
        self.shared_mean(J)
        for a in range(3):
            d = [0, 0, 0]
            d[a] = 1
            J[a] = self.sync(J[a], d, copy=True)
        self.J = J
        around = []
        for a in range(3):
            c, e = [x for x in range(3) if x != a]
            around += [J[a], _at(J[a], c, 1), _at(J[a], e, 1), _at(_at(J[a], c, 1), e, 1)]
        around = torch.stack(around)
        new = torch.stack([(self.wj[12 * c:12 * c + 12] * around).sum(0) for c in range(3)])
        Jc = self.owned(new, self.Jc, one)
        if not self.wraps:
            for f in range(6):
                if self.bc[f] == sim.BC_FARFIELD:
                    self.extend(Jc, one, f)
            for f in range(6):
                if self.bc[f] == sim.BC_WALL:
                    a, up, w = f // 2, f & 1, [slice(G, G + m) for m in self.m]
                    w[a] = slice(G + self.m[a] - 2, G + self.m[a]) if up else slice(G, G + 2)
                    Jc[(slice(None),) + tuple(w)] = 0.0
                    self.extend(Jc, one, f)
            self.Jc = self.corners(Jc, one)
        else:
            self.Jc = self.periodic(Jc, one, 3)
        self.pv, rho = [], []
        for U, coeff in zip(self.U, (P.state_coeff_H, P.state_coeff_Na)):
            r = torch.clamp(U[0], min=1e-12)
            v = U[1:4] / r
            e = (U[4] - 0.5 * r * (v * v).sum(0)).clamp(min=0.0)
            p = ((P.gamma - 1.0) * e).clamp(min=1e-12)
            self.pv.append((v, p, p / (r * coeff)))
            rho.append(torch.clamp(U[0], min=0.0))
        self.n, self.eff, self.chi, self.w = self.limiter(rho)
        self.up = sum(c * torch.where(r > 1e-20, p[0], torch.zeros_like(p[0])) for c, r, p in zip(self.chi, rho, self.pv))
        self.ucon = []
        for a in range(3):
            k = 0.5 * (self.JD[a] + _at(self.JD[a], a, 1))
            self.ucon.append((k * self.up).sum(0) / (self.jac.abs() + 1e-30))

    def time_step(self):
        P, s = self.P, self.inside((0, 0, 0), self.m)
        V = self.jac.abs()
        best = 1e100
        for U in self.U:
            rho = torch.clamp(U[0], min=1e-2)
            u = U[1:4] / rho
            pr = (P.gamma - 1.0) * (U[4] - 0.5 * rho * (u * u).sum(0))
            cs2, vA2 = P.gamma * pr / rho, P.inver_MA2 * (self.Bc * self.Bc).sum(0) / rho
            den = torch.zeros_like(rho)
            for a in range(3):
                for n in (0, 1):
                    S = _at(self.JD[a], a, n)
                    A = torch.sqrt((S * S).sum(0))
                    nrm = S / A
                    vn2 = P.inver_MA2 * (self.Bc * nrm).sum(0) ** 2 / rho
                    t = cs2 + vA2
                    cf = torch.sqrt(0.5 * (t + torch.sqrt((t * t - 4.0 * cs2 * vn2).clamp(min=0.0))))
                    den = den + ((u * nrm).sum(0).abs() + cf) * A
            best = min(best, float((P.cfl * V / den)[s].min()))
        return best

    # --- right-hand sides ---------------------------------------------------------------------
    def rusanov(self, a, U, pv, far):
        """Flux through every lower face along axis a."""
        gm, S = self.P.gamma, self.JD[a]
        sides = []
        for n in (-1, 0):
            r, v, p = _at(U[0], a, n), _at(pv[0], a, n), _at(pv[1], a, n)
            un = (S * v).sum(0)
            E = p / (gm - 1.0) + 0.5 * r * (v * v).sum(0)
            c = torch.sqrt((gm * p / torch.clamp(r, min=1e-30)).clamp(min=0.0))
            q = torch.cat([r[None], r * v, E[None]])
            f = torch.cat([(r * un)[None], r * un * v + S * p, (un * (E + p))[None]])
            sides.append((q, f, un.abs() + c * torch.sqrt((S * S).sum(0))))
        (qL, fL, sL), (qR, fR, sR) = sides
        return 0.5 * (fL + fR) - 0.5 * torch.maximum(sL, sR) * (qR - qL)

    def fluid(self):
        P = self.P
        B, J, V = self.Bc, self.Jc, self.jac.abs()
        cross = lambda x, y: torch.stack([x[1] * y[2] - x[2] * y[1], x[2] * y[0] - x[0] * y[2], x[0] * y[1] - x[1] * y[0]])  # noqa: E731
        jxb = cross(J, B)
        ambi = P.ambipolar_enabled != 0.0
        if ambi:
            pe = self.pv[0][1] + self.pv[1][1]
            grad = 0.0
            for a in range(3):
                grad = grad + 0.5 * (_at(self.JD[a], a, -1) + self.JD[a]) / V * (_at(pe, a, 1) - _at(pe, a, -1))
            grad = 0.5 * grad
        x, y, z = self.centre
        dark = (x < 0.0) & (torch.sqrt(y * y + z * z) < 1.0)
        nu = torch.where(dark, torch.full_like(x, P.nu_shadow), torch.full_like(x, P.nu_lit))
        out = []
        for s, U in enumerate(self.U):
            v, p, T = self.pv[s]
            r = torch.zeros_like(U)
            for a in range(3):
                f = self.rusanov(a, U, self.pv[s], None)
                r = r - (_at(f, a, 1) - f) / self.jac
            rho = torch.clamp(U[0], min=0.0)
            M = (P.M_H, P.M_Na)[s]
            force = cross(v - self.up, B)
            r[1:4] += P.c_ind * self.n[s] * force + P.c_hall * self.w[s] * jxb
            r[4] += P.c_ind * self.n[s] * (force * v).sum(0) + P.c_hall * self.w[s] * (jxb * v).sum(0)
            if ambi:
                r[1:4] -= self.w[s] * grad
                r[4] -= self.w[s] * (grad * v).sum(0)
            if s == 1:
                r[0] += P.a1_Na * self.photo
                r[4] += P.a6 * self.photo * P.Tn0
            drag = P.a4 * rho * nu
            v2 = (v * v).sum(0)
            r[1:4] -= drag * v
            r[4] += -drag * v2 + P.a5 * self.n[s] * nu * (P.Tn0 - T * P.T_ref) * (M / (M + P.M_Na)) + drag * v2 * (P.M_Na / (M + P.M_Na))
            out.append(r)
        return out

    def electric(self):
        """The edge EMF with every contribution, boundary conditions included."""
        P = self.P
        tot = [b + c for b, c in zip(self.Bf, self.Badd)]
        mid = lambda f, a: 0.5 * (f[a] + _at(f[a], a, 1))  # noqa: E731
        bt, bi = [mid(tot, a) for a in range(3)], [mid(self.Bf, a) for a in range(3)]

        def flux(b, f):
            """Transport of the b flux through a lower f face."""
            side = lambda x, n: _at(x, f, n)  # noqa: E731
            g = [side(self.ucon[f], n) * side(bt[b], n) - side(self.ucon[b], n) * tot[f] for n in (-1, 0)]
            speed = torch.maximum(side(self.ucon[f], -1).abs(), self.ucon[f].abs())
            return 0.5 * (g[0] + g[1]) - 0.5 * speed * (bi[b] - side(bi[b], -1))

        rho, pe = [U[0] for U in self.U], self.pv[0][1] + self.pv[1][1]
        node = pe
        for a in range(3):
            node = node + _at(node, a, -1)
        node = 0.125 * node
        alpha_c = P.hall_coef / self.eff
        B, J = self.Bc, self.Jc
        ehc = alpha_c * torch.stack([J[1] * B[2] - J[2] * B[1], J[2] * B[0] - J[0] * B[2], J[0] * B[1] - J[1] * B[0]])
        hb = alpha_c.abs() * torch.sqrt((B * B).sum(0))
        E, H = [], []
        for a in range(3):
            c, e = (a + 1) % 3, (a + 2) % 3
            around = lambda x: [x, _at(x, c, -1), _at(x, e, -1), _at(_at(x, c, -1), e, -1)]  # noqa: E731
            most = lambda x: torch.stack(around(x)).amax(0)  # noqa: E731
            mean = lambda x: 0.25 * sum(around(x))  # noqa: E731
            # the face EMF along a: through c faces it is -flux of e, through e faces +flux of c
            on_c, on_e = -flux(e, c), flux(c, e)
            centre = 0.25 * (on_c + _at(on_c, e, -1) + on_e + _at(on_e, c, -1))
            de, dc = self.Bf[e] - _at(self.Bf[e], c, -1), self.Bf[c] - _at(self.Bf[c], e, -1)
            x = centre + 0.25 * (most(self.ucon[c].abs()) * de - most(self.ucon[e].abs()) * dc)
            if P.ambipolar_enabled != 0.0:
                x = x - P.pressure_coef * (_at(node, a, 1) - node) / self.limiter([mean(r) for r in rho])[1]
            if P.local_enabled != 0.0 and P.local_eta_max > 0.0 and P.local_r_decay > 0.0:
                x = x + self.leta[a] * self.J[a]
            hall = sum(mean(ehc[k]) * self.dr[a][k] for k in range(3))
            L, b4 = torch.clamp(self.dl[a], min=1e-14), 0.1 * most(hb)
            Ae = 0.5 * (self.area[e] + _at(self.area[e], c, -1))
            Ac = 0.5 * (self.area[c] + _at(self.area[c], e, -1))
            hall = hall + 0.5 * b4 * (L / torch.clamp(Ae, min=1e-14)) ** 2 * de - 0.5 * b4 * (L / torch.clamp(Ac, min=1e-14)) ** 2 * dc
            d = [0, 0, 0]
            d[a] = 1
            E.append(self.owned(x, self.zero, d))
            H.append(self.owned(self.taper[a] * hall, self.zero, d))
        self.shared_mean(E)
        E = [x + y for x, y in zip(E, H)]
        u, Bi = P.q_pv_inf, P.B_imf
        far = self.vector((Bi[1] * u[2] - Bi[2] * u[1], Bi[2] * u[0] - Bi[0] * u[2], Bi[0] * u[1] - Bi[1] * u[0]))
        for a in range(3):
            d = [0, 0, 0]
            d[a] = 1
            for f in range(6):
                if self.bc[f] == sim.BC_WALL and f // 2 != a:
                    E[a][self._slab(d, f, False)] = 0.0
            for f in range(6):
                if self.bc[f] == sim.BC_FARFIELD:
                    s = self._slab(d, f, False)
                    E[a][s] = (far.view(3, 1, 1, 1) * self.dr[a]).sum(0)[s]
            if self.wraps:
                E[a] = self.periodic(E[a], d, 3)
        return E

    def advance(self, dt):
        rhs, E = self.fluid(), self.electric()
        for s in range(2):
            self.U[s] = self.owned(self.U[s] + dt * rhs[s], self.U[s], (1, 1, 1))
        for a in range(3):
            c, e = (a + 1) % 3, (a + 2) % 3
            curl = (_at(E[e], c, 1) - E[e]) - (_at(E[c], e, 1) - E[c])
            d = [1, 1, 1]
            d[a] = 0
            self.Bf[a] = self.owned(self.Bf[a] - dt * curl, self.Bf[a], d)
        self.sync_state()
        self.sync_faces(self.Bf)
        self.derive()


def _exact_steps(case, seed):
    problem = _problem(case, seed)
    ctx = hip.Mercury(problem)
    blocks = [_Block(ctx, problem, b) for b in range(problem.nb)]
    ctx.close()
    for b in blocks:
        b.sync_faces(b.Badd, copy=True)
        b.sync_faces(b.Bf)
        b.derive()
    dts = []
    for _ in range(case["steps"]):
        dt = min(b.time_step() for b in blocks)
        dts.append(dt)
        before = [([u.clone() for u in b.U], [f.clone() for f in b.Bf]) for b in blocks] if case.get("rk2") else None
        for _ in range(2 if before else 1):
            for b in blocks:
                b.advance(dt)
        if before:
            for b, (U, F) in zip(blocks, before):
                b.U = [b.owned(0.5 * (x + y), y, (1, 1, 1)) for x, y in zip(U, b.U)]
                for a in range(3):
                    d = [1, 1, 1]
                    d[a] = 0
                    b.Bf[a] = b.owned(0.5 * (F[a] + b.Bf[a]), b.Bf[a], d)
                b.sync_state()
                b.sync_faces(b.Bf)
                b.derive()
    out = {"dt": np.array(dts)} if case.get("eager") else {}
    for i, b in enumerate(blocks):
        own = (slice(None),) + b.inside((0, 0, 0), b.m)
        out["U_H.%d" % i], out["U_Na.%d" % i], out["B.%d" % i] = b.U[0][own], b.U[1][own], torch.stack(b.Bf)[own]
        out["B_cell.%d" % i], out["J_cell.%d" % i] = b.Bc[own], b.Jc[own]
    return out


def _exact_forms(case, seed):
    s = _Forms(case, seed)
    A, m = s.A, s.m

    def owned(x, d):
        out = torch.zeros_like(x)
        w = tuple(slice(G, G + m[a] + 1 - d[a]) for a in range(3))
        out[w] = x[w]
        return out

    grad, curl, B = [], [], []
    for a in range(3):
        c, e = (a + 1) % 3, (a + 2) % 3
        edge, face = [0, 0, 0], [1, 1, 1]
        edge[a], face[a] = 1, 0
        grad.append(owned(_at(s.node, a, 1) - s.node, edge))
        curl.append(owned((_at(A[e], c, 1) - A[e]) - (_at(A[c], e, 1) - A[c]), face))
        B.append(s.B0[a] - _DT * curl[a])
    return {"grad": grad, "curl": curl, "div": None, "B": B, "worst": None}  # div curl is rounding alone


def exact(case, seed):
    if case["kind"] == "dec":
        return _exact_forms(case, seed)
    if case["kind"] in ("cube", "shell"):
        return _exact_steps(case, seed)
    return None  # connected, patched, resistive and batched runs: the same passes, on topologies that need their own plans
