"""What the framework is timed on: time steps of flows past a sphere, Poisson solves, relaxation
sweeps and force evaluations on block octrees, through the Python binding of the C ABI.

A case is a dict of plain values; its `kind` says which entry points it runs:

* step    : one `Context.step` (Solver::Update) of one or several resident flows past a sphere
* poisson : one pressure Poisson solve from x = 0 (`solve_mixed`, `bicgstab` or `cg`)
* sweeps  : a fixed number of RBGS or Jacobi iterations from x = 0
* forces  : what a run reads after a step: ghost fills, pressure and viscous force, the CFL guard

Linear solves run to a relative residual of 1e-12.  At the 1e-8 to 1e-10 at which a flow run stops,
a solution shows where its solver stopped in the seventh to ninth digit; at 1e-12 it is the
system's solution to nine digits, whichever way it was reached.

Fields stay on the device, as in a flow run: `run` returns them by name and a field is read to the
host when it is looked up.
"""
import functools
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ffv-hc_amd"))
import ffvhc  # noqa: E402
import flows  # noqa: E402
from serve import uniform_flow_init  # noqa: E402

N, G = 16, 2
NP = N + 2 * G
EPS = 1e-12
METHOD, OMEGA = 26, 1.6  # the mixed-precision schedule that the autotuner picks for these systems
SWEEPS = 100             # countMax of the reference's stationary solvers
INNER = (slice(None),) + (slice(G, G + N),) * 3
DEV = "cuda"


# ------------------------------------------------------------------------------------- cases

def listed():
    return [
        # a small case of a served stream: launches and their latency are all there is
        _step("step_sphere_16", (4, 2, 2), 2.0, 1),
        # the single-level flow past a sphere (524,288 cells), with the tuned solver and with the
        # reference's own FP64 Jacobi-BiCGSTAB
        _step("step_sphere_128", (8, 4, 4), 2.0, 1),
        _step("step_sphere_128_fp64", (8, 4, 4), 2.0, 1, solver="fp64"),
        # sphere and wake refined to three levels, implicit velocities: a moderate tree, and the
        # resolution of the reference configuration's sphere example (h = D/64, 10.2 M cells)
        _step("step_wake_520", (8, 4, 4), 2.0, 3, implicit=True),
        _step("step_wake_2480", (8, 4, 4), 1.0, 3, implicit=True),
        # a batched parameter sweep: flows of 16 to 324 blocks on one to three levels in one context
        _step("step_batch_8", (4, 2, 2), 2.0, 3, implicit=True, ncases=8),
        # the standalone Poisson benchmark: roots 8^3, level 1 in a ball, 1,128 blocks
        _poisson("poisson_1128", (8, 8, 8), True, "mixed"),
        # the reference's FP64 solvers: BiCGSTAB on a two-level tree around a body, PCG on a
        # single-level box
        _poisson("poisson_288_bicgstab", (4, 4, 4), True, "bicgstab", body=True),
        _poisson("poisson_60_cg", (5, 4, 3), False, "cg"),
        # the reference's stationary solvers at their default iteration limit: FP64 RBGS on the
        # two-level benchmark tree around a body, FP32 Jacobi on a small box of odd sizes
        _sweeps("rbgs_1128", (8, 8, 8), True, "rbgs", 8, body=True),
        _sweeps("jacobi_30_fp32", (5, 3, 2), False, "jacobi", 4),
        # drag and guard of the single-level flow after a step: the shortest calls
        _forces("forces_128", (8, 4, 4), 2.0, 1),
    ]


def _step(name, root, edge, levels, solver="mixed", implicit=False, ncases=1):
    return {"name": name, "kind": "step", "nx": root[0], "ny": root[1], "nz": root[2], "edge": edge, "levels": levels,
            "solver": solver, "implicit": implicit, "ncases": ncases, "re": 100.0}


def _poisson(name, root, ball, solver, body=False):
    return {"name": name, "kind": "poisson", "nx": root[0], "ny": root[1], "nz": root[2], "ball": ball,
            "solver": solver, "body": body}


def _sweeps(name, root, ball, smoother, prec, body=False):
    return {"name": name, "kind": "sweeps", "nx": root[0], "ny": root[1], "nz": root[2], "ball": ball,
            "smoother": smoother, "prec": prec, "body": body}


def _forces(name, root, edge, levels):
    return {"name": name, "kind": "forces", "nx": root[0], "ny": root[1], "nz": root[2], "edge": edge,
            "levels": levels}


def draw(rng):
    """One more case of the same ranges: trees of 4 to 1,700 blocks, any solver, both precisions."""
    kind = rng.choice(["step", "step", "poisson", "poisson", "sweeps", "forces"])
    if kind in ("step", "forces"):
        while True:
            k = max(2, int(round(2.0 * 4.0 ** rng.random())))  # roots (2k +- 1) x k x k
            root = (2 * k + rng.randint(-1, 1), k, k)
            edge = rng.choice([1.0, 2.0])
            levels = rng.randint(1, 3)
            nblk = _flow_tree(root, edge, levels).nblk
            if nblk <= 1700:
                break
        if kind == "forces":
            c = _forces("", root, edge, levels)
        else:
            fp64 = rng.random() < 0.25 and nblk <= 300
            re = round(rng.uniform(50.0, 300.0), 1)
            # the explicit form is stable on the coarse single-level grids alone
            explicit = levels == 1 and edge == 2.0 and re >= 100.0
            c = _step("", root, edge, levels, solver="fp64" if fp64 else "mixed", implicit=not explicit,
                      ncases=rng.choice([1, 1, 2, 4]) if nblk <= 200 else 1)
            c["re"] = re
    else:
        root = tuple(max(2, int(round(2.0 * 5.0 ** rng.random()))) for _ in range(3))
        ball = rng.random() < 0.6
        body = rng.random() < 0.5
        if kind == "poisson":
            solver = rng.choice(["mixed", "mixed", "bicgstab", "cg"])
            if solver == "cg":  # a symmetric system only
                ball = body = False
            c = _poisson("", root, ball, solver, body)
        else:
            c = _sweeps("", root, ball, rng.choice(["rbgs", "rbgs", "jacobi"]), rng.choice([8, 8, 4]), body)
    del c["name"]
    return c


# -------------------------------------------------------------------------- trees and systems
# Trees, geometry and matrix bands depend on the case alone; a program builds them once and keeps
# them.

def _root(case):
    return case["nx"], case["ny"], case["nz"]


@functools.lru_cache(maxsize=None)
def _flow_tree(root, edge, levels):
    return ffvhc.Tree(root=root, root_length=edge, regions=flows.sphere_regions(_centre(root, edge), 1.0,
                                                                               root[0] * edge, levels))


def _centre(root, edge):
    """A quarter of the length downstream, the middle across."""
    return 0.25 * root[0] * edge, 0.5 * root[1] * edge, 0.5 * root[2] * edge


@functools.lru_cache(maxsize=6)
def _flow_geometry(root, edge, levels):
    return _flow_tree(root, edge, levels).geometry_sphere(center=_centre(root, edge), radius=0.5, cut_id=1)[:3]


@functools.lru_cache(maxsize=None)
def _box_tree(root, ball):
    """A box of roots of edge 1, refined once in a ball of a quarter of the shortest side."""
    regions = [dict(kind="ball", a=tuple(0.5 * r for r in root), r=0.25 * min(root), level=1)] if ball else []
    return ffvhc.Tree(root=root, root_length=1.0, margin=1.0, regions=regions)


def _batch(case):
    """(root, edge, levels, Reynolds number) of each flow of a step case: the case's own tree first,
    then the same domain on one to three levels in turn."""
    return [(_root(case), case["edge"], case["levels"] if q == 0 else 1 + q % case["levels"],
             case["re"] * (1.0 + 0.25 * q)) for q in range(case["ncases"])]


@functools.lru_cache(maxsize=2)
def _solid(root, ball):
    """Cells inside a ball of an eighth of the shortest side: a body in a staircase."""
    tree = _box_tree(root, ball)
    tb = tree.table()
    at = np.arange(N) + 0.5
    d2 = 0.0
    for axis in range(3):
        p = tb["org"][:, axis, None] + tb["dx"][:, None] * at - 0.5 * root[axis] - 0.2
        shape = [p.shape[0], 1, 1, 1]
        shape[3 - axis] = N
        d2 = d2 + (p * p).reshape(shape)
    return d2 < (0.125 * min(root)) ** 2


@functools.lru_cache(maxsize=2)
def _bands(root, ball, body):
    """The padded bands {Ap, Aw, Ae, As, An, Ab, At} of the pressure matrix (bcut_calc_ab_p) with the
    outer conditions folded in: Dirichlet 0 on X+, Neumann 0 elsewhere.  Within a block, faces
    between a fluid cell and the body carry no flux; a solid cell has the reference's row
    (-6; 1, ..., 1)."""
    tree = _box_tree(root, ball)
    tb = tree.table()
    nb = tree.nblk
    lap = np.broadcast_to((1.0 / (tb["dx"] * tb["dx"]))[:, None, None, None], (nb, N, N, N))
    off = [lap.copy() for _ in range(6)]
    solid = _solid(root, ball) if body else np.zeros((nb, N, N, N), bool)
    for f in range(6):
        dim = 3 - f // 2
        beside = np.zeros_like(solid)  # the neighbour across face f is solid
        a, b = [slice(None)] * 4, [slice(None)] * 4
        a[dim], b[dim] = (slice(0, N - 1), slice(1, N)) if f & 1 else (slice(1, N), slice(0, N - 1))
        beside[tuple(a)] = solid[tuple(b)]
        off[f][beside] = 0.0
    diag = -(off[0] + off[1]) - (off[2] + off[3]) - (off[4] + off[5])
    diag[solid] = -6.0
    for f in range(6):
        off[f][solid] = 1.0
    for f in range(6):
        at = [slice(None)] * 4
        at[0] = tb["ftype"][:, f] == 0
        at[3 - f // 2] = N - 1 if f & 1 else 0
        at = tuple(at)
        diag[at] += -off[f][at] if f == ffvhc.X_P else off[f][at]
        off[f][at] = 0.0
    out = []
    for band in [diag] + off:
        p = np.zeros((nb, NP, NP, NP))
        p[INNER] = band
        out.append(p)
    return out


def _rhs(case, seed):
    """The Poisson benchmark's right-hand side: uniform[-1, 1] with the mean removed, 0 in a body."""
    root, ball = _root(case), case["ball"]
    v = np.random.default_rng(seed).uniform(-1.0, 1.0, (_box_tree(root, ball).nblk, N, N, N))
    v -= v.mean()
    if case["body"]:
        v[_solid(root, ball)] = 0.0
    b = np.zeros((v.shape[0], NP, NP, NP))
    b[INNER] = v
    return b


P_BC = [(ffvhc.NEUMANN, 0.0), (ffvhc.DIRICHLET, 0.0)] + [(ffvhc.NEUMANN, 0.0)] * 4


def _velocity(tb, seed):
    """A smooth seeded flow past the sphere's position for the force evaluation: padded ux, uy, uz, p."""
    r = np.random.default_rng(seed)
    at = np.arange(-G, N + G) + 0.5
    out = []
    for mean in (1.0, 0.0, 0.0, 0.0):
        v = mean
        for _ in range(3):
            w = r.uniform(0.2, 1.2, 3)
            s = [np.sin(w[d] * (tb["org"][:, d, None] + tb["dx"][:, None] * at) + r.uniform(0, 6.28)) for d in range(3)]
            v = v + r.uniform(0.05, 0.3) * s[2][:, :, None, None] * s[1][:, None, :, None] * s[0][:, None, None, :]
        out.append(np.ascontiguousarray(v))
    return out


class Fields(dict):
    """Device fields of a context by name (or (case id, field)): a lookup reads the field, padded,
    to the host."""

    def __init__(self, ctx, handles, dtype=np.float64):
        super().__init__(handles)
        self.ctx, self.dtype = ctx, dtype

    def __getitem__(self, name):
        case_id, field = super().__getitem__(name)
        return self.ctx.download(field, case_id, dtype=self.dtype)


# ----------------------------------------------------------------------------- prepare and run

def prepare(case, seed):
    return {"step": _prepare_step, "poisson": _prepare_system, "sweeps": _prepare_system,
            "forces": _prepare_forces}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_step(case, seed):
    """The resident flows: geometry, fields and the noisy uniform flow that a run starts from."""
    batch = _batch(case)
    ctx = ffvhc.Context(max_blocks=sum(_flow_tree(*b[:3]).nblk for b in batch))
    F = ctx.step_fields()
    ids = []
    for q, (root, edge, levels, re) in enumerate(batch):
        tree = _flow_tree(root, edge, levels)
        # CFL 0.3 on the finest cells, as a run of the sphere example; the single-level explicit flow
        # takes its configuration's dt = 0.01
        dt = flows.cfl_dt(tree, 0.3) if case["implicit"] else 0.01
        ids.append(ctx.add_case(tree, flows.flow_params(re, dt), geometry=_flow_geometry(root, edge, levels)))
        uniform_flow_init(16 * seed + q)(ctx, ids[-1], F)
    ctx.select(ids)
    kw = dict(solver=3, count_max=5000, eps=EPS, ncases=len(ids))
    kw.update(omega=OMEGA, mixed=True, mixed_method=METHOD) if case["solver"] == "mixed" else kw.update(omega=1.0)
    if case["implicit"]:
        kw.update(implicit_u=True, alpha_u=1.0, omega_u=1.0, count_max_u=1000, eps_u=EPS)
    return {"run": _run_step, "ctx": ctx, "F": F, "ids": ids, "kw": kw}


def _run_step(state):
    ctx, F = state["ctx"], state["F"]
    _, _, rc = ctx.step(F, **state["kw"])
    if rc:
        raise RuntimeError("step: status %d" % rc)
    names = {"ux": F.ux, "uy": F.uy, "uz": F.uz, "p": F.p, "lapp": F.lapp}
    names.update(("v%d" % q, F.v[q]) for q in range(6))
    if len(state["ids"]) == 1:  # the terms that the next step's Adams-Bashforth reads
        for d, axis in enumerate("xyz"):
            names["convection_" + axis], names["diffusion_" + axis] = F.ucp[d], F.udp[d]
        return Fields(ctx, {k: (state["ids"][0], f) for k, f in names.items()})
    return {"flow%d" % i: Fields(ctx, {k: (i, f) for k, f in names.items() if k in ("ux", "uy", "uz", "p")})
            for i in state["ids"]}


def _prepare_system(case, seed):
    root, ball = _root(case), case["ball"]
    tree = _box_tree(root, ball)
    ctx = ffvhc.Context(max_blocks=tree.nblk)
    cid = ctx.add_case(tree, ffvhc.case_params(bc={ffvhc.BC_P: P_BC}))
    prec = case.get("prec", 8)
    dtype = np.float64 if prec == 8 else np.float32
    A = [ctx.field(prec) for _ in range(7)]
    b, x = ctx.field(prec), ctx.field(prec)
    for q, band in enumerate(_bands(root, ball, case["body"])):
        ctx.upload(A[q], cid, band.astype(dtype, copy=False))
    ctx.upload(b, cid, _rhs(case, seed).astype(dtype, copy=False))
    return {"run": _run_poisson if case["kind"] == "poisson" else _run_sweeps, "ctx": ctx, "cid": cid, "A": A, "b": b,
            "x": x, "how": case.get("solver") or case["smoother"], "dtype": dtype}


def _run_poisson(state):
    ctx, x, A, b = state["ctx"], state["x"], state["A"], state["b"]
    ctx.fill(x, 0.0)
    if state["how"] == "mixed":
        rc = ctx.solve_mixed(METHOD, x, A, b, ffvhc.BC_P, OMEGA, 5000, EPS, 0.1)[-1]
    elif state["how"] == "bicgstab":
        rc = ctx.bicgstab(x, A, b, ffvhc.BC_P, 1.0, 1, 20000, EPS)[-1]
    else:
        rc = ctx.cg(x, A, b, ffvhc.BC_P, 1.0, 1, 20000, EPS)[-1]
    if rc:
        raise RuntimeError("solve: status %d" % rc)
    return Fields(ctx, {"x": (state["cid"], x)})


def _run_sweeps(state):
    ctx, x = state["ctx"], state["x"]
    ctx.fill(x, 0.0)
    go = ctx.rbgs if state["how"] == "rbgs" else ctx.jacobi
    omega = 1.2 if state["how"] == "rbgs" else 0.8
    go(x, state["A"], state["b"], ffvhc.BC_P, omega, SWEEPS, 0.0)
    return Fields(ctx, {"x": (state["cid"], x)}, state["dtype"])


def _prepare_forces(case, seed):
    root, edge, levels = _root(case), case["edge"], case["levels"]
    tree = _flow_tree(root, edge, levels)
    ctx = ffvhc.Context(max_blocks=tree.nblk)
    cid = ctx.add_case(tree, flows.flow_params(100.0, 0.001), geometry=_flow_geometry(root, edge, levels))
    f = [ctx.field(8) for _ in range(4)]
    for field, v in zip(f, _velocity(tree.table(), seed)):
        ctx.upload(field, cid, v)
    return {"run": _run_forces, "ctx": ctx, "cid": cid, "f": f}


def _run_forces(state):
    ctx, (ux, uy, uz, p) = state["ctx"], state["f"]
    for d, u in enumerate((ux, uy, uz)):
        ctx.ghost_fill(u, ffvhc.BC_UX + d, 5)
    ctx.ghost_fill(p, ffvhc.BC_P, 1)
    out = {"force_p": ctx.force_p(p, 1), "force_v": ctx.force_v(ux, uy, uz, 1), "cfl": ctx.cfl(ux)[0]}
    out["fields"] = Fields(ctx, {k: (state["cid"], f) for k, f in zip(("ux", "uy", "uz", "p"), state["f"])})
    return out


def work(case):
    """Bytes and operations of one pass that no solver can do without: each array in and out once."""
    if case["kind"] == "step":
        cells = sum(_flow_tree(*b[:3]).nblk for b in _batch(case)) * N ** 3
        # in: u, p, the previous terms, face velocities and the cut geometry; out: those and the
        # Poisson system, lapp
        return {"bytes": cells * (16 * 8 + 28 + 25 * 8), "flops": cells * 300}
    if case["kind"] == "forces":
        cells = _flow_tree(_root(case), case["edge"], case["levels"]).nblk * N ** 3
        return {"bytes": cells * 4 * 8, "flops": cells * 10}
    cells = _box_tree(_root(case), case["ball"]).nblk * N ** 3
    turns = SWEEPS if case["kind"] == "sweeps" else 1
    return {"bytes": cells * 9 * case.get("prec", 8), "flops": cells * 15 * turns}


# ---------------------------------------------------------------------------------- in 64 bits

def exact(case, seed):
    """What run returns, in 64 bits by plain torch: the solution of the Poisson system (its residual at
    1e-14), the iterates of the sweeps, the ghost layers and forces.  None for a time step: what it
    returns is set by where its solves stop."""
    if case["kind"] == "step":
        return None
    if case["kind"] == "forces":
        return _exact_forces(case, seed)
    tb = _tables(_box_tree(_root(case), case["ball"]).table())
    A = [_t(a[INNER]) for a in _bands(_root(case), case["ball"], case["body"])]
    b = _t(_rhs(case, seed)[INNER])
    if case["kind"] == "poisson":
        x = _solve(tb, A, b)
    else:
        if case["prec"] == 4:
            A, b = [a.float().double() for a in A], b.float().double()
        x = _sweep(tb, A, b, case["smoother"])
    return {"x": _pad(_with_ghosts(tb, x, P_BC))}


def _t(a):
    return torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=DEV)


def _tables(tb):
    """Per face, the blocks of each neighbour kind with what their ghost values come from."""
    out = {"dx": _t(tb["dx"]), "faces": []}
    ix = lambda a: torch.tensor(a, dtype=torch.long, device=DEV)  # noqa: E731
    for f in range(6):
        kind, nbr, sub = tb["ftype"][:, f], tb["nbr"][:, f], tb["sub"][:, f]
        pick = [np.nonzero(kind == q)[0] for q in range(4)]
        out["faces"].append({"outer": ix(pick[0]), "same": ix(pick[1]), "same_of": ix(nbr[pick[1], 0]),
                             "coarser": ix(pick[2]), "coarser_of": ix(nbr[pick[2], 0]), "sub": sub[pick[2]],
                             "finer": ix(pick[3]), "finer_of": ix(nbr[pick[3]])})
    return out


def _quarter(f, sub):
    """Origin (along the face's slow axis, its fast axis) of quarter `sub` of face f: the quarters
    count the axes y, z on X faces, z, x on Y faces and x, y on Z faces."""
    o0, o1 = sub & 1, sub >> 1
    return (o0, o1) if f // 2 == 1 else (o1, o0)


@functools.lru_cache(maxsize=None)
def _weights(o):
    """Linear interpolation of 16 coarse cells to the 16 fine cells of half o, extrapolated at the ends."""
    w = np.zeros((N, N))
    for a in range(N):
        i = a + 1 + N * o
        ic, r = i // 2, 0.25 + 0.5 * (i % 2)
        if i < 2:
            ic, r = 1, -0.25
        elif i > 2 * N - 1:
            ic, r = N - 1, 1.25
        w[a, ic - 1], w[a, ic] = 1.0 - r, r
    return _t(w)


def _layer(x, f, depth=0):
    """The layer of interior cells `depth` cells inside face f: (blocks, slow axis, fast axis)."""
    return x.select(3 - f // 2, N - 1 - depth if f & 1 else depth)


def _with_ghosts(tb, x, bc, updater=1):
    """(blocks, 18, 18, 18): the interior x and one ghost layer a face (edges and corners 0).  Same
    level: the neighbour's cells; finer neighbours: means of 8; a coarser one: trilinear (updater 1)
    or the own cell plus half the coarse jump (updater 5); outer faces: Dirichlet / Neumann."""
    g = torch.zeros((x.shape[0], N + 2, N + 2, N + 2), dtype=x.dtype, device=x.device)
    g[:, 1:-1, 1:-1, 1:-1] = x
    ghost = [torch.zeros((x.shape[0], N, N), dtype=x.dtype, device=x.device) for _ in range(6)]
    for f, T in enumerate(tb["faces"]):
        kind, value = bc[f]
        o = T["outer"]
        if len(o):
            adj = _layer(x, f)[o]
            step = (value * tb["dx"][o])[:, None, None]
            ghost[f][o] = 2.0 * value - adj if kind == ffvhc.DIRICHLET else adj + step if f & 1 else adj - step
        if len(T["same"]):
            ghost[f][T["same"]] = _layer(x, f ^ 1)[T["same_of"]]
        for q in range(4) if len(T["finer"]) else ():
            src = T["finer_of"][:, q]
            two = 0.5 * (_layer(x, f ^ 1)[src] + _layer(x, f ^ 1, 1)[src])
            ob, oa = _quarter(f, q)
            mean = two.reshape(-1, N // 2, 2, N // 2, 2).mean(dim=(2, 4))
            ghost[f][T["finer"][:, None, None], torch.arange(8 * ob, 8 * ob + 8, device=x.device)[:, None],
                     torch.arange(8 * oa, 8 * oa + 8, device=x.device)] = mean
    for f, T in enumerate(tb["faces"]):
        for q in range(4) if len(T["coarser"]) else ():
            at = torch.tensor(np.nonzero(T["sub"] == q)[0], dtype=torch.long, device=x.device)
            if not len(at):
                continue
            me, src = T["coarser"][at], T["coarser_of"][at]
            ob, oa = _quarter(f, q)
            if updater == 1:
                # the fine ghost centre lies a quarter of a coarse cell inside the coarse block
                p = 1.25 * _layer(x, f ^ 1)[src] - 0.25 * _layer(x, f ^ 1, 1)[src]
                ghost[f][me] = _weights(ob) @ p @ _weights(oa).T
            else:
                jump = 0.5 * (_layer(x, f ^ 1)[src] - ghost[f ^ 1][src])
                jump = jump[:, 8 * ob:8 * ob + 8, 8 * oa:8 * oa + 8]
                ghost[f][me] = _layer(x, f)[me] + jump.repeat_interleave(2, 1).repeat_interleave(2, 2)
    for f in range(6):
        at = [slice(None)] + [slice(1, -1)] * 3
        at[3 - f // 2] = N + 1 if f & 1 else 0
        g[tuple(at)] = ghost[f]
    return g


def _pad(g):
    out = torch.zeros((g.shape[0], NP, NP, NP), dtype=g.dtype, device=g.device)
    out[:, 1:-1, 1:-1, 1:-1] = g
    return out


def _around(g):
    """The six neighbour values w, e, s, n, b, t of every interior cell."""
    c = slice(1, -1)
    lo, hi = slice(0, -2), slice(2, None)
    return (g[:, c, c, lo], g[:, c, c, hi], g[:, c, lo, c], g[:, c, hi, c], g[:, lo, c, c], g[:, hi, c, c])


def _off(A, g):
    return sum(a * v for a, v in zip(A[1:], _around(g)))


NULL_BC = [(ffvhc.NEUMANN, 0.0)] * 6


def _solve(tb, A, b):
    """Jacobi-preconditioned BiCGSTAB from 0, restarted from the true residual until that is 1e-14."""
    mul = lambda v: A[0] * v + _off(A, _with_ghosts(tb, v, NULL_BC))  # noqa: E731
    x = torch.zeros_like(b)
    r = b.clone()
    bb = float(b.norm())
    for _ in range(20):
        if float(r.norm()) <= 1e-14 * bb:
            break
        r0, p, rho, goal = r.clone(), r.clone(), (r * r).sum(), max(1e-14 * bb, 1e-9 * float(r.norm()))
        for it in range(1500):
            y = p / A[0]
            q = mul(y)
            alpha = rho / (q * r0).sum()
            s = r - alpha * q
            z = s / A[0]
            t = mul(z)
            gamma = (t * s).sum() / (t * t).sum()
            x += alpha * y + gamma * z
            r = s - gamma * t
            if it % 10 == 9 and float(r.norm()) <= goal:
                break
            new = (r * r0).sum()
            p = r + (new / rho) * (alpha / gamma) * (p - gamma * q)
            rho = new
        r = b - mul(x)
    return x


def _sweep(tb, A, b, smoother):
    x = torch.zeros_like(b)
    k = torch.arange(N, device=b.device)
    red = (k[:, None, None] + k[:, None] + k) % 2 == 0
    for _ in range(SWEEPS):
        g = _with_ghosts(tb, x, P_BC)
        if smoother == "jacobi":
            x = x - 0.8 * (x - (b - _off(A, g)) / A[0])
            continue
        for colour in (red, ~red):
            x = torch.where(colour, x - 1.2 * (x - (b - _off(A, g)) / A[0]), x)
            g[:, 1:-1, 1:-1, 1:-1] = x
    return x


def _exact_forces(case, seed):
    root, edge, levels = _root(case), case["edge"], case["levels"]
    tree = _flow_tree(root, edge, levels)
    table = tree.table()
    tb = _tables(table)
    cut, cid, pid = _flow_geometry(root, edge, levels)
    shape = (tree.nblk, NP, NP, NP)
    cut = [_t(c.reshape(shape)[INNER]) for c in cut]
    fluid = _t(pid.reshape(shape)[INNER]) == 1
    mask = [((_t(c.reshape(shape)[INNER]) == 1) & fluid).double() for c in cid]
    hit = [_t(c.reshape(shape)[INNER]) == 1 for c in cid]
    dx = tb["dx"][:, None, None, None]
    v = [_t(a[INNER]) for a in _velocity(table, seed)]
    bc = [flows.FLOW_BC[k] for k in (ffvhc.BC_UX, ffvhc.BC_UY, ffvhc.BC_UZ, ffvhc.BC_P)]
    g = [_with_ghosts(tb, v[d], bc[d], 5) for d in range(3)] + [_with_ghosts(tb, v[3], bc[3], 1)]
    # pressure: extrapolated to the cut face from the cell and its opposite neighbour
    near = _around(g[3])
    face = [v[3] + 0.5 * (v[3] - near[f ^ 1]) for f in range(6)]
    fp = [((mask[2 * a + 1] * face[2 * a + 1] - mask[2 * a] * face[2 * a]) * dx * dx).sum() for a in range(3)]
    # viscous: the no-slip wall value behind a cut face, at the cut distance
    mu = 1.0 / 100.0
    un = [[torch.where(hit[f], (1.0 - 1.0 / cut[f]) * v[a], n) for f, n in enumerate(_around(g[a]))] for a in range(3)]
    fv = []
    for a in range(3):
        total = 0.0
        for ax in range(3):
            lo, hi = v[a] - un[a][2 * ax], un[a][2 * ax + 1] - v[a]
            if ax == a:
                lo, hi = 2.0 * lo, 2.0 * hi
            else:
                cross = 0.5 * (un[ax][2 * a + 1] - un[ax][2 * a])
                lo, hi = lo + cross, hi + cross
            total = total + mu / dx * (lo * mask[2 * ax] - hi * mask[2 * ax + 1])
        fv.append((total * dx * dx).sum())
    cfl = v[0].abs().max() * 0.001 / (edge / 2 ** tree.max_level)
    out = {"force_p": torch.stack(fp)[None], "force_v": torch.stack(fv)[None], "cfl": cfl[None]}
    out["fields"] = {k: _pad(w) for k, w in zip(("ux", "uy", "uz", "p"), g)}
    return out
