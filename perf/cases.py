"""The measured workloads of the framework: calls that a simulation program makes, through the
public binding (``cipc.gpu``) of the device library, over the sizes that it makes them at.

Kinds of a case (``kind``):

* ``iteration``: the non-linear stages of one Newton iteration (active set, assembly, step
  bound, line-search energy), the matrix left on the device for the solve; the gradient and
  the right-hand side are read back, as a program with its own convergence test does;
* ``system``: active set and assembled system handed to the program (it factorises the matrix
  on the host), through the C interface into buffers that the program keeps;
* ``solve``: the Newton linear solve of an assembled system to the default 1e-6;
* ``line_search``: one trial step (move, intersection test, energy) and the positions it reached;
* ``time_step``: one whole implicit time step.

Bodies (``body``): ``cubes``, lattice cubes stacked in contact on the ground (``count`` cubes of
``cells``^3 cells); ``cloth``, a cloth of ``cells``^2 quads folded over a ball collider;
``batch``, ``count`` independent cubes of up to ``cells``^3 cells, at the frame where each
reaches the ground, in one batch context.  The seed sets the vertex jitter, the rotations, the
velocities and the direction; the sizes are the case's.
"""
import ctypes
import dataclasses
import functools
import math
import os
import sys

import numpy as np

_PACKAGE = os.path.abspath("cpu-ipc_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from cipc import gpu, scenes  # noqa: E402

_DP, _IP, _I64P = (ctypes.POINTER(t) for t in (ctypes.c_double, ctypes.c_int, ctypes.c_int64))
_FP64, _MIXED = 0, 1                 # solve precisions
_JACOBI, _FSAI = 0, 1                # solve preconditioners
_ALPHA = 0.05                        # the trial step of a line search that has been cut back a few times


def listed():
    return [
        # a small interactive scene whose program solves on the host: latency of every launch and read-back
        dict(name="system-cubes-2x4", kind="system", body="cubes", count=2, cells=4),
        # the same path for the hinge-angle cloth, the other bending model
        dict(name="system-cloth-41-hinge", kind="system", body="cloth", cells=41, bending=1),
        # an odd-sized middling scene: launch-bound
        dict(name="iteration-cubes-2x11", kind="iteration", body="cubes", count=2, cells=11, mixed=False),
        # the benchmark's own scene (37,044 vertices, 160,000 tets)
        dict(name="iteration-cubes-4x20", kind="iteration", body="cubes", count=4, cells=20, mixed=False),
        # a large scene (143,748 vertices, 655,360 tets), elastic Hessian blocks in the mixed form
        dict(name="iteration-cubes-4x32-mixed", kind="iteration", body="cubes", count=4, cells=32, mixed=True),
        # cloth in self-contact (triangles, quadratic bending): no tet to speak of, contacts dominate
        dict(name="iteration-cloth-128", kind="iteration", body="cloth", cells=128, bending=0, mixed=False),
        # many independent scenes in one context, as for data generation
        dict(name="iteration-batch-40x24", kind="iteration", body="batch", count=40, cells=24, mixed=False),
        # the solve of a small system with the plain preconditioner: per-iteration latency
        dict(name="solve-cubes-2x9-jacobi", kind="solve", body="cubes", count=2, cells=9, precision=_FP64, preconditioner=_JACOBI),
        # the default solve of the time step (FP64, block FSAI) on the benchmark's system
        dict(name="solve-cubes-4x20-fsai", kind="solve", body="cubes", count=4, cells=20, precision=_FP64, preconditioner=_FSAI),
        # lock-step solves of a batch, FP32 inside FP64 refinement
        dict(name="solve-batch-24x20-mixed", kind="solve", body="batch", count=24, cells=20, precision=_MIXED, preconditioner=_FSAI),
        # one trial step of the line search on the benchmark's scene
        dict(name="line_search-cubes-4x20", kind="line_search", body="cubes", count=4, cells=20),
        # a whole implicit step of a small scene: every stage, tens of times over
        dict(name="time_step-cubes-2x6", kind="time_step", body="cubes", count=2, cells=6),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["system", "iteration", "iteration", "iteration", "solve", "solve", "line_search", "time_step"])
    bodies = {"system": ["cubes", "cloth"], "iteration": ["cubes", "cubes", "cloth", "batch"], "solve": ["cubes", "cubes", "batch"],
              "line_search": ["cubes", "cloth", "batch"], "time_step": ["cubes"]}
    body = rng.choice(bodies[kind])
    case = dict(kind=kind, body=body)
    if body == "cubes":
        top = {"system": 16, "iteration": 30, "solve": 20, "line_search": 28, "time_step": 6}[kind]
        case.update(count=rng.randint(2, 2 if kind == "time_step" else 4), cells=_between(rng, 4, top))
    elif body == "cloth":
        case.update(cells=_between(rng, 16, 60 if kind == "system" else 128), bending=rng.randint(0, 1))
    else:
        case.update(count=_between(rng, 3, 40 if kind != "solve" else 24), cells=rng.randint(9, 24 if kind != "solve" else 20))
    if kind == "iteration":
        case.update(mixed=rng.random() < 0.3)
    if kind == "solve":
        case.update(precision=rng.choice([_FP64, _MIXED]), preconditioner=rng.choice([_JACOBI, _FSAI, _FSAI]))
    return case


# ---- scenes ------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _lattice(cells):
    """One unperturbed cube of unit cells as a scene: the topology, which no seed changes."""
    x, tets = scenes.lattice(cells, 1.0)
    return scenes.finalize(f"cube{cells}", x, tets, scenes.Material())


def _bodies(parts, material, velocities, diag2=None):
    """A scene of lattice cubes [(template, positions)], with the set-up rules of
    ``scenes.finalize`` but the templates' surfaces."""
    off = np.cumsum([0] + [len(x) for _, x in parts])
    toff = np.cumsum([0] + [t.T for t, _ in parts])
    x = np.concatenate([x for _, x in parts])
    tets = np.concatenate([t.tets + o for (t, _), o in zip(parts, off)])
    faces = np.concatenate([t.faces + np.array([o, o, o, k]) for (t, _), o, k in zip(parts, off, toff)])
    sv = np.concatenate([t.surf_verts + o for (t, _), o in zip(parts, off)])
    se = np.concatenate([t.surf_edges + o for (t, _), o in zip(parts, off)])
    dm_inv, vol = scenes.dm_inverse_colmajor(x, tets)
    masses = np.bincount(tets.reshape(-1), np.repeat(vol * material.density / 4.0, 4), len(x))
    if diag2 is None:
        diag2 = float(np.sum((x.max(axis=0) - x.min(axis=0)) ** 2))
    elen = float(np.linalg.norm(x[se[:, 0]] - x[se[:, 1]], axis=1).sum() / (3 * len(se)))
    return scenes.Scene(name="cubes", x=x.copy(), v_rest=x.copy(), V_prev=x.copy(), velocities=velocities, tets=tets.astype(np.int32),
                        dm_inv=dm_inv, volumes=vol, masses=masses, boundary=np.zeros(len(x), np.int32), faces=faces.astype(np.int32),
                        surf_verts=sv.astype(np.int32), surf_edges=se.astype(np.int32), material=material, bbox_diag2=diag2,
                        hhat=material.rel_dhat ** 2 * diag2, fhat=material.fhat_rel * diag2, dtol=material.dtol_rel * diag2,
                        mean_mass=float(masses.mean()), avg_edge_len=elen)


def _stacked(count, cells, seed):
    """Cubes of cell edge 0.1 m, yawed at random, stacked with 1e-3 m gaps (below the contact
    distance) on the ground, each moving at up to 0.5 m/s per axis; friction 0.3."""
    rng = np.random.default_rng([seed, 1])
    template, parts, vel, floor = _lattice(cells), [], [], scenes.GROUND_Y + 1e-3
    for _ in range(count):
        x = (template.v_rest + rng.uniform(-0.01, 0.01, template.v_rest.shape) - 0.5 * cells) * 0.1
        x = x @ scenes.yaw_rotation(rng).T
        lo, hi = x.min(axis=0), x.max(axis=0)
        x = x + np.array([-0.5 * (lo[0] + hi[0]), floor - lo[1], -0.5 * (lo[2] + hi[2])])
        floor = x[:, 1].max() + 1e-3
        parts.append((template, x))
        vel.append(np.tile(rng.uniform(-0.5, 0.5, 3), (len(x), 1)))
    return _bodies(parts, scenes.Material(friction=0.3), np.concatenate(vel))


def _landed(count, cells, seed):
    """Independent unit cubes, cell counts spread over 8..cells, stiffness per scene, the lowest
    point 0.2-0.9 contact distances above the ground, at the speed of a 0.02-0.2 m drop."""
    rng = np.random.default_rng([seed, 2])
    out = []
    for k in range(count):
        n = int(round(8 * (cells / 8) ** (k / max(count - 1, 1))))
        mat = scenes.Material(youngs=math.exp(rng.uniform(math.log(1e4), math.log(1e6))), poisson=rng.uniform(0.3, 0.45), friction=0.2)
        t = _lattice(n)
        x = (t.v_rest + rng.uniform(-0.01, 0.01, t.v_rest.shape)) / n
        height = rng.uniform(0.2, 0.9) * mat.rel_dhat * math.sqrt(3.0)
        x = x + np.array([3.0 * k, scenes.GROUND_Y + height, 0.0]) - x.min(axis=0)
        v = np.tile([0.0, -math.sqrt(2 * 9.8 * rng.uniform(0.02, 0.2)), 0.0], (len(x), 1))
        out.append(_bodies([(t, x)], mat, v, diag2=3.0))
    return out


@functools.lru_cache(maxsize=4)
def _cloth_template(cells, bending):
    return scenes.cloth_on_sphere(n=cells, sphere_cells=8, bending=bending, fold=cells // 2)


def _cloth(cells, bending, seed):
    """The folded cloth, every cloth vertex displaced by up to 2% of a cell in its plane and 2% of
    the layer gap in height, falling at up to 0.5 m/s."""
    t = _cloth_template(cells, bending)
    rng = np.random.default_rng([seed, 3])
    free = (t.boundary == 0)[:, None]
    x = t.x + free * rng.uniform(-1.0, 1.0, t.x.shape) * np.array([0.02 / cells, 1.2e-5, 0.02 / cells])
    v = free * np.array([0.1, -0.5, 0.05]) * rng.uniform(0.5, 1.0)
    return dataclasses.replace(t, x=x, V_prev=x.copy(), velocities=v)


def _scene(case, seed):
    if case["body"] == "cubes":
        return _stacked(case["count"], case["cells"], seed)
    if case["body"] == "cloth":
        return _cloth(case["cells"], case["bending"], seed)
    return _landed(case["count"], case["cells"], seed)


# ---- one case ----------------------------------------------------------------------------
class _State:
    pass


def _probe(case, seed):
    """(scenes, inertial targets, step-start positions, directions, stiffness), each per scene:
    a Newton state in the middle of a step, the direction as the inertia alone gives it."""
    s = _scene(case, seed)
    many = s if isinstance(s, list) else [s]
    probes = [scenes.newton_probe_state(sc, seed=seed % (1 << 31) + 7) for sc in many]
    kappa = [scenes.suggest_kappa(sc.hhat, sc.bbox_diag2, sc.mean_mass) for sc in many]
    return many, [xt for xt, _ in probes], [sc.x - sc.velocities * sc.material.dt for sc in many], [p for _, p in probes], np.array(kappa)


def prepare(case, seed):
    st = _State()
    st.case = case
    many, xt, prev, p, kappa = _probe(case, seed)
    batch = case["body"] == "batch"
    st.kappa = kappa if batch else float(kappa[0])
    st.ctx = gpu.BatchContext(many, xtildes=xt) if batch else gpu.GpuContext(many[0], xtilde=xt[0])
    if case["kind"] == "time_step":
        st.start = (many[0].x, many[0].V_prev, xt[0], many[0].velocities)
        st.params = gpu.step_params(many[0])
        return st
    st.p = np.concatenate(p)
    st.ctx.set_state(V_prev=np.concatenate(prev))
    st.ctx.active_set()
    st.ctx.friction_update(st.kappa)
    st.ctx.set_direction(st.p)
    if case.get("mixed"):
        st.ctx.set_hessian_precision(1)
    if case["kind"] == "solve":
        st.ctx.newton_iteration(st.kappa)
    if case["kind"] == "line_search":
        st.ctx.save_positions()
        st.x = np.zeros((st.ctx.V, 3))
    if case["kind"] == "iteration":
        st.gradient, st.rhs = np.zeros((st.ctx.V, 3)), np.zeros(3 * st.ctx.V)
    if case["kind"] == "system":
        st.buffers = _buffers(case)
    return st


def _call(name, ctx, *args):
    lib = gpu.load()
    if getattr(lib, "cipc_gpu_" + name)(ctx.h, *args) != gpu.OK:
        raise RuntimeError(lib.cipc_gpu_last_error().decode())


def _at(a, pointer=_DP):
    return None if a is None else a.ctypes.data_as(pointer)


def _buffers(case):
    """What a program that solves on the host keeps: arrays as large as its scene can need."""
    V, _, nnz, F, _ = _counts(case)
    room = 8 * F + 1024                          # contacts and pairs of a scene with layers in contact
    return dict(counts=np.zeros(4, np.int64), self_set=np.zeros((room, 4), np.int32), ee_set=np.zeros((room, 4), np.int32),
                ee_ie=np.zeros((room, 2), np.int32), ccd_set=np.zeros((4 * room, 2), np.int32), env_set=np.zeros(V, np.int32),
                nnz=np.zeros(1, np.int64), collisions=np.zeros(1, np.int32), gradient=np.zeros((V, 3)), outer=np.zeros(3 * V + 1, np.int32),
                inner=np.zeros(nnz + 40 * room, np.int32), values=np.zeros(nnz + 40 * room), rhs=np.zeros(3 * V))


def _system(ctx, kappa, b):
    _call("active_set", ctx, _at(b["counts"], _I64P))
    if max(b["counts"][0], b["counts"][1]) > len(b["self_set"]) or b["counts"][2] > len(b["ccd_set"]):
        raise RuntimeError("the program's contact arrays are too small")
    _call("get_active_set", ctx, *[_at(b[k], _IP) for k in ("self_set", "ee_set", "ee_ie", "ccd_set", "env_set")])
    _call("assemble", ctx, kappa, _at(b["nnz"], _I64P), _at(b["collisions"], _IP))
    if b["nnz"][0] > len(b["values"]):
        raise RuntimeError("the program's matrix arrays are too small")
    _call("get_gradient", ctx, _at(b["gradient"]))
    _call("get_csr", ctx, _at(b["outer"], _IP), _at(b["inner"], _IP), _at(b["values"]), _at(b["rhs"]))
    return b


_BATCH_VALUES = ("alpha_scenes", "energy_scenes", "nnz", "contacts", "collisions")
_VALUES = ("alpha", "bound_ground", "bound_partial", "bound_cfl", "bound_full", "energy", "nnz", "contacts", "collisions")


def run(st):
    case, ctx = st.case, st.ctx
    kind = case["kind"]
    if kind == "iteration":
        t = ctx.newton_iteration(st.kappa)
        out = {k: t[k] for k in (_BATCH_VALUES if case["body"] == "batch" else _VALUES)}
        _call("get_gradient", ctx, _at(st.gradient))
        _call("get_csr", ctx, None, None, None, _at(st.rhs))
        return dict(out, gradient=st.gradient, rhs=st.rhs)
    if kind == "system":
        return _system(ctx, st.kappa, st.buffers)
    if kind == "solve":
        return ctx.solve(precision=case["precision"], preconditioner=case["preconditioner"])[0]
    if kind == "line_search":
        ctx.step_forward(_ALPHA)
        hit = ctx.is_intersected()
        terms = ctx.energy_terms(st.kappa)
        _call("get_positions", ctx, _at(st.x))
        return {"hit": np.asarray(hit), "terms": [terms[..., k] for k in range(9)], "x": st.x}
    x, prev, xt, v = st.start
    ctx.set_state(x, prev, xt)
    ctx.set_velocities(v)
    kappa, stats = ctx.time_step(0.0, st.params)
    x, _, _, v = ctx.state()
    return {"x": x, "velocities": v, "kappa": kappa}


# ---- what a pass cannot do without ---------------------------------------------------------
def _counts(case):
    """(V, T, nonzeros of the lower elastic matrix, surface faces, triangles): a lattice of c^3
    cells has 3 c (c+1)^2 axis edges and 3 c^2 (c+1) face diagonals."""
    if case["body"] == "cloth":
        c, b = case["cells"], 8
        v = (c + 1) ** 2
        return v + (b + 1) ** 3, 5 * b ** 3, 6 * v + 9 * (3 * c * c + 2 * c) + 9 * 3 * c * c, 2 * c * c + 12 * b * b, 2 * c * c
    if case["body"] == "cubes":
        sizes = [case["cells"]] * case["count"]
    else:
        sizes = [int(round(8 * (case["cells"] / 8) ** (k / max(case["count"] - 1, 1)))) for k in range(case["count"])]
    V, T = sum((c + 1) ** 3 for c in sizes), sum(5 * c ** 3 for c in sizes)
    E = sum(3 * c * (c + 1) ** 2 + 3 * c * c * (c + 1) for c in sizes)
    return V, T, 6 * V + 9 * E, sum(12 * c * c for c in sizes), 0


def work(case):
    """Bytes: positions, step start and target, direction, mass, topology and rest shape in, each
    output out, once.  Flops: about 2,000 per projected tet stiffness with its gradient, 600 per
    triangle, 60 per energy evaluation of an element; for a solve one product with the matrix
    and the vector updates of one iteration (how many are needed depends on the method)."""
    V, T, nnz, F, tri = _counts(case)
    elements = 96 * T + 60 * tri
    surface = F * (12 + 12)                      # faces and the 1.5 edges of each
    system = 12 * nnz + 4 * (3 * V + 1)
    kind = case["kind"]
    if kind == "solve":
        return {"bytes": system + 48 * V, "flops": 4 * nnz + 30 * V}
    if kind == "line_search":
        return {"bytes": 24 * 4 * V + 8 * V + elements + surface, "flops": 60 * (T + tri) + 30 * V}
    flops = 2000 * T + 600 * tri + 60 * (T + tri)
    if kind == "time_step":
        return {"bytes": 24 * 7 * V + 8 * V + elements + surface, "flops": 2 * flops}
    return {"bytes": 24 * 4 * V + 8 * V + elements + surface + system + 48 * V, "flops": flops}


def tolerance(case):
    """FP64 sums in another order, and contact projections that cancel: 1e-10, the mixed form too
    (its blocks are rounded before any sum).  A solve stops at a relative residual of 1e-6:
    over bodies, sizes, precisions and preconditioners its direction lies up to 4.1e-6 (2-norm)
    and 7.2e-5 (largest entry over the root mean square) from the one of a residual of 1e-11.  A
    time step's velocities differ by up to 7.3e-6 and 1.0e-4 between preconditioners and
    precisions of its solves.  About four times each."""
    if case["kind"] == "solve":
        return {"rel": 2e-5, "max": 3e-4}
    if case["kind"] == "time_step":
        return {"rel": 3e-5, "max": 4e-4}
    return {"rel": 1e-10, "max": 1e-8}


# ---- the same in plain numpy ---------------------------------------------------------------
def _elastic(sc, x):
    """(F, I2, J) of every tet and its (mu, lambda)-rates."""
    d = np.stack([x[sc.tets[:, k]] - x[sc.tets[:, 0]] for k in (1, 2, 3)], axis=2)
    F = d @ sc.dm_inv.reshape(-1, 3, 3).transpose(0, 2, 1)
    return F, np.einsum("tij,tij->t", F, F), np.linalg.det(F), sc.material.length_rate, sc.material.volume_rate


def _elastic_energy(sc, x):
    _, I2, J, u, r = _elastic(sc, x)
    return float(np.sum(sc.volumes * (0.5 * u * (I2 - 3) + 0.5 * r * (J - 1 - 3 * u / (4 * r)) ** 2 - 0.5 * u * np.log(I2 + 1))))


def _elastic_gradient(sc, x):
    F, I2, J, u, r = _elastic(sc, x)
    cof = np.stack([np.cross(F[:, :, 1], F[:, :, 2]), np.cross(F[:, :, 2], F[:, :, 0]), np.cross(F[:, :, 0], F[:, :, 1])], axis=2)
    P = (u * (1 - 1 / (I2 + 1)))[:, None, None] * F + (r * (J - 1 - 3 * u / (4 * r)))[:, None, None] * cof
    H = sc.volumes[:, None, None] * (P @ sc.dm_inv.reshape(-1, 3, 3))       # columns: forces on corners 1..3
    g = np.zeros_like(x)
    for k in (1, 2, 3):
        np.add.at(g, sc.tets[:, k], H[:, :, k - 1])
        np.add.at(g, sc.tets[:, 0], -H[:, :, k - 1])
    return g


def _landed_exact(sc, xt, prev, kappa):
    """(energy, gradient) of a landed cube: elasticity, inertia, the ground's barrier and its
    lagged friction (the cube meets nothing else)."""
    x, m, dt2, hhat = sc.x, sc.masses, sc.material.dt ** 2, sc.hhat
    dx = x - xt
    e = dt2 * _elastic_energy(sc, x) + 0.5 * float(np.sum(m * np.sum(dx * dx, axis=1)))
    g = dt2 * _elastic_gradient(sc, x) + m[:, None] * dx
    h = x[sc.surf_verts, 1] - scenes.GROUND_Y
    near = h * h < hhat
    v, h = sc.surf_verts[near], h[near]
    d = h * h
    slope = (hhat - d) * (2 * np.log(d / hhat) - hhat / d + 1)
    e += kappa * float(np.sum(-(d - hhat) ** 2 * np.log(d / hhat)))
    g[v, 1] += kappa * slope * 2 * h
    lam = -kappa * slope * 2 * h
    eps = math.sqrt(sc.fhat * dt2)
    t = (x - prev)[v] * np.array([1.0, 0.0, 1.0])
    s = np.linalg.norm(t, axis=1)
    e += sc.material.friction * float(np.sum(lam * np.where(s > eps, s - 0.5 * eps, 0.5 * s * s / eps)))
    g[v] += (sc.material.friction * lam / np.maximum(s, eps))[:, None] * t
    return e, g


def exact(case, seed):
    """What has a closed form: the batch's energies and gradients, the ground and displacement
    bounds of a step, the elastic and inertial energies of a trial step.  The contact terms and
    the systems that hold them would need the whole contact search restated; a solve's and a
    time step's results are the iterates that first meet a threshold."""
    many, xt, prev, p, kappa = _probe(case, seed)
    if case["kind"] == "iteration" and case["body"] == "batch":
        eg = [_landed_exact(sc, a, b, k) for sc, a, b, k in zip(many, xt, prev, kappa)]
        return {"alpha_scenes": None, "energy_scenes": np.array([e for e, _ in eg]), "nnz": None, "contacts": None, "collisions": None,
                "gradient": np.concatenate([g for _, g in eg]), "rhs": np.concatenate([g.reshape(-1) for _, g in eg])}
    if case["kind"] == "iteration":
        sc, sv = many[0], many[0].surf_verts
        out = dict.fromkeys(_VALUES + ("gradient", "rhs"))
        fall, h = p[0][sv, 1], sc.x[sv, 1] - scenes.GROUND_Y
        out["bound_ground"] = float(np.min(np.where(fall > 0, 0.8 * h / np.where(fall > 0, fall, 1.0), 1.0), initial=1.0))
        out["bound_cfl"] = float(math.sqrt(sc.hhat) / (2 * np.linalg.norm(p[0][sv], axis=1).max()))
        return out
    if case["kind"] == "line_search":
        rows, moved = [], []
        for sc, a, q in zip(many, xt, p):
            x = np.where((sc.boundary == 0)[:, None], sc.x - _ALPHA * q, sc.x)
            moved.append(x)
            rows.append([_elastic_energy(sc, x) if sc.T else 0.0, 0.5 * float(np.sum(sc.masses * np.sum((x - a) ** 2, axis=1)))])
        rows = np.array(rows)
        first = rows if case["body"] == "batch" else rows[0]
        return {"hit": None, "terms": [first[..., 0], first[..., 1]] + [None] * 7, "x": np.concatenate(moved)}
    return None
