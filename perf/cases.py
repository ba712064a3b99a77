"""The workloads this library is timed on, through its public entry points (optcuts_amd.capi over the C ABI).

Every case is one pass over a height-field disc (optcuts_amd.meshgen), the library's synthetic mesh class, in one of
these kinds:

  energy    the Energy interface of the reference's line search: a new map, its energy, its gradient and the
            injectivity bound along a direction
  triplets  the projected Hessian as triplets in the reference's order (the drop-in path's assembly)
  solver    the LinSysSolver drop-in: new values on a kept pattern, factorize, one solve
  step      one Newton iteration of the device-resident driver from a given map (the pattern, the set-up and the
            solver's buffers are kept, as they are across the iterations of a solve)
  charts    the same for many independent charts in one batch
  scaffold  a whole call of the joint mode: new map and air mesh, set-up, three Newton iterations with their
            air-mesh updates
  train     one training step's gradient of the learned preconditioner's network on one Newton system

A step is repeated from the same map by setting the map again: the energy that the line search starts from is then
the one the previous pass accepted, which the same step reaches and does not exceed, so every pass takes the same
step (the relative-decrease stop is off).
"""
import math

import numpy as np
import torch

from optcuts_amd import capi, learned
from optcuts_amd import scaffold as air
from optcuts_amd.meshgen import height_field_disc, union_of_charts

PRECOND = {"jacobi": capi.PRECOND_JACOBI, "amg": capi.PRECOND_AMG, "ic0": capi.PRECOND_IC0,
           "learned": capi.PRECOND_LEARNED}


def listed():
    return [
        # 1,922 faces: a local problem's energy test, where latency and launches count
        {"name": "energy_2k", "kind": "energy", "m": 32},
        # 19,602 faces: one drop-in assembly of an ordinary mesh
        {"name": "triplets_20k", "kind": "triplets", "m": 100},
        # 100,352 faces: the drop-in solve with the multigrid, at the solver's default tolerance
        {"name": "solver_100k_amg", "kind": "solver", "m": 225, "precond": "amg"},
        # 1,922 faces: the plain (parity) form on a small mesh, one Jacobi-PCG solve of a few hundred iterations
        {"name": "step_2k_jacobi", "kind": "step", "m": 32, "precond": "jacobi", "mixed": False, "tol": 1e-10},
        # 199,712 faces (the benchmark's disc): the plain form
        {"name": "step_200k_jacobi", "kind": "step", "m": 317, "precond": "jacobi", "mixed": False, "tol": 1e-10},
        # the chosen form on an ordinary, on the benchmark's and on the largest size (199,712 and 1,000,000 faces),
        # at the benchmark's tolerance
        {"name": "step_200k_amg", "kind": "step", "m": 317, "precond": "amg", "mixed": False, "tol": 1e-3},
        {"name": "step_1m_amg", "kind": "step", "m": 708, "precond": "amg", "mixed": False, "tol": 1e-3},
        # the mixed form (FP32 element terms, FP32-stored multigrid)
        {"name": "step_200k_mixed", "kind": "step", "m": 317, "precond": "amg", "mixed": True, "tol": 1e-3},
        # the learned factor with FP32 element terms on an odd size (49,928 faces)
        {"name": "step_50k_learned", "kind": "step", "m": 159, "precond": "learned", "mixed": True, "tol": 5e-3},
        # the benchmark's batch: 64 charts of 500 to 20,000 faces
        {"name": "charts_64", "kind": "charts", "n": 64, "lo": 500, "hi": 20000},
        # 49,928 faces and their air mesh: the joint mode from set-up on
        {"name": "scaffold_50k", "kind": "scaffold", "m": 159},
        # 10,082 faces, the upper end of the training set's meshes; four probes as learned.train uses
        {"name": "train_10k", "kind": "train", "m": 72, "probes": 4},
    ]


def _grid(rng, lo, hi):
    """Grid size of a disc whose face count is drawn over [lo, hi] by its logarithm."""
    faces = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(3, int(round(math.sqrt(faces / 2.0))) + 1)


def draw(rng):
    kind = rng.choice(("energy", "triplets", "solver", "step", "step", "step", "step", "charts", "scaffold", "train"))
    if kind == "energy":
        return {"kind": kind, "m": _grid(rng, 200, 400000)}
    if kind == "triplets":
        return {"kind": kind, "m": _grid(rng, 200, 60000)}
    if kind == "solver":
        precond = rng.choice(("amg", "amg", "ic0", "jacobi"))
        return {"kind": kind, "m": _grid(rng, 500, 100000 if precond == "amg" else 50000), "precond": precond}
    if kind == "step":
        precond, mixed, tol, hi = rng.choice((("jacobi", False, 1e-10, 200000), ("amg", False, 1e-3, 1000000),
                                              ("amg", False, 1e-3, 1000000), ("amg", True, 1e-3, 400000),
                                              ("learned", True, 5e-3, 200000), ("ic0", False, 5e-3, 200000)))
        return {"kind": kind, "m": _grid(rng, 500, hi), "precond": precond, "mixed": mixed, "tol": tol}
    if kind == "charts":
        return {"kind": kind, "n": rng.randint(3, 64), "lo": 500, "hi": rng.randint(2000, 20000)}
    if kind == "scaffold":
        return {"kind": kind, "m": _grid(rng, 1000, 50000)}
    return {"kind": kind, "m": _grid(rng, 500, 20000), "probes": rng.choice((2, 4, 4, 8))}


# ---- inputs -------------------------------------------------------------------------------------------------------
def _distorted(m, seed):
    """A disc and a map of it away from its start: the projection with each vertex moved by up to 0.2 of the grid
    spacing (every triangle keeps its orientation)."""
    V, F, UV = height_field_disc(m, seed=seed)
    rng = np.random.default_rng([seed, 1])
    return V, F, UV + rng.uniform(-0.2, 0.2, UV.shape) / (m - 1)


def _direction(m, UV, seed):
    """A search direction whose injectivity bound lies below a full step."""
    return np.random.default_rng([seed, 2]).normal(size=UV.size) * (0.5 / (m - 1))


def _neighbours(F, nV):
    e = np.concatenate([F[:, [0, 1]], F[:, [1, 2]], F[:, [2, 0]]])
    e = np.unique(np.concatenate([e, e[:, ::-1]]), axis=0)
    ptr = np.concatenate([[0], np.cumsum(np.bincount(e[:, 0], minlength=nV))])
    return ptr.astype(np.int32), e[:, 1].astype(np.int32)


def _context(V, F, UV, fixed=(0,)):
    ctx = capi.Context(0)
    ctx.set_mesh(V, F, fixed=fixed)
    ctx.set_uv(UV)
    return ctx


def _charts(case, seed):
    """Discs of log-uniform face counts; the counts belong to the case, the shapes to the seed."""
    sizes = np.exp(np.random.default_rng(case["n"]).uniform(math.log(case["lo"]), math.log(case["hi"]), case["n"]))
    return [height_field_disc(max(3, int(round(math.sqrt(f / 2.0))) + 1), seed=[seed, k]) for k, f in enumerate(sizes)]


def _train_system(m, seed):
    """The Newton system of a distorted disc as the network sees one: block CSR, block values, fixed mask."""
    V, F, UV = _distorted(m, seed)
    return _block_system(F, _terms(V, F, UV)[2], len(V)) + (np.arange(len(V)) == 0,)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "charts":
        V, F, UV, vs, fs, fixed = union_of_charts(_charts(case, seed))
        ctx = _context(V, F, UV, fixed)
        ctx.set_charts(vs, fs)
        ctx.newton_init(a0=1.0, rel_gl2_tol=1e-30, allow_edec_rel_tol=False, precond=capi.PRECOND_AMG, pcg_rel_tol=1e-4,
                        pcg_max_iter=1000)
        return {"kind": kind, "ctx": ctx, "uv": UV}
    m = case["m"]
    if kind == "train":
        net = capi.Gnn(0)
        net.set_params(np.load(learned.DEFAULT_WEIGHTS))
        net.set_system(*_train_system(m, seed))
        return {"kind": kind, "net": net, "probes": case["probes"], "seed": seed}
    if kind in ("energy", "triplets", "solver"):
        V, F, UV = _distorted(m, seed)
        ctx = _context(V, F, UV)
        state = {"kind": kind, "ctx": ctx, "uv": UV}
        if kind == "energy":
            state["dir"] = _direction(m, UV, seed)
        if kind == "solver":
            I, J, vals = ctx.hessian_triplets()
            ctx.solver_set_pattern(len(V), *_neighbours(F, len(V)), fixed=(0,))
            ctx.solver_set_params(PRECOND[case["precond"]], 1e-10, 100000)
            ctx.solver_set_coords(UV)
            ctx.solver_update_a(I, J, vals)
            state["a"] = ctx.solver_get_a()
            state["rhs"] = -ctx.gradient()
        return state
    V, F, UV = height_field_disc(m, seed=seed)
    ctx = _context(V, F, UV)
    state = {"kind": kind, "ctx": ctx, "uv": UV}
    if kind == "scaffold":
        edge = (2.0 + math.sqrt(2.0)) / (3.0 * (m - 1))  # the map's mean edge, so that a case has one air mesh size
        state["air"] = air.initial_air_mesh(UV, F, edge) + (air.area_threshold(edge), 0.01 * JOINT_A0)
        ctx.set_forcing(0.1, 0.2)
        return state
    if case["precond"] == "learned":
        net = state["net"] = capi.Gnn(0)
        net.set_params(np.load(learned.DEFAULT_WEIGHTS))
        ctx.set_learned(net)
    ctx.newton_init(a0=1.0, rel_gl2_tol=1e-30, allow_edec_rel_tol=False, precond=PRECOND[case["precond"]],
                    pcg_rel_tol=case["tol"], pcg_max_iter=1000 if case["precond"] == "amg" else 200000,
                    precision=capi.PRECISION_MIXED if case["mixed"] else capi.PRECISION_FP64)
    return state


JOINT_A0 = 1.0 - 0.999  # the joint mode's weight of the distortion energy


# ---- passes -------------------------------------------------------------------------------------------------------
def run(state):
    kind, ctx = state["kind"], state.get("ctx")
    if kind == "energy":
        ctx.set_uv(state["uv"])
        return {"E": ctx.energy(), "g": ctx.gradient(), "bound": ctx.init_step_size(state["dir"], 1.0)}
    if kind == "triplets":
        ctx.set_uv(state["uv"])
        I, J, vals = ctx.hessian_triplets()
        return {"I": I, "J": J, "V": vals}
    if kind == "solver":
        ctx.solver_set_a(state["a"])
        ctx.solver_factorize()
        return {"x": ctx.solver_solve(state["rhs"])}
    if kind == "train":
        net = state["net"]
        net.zero_grad()
        loss = net.loss_grad(state["probes"], state["seed"])
        return {"loss": loss, "grad": net.get_grads()}
    ctx.set_uv(state["uv"])
    if kind == "scaffold":
        ctx.set_air_mesh(*state["air"])
        energies = [ctx.newton_init(a0=JOINT_A0, rel_gl2_tol=1e-12, allow_edec_rel_tol=False, precond=capi.PRECOND_AMG,
                                    pcg_rel_tol=1e-3, pcg_max_iter=100)]
        for _ in range(3):
            s, _ = ctx.newton_step()
            energies += [s["E_total"], s["E_SD"], ctx.scaffold_update()[0]]
        return {"uv": ctx.get_uv(), "air": ctx.air_mesh_get()[0], "E": np.array(energies)}
    s, _ = ctx.newton_step()
    out = {"uv": ctx.get_uv(), "E": s["E_total"], "grad_sq": s["grad_sq"], "step": s["step"]}
    if kind == "charts":
        chart = ctx.charts_state()
        out.update(charts_E=chart["E_SD"], charts_grad_sq=chart["grad_sq"], charts_step=chart["step"])
    return out


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def _products(case, faces):
    """Products with the Newton matrix that one solve of a case needs (iterations as measured, growing with the
    square root of the size for the point and incomplete factors; a multigrid iteration counts its V-cycle's six
    fine-level products over 1.2, the coarse levels' share)."""
    precond, tol = case.get("precond", "amg"), case.get("tol", 1e-10 if case["kind"] == "solver" else 1e-3)
    root = math.sqrt(faces / 200000.0)
    if precond == "amg":
        return 7.0 * (25 if tol < 1e-6 else 9)
    if precond == "learned":
        return 2.0 * max(4.0, 40 * root)
    if precond == "ic0":
        return 3.0 * max(4.0, (900 if tol < 1e-6 else 34) * root)
    return max(20.0, 6000 * root)


def work(case):
    kind = case["kind"]
    if kind == "charts":
        faces = case["n"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
    else:
        faces = 2.0 * (case["m"] - 1) ** 2
    verts, blocks = faces / 2.0, 3.5 * faces
    element = 52.0 * faces  # vertex ids and rest features of a triangle
    if kind == "energy":
        return {"bytes": element + (16 + 16 + 16) * verts, "flops": 120.0 * faces}
    if kind == "triplets":
        return {"bytes": element + 16 * verts + 36 * 16 * faces, "flops": 900.0 * faces}
    if kind == "train":
        edges = 6.0 * verts
        per_layer = 2 * 32 * 80 * edges + 2 * 32 * 64 * verts  # message and update products, three times (fwd, bwd)
        return {"bytes": 36.0 * blocks + 2 * 4 * 14599, "flops": 3 * 3 * per_layer}
    products = _products(case, faces) * (3 if kind == "scaffold" else 1)
    matrix = 36.0 * blocks + 48.0 * verts  # blocks with their columns, a vector gathered once, one written
    bytes_ = products * matrix + (24.0 * blocks if kind == "solver" else element + 32 * verts)
    return {"bytes": bytes_, "flops": 8.0 * blocks * products + (0 if kind == "solver" else 900.0 * faces)}


def tolerance(case):
    """Relative differences of another correct implementation: about four times what the sums in another order, the
    same path in 64 bits (exact) or, for a solve stopped at a loose tolerance, one stopped an iteration earlier or
    later give over the declared sizes."""
    kind = case["kind"]
    if kind in ("energy", "triplets"):
        return {"rel": 1e-11, "max": 1e-9}
    if kind == "train":  # bf16 operands, FP32 sums
        return {"rel": 1e-3, "max": 0.02}
    if kind == "solver":
        return {"rel": 1e-8, "max": 1e-7}
    if kind == "step" and case["precond"] == "jacobi":
        return {"rel": 1e-9, "max": 1e-8}
    if kind == "step" and case["tol"] > 1e-3:
        return {"rel": 5e-3, "max": 0.02}
    return {"rel": 6e-4, "max": 4e-3}


# ---- the same in plain numpy and torch, 64 bits ---------------------------------------------------------------------
def _features(V, F):
    a, b = V[F[:, 1]] - V[F[:, 0]], V[F[:, 2]] - V[F[:, 0]]
    area2 = 0.25 * (np.cross(a, b) ** 2).sum(1)
    area = np.sqrt(area2)
    forms = [(x * y).sum(1) / (2 * area2) for x, y in ((a, a), (b, b), (a, b))]
    return [area / area.sum(), area2] + forms


_DA, _DB = np.array([-1.0, 1.0, 0.0]), np.array([-1.0, 0.0, 1.0])


def _terms(V, F, UV, hessian=True):
    """Per triangle: energy, gradient (F x 6) and projected Hessian (F x 6 x 6) of w (1 + A^2 / a^2) R(x) with a the
    signed area of the map's triangle and R the quadratic form of the rest metric."""
    w, A2, E0, E1, E01 = _features(V, F)
    X = UV[F]                                     # F x 3 x 2
    p, q = X[:, 1] - X[:, 0], X[:, 2] - X[:, 0]
    a = 0.5 * (p[:, 0] * q[:, 1] - p[:, 1] * q[:, 0])
    K = np.outer(_DA, _DB) - np.outer(_DB, _DA)   # a = x_0^T K x_1 / 2
    Q3 = (E0[:, None, None] * np.outer(_DB, _DB) + E1[:, None, None] * np.outer(_DA, _DA) -
          E01[:, None, None] * (np.outer(_DA, _DB) + np.outer(_DB, _DA)))
    dR = np.einsum("fij,fjd->fid", Q3, X)
    R = 0.5 * np.einsum("fid,fid->f", X, dR)
    da = 0.5 * np.stack([X[:, :, 1] @ K.T, X[:, :, 0] @ K], 2)
    L, L1, L2 = 1 + A2 / a ** 2, -2 * A2 / a ** 3, 6 * A2 / a ** 4
    g = w[:, None, None] * ((R * L1)[:, None, None] * da + L[:, None, None] * dR)
    n = len(F)
    if not hessian:
        return w * L * R, g.reshape(n, 6), None
    d2a = np.zeros((3, 2, 3, 2))
    d2a[:, 0, :, 1] = 0.5 * K
    d2a[:, 1, :, 0] = 0.5 * K.T
    va, vr = da.reshape(n, 6), dR.reshape(n, 6)
    cross = va[:, :, None] * vr[:, None, :]
    H = ((R * L2)[:, None, None] * va[:, :, None] * va[:, None, :] + (R * L1)[:, None, None] * d2a.reshape(6, 6) +
         L1[:, None, None] * (cross + cross.transpose(0, 2, 1)) +
         L[:, None, None] * np.einsum("fij,de->fidje", Q3, np.eye(2)).reshape(n, 6, 6)) * w[:, None, None]
    lam, vec = np.linalg.eigh(H)
    return w * L * R, g.reshape(n, 6), (vec * np.maximum(lam, 0.0)[:, None, :]) @ vec.transpose(0, 2, 1)


def _gradient(F, g, nV):
    out = np.zeros((nV, 2))
    np.add.at(out, F, g.reshape(-1, 3, 2))
    out[0] = 0.0
    return out


def _block_system(F, H, nV):
    """Block CSR (row pointers, columns, 2x2 blocks) of the summed element Hessians, vertex 0 fixed (identity)."""
    rows, cols = np.repeat(F, 3, 1).ravel(), np.tile(F, (1, 3)).ravel()
    blocks = H.reshape(-1, 3, 2, 3, 2).transpose(0, 1, 3, 2, 4).reshape(-1, 2, 2)
    free = (rows != 0) & (cols != 0)
    rows, cols = np.append(rows[free], 0), np.append(cols[free], 0)
    blocks = np.concatenate([blocks[free], np.eye(2)[None]])
    key, at = np.unique(rows.astype(np.int64) * nV + cols, return_inverse=True)
    vals = np.zeros((len(key), 2, 2))
    np.add.at(vals, at, blocks)
    ptr = np.concatenate([[0], np.cumsum(np.bincount(key // nV, minlength=nV))])
    return ptr.astype(np.int32), (key % nV).astype(np.int32), vals


def _bound(F, UV, d):
    """First positive root of the map's triangle areas along d, at most 1."""
    X, D = UV[F], d.reshape(-1, 2)[F]
    p, q, s, t = X[:, 1] - X[:, 0], X[:, 2] - X[:, 0], D[:, 1] - D[:, 0], D[:, 2] - D[:, 0]
    det = lambda x, y: x[:, 0] * y[:, 1] - x[:, 1] * y[:, 0]  # noqa: E731
    a, b, c = det(s, t), det(p, t) + det(s, q), det(p, q)
    with np.errstate(all="ignore"):
        root = np.sqrt(b * b - 4 * a * c)
        r = np.stack([2 * c / (-b + root), 2 * c / (-b - root)])
    r[~(r > 0)] = np.inf
    return min(1.0, float(r.min()))


def _solve(ptr, col, vals, rhs):
    """Solution of a symmetric block CSR system: dense, or beyond a few thousand unknowns diagonally preconditioned
    conjugate gradients to a residual of 1e-14."""
    n = len(ptr) - 1
    row = np.repeat(np.arange(n), np.diff(ptr))
    if n <= 3000:
        A = np.zeros((n, 2, n, 2))
        A[row, :, col, :] = vals
        return np.linalg.solve(A.reshape(2 * n, 2 * n), rhs)
    at = "cuda" if torch.cuda.is_available() else "cpu"
    i = (2 * row[:, None, None] + np.arange(2)[:, None] + np.zeros((2, 2), int)).ravel()
    j = (2 * col.astype(np.int64)[:, None, None] + np.arange(2) + np.zeros((2, 2), int)).ravel()
    A = torch.sparse_coo_tensor(np.stack([i, j]), vals.ravel(), (2 * n, 2 * n), dtype=torch.float64, device=at)
    A = A.coalesce().to_sparse_csr()
    M = torch.from_numpy(1.0 / vals[row == col][:, [0, 1], [0, 1]].ravel()).to(at)
    r = torch.from_numpy(np.ascontiguousarray(rhs)).to(at)
    x, z, stop = torch.zeros_like(r), M * r, 1e-28 * float(r @ r)
    p, rz = z.clone(), r @ z
    for it in range(100000):
        q = A @ p
        alpha = rz / (p @ q)
        x += alpha * p
        r -= alpha * q
        if it % 64 == 63 and float(r @ r) <= stop:
            break
        z = M * r
        rz, old = r @ z, rz
        p = z + (rz / old) * p
    return x.cpu().numpy()


def _exact_step(m, seed, solve):
    V, F, UV = height_field_disc(m, seed=seed)
    E, g, H = _terms(V, F, UV, solve)
    grad = _gradient(F, g, len(V)).ravel()
    out = {"uv": None, "E": None, "grad_sq": float(grad @ grad), "step": None}
    if not solve:
        return out
    d = _solve(*_block_system(F, H, len(V)), -grad)
    step, e0 = 0.99 * _bound(F, UV, d), E.sum()
    while True:
        new = UV + step * d.reshape(-1, 2)
        e = _terms(V, F, new, False)[0].sum()
        if e <= e0:
            return dict(out, uv=new, E=float(e), step=step)
        step /= 2


def _probe(n2, seed, j):
    """The +-1 probe vector j of a seed (the library's hash)."""
    M = np.uint64(0xFFFFFFFF)
    x = (np.arange(n2, dtype=np.uint64) * np.uint64(0x9E3779B1) + np.uint64(seed & 0xFFFFFFFF) * np.uint64(0x85EBCA77) +
         np.uint64(j) * np.uint64(0xC2B2AE3D)) & M
    for shift, mul in ((16, 0x7FEB352D), (15, 0x846CA68B), (16, None)):
        x ^= x >> np.uint64(shift)
        if mul:
            x = (x * np.uint64(mul)) & M
    return torch.from_numpy(np.where(x & np.uint64(1), 1.0, -1.0)).reshape(-1, 2)


def _exact_train(m, probes, seed):
    ptr, col, vals, fixed = _train_system(m, seed)
    nV = len(ptr) - 1
    row = np.repeat(np.arange(nV), np.diff(ptr))
    diag = row == col
    C = torch.linalg.inv(torch.linalg.cholesky(torch.from_numpy(vals[diag])))
    eu, ew, A = (torch.from_numpy(x[~diag]) for x in (row, col.astype(np.int64), vals))
    A = C[eu] @ A @ C[ew].transpose(1, 2)
    deg = torch.bincount(eu, minlength=nV).double()
    trace = torch.from_numpy(np.log(vals[diag][:, 0, 0] + vals[diag][:, 1, 1]))
    free = torch.from_numpy(~fixed)
    x = torch.stack([torch.ones(nV).double(), deg / 8, torch.where(free, trace - trace[free].mean(), 0.0),
                     (~free).double()], 1)
    e = torch.cat([A.reshape(-1, 4), A.pow(2).sum((1, 2)).sqrt()[:, None], (ew < eu)[:, None].double(),
                   (ew > eu)[:, None].double(), torch.zeros(len(eu), 9).double()], 1)
    theta = torch.from_numpy(np.load(learned.DEFAULT_WEIGHTS).astype(np.float64)).requires_grad_()
    at = [0]

    def take(*shape):
        n = int(np.prod(shape))
        at[0] += n
        return theta[at[0] - n:at[0]].reshape(shape)

    sums = lambda v: torch.zeros(nV, *v.shape[1:]).double().index_add(0, eu, v)  # noqa: E731
    h = torch.relu(x @ take(32, 4).T + take(32))
    for _ in range(3):
        msg = torch.relu(torch.cat([h[eu], h[ew], e], 1) @ take(32, 80).T + take(32))
        h = h + torch.relu(torch.cat([h, sums(msg) / deg.clamp(min=1)[:, None]], 1) @ take(32, 64).T + take(32))
    low = ew < eu
    lu, lw = eu[low], ew[low]
    G = (torch.cat([h[lu], h[lw], e[low]], 1) @ take(4, 80).T + take(4)).reshape(-1, 2, 2)
    d = h @ take(3, 32).T + take(3)
    D = torch.stack([d[:, 0].exp(), torch.zeros(nV).double(), d[:, 1], d[:, 2].exp()], 1).reshape(-1, 2, 2)
    D = torch.where(free[:, None, None], D, torch.eye(2).double())
    mul = lambda B, v: (B @ v[:, :, None])[:, :, 0]  # noqa: E731
    loss = 0.0
    for j in range(probes):
        v = _probe(2 * nV, seed, j)
        y = mul(D.transpose(1, 2), v).index_add(0, lw, mul(G.transpose(1, 2), v[lu]))
        y = y + sums(mul(A, y[ew]))
        loss = loss + (mul(D, y).index_add(0, lu, mul(G, y[lw])) - v).pow(2).sum()
    loss = loss / (probes * 2 * nV)
    loss.backward()
    return {"loss": float(loss.detach()), "grad": theta.grad.numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "energy":
        V, F, UV = _distorted(case["m"], seed)
        E, g, _ = _terms(V, F, UV, False)
        return {"E": float(E.sum()), "g": _gradient(F, g, len(V)).ravel(),
                "bound": _bound(F, UV, _direction(case["m"], UV, seed))}
    if kind == "triplets":
        V, F, UV = _distorted(case["m"], seed)
        H = _terms(V, F, UV)[2].reshape(-1, 3, 2, 3, 2).transpose(0, 1, 3, 2, 4)  # triangle, corner, corner, 2, 2
        free = ((F != 0)[:, :, None] & (F != 0)[:, None, :])
        at = 2 * np.broadcast_to(F[:, :, None, None, None], H.shape) + np.arange(2)[:, None]
        to = 2 * np.broadcast_to(F[:, None, :, None, None], H.shape) + np.arange(2)
        end = np.array([0, 1])
        return {"I": np.append(at[free], end), "J": np.append(to[free], end), "V": np.append(H[free], [1.0, 1.0])}
    if kind == "solver":
        V, F, UV = _distorted(case["m"], seed)
        _, g, H = _terms(V, F, UV)
        return {"x": _solve(*_block_system(F, H, len(V)), -_gradient(F, g, len(V)).ravel())}
    if kind == "step":  # a solve stopped at a loose tolerance has no exact value of its own, its gradient has
        return _exact_step(case["m"], seed, case["tol"] < 1e-6)
    if kind == "train":
        return _exact_train(case["m"], case["probes"], seed)
    return None  # truncated solves
