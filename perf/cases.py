"""The work that the assembly library is measured on: one pass of each public entry point, from a 64 x 64 quad4 mesh, where
launches and host calls are the time, to meshes whose CSR values fill gigabytes.

Every case is a mesh, a physics, a Dirichlet set and a call:

    step        residual and CSR Jacobian in one call (what each Newton iteration assembles)
    residual    the residual alone (line searches, explicit steps)
    mf_action   matrix-free Jacobian action, asm_action the assembled one (Krylov methods without a stored matrix)
    mass        consistent mass matrix on the Jacobian's pattern
    solve       one Newton iteration: residual and Jacobian, Jacobi-preconditioned CG, update of the unknowns
    update      batched learned material update of n quadrature points (network, check of its output, plain fallback)
    gradient    loss and gradient of the learned material's network over n samples (one minibatch of its training)

Meshes are bricks of nx x ny x nz cells (quad4, hex8, or 6 tet10 per cell with jittered vertices), numbered as the
library's own generators number them. Fields are smooth sums of sines and cosines; the finite displacements' gradients
stay below 1 in norm, so that no element folds for any seed.
"""
import ctypes
import functools

import numpy as np
import torch

import __graft_entry__

DEV = "cuda:0"
F64 = torch.float64


def _fec():
    return __graft_entry__.load_package()


# ------------------------------------------------------------------ the cases
def _brick(name, call, elem, physics, nx, ny, nz=0, bc="none", blocks=1):
    c = {"call": call, "elem": elem, "physics": physics, "nx": nx, "ny": ny, "nz": nz, "bc": bc, "blocks": blocks}
    return {"name": name, **c} if name else c


def _points(name, call, net, n):
    c = {"call": call, "net": net, "n": n}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest real problem: the 64 x 64 Poisson square of the reference's test, all edges fixed; the time is
        # host calls, launches and the wait at the end
        _brick("poisson_quad4_step", "step", "quad4", "poisson", 64, 64, bc="all"),
        # the largest scalar problem: diffusion on 2.1 million hex8, 57 million CSR values
        _brick("poisson_hex8_step", "step", "hex8", "poisson", 128, 128, 128),
        # the headline: large-deformation solid on a structured mesh, 217 million CSR values
        _brick("neohookean_hex8_step", "step", "hex8", "neohookean", 96, 96, 96),
        # a load step of plasticity with its state, boundary driven
        _brick("j2_hex8_step", "step", "hex8", "j2", 64, 64, 64, bc="all"),
        # the largest unstructured problem: quadratic tetrahedra, 663,552 elements, 232 million CSR values
        _brick("neohookean_tet10_step", "step", "tet10", "neohookean", 48, 48, 48),
        # a part made of two materials on rollers (single components fixed), with odd sizes: the general hex8 path and
        # the dof-level CSR
        _brick("two_material_hex8_step", "step", "hex8", "neohookean", 43, 37, 51, bc="roller", blocks=2),
        # a residual evaluation on tetrahedra, as a line search makes
        _brick("neohookean_tet10_residual", "residual", "tet10", "neohookean", 33, 39, 35),
        # one Krylov product without a matrix on an odd-sized mesh
        _brick("neohookean_hex8_mf_action", "mf_action", "hex8", "neohookean", 83, 67, 71),
        # one whole linear step of a clamped elastic block, solved tightly
        _brick("elastic_hex8_solve", "solve", "hex8", "elastic", 40, 32, 36, bc="face"),
        # the mass matrix of a dynamics run
        _brick("elastic_hex8_mass", "mass", "hex8", "elastic", 64, 64, 64),
        # a learned material evaluated at the quadrature points of the 64^3 plasticity problem
        _points("j2_network_update", "update", "j2", 2097152),
        # one minibatch of the training of the larger network: forward and backward
        _points("neohookean_network_gradient", "gradient", "neohookean", 16384),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _box(rng, lo, hi, cells):
    """Three edge lengths in [lo, hi], cubes and slabs alike, of at most `cells` cells."""
    while True:
        n = _log_int(rng, lo, hi)
        d = [max(2, min(hi, int(round(n * rng.uniform(0.6, 1.5))))) for _ in range(3)]
        if d[0] * d[1] * d[2] <= cells:
            return d


def draw(rng):
    kind = rng.choice(["quad4", "poisson", "solid", "solid", "tet10", "tet10", "vector", "vector", "solve", "mass", "network"])
    bc = lambda: rng.choice(["none", "all", "face", "roller"])  # noqa: E731
    if kind == "quad4":
        physics = rng.choice(["poisson", "plane_strain"])
        fixed = rng.choice(["all", "face"])
        return _brick(None, "step", "quad4", physics, _log_int(rng, 16, 512), _log_int(rng, 16, 512), bc=fixed)
    if kind == "poisson":
        return _brick(None, "step", "hex8", "poisson", *_box(rng, 8, 128, 128 ** 3), bc=rng.choice(["none", "all", "face"]))
    if kind == "solid":
        physics = rng.choice(["neohookean", "elastic", "j2"])
        blocks = 2 if physics == "neohookean" and rng.random() < 0.4 else 1
        return _brick(None, "step", "hex8", physics, *_box(rng, 6, 96, 64 ** 3), bc=bc(), blocks=blocks)
    if kind == "tet10":
        physics = rng.choice(["neohookean", "elastic", "poisson"])
        return _brick(None, "step", "tet10", physics, *_box(rng, 4, 48, 32 ** 3), bc=rng.choice(["none", "all", "face"]))
    if kind == "vector":
        call = rng.choice(["residual", "mf_action", "asm_action"])
        elem = rng.choice(["hex8", "hex8", "tet10"])
        physics = rng.choice(["poisson", "neohookean", "elastic"] + (["j2"] if elem == "hex8" else []))
        return _brick(None, call, elem, physics, *_box(rng, 6, 96, 72 ** 3 if elem == "hex8" else 40 ** 3),
                      bc=rng.choice(["none", "all", "face"]))
    if kind == "solve":
        physics = rng.choice(["elastic", "poisson"])
        return _brick(None, "solve", "hex8", physics, *_box(rng, 8, 44, 36 ** 3), bc="face")
    if kind == "mass":
        elem = rng.choice(["hex8", "tet10"])
        return _brick(None, "mass", elem, rng.choice(["elastic", "poisson"]),
                      *_box(rng, 6, 72, 56 ** 3 if elem == "hex8" else 28 ** 3), bc=rng.choice(["none", "face"]))
    if rng.random() < 0.5:
        return _points(None, "update", rng.choice(["j2", "neohookean"]), _log_int(rng, 4096, 2097152))
    return _points(None, "gradient", rng.choice(["j2", "neohookean"]), _log_int(rng, 1024, 131072))


# ------------------------------------------------------------------ meshes, fields, Dirichlet sets
_HEX = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
_TET_EDGES = [(0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3)]


def _grid(*n):
    """Coordinates of an integer grid, first index slowest."""
    return [a.ravel() for a in np.meshgrid(*(np.arange(m) for m in n), indexing="ij")]


def _mesh(case, seed):
    """(node coordinates NN x nd, connectivity NE x nnpe 0-based, block label per element)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["elem"] == "quad4":
        j, i = _grid(ny + 1, nx + 1)
        coords = np.stack([i / nx, j / ny], axis=1)
        ex, ey = _grid(nx, ny)
        node = lambda a, b: a + (nx + 1) * b  # noqa: E731
        conn = np.stack([node(ex, ey), node(ex + 1, ey), node(ex + 1, ey + 1), node(ex, ey + 1)], axis=1)
        return coords, conn, np.zeros(len(conn), np.int64)
    ex, ey, ez = _grid(nx, ny, nz)
    if case["elem"] == "hex8":
        k, j, i = _grid(nz + 1, ny + 1, nx + 1)
        n = np.array([nx, ny, nz])
        at = np.stack([i, j, k], axis=1)
        coords = at / n
        if case["call"] == "mass" or case["blocks"] == 2:  # a mesh as a generator delivers it: interior nodes off the lattice
            inside = ((at > 0) & (at < n)).all(axis=1)
            coords += inside[:, None] * np.random.default_rng(seed).uniform(-0.2, 0.2, at.shape) / n
        conn = np.stack([(ex + a) + (nx + 1) * ((ey + b) + (ny + 1) * (ez + c)) for a, b, c in _HEX], axis=1)
        return coords, conn, (2 * ex >= nx).astype(np.int64) if case["blocks"] == 2 else np.zeros(len(conn), np.int64)
    # 6 tetrahedra per cell around the diagonal (0,0,0)-(1,1,1); edge midpoints are points of the twice finer grid
    n = np.array([nx, ny, nz])
    kk, jj, ii = _grid(*(2 * n[::-1] + 1))
    fine = np.stack([ii, jj, kk], axis=1)
    k, j, i = _grid(*(n[::-1] + 1))
    vert = np.stack([i, j, k], axis=1)
    inside = ((vert > 0) & (vert < n)).all(axis=1)
    shift = np.random.default_rng(seed).uniform(-0.2, 0.2, vert.shape)
    x = (vert + inside[:, None] * shift) / n
    vid = lambda p: p[:, 0] + (nx + 1) * (p[:, 1] + (ny + 1) * p[:, 2])  # noqa: E731
    odd = fine % 2
    coords = 0.5 * (x[vid((fine - odd) // 2)] + x[vid((fine + odd) // 2)])
    base = 2 * np.stack([ex, ey, ez], axis=1)
    conn = np.zeros((len(ex), 6, 10), np.int64)
    for t, p in enumerate([(0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)]):
        a = np.zeros(3, np.int64)
        a[p[0]] = 2
        b = a.copy()
        b[p[1]] = 2
        if t in (1, 2, 5):
            a, b = b, a
        corners = [np.zeros(3, np.int64), a, b, np.array([2, 2, 2])]
        for c, q in enumerate(corners + [(corners[u] + corners[v]) // 2 for u, v in _TET_EDGES]):
            w = base + q
            conn[:, t, c] = w[:, 0] + (2 * nx + 1) * (w[:, 1] + (2 * ny + 1) * w[:, 2])
    conn = conn.reshape(-1, 10)
    return coords, conn, np.zeros(len(conn), np.int64)


def _nf(case):
    return 1 if case["physics"] == "poisson" else (2 if case["elem"] == "quad4" else 3)


def _field(X, nf, seed, amp):
    """Smooth field on the unit brick: sines and cosines up to four half waves, gradient entries below `amp` / 2."""
    r = np.random.default_rng(seed)
    u = np.zeros((len(X), nf))
    for k in range(1, 5):
        a = r.standard_normal((2, nf))
        a *= amp / (16 * np.pi * k) / np.maximum(1.0, np.abs(a))
        u += np.prod(np.sin(k * np.pi * X), axis=1)[:, None] * a[0] + np.prod(np.cos(k * np.pi * X), axis=1)[:, None] * a[1]
    return u


# amplitude of the displacement (or temperature) by physics: finite strain; small strain past yield; small strain
_AMP = {"poisson": 8.0, "neohookean": 0.6, "j2": 0.05, "elastic": 0.02, "plane_strain": 0.02}


def _fixed(case, X):
    """Fixed (node, component) pairs as {component: nodes}: the whole boundary, one face, or rollers on three faces."""
    nf, nd = _nf(case), X.shape[1]
    if case["bc"] == "all":
        on = ((X < 1e-12) | (X > 1 - 1e-12)).any(axis=1)
        return {d: np.flatnonzero(on) for d in range(nf)}
    if case["bc"] == "face":
        return {d: np.flatnonzero(X[:, 0] < 1e-12) for d in range(nf)}
    if case["bc"] == "roller":
        return {d: np.flatnonzero(X[:, d % nd] < 1e-12) for d in range(nf)}
    return {}


_PROPS = {"elastic": (1e3, 10.0, 1.0), "plane_strain": (1e3, 10.0, 1.0), "neohookean": (1.0, 0.5), "j2": (200.0, 0.3, 0.25, 2.0)}


def _inputs(case, seed):
    """Everything of a mesh case on the host: mesh, full field U, direction V, free-dof mask, old J2 state."""
    X, conn, label = _mesh(case, seed)
    nf = _nf(case)
    U = _field(X, nf, seed + 1, _AMP[case["physics"]])
    V = _field(X, nf, seed + 2, 1.0)
    free = np.ones((len(X), nf), bool)
    for d, nodes in _fixed(case, X).items():
        free[nodes, d] = False
    if case["call"] == "solve":
        U[~free] += _field(X, nf, seed + 3, _AMP[case["physics"]])[~free]
    V[~free] = 0.0
    state = None
    if case["physics"] == "j2":  # plastic strain of earlier load steps: symmetric, deviatoric, with its hardening variable
        r = np.random.default_rng(seed + 4)
        e = 5e-4 * r.standard_normal((len(conn), 8, 6), dtype=np.float32)
        m = (e[..., 0] + e[..., 3] + e[..., 5]) / 3
        for c in (0, 3, 5):
            e[..., c] -= m
        eq = np.sqrt(2.0 / 3.0 * (e[..., [0, 3, 5]] ** 2).sum(-1) + 4.0 / 3.0 * (e[..., [1, 2, 4]] ** 2).sum(-1))
        state = np.ascontiguousarray(np.concatenate([e, eq[..., None].astype(np.float32)], axis=-1))
    return X, conn, label, U, V, free, state


# ------------------------------------------------------------------ what a user's program holds, and one pass
def prepare(case, seed):
    if case["call"] in ("update", "gradient"):
        return _prepare_network(case, seed)
    fec = _fec()
    X, conn, label, U, V, free, state = _inputs(case, seed)
    nf = _nf(case)
    kind = case["elem"].upper()
    sets = {"fixed_%d" % d: nodes + 1 for d, nodes in _fixed(case, X).items()}
    if case["blocks"] == 2:
        mesh = fec.split_into_blocks(fec.BlockMesh(X, [("all", conn + 1)], kind, sets), label, ["left", "right"])
        mesh.nodeset_nodes = sets
    else:
        mesh = fec.BlockMesh(X, [("block_1", conn + 1)], kind, sets)
    space = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    var = fec.ScalarFunction(space, "u") if nf == 1 else fec.VectorFunction(space, "displ")
    asm = fec.SparseMatrixAssembler(var, sparse_matrix_type="csr")
    kinds = {"poisson": lambda: fec.Poisson("constant", 1.0), "neohookean": fec.NeoHookean, "j2": fec.J2Plasticity,
             "elastic": lambda: fec.Mechanics(fec.ThreeDimensional(), *_PROPS["elastic"]),
             "plane_strain": lambda: fec.Mechanics(fec.PlaneStrain(), *_PROPS["plane_strain"])}
    physics = kinds[case["physics"]]()
    if case["blocks"] == 2:
        physics = {"left": physics, "right": kinds["elastic"]()}

    def value(d):
        nodes = sets["fixed_%d" % d] - 1
        at = {tuple(x): U[n, d] for x, n in zip(X[nodes].tolist(), nodes)}
        return lambda P, t: np.array([at[tuple(p)] for p in P.tolist()])

    names = var.names
    bcs = [fec.DirichletBC(names[d], value(d), nset_name="fixed_%d" % d) for d in range(nf) if "fixed_%d" % d in sets]
    p = fec.create_parameters(mesh, asm, physics, dirichlet_bcs=bcs)
    if state is not None:
        asm.ctx.call("fecx_set_state_old", state.ctypes.data_as(ctypes.c_void_p))
    dofs = asm.dof.unknown_dofs - 1
    s = {"call": case["call"], "fec": fec, "asm": asm, "p": p,
         "Uu": torch.from_numpy(U.reshape(-1)[dofs]).to(DEV), "Vu": torch.from_numpy(V.reshape(-1)[dofs]).to(DEV)}
    if case["call"] == "solve":
        s["solver"] = fec.IterativeLinearSolver(asm, "cg", fec.IterativeLinearSolverSettings(rtol=1e-10, atol=0.0))
        s["x"] = torch.empty_like(s["Uu"])
    return s


def run(state):
    fec, call = state["fec"], state["call"]
    if call == "update":
        return fec.surrogate.material_update(state["asm"], state["kind"], state["X"])
    if call == "gradient":
        return state["net"].gradient(state["X"], state["T"])
    asm, p, Uu, Vu = state["asm"], state["p"], state["Uu"], state["Vu"]
    if call == "step":
        fec.assemble_vector_and_stiffness_(asm, Uu, p)
        return fec.residual(asm), fec.stiffness(asm).values
    if call == "residual":
        fec.assemble_vector_(asm, fec.residual, Uu, p)
        return fec.residual(asm)
    if call == "mf_action":
        fec.assemble_matrix_free_action_(asm, fec.stiffness_action, Uu, Vu, p)
        return fec.hvp(asm, Vu)
    if call == "asm_action":
        fec.assemble_matrix_action_(asm, fec.stiffness, Uu, Vu, p)
        return fec.hvp(asm, Vu)
    if call == "mass":
        fec.assemble_mass_(asm, fec.mass, Uu, p)
        return fec.mass(asm).values
    state["x"].copy_(Uu)  # the iterate starts from the last accepted one
    state["solver"].solve(state["x"], p)
    return state["x"]


# ------------------------------------------------------------------ the learned material's network
_NET = {"j2": [13, 128, 128, 128, 13], "neohookean": [9, 256, 256, 15]}


def _network(net, features, targets, seed, steps):
    """Weights (out x in and bias per layer) and standardisation of a network, fitted by `steps` Adam steps."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    d = _NET[net]
    scale = [features.mean(0), features.std(0).clamp_min(1e-12), targets.mean(0), targets.std(0).clamp_min(1e-12)]
    x, y = (features - scale[0]) / scale[1], (targets - scale[2]) / scale[3]
    w = []
    for a, b in zip(d, d[1:]):
        w += [torch.randn(b, a, device=DEV, generator=g) * (2.0 / a) ** 0.5, torch.zeros(b, device=DEV)]
    m, v = [torch.zeros_like(t) for t in w], [torch.zeros_like(t) for t in w]
    for k in range(1, steps + 1):
        at = torch.randint(0, len(x), (8192,), device=DEV, generator=g)
        _, grad = _loss_gradient(w, x[at], y[at])
        for i, t in enumerate(grad):
            m[i] = 0.9 * m[i] + 0.1 * t
            v[i] = 0.999 * v[i] + 0.001 * t * t
            w[i] = w[i] - 3e-3 * (1 - 0.9 * k / steps) * (m[i] / (1 - 0.9 ** k)) / ((v[i] / (1 - 0.999 ** k)).sqrt() + 1e-8)
    return w, scale


def _loss_gradient(w, x, y):
    """Mean squared error over samples and outputs, and its gradient, of the tanh-form GELU network."""
    leaf = [t.detach().requires_grad_(True) for t in w]
    h = x
    for i in range(0, len(leaf), 2):
        h = h @ leaf[i].T + leaf[i + 1]
        if i + 2 < len(leaf):
            h = torch.nn.functional.gelu(h, approximate="tanh")
    loss = ((h - y) ** 2).mean()
    return loss.detach(), torch.autograd.grad(loss, leaf)


def _features(net, X):
    if net == "neohookean":
        return X
    H = X[:, :9].reshape(-1, 3, 3)
    S = 0.5 * (H + H.transpose(1, 2))
    return torch.cat([S[:, [0, 1, 2, 1, 2, 2], [0, 0, 0, 1, 1, 2]], X[:, 9:]], dim=1)


def _samples(case, seed):
    """Raw network inputs and their plain-model outputs, in 64 bits."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    n = case["n"]
    if case["net"] == "neohookean":
        X = (0.1 * torch.randn(n, 9, device=DEV, generator=g).clamp(-3, 3)).float()
        P, _ = _neohookean(X.double().reshape(n, 3, 3), False)
        F = torch.eye(3, dtype=F64, device=DEV) + X.double().reshape(n, 3, 3)
        Ci = torch.linalg.inv(F.transpose(1, 2) @ F) - torch.eye(3, dtype=F64, device=DEV)
        return X, torch.cat([P.reshape(n, 9), Ci[:, [0, 1, 2, 1, 2, 2], [0, 0, 0, 1, 1, 2]]], dim=1)
    E = 3e-3 * torch.randn(n, 3, 3, device=DEV, generator=g)
    E = 0.5 * (E + E.transpose(1, 2))
    e = 1e-3 * torch.randn(n, 6, device=DEV, generator=g)
    e[:, [0, 3, 5]] -= e[:, [0, 3, 5]].mean(1, keepdim=True)
    eq = (2 / 3 * (e[:, [0, 3, 5]] ** 2).sum(1) + 4 / 3 * (e[:, [1, 2, 4]] ** 2).sum(1)).sqrt()
    X = torch.cat([E.reshape(n, 9), e, eq[:, None]], dim=1).contiguous()
    P, _, new = _j2(X[:, :9].double().reshape(n, 3, 3), X[:, 9:].double(), False)
    return X, torch.cat([P[:, [0, 1, 2, 1, 2, 2], [0, 0, 0, 1, 1, 2]], new - X[:, 9:].double()], dim=1)


def _prepare_network(case, seed):
    fec = _fec()
    X, T = _samples(case, seed)
    w, scale = _network(case["net"], _features(case["net"], X), T.float(), seed, 300 if case["call"] == "update" else 20)
    mesh = fec.StructuredMesh("hex", (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), (3, 3, 3))
    var = fec.VectorFunction(fec.FunctionSpace(mesh, "H1Field", "Lagrange"), "displ")
    asm = fec.SparseMatrixAssembler(var, sparse_matrix_type="csr")
    j2 = case["net"] == "j2"
    fec.create_parameters(mesh, asm, fec.J2Surrogate() if j2 else fec.NeoHookeanSurrogate())
    net = fec.Surrogate(asm, fec.surrogate.MLP_J2 if j2 else fec.surrogate.MLP_NH, seed=0)
    net.set_params(torch.cat([t.reshape(-1) for t in w]).cpu().numpy())
    net.set_scaling(*[t.cpu().numpy() for t in scale])
    net.set_tolerance(0.05)
    return {"call": case["call"], "fec": fec, "asm": asm, "net": net, "X": X.contiguous(), "T": T.float().contiguous(),
            "kind": fec._lib.J2_SURROGATE if j2 else fec._lib.NH_SURROGATE, "w": w, "scale": scale}


# ------------------------------------------------------------------ what a pass cannot do without
_ELEM = {"quad4": (4, 2, 4), "hex8": (8, 3, 8), "tet10": (10, 3, 4)}  # nodes, dimensions, quadrature points


@functools.lru_cache(maxsize=64)
def _sizes(elem, nx, ny, nz):
    """(nodes, elements, node pairs that share an element, each with itself) of a brick."""
    if elem == "quad4":
        return (nx + 1) * (ny + 1), nx * ny, (3 * nx + 1) * (3 * ny + 1)
    if elem == "hex8":
        return (nx + 1) * (ny + 1) * (nz + 1), nx * ny * nz, (3 * nx + 1) * (3 * ny + 1) * (3 * nz + 1)
    cells = nx * ny * nz
    return (2 * nx + 1) * (2 * ny + 1) * (2 * nz + 1), 6 * cells, int(230 * cells * (1 + 0.2 / nx + 0.2 / ny + 0.2 / nz))


def work(case):
    """Inputs read once and outputs written once; operations of the closed-form element algebra (per quadrature point and
    node: map, gradients, stress and force; per unordered node pair: the block)."""
    if case["call"] in ("update", "gradient"):
        d = _NET[case["net"]]
        raw, out = (16, 13) if case["net"] == "j2" else (9, 15)
        flops = 2.0 * sum(a * b for a, b in zip(d, d[1:])) * case["n"]
        if case["call"] == "update":
            return {"bytes": 4.0 * case["n"] * (raw + out), "flops": flops}
        return {"bytes": 4.0 * case["n"] * (raw + out) + 8.0 * sum(a * b + b for a, b in zip(d, d[1:])), "flops": 3 * flops}
    nnpe, nd, nq = _ELEM[case["elem"]]
    nn, ne, pairs = _sizes(case["elem"], case["nx"], case["ny"], case["nz"])
    nf = _nf(case)
    byte = 4.0 * ne * nnpe + 8.0 * nn * nd + 8.0 * nn * nf
    state = 4.0 * 7 * nq * ne if case["physics"] == "j2" else 0.0
    point = nnpe * (2 * nd * nd + 2 * nd * nd + 2 * nf * nd) + 40 + 2 * nf * nf * nd * nd
    vector = ne * nq * (point + 2.0 * nnpe * nf * nd)
    block = 6.0 if nf == 1 else 6.0 * nf * nf
    matrix = ne * nq * (nnpe * (nnpe + 1) / 2) * block
    csr = 8.0 * pairs * nf * nf
    if case["call"] == "residual":
        return {"bytes": byte + 2 * state + 8.0 * nn * nf, "flops": vector}
    if case["call"] in ("mf_action", "asm_action"):
        return {"bytes": byte + state + 16.0 * nn * nf, "flops": 2 * vector}
    if case["call"] == "mass":
        return {"bytes": 4.0 * ne * nnpe + 8.0 * nn * nd + csr, "flops": ne * nq * (nnpe * (nnpe + 1) / 2) * 2.0}
    step = {"bytes": byte + 2 * state + 8.0 * nn * nf + csr, "flops": vector + matrix}
    if case["call"] == "step":
        return step
    # CG to 1e-10: about 20 iterations per cell along the longest edge, each reading the matrix once
    its = 20.0 * max(case["nx"], case["ny"], case["nz"])
    return {"bytes": step["bytes"] + its * (csr + 4.0 * pairs + 80.0 * nn * nf),
            "flops": step["flops"] + its * (2.0 * pairs * nf * nf + 12.0 * nn * nf)}


# ------------------------------------------------------------------ the same in 64 bits, with torch alone
def _rule(elem):
    """Shape values (nq x nnpe), their reference gradients (nq x nnpe x nd) and the weights of an element kind."""
    if elem == "tet10":
        a, b = (5 - 5 ** 0.5) / 20, (5 + 3 * 5 ** 0.5) / 20
        pts = np.array([[a, a, a], [b, a, a], [a, b, a], [a, a, b]])
        L = np.concatenate([1 - pts.sum(1, keepdims=True), pts], axis=1)
        dL = np.concatenate([-np.ones((1, 3)), np.eye(3)])
        N = [L[:, v] * (2 * L[:, v] - 1) for v in range(4)] + [4 * L[:, p] * L[:, r] for p, r in _TET_EDGES]
        dN = [(4 * L[:, v, None] - 1) * dL[v] for v in range(4)]
        dN += [4 * (L[:, r, None] * dL[p] + L[:, p, None] * dL[r]) for p, r in _TET_EDGES]
        w = np.full(4, 1 / 24)
        return [torch.from_numpy(np.ascontiguousarray(t)).to(DEV) for t in (np.stack(N, 1), np.stack(dN, 1), w)]
    nd = 2 if elem == "quad4" else 3
    corner = 2.0 * np.array([c[:nd] for c in _HEX[: 2 ** nd]]) - 1
    pts = np.stack(_grid(*[2] * nd)[::-1], axis=1) * 2.0 - 1
    pts /= 3 ** 0.5
    f = 1 + pts[:, None, :] * corner[None]
    N = f.prod(-1) / 2 ** nd
    dN = np.stack([corner[None, :, j] * np.delete(f, j, axis=-1).prod(-1) for j in range(nd)], axis=-1) / 2 ** nd
    return [torch.from_numpy(np.ascontiguousarray(t)).to(DEV) for t in (N, dN, np.ones(len(pts)))]


def _eye(n):
    return torch.eye(n, dtype=F64, device=DEV)


def _elastic(H, tangent):
    _, K, G = _PROPS["elastic"]
    n = H.shape[-1]
    I = _eye(n)
    lam = K - 2 * G / 3
    P = G * (H + H.transpose(-1, -2)) + lam * H.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None] * I
    if not tangent:
        return P, None
    A = lam * torch.einsum("ij,kl->ijkl", I, I) + G * (torch.einsum("ik,jl->ijkl", I, I) + torch.einsum("il,jk->ijkl", I, I))
    return P, A.expand(*H.shape[:-2], n, n, n, n)


def _neohookean(H, tangent):
    lam, mu = _PROPS["neohookean"]
    F = _eye(3) + H
    Fi = torch.linalg.inv(F)
    FiT = Fi.transpose(-1, -2)
    lnJ = torch.log(torch.linalg.det(F))[..., None, None]
    P = mu * (F - FiT) + lam * lnJ * FiT
    if not tangent:
        return P, None
    c = (mu - lam * lnJ)[..., None, None]
    A = mu * torch.einsum("ik,jl->ijkl", _eye(3), _eye(3))
    return P, A + c * torch.einsum("...li,...jk->...ijkl", Fi, Fi) + lam * torch.einsum("...ji,...lk->...ijkl", Fi, Fi)


def _j2(H, old, tangent):
    E, nu, sy, hard = _PROPS["j2"]
    mu, kap = E / (2 * (1 + nu)), E / (3 * (1 - 2 * nu))
    I = _eye(3)
    ep = old[..., [0, 1, 2, 1, 3, 4, 2, 4, 5]].reshape(H.shape)
    ee = 0.5 * (H + H.transpose(-1, -2)) - ep
    tr = ee.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None]
    s = 2 * mu * (ee - tr / 3 * I)
    norm = s.square().sum((-1, -2)).sqrt()[..., None, None]
    f = norm - (2 / 3) ** 0.5 * (sy + hard * old[..., 6, None, None])
    plastic = f > 0
    n = torch.where(plastic, s / norm.clamp_min(1e-300), torch.zeros_like(s))
    dg = torch.where(plastic, f / (2 * mu + 2 * hard / 3), torch.zeros_like(f))
    P = s - 2 * mu * dg * n + kap * tr * I
    new = (ep + dg * n).flatten(-2)[..., [0, 3, 6, 4, 7, 8]]
    new = torch.cat([new, old[..., 6:] + (2 / 3) ** 0.5 * dg[..., 0]], dim=-1)
    if not tangent:
        return P, None, new
    th = torch.where(plastic, 1 - 2 * mu * dg / norm.clamp_min(1e-300), torch.ones_like(dg))
    tb = torch.where(plastic, 1 / (1 + hard / (3 * mu)) - (1 - th), torch.zeros_like(dg))
    II = torch.einsum("ij,kl->ijkl", I, I)
    sym = 0.5 * (torch.einsum("ik,jl->ijkl", I, I) + torch.einsum("il,jk->ijkl", I, I))
    A = kap * II + 2 * mu * th[..., None, None] * (sym - II / 3)
    return P, A - 2 * mu * tb[..., None, None] * torch.einsum("...ij,...kl->...ijkl", n, n), new


def _material(physics, H, old, tangent):
    """Flux (... x nf x nd) and, where asked for, its derivative (... x nf x nd x nf x nd)."""
    if physics == "poisson":
        return H, _eye(H.shape[-1])[None, :, None, :].expand(*H.shape[:-2], 1, H.shape[-1], 1, H.shape[-1]) if tangent else None
    if physics == "neohookean":
        return _neohookean(H, tangent)
    if physics == "j2":
        return _j2(H, old, tangent)[:2]
    return _elastic(H, tangent)


def _pattern(conn, nn):
    """Node-block CSR of a mesh: row pointers, and for every element its pairs' positions among the blocks."""
    key = (conn[:, :, None] * nn + conn[:, None, :]).reshape(-1)
    blocks, at = torch.unique(key, return_inverse=True)
    ptr = torch.searchsorted(blocks, torch.arange(nn + 1, device=DEV) * nn)
    return ptr, blocks % nn, at.reshape(conn.shape[0], conn.shape[1], conn.shape[1])


def _exact_mesh(case, seed, vector, matrix, V=None):
    """(vector over all dofs, block matrix and its pattern) of a mesh case."""
    X, conn, label, U, Vh, free, state = _inputs(case, seed)
    nf = _nf(case)
    N, dN, w0 = _rule(case["elem"])
    X, U, Vh = (torch.from_numpy(np.ascontiguousarray(t)).to(DEV) for t in (X, U, Vh))
    conn = torch.from_numpy(conn).to(DEV)
    nn = len(X)
    out = torch.zeros(nn, nf, dtype=F64, device=DEV) if vector else None
    vals = pat = None
    if matrix:
        pat = _pattern(conn, nn)
        vals = torch.zeros(len(pat[1]), nf, nf, dtype=F64, device=DEV)
    chunk = 16384 if matrix or case["call"] == "asm_action" else 65536
    for mat in range(case["blocks"]):
        physics = "elastic" if mat else case["physics"]
        ids = torch.from_numpy(np.flatnonzero(label == mat)).to(DEV)
        for e in ids.split(chunk):
            c = conn[e]
            J = torch.einsum("eai,qaj->eqij", X[c], dN)
            g = torch.einsum("qaj,eqji->eqai", dN, torch.linalg.inv(J))
            w = torch.linalg.det(J) * w0
            if case["call"] == "mass":
                rho = _PROPS["elastic"][0] if physics != "poisson" else 1.0
                m = torch.einsum("eq,qa,qb->eab", rho * w, N, N)
                vals.view(-1, nf * nf).index_add_(0, pat[2][e].reshape(-1), m.reshape(-1, 1) * _eye(nf).reshape(1, -1))
                continue
            H = torch.einsum("eai,eqaj->eqij", U[c], g)
            old = torch.from_numpy(state[e.cpu().numpy()]).to(DEV).double() if state is not None else None
            P, A = _material(physics, H, old, matrix or V)
            if V:
                P = torch.einsum("eqijkl,eqkl->eqij", A, torch.einsum("eai,eqaj->eqij", Vh[c], g))
            if vector:
                r = torch.einsum("eq,eqij,eqaj->eai", w, P, g)
                if physics == "poisson" and not V:
                    r -= torch.einsum("eq,qa->ea", w, N)[..., None]
                out.index_add_(0, c.reshape(-1), r.reshape(-1, nf))
            if matrix:
                K = torch.empty(len(e), c.shape[1], c.shape[1], nf, nf, dtype=F64, device=DEV)
                for i in range(nf):
                    for k in range(nf):
                        t = w[..., None, None] * (g @ A[:, :, i, :, k, :])
                        K[..., i, k] = (t @ g.transpose(-1, -2)).sum(1)
                vals.index_add_(0, pat[2][e].reshape(-1), K.reshape(-1, nf, nf))
    return out, vals, pat, torch.from_numpy(free).to(DEV), U


def _csr(vals, pat, free):
    """The block matrix's values over free rows and columns in row order, with the row and column of each."""
    ptr, col, _ = pat
    nn, nf = free.shape
    deg = ptr[1:] - ptr[:-1]
    row = torch.repeat_interleave(torch.arange(nn, device=DEV), deg)
    slot = torch.arange(len(col), device=DEV) - ptr[row]
    flat = torch.empty(vals.numel(), dtype=F64, device=DEV)
    keep = torch.empty(vals.numel(), dtype=torch.bool, device=DEV)
    at = nf * nf * ptr[row] + nf * slot
    for i in range(nf):
        for k in range(nf):
            flat[at + i * nf * deg[row] + k] = vals[:, i, k]
            keep[at + i * nf * deg[row] + k] = free[row, i] & free[col, k]
    return flat[keep], keep


def _solve(case, seed):
    """U - K^-1 R over the free dofs, by conjugate gradients in 64 bits to 1e-13."""
    R, vals, pat, free, U = _exact_mesh(case, seed, True, True)
    ptr, col, _ = pat
    nn, nf = free.shape
    row = torch.repeat_interleave(torch.arange(nn, device=DEV), ptr[1:] - ptr[:-1])
    c = torch.arange(nf, device=DEV)
    i = (row[:, None, None] * nf + c[None, :, None]).expand(-1, nf, nf).reshape(-1)
    j = (col[:, None, None] * nf + c[None, None, :]).expand(-1, nf, nf).reshape(-1)
    A = torch.sparse_coo_tensor(torch.stack([i, j]), vals.reshape(-1), (nn * nf, nn * nf)).coalesce().to_sparse_csr()
    m = free.reshape(-1).double()
    diag = vals[row == col]
    d = torch.diagonal(diag, dim1=-2, dim2=-1).reshape(-1)
    b = R.reshape(-1) * m
    x = torch.zeros_like(b)
    r = b.clone()
    z = r / d
    p = z.clone()
    rz = r @ z
    stop = 1e-13 * b.norm()
    for k in range(4000):
        q = (A @ (p * m)[:, None])[:, 0] * m
        a = rz / (p @ q)
        x += a * p
        r -= a * q
        if k % 25 == 0 and r.norm() <= stop:
            break
        z = r / d
        new = r @ z
        p = z + new / rz * p
        rz = new
    return (U.reshape(-1) - x)[free.reshape(-1)]


def exact(case, seed):
    call = case["call"]
    if call == "update":
        return None  # a 16-bit network decides point by point whether its own output is taken
    if call == "gradient":
        X, T = _samples(case, seed)
        w, scale = _network(case["net"], _features(case["net"], X), T.float(), seed, 20)
        f = (_features(case["net"], X).double() - scale[0].double()) / scale[1].double()
        y = (T.float().double() - scale[2].double()) / scale[3].double()
        loss, grad = _loss_gradient([t.double() for t in w], f, y)
        return float(loss), torch.cat([t.reshape(-1) for t in grad])
    if call == "solve":
        return _solve(case, seed)
    R, vals, pat, free, _ = _exact_mesh(case, seed, call != "mass", call in ("step", "mass"), V=call in ("mf_action", "asm_action"))
    if call == "mass":
        return _csr(vals, pat, free)[0]
    R = R.reshape(-1)[free.reshape(-1)]
    return R if call != "step" else (R, _csr(vals, pat, free)[0])
