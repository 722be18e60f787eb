"""The SpMV and the two-kernel CG iteration over every row form they dispatch on (1, 2 or 3 fields per node, the dof-level CSR
of a Dirichlet set that splits nodes), at the sizes where lane groups and work-group ranges end: a single unknown node, rows
narrower and far wider than a lane group's pass, unknown counts around the work-group sizes.

Tolerances, derived beforehand: SpMV sums at most ~500 products, |error| <= 500 eps (|A| |x|) row by row with
eps = 2^-53; a CG of 8 iterations on a mass matrix (condition number below ~1e2 after Jacobi scaling) amplifies the
FP64 rounding of its dot products by at most its condition number per iteration, well under 1e-9 of the iterate."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _mesh(fec, name):
    """(mesh, nf, fixed nodes per component)"""
    if name.startswith("quad4"):
        n = int(name.split()[1])
        m = fec.StructuredMesh("quad", (0.0, 0.0), (1.0, 1.0), (n + 1, n + 1))
        return m, 2 if "nf2" in name else 1, {}
    if name == "hex8 one node":  # 2^3 elements, every node fixed but the centre
        m = fec.StructuredMesh("hex", (0.0,) * 3, (1.0,) * 3, (3, 3, 3))
        edge = fec.boundary_nodes(m)
        return m, 3, {0: edge, 1: edge, 2: edge}
    if name.startswith("hex8"):
        n = int(name.split()[1])
        m = fec.StructuredMesh("hex", (0.0,) * 3, (1.0,) * 3, (n + 1,) * 3)
        fixed = {d: np.flatnonzero(m.coords[:, d] < 1e-12) + 1 for d in range(3)} if "roller" in name else {}
        return m, 1 if "nf1" in name else 3, fixed
    return fec.fan_tet10_mesh(int(name.split()[1])), 1 if "nf1" in name else 3, {}


CASES = ["quad4 1", "quad4 7", "quad4 31 nf2", "hex8 one node", "hex8 1", "hex8 6", "hex8 9 nf1", "hex8 14", "hex8 5 roller",
         "fan 5", "fan 32", "fan 32 nf1"]


@pytest.mark.parametrize("name", CASES)
def test_spmv_and_cg_iterations(fec, gpu, name):
    print(f"[krylov] {name}", flush=True)
    mesh, nf, fixed = _mesh(fec, name)
    space = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    var = fec.ScalarFunction(space, "u") if nf == 1 else fec.VectorFunction(space, "displ")
    asm = fec.SparseMatrixAssembler(var, sparse_matrix_type="csr", device=0)
    for d, nodes in fixed.items():
        mesh.nodeset_nodes[f"_f{d}"] = nodes
    bcs = [fec.DirichletBC(var.names[d], lambda X, t: 0.0, nset_name=f"_f{d}") for d in fixed]
    physics = fec.Poisson() if nf == 1 else fec.Mechanics(fec.PlaneStrain() if nf == 2 else None)
    p = fec.create_parameters(mesh, asm, physics, dirichlet_bcs=bcs)
    Uu = fec.create_unknowns(asm)
    fec.assemble_mass_(asm, fec.mass, Uu, p)
    M = fec.mass(asm)
    A = M.to_scipy()
    n = A.shape[0]
    g = np.random.default_rng(1)
    # SpMV with arbitrary values on the pattern
    vals = torch.from_numpy(g.standard_normal(asm.nnz)).to(gpu)
    x = g.standard_normal(n)
    y = torch.full_like(Uu, np.nan)
    xd = torch.from_numpy(x).to(gpu)
    asm.ctx.call("fecx_csr_spmv", fec.assembler._ptr(vals), fec.assembler._ptr(xd), fec.assembler._ptr(y))
    B = A.copy()
    B.data = vals.cpu().numpy()
    bound = 500 * 2.0 ** -53 * (abs(B) @ np.abs(x)) + 1e-300
    assert np.all(np.abs(y.cpu().numpy() - B @ x) <= bound)
    # eight CG iterations on the mass matrix from a nonzero start, with and without the preconditioner
    b = g.standard_normal(n)
    bd = torch.from_numpy(b).to(gpu)
    for pre in (1, 0):
        xg = torch.from_numpy(x).to(gpu)
        it, res = ctypes.c_int(-1), ctypes.c_double(-1.0)
        asm.ctx.call("fecx_cg_solve", fec.assembler._ptr(M.values), fec.assembler._ptr(bd), fec.assembler._ptr(xg),
                     ctypes.c_double(1e-9), ctypes.c_double(0.0), ctypes.c_int(8), ctypes.c_int(pre), ctypes.byref(it),
                     ctypes.byref(res))
        d = 1.0 / A.diagonal() if pre else np.ones(n)
        xs, r = x.copy(), b - A @ x
        z = d * r
        q, rz, k = z.copy(), r @ z, 0
        while k < 8 and np.linalg.norm(r) > 1e-9 * np.linalg.norm(b):
            Aq = A @ q
            a = rz / (q @ Aq)
            xs, r = xs + a * q, r - a * Aq
            z = d * r
            new = r @ z
            q, rz, k = z + new / rz * q, new, k + 1
        assert it.value == k
        assert np.linalg.norm(xg.cpu().numpy() - xs) <= 1e-9 * np.linalg.norm(xs)
        assert abs(res.value - np.linalg.norm(r)) <= 1e-9 * np.linalg.norm(b)


def _quads(fec, name):
    """(mesh, 2, fixed) of a square or of quadrilaterals around a point (rows of up to 2 (2 m + 1) columns), on rollers"""
    m = int(name.split()[1])
    if name.startswith("quadfan"):
        t = np.pi * np.arange(2 * m) / m
        ring = np.stack([np.cos(t), np.sin(t)], axis=1) * np.where(np.arange(2 * m) % 2, 1.4, 1.0)[:, None]
        conn = np.array([[0, 1 + 2 * i, 2 + 2 * i, 1 + (2 * i + 2) % (2 * m)] for i in range(m)]) + 1
        mesh = fec.BlockMesh(np.concatenate([np.zeros((1, 2)), ring]), [("b", conn)], "QUAD4")
    else:
        mesh = fec.StructuredMesh("quad", (0.0, 0.0), (1.0, 1.0), (m + 1, m + 1))
    return mesh, 2, {d: np.flatnonzero(mesh.coords[:, d] < mesh.coords[:, d].min() + 1e-12) + 1 for d in range(2)}


def _loose(fec, name):
    """(mesh, nf, fixed): a brick or square with a loose node (of no element) before, between and after the others', the last
    rows of the matrix being empty; "alone": every node of an element is fixed, so that the matrix has no entry"""
    m, nf, fixed = _quads(fec, name) if name.startswith("quad") and "roller" in name else _mesh(fec, name.replace(" alone", ""))
    n = m.num_nodes
    at = np.concatenate([[-1], np.arange(n // 2), [-1], np.arange(n // 2, n), [-1, -1]])  # new node -> old node
    new = np.empty(n, np.int64)
    new[at[at >= 0]] = np.flatnonzero(at >= 0)
    coords = np.where(at[:, None] >= 0, m.coords[at], 1.7)
    mesh = fec.BlockMesh(coords, [("b", new[m.conn - 1] + 1)], m.element_type)
    fixed = {d: new[nodes - 1] + 1 for d, nodes in fixed.items()}
    if "alone" in name:
        fixed = {d: new + 1 for d in range(nf)}
    return mesh, nf, fixed, np.flatnonzero(at < 0)


@pytest.mark.parametrize("name", ["hex8 3 nf1", "hex8 3", "hex8 3 roller", "quad4 5 nf2", "quad4 2 nf2 roller", "quad4 7 nf2 roller",
                                  "quadfan 5 nf2 roller", "quadfan 6 nf2 roller", "quadfan 40 nf2 roller", "hex8 2 nf1 alone",
                                  "hex8 2 alone"])
def test_rows_of_loose_nodes(fec, gpu, name):
    """Nodes that no element touches have empty rows: a product of zero, a unit preconditioner, and an unknown that CG leaves at its
    start (b is zero there, or the matrix has no entry). Tolerances as above."""
    print(f"[krylov] loose nodes {name}", flush=True)
    mesh, nf, fixed, loose = _loose(fec, name)
    space = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    var = fec.ScalarFunction(space, "u") if nf == 1 else fec.VectorFunction(space, "displ")
    asm = fec.SparseMatrixAssembler(var, sparse_matrix_type="csr", device=0)
    for d, nodes in fixed.items():
        mesh.nodeset_nodes[f"_f{d}"] = nodes
    bcs = [fec.DirichletBC(var.names[d], lambda X, t: 0.0, nset_name=f"_f{d}") for d in fixed]
    physics = fec.Poisson() if nf == 1 else fec.Mechanics(fec.PlaneStrain() if nf == 2 else None)
    p = fec.create_parameters(mesh, asm, physics, dirichlet_bcs=bcs)
    Uu = fec.create_unknowns(asm)
    fec.assemble_mass_(asm, fec.mass, Uu, p)
    A = fec.mass(asm).to_scipy()
    n = A.shape[0]
    empty = np.isin((asm.dof.unknown_dofs - 1) // nf, loose)
    assert np.array_equal(np.diff(A.indptr) == 0, empty) and empty[-1]
    g = np.random.default_rng(2)
    P = fec.assembler._ptr
    values = fec.mass(asm).values if asm.nnz else torch.full((1,), float("nan"), dtype=torch.float64, device=gpu)
    x, b = g.standard_normal(n), g.standard_normal(n)
    if asm.nnz:
        b[empty] = 0.0
    xd, bd = torch.from_numpy(x).to(gpu), torch.from_numpy(b).to(gpu)
    y, dinv = torch.full_like(Uu, np.nan), torch.full_like(Uu, np.nan)
    asm.ctx.call("fecx_csr_spmv", P(values), P(xd), P(y))
    assert np.all(np.abs(y.cpu().numpy() - A @ x) <= 500 * 2.0 ** -53 * (abs(A) @ np.abs(x)))
    asm.ctx.call("fecx_csr_diagonal_inverse", P(values), P(dinv))
    diag = A.diagonal()
    assert np.array_equal(dinv.cpu().numpy(), np.where(diag != 0.0, 1.0 / np.where(diag != 0.0, diag, 1.0), 1.0))
    for pre in (1, 0):
        xg = xd.clone()
        it, res = ctypes.c_int(-1), ctypes.c_double(-1.0)
        asm.ctx.call("fecx_cg_solve", P(values), P(bd), P(xg), ctypes.c_double(1e-9), ctypes.c_double(0.0), ctypes.c_int(5),
                     ctypes.c_int(pre), ctypes.byref(it), ctypes.byref(res))
        d = dinv.cpu().numpy() if pre else np.ones(n)
        xs, r = x.copy(), b - A @ x
        q = d * r
        rz = r @ q
        for _ in range(5):
            Aq = A @ q
            a = rz / (q @ Aq) if asm.nnz else 0.0
            xs, r = xs + a * q, r - a * Aq
            new = r @ (d * r)
            q, rz = d * r + new / rz * q, new
        assert it.value == 5
        assert np.linalg.norm(xg.cpu().numpy() - xs) <= 1e-9 * np.linalg.norm(xs)
        assert abs(res.value - np.linalg.norm(r)) <= 1e-9 * np.linalg.norm(b)
        assert np.array_equal(xg.cpu().numpy()[empty], x[empty])


@pytest.mark.parametrize("name", ["quad4 260", "hex8 40 nf1", "quad4 150 nf2", "quad4 130 nf2 roller", "hex8 25", "hex8 18 roller",
                                  "tet10 13"])
def test_cg_over_many_lines_and_batches(fec, gpu, name):
    """Matrices of more lines than the product's 1,024 work-groups have lane groups, so that each takes two or three and the last
    ranges are ragged (quad4 260: 2,129 units of 32 rows; tet10: rows of up to 195 columns, two passes of a lane group), and solves
    of more iterations than two batches of 8, stopped around their ends or converged. The matrix: -U(0.5, 1.5) off the diagonal,
    symmetric, diagonal 1.1 times the row's sum, so its condition number is at most 2.1 / 0.1 = 21 after Jacobi scaling and, the
    row sums within a factor of 13, 273 without. Rounding of k iterations' sums over n <= 7e4 unknowns, taken as random, moves the
    iterate by condition sqrt(n) k eps: 3e-11 for the 50 iterations that the first condition number allows, 1.2e-9 for the 150 of
    the second; 2e-9 is asked for."""
    print(f"[krylov] many lines {name}", flush=True)
    if name.startswith("tet10"):
        mesh, nf, fixed = fec.kuhn_tet10_mesh(int(name.split()[1])), 3, {}
    else:
        mesh, nf, fixed = _quads(fec, name) if name.startswith("quad") and "roller" in name else _mesh(fec, name)
    space = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    var = fec.ScalarFunction(space, "u") if nf == 1 else fec.VectorFunction(space, "displ")
    asm = fec.SparseMatrixAssembler(var, sparse_matrix_type="csr", device=0)
    for d, nodes in fixed.items():
        mesh.nodeset_nodes[f"_f{d}"] = nodes
    bcs = [fec.DirichletBC(var.names[d], lambda X, t: 0.0, nset_name=f"_f{d}") for d in fixed]
    physics = fec.Poisson() if nf == 1 else fec.Mechanics(fec.PlaneStrain() if nf == 2 else None)
    fec.create_parameters(mesh, asm, physics, dirichlet_bcs=bcs)
    rp, cv = (t.cpu().numpy() for t in asm.pattern())
    n = rp.size - 1
    import scipy.sparse as sp
    g = np.random.default_rng(4)
    A = sp.csr_matrix((-0.25 - 0.5 * g.random(cv.size), cv, rp), shape=(n, n))
    A = (A + A.T).tocsr()
    A.sort_indices()
    assert np.array_equal(A.indptr, rp) and np.array_equal(A.indices, cv)
    rows = np.repeat(np.arange(n), np.diff(rp))
    A.data[cv == rows] = 0.0
    A.data[cv == rows] = 1.1 * -np.asarray(A.sum(axis=1)).ravel()
    vals, diag = torch.from_numpy(A.data).to(gpu), A.diagonal()
    b, x0 = g.standard_normal(n), g.standard_normal(n)
    bd = torch.from_numpy(b).to(gpu)
    tol = 1e-9 * np.linalg.norm(b)
    P = fec.assembler._ptr
    for pre in (1, 0):
        d = 1.0 / diag if pre else np.ones(n)
        x, r = x0.copy(), b - A @ x0
        q = d * r
        rz, k, at = r @ q, 0, {}
        while np.linalg.norm(r) > tol:
            at[k] = x.copy(), np.linalg.norm(r)
            Aq = A @ q
            a = rz / (q @ Aq)
            x, r = x + a * q, r - a * Aq
            new = r @ (d * r)
            q, rz, k = d * r + new / rz * q, new, k + 1
        at[k] = x, np.linalg.norm(r)
        assert 24 < k < 1000
        for maxit in (0, 7, 8, 9, 16, 17, 24, k - 1, k, k + 1, k + 30):
            xg = torch.from_numpy(x0).to(gpu)
            it, res = ctypes.c_int(-1), ctypes.c_double(-1.0)
            asm.ctx.call("fecx_cg_solve", P(vals), P(bd), P(xg), ctypes.c_double(1e-9), ctypes.c_double(0.0), ctypes.c_int(maxit),
                         ctypes.c_int(pre), ctypes.byref(it), ctypes.byref(res))
            want = min(maxit, k)
            assert it.value == want, (pre, maxit)
            xs, rs = at[want]
            assert np.linalg.norm(xg.cpu().numpy() - xs) <= 2e-9 * np.linalg.norm(xs), (pre, maxit)
            assert abs(res.value - rs) <= 2e-9 * np.linalg.norm(b), (pre, maxit)
