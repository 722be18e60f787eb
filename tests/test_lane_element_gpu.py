"""tet10 residuals and matrix-free actions with one lane per element: the smallest mesh that takes it and a ragged one, every
material, fixed nodes. The residual has the bits of the residual + Jacobian call, which forms it on 16 lanes per element in the
same order; the action agrees with the one from the element blocks, each within 1e-6 of exact arithmetic (FP32 element algebra,
relative 2-norm), so within 2e-6 of each other. A folded element raises from either."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [18, 23])
@pytest.mark.parametrize("physics", ["poisson", "elastic", "neohookean"])
def test_rows_of_the_other_kernels(fec, gpu, n, physics):
    print(f"[lane element] {physics} {n}", flush=True)
    mesh = fec.workloads.kuhn_tet10_mesh(n, jitter=0.2, seed=n)
    assert mesh.num_elements > 1 << 15 and mesh.num_elements % 64 != 0
    V = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    var = fec.ScalarFunction(V, "u") if physics == "poisson" else fec.VectorFunction(V, "displ")
    mat = {"poisson": lambda: fec.Poisson("sines", 1.5), "elastic": lambda: fec.Mechanics(K=1.3, G=0.7),
           "neohookean": lambda: fec.NeoHookean(1.0, 0.5)}[physics]()
    asm = fec.SparseMatrixAssembler(var, sparse_matrix_type="csr", device=gpu.index or 0)
    X = np.asarray(mesh.coords)
    mesh.nodeset_nodes["_bc"] = np.flatnonzero(X[:, 0] < 1e-9) + 1
    p = fec.create_parameters(mesh, asm, mat, dirichlet_bcs=[fec.DirichletBC(v, lambda X, t: 0.0, nset_name="_bc") for v in var.names])
    g = np.random.default_rng(n)
    nf = len(var.names)
    U = np.stack([0.03 * X[:, 0] * np.sin(3 * X @ g.standard_normal(3) + i) for i in range(nf)], axis=1).ravel()  # 0 at x = 0
    unk = asm.dof.unknown_dofs - 1
    Uu = torch.from_numpy(U[unk].copy()).to(gpu)
    Vu = torch.from_numpy(g.standard_normal(unk.size)).to(gpu)
    fec.assemble_vector_and_stiffness_(asm, Uu, p)
    both = fec.residual(asm).clone()
    fec.assemble_vector_(asm, fec.residual, Uu, p)
    assert torch.equal(fec.residual(asm), both)
    fec.assemble_matrix_action_(asm, fec.stiffness, Uu, Vu, p)
    blocks = fec.hvp(asm, Vu).clone()
    fec.assemble_matrix_free_action_(asm, fec.stiffness_action, Uu, Vu, p)
    assert (fec.hvp(asm, Vu) - blocks).norm().item() <= 2e-6 * blocks.norm().item()
    if physics == "neohookean":
        Uu[Uu.numel() // 2] = 1e3
        with pytest.raises(Exception):
            fec.assemble_vector_(asm, fec.residual, Uu, p)
