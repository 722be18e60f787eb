"""The dof-level CSR of rollers and other partial Dirichlet sets, which the reductions and the fused kernel write in place: on
every kernel that writes it, the values equal the unconstrained assembly's at the unknown rows and columns, bit for bit (the
same element matrices, the same contributions in the same order). Meshes cover light and heavy rows of every element kind,
rows on the slot-owner kernel (70 to 165 blocks, hex8 nodes with 12 incidences), sizes that are no multiple of a work-group's
rows, and every scatter design of a structured mesh (FP64 atomics, whose order of arrival differs: 1e-13)."""
import ctypes

import numpy as np
import pytest
import torch

from test_mass_rows_gpu import _mesh

pytestmark = pytest.mark.gpu

FUSED, TWO_PHASE, ATOMIC, COLOURED, AUTO = 0, 1, 2, 3, 4
CASES = [("quad4 6", AUTO), ("hex8 5", FUSED), ("hex8 9", FUSED), ("hex8 5", TWO_PHASE), ("hex8 5", ATOMIC), ("hex8 5", COLOURED),
         ("hexfan 6", AUTO), ("tet10 2", AUTO), ("tet10 3", "two launches"), ("fan 5", AUTO), ("fan 13", AUTO), ("fan 32", AUTO)]


def _assemble(fec, mesh, fixed, design):
    space = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    var = fec.VectorFunction(space, "displ")
    nf = var.nf
    asm = fec.SparseMatrixAssembler(var, sparse_matrix_type="csr", device=0)
    U = 0.02 * np.sin(1.0 + np.arange(nf * mesh.num_nodes)).reshape(-1, nf) * np.abs(mesh.coords).max() / mesh.num_nodes
    bcs = []
    for d, nodes in fixed.items():
        mesh.nodeset_nodes[f"_p{d}"] = nodes
        bcs.append(fec.DirichletBC(var.names[d], lambda X, t, v=U[nodes - 1, d]: v, nset_name=f"_p{d}"))
    p = fec.create_parameters(mesh, asm, fec.Mechanics(fec.PlaneStrain()) if nf == 2 else fec.NeoHookean(), dirichlet_bcs=bcs)
    if design == "two launches":
        asm.ctx.call("fecx_set_merged_rows", ctypes.c_int(0))
    else:
        asm.ctx.call("fecx_set_scatter", ctypes.c_int(design))
    Uu = torch.from_numpy(U.ravel()[asm.dof.unknown_dofs - 1]).to("cuda:0")
    fec.assemble_vector_and_stiffness_(asm, Uu, p)
    return asm, fec.residual(asm).cpu().numpy(), fec.stiffness(asm).to_scipy()


@pytest.mark.parametrize("name,design", CASES)
def test_partial_rows_equal_unconstrained(fec, gpu, name, design):
    print(f"[partial rows] {name} {design}", flush=True)
    mesh = _mesh(fec, name)
    nd = mesh.coords.shape[1]
    g = np.random.default_rng(3)
    # rollers on the low faces, and single components of a few nodes in between
    fixed = {d: np.unique(np.concatenate([np.flatnonzero(mesh.coords[:, d] < mesh.coords[:, d].min() + 1e-12),
                                          g.integers(0, mesh.num_nodes, 3)])) + 1 for d in range(nd)}
    _, R0, K0 = _assemble(fec, mesh, {}, design)
    asm, R, K = _assemble(fec, mesh, fixed, design)
    u = asm.dof.unknown_dofs - 1
    ref = K0[u][:, u].tocsr()
    ref.sort_indices()
    assert np.array_equal(K.indptr, ref.indptr) and np.array_equal(K.indices, ref.indices)
    if design == ATOMIC:
        assert np.abs(K.data - ref.data).max() <= 1e-13 * np.abs(ref.data).max()
    else:
        assert np.array_equal(K.data, ref.data) and np.array_equal(R, R0[u])


@pytest.mark.parametrize("name", ["quad4 6", "hex8 5", "tet10 2", "fan 32"])
def test_split_node_of_no_element(fec, gpu, name):
    """The only node with some fixed and some free components belongs to no element: a dof-level CSR whose rows are all complete."""
    print(f"[partial rows] split loose node, {name}", flush=True)
    m = _mesh(fec, name)
    n = m.num_nodes
    mesh = fec.BlockMesh(np.vstack([m.coords, m.coords.mean(axis=0)]), [("b", m.conn)], m.element_type)
    _, R0, K0 = _assemble(fec, mesh, {}, AUTO)
    asm, R, K = _assemble(fec, mesh, {1: np.array([n + 1])}, AUTO)
    u = asm.dof.unknown_dofs - 1
    ref = K0[u][:, u].tocsr()
    ref.sort_indices()
    assert K.nnz == K0.nnz and K.shape[0] == K0.shape[0] - 1
    assert np.array_equal(K.indptr, ref.indptr) and np.array_equal(K.indices, ref.indices)
    assert np.array_equal(K.data, ref.data) and np.array_equal(R, R0[u])
