"""The consistent mass of 2 and 3 fields, reduced from one word per node pair and written out as blocks m I, over the row
shapes its kernels dispatch on: light rows (at most 8 incidences and 32 blocks) of every element kind, heavier ones on a
wavefront (hex8 nodes with 12 incidences, tet10 vertices with 24, rows of 70 and of 165 blocks), meshes of one element, row
counts that are no multiple of the work-groups' and the dof-level CSR of rollers.

Tolerance: 1e-6 relative error against the FP64 oracle (2-norm and max-norm; FP32 element arithmetic, FP64 sums), the bound
of the other mass tests; entries that couple different components are exactly zero and the matrix is symmetric bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _hex_fan(m, layers):
    """m hex8 around a common edge, `layers` of them on top of each other: the inner edge's nodes have 2 m incidences."""
    t = 2 * np.pi * np.arange(m) / m
    ring = np.stack([np.cos(t), np.sin(t)], axis=1)
    outer = 1.3 * np.stack([np.cos(t + np.pi / m), np.sin(t + np.pi / m)], axis=1)
    flat = np.concatenate([np.zeros((1, 2)), ring, outer])
    coords = np.concatenate([np.column_stack([flat, np.full(len(flat), 0.7 * z)]) for z in range(layers + 1)])
    n = len(flat)
    quad = np.array([[0, 1 + i, 1 + m + i, 1 + (i + 1) % m] for i in range(m)])
    conn = np.concatenate([np.concatenate([quad + n * z, quad + n * (z + 1)], axis=1) for z in range(layers)])
    return coords, conn + 1


def _mesh(fec, name):
    kind, *a = name.split()
    if kind == "quad4":
        return fec.StructuredMesh("quad", (0.0, 0.0), (1.0, 1.0), (int(a[0]) + 1,) * 2)
    if kind == "hex8":
        return fec.StructuredMesh("hex", (0.0,) * 3, (1.0,) * 3, (int(a[0]) + 1,) * 3)
    if kind == "hexfan":
        coords, conn = _hex_fan(int(a[0]), 2)
        return fec.BlockMesh(coords, [("b", conn)], "HEX8")
    return fec.fan_tet10_mesh(int(a[0])) if kind == "fan" else fec.kuhn_tet10_mesh(int(a[0]))


CASES = ["quad4 1", "quad4 9", "hex8 1", "hex8 5", "hex8 7 roller", "hexfan 6", "hexfan 13", "tet10 1", "tet10 3", "tet10 2 roller",
         "fan 4", "fan 13", "fan 32"]


@pytest.mark.parametrize("name", CASES)
def test_consistent_mass_rows(fec, orc, gpu, name):
    print(f"[mass rows] {name}", flush=True)
    mesh = _mesh(fec, name)
    space = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    var = fec.VectorFunction(space, "displ")
    nf = var.nf
    asm = fec.SparseMatrixAssembler(var, sparse_matrix_type="csr", device=0)
    bcs = []
    if "roller" in name:
        for d in range(nf):
            mesh.nodeset_nodes[f"_r{d}"] = np.flatnonzero(mesh.coords[:, d] < 1e-12) + 1
            bcs.append(fec.DirichletBC(var.names[d], lambda X, t: 0.0, nset_name=f"_r{d}"))
    p = fec.create_parameters(mesh, asm, fec.Mechanics(fec.PlaneStrain() if nf == 2 else None), dirichlet_bcs=bcs)
    fec.assemble_mass_(asm, fec.mass, fec.create_unknowns(asm), p)
    M = fec.mass(asm)
    unknown = asm.dof.unknown_dofs
    _, d2u = orc.update_dofs(nf * mesh.num_nodes, asm.dof.dirichlet_dofs)
    kind = {"QUAD4": orc.QUAD4, "HEX8": orc.HEX8, "TET10": orc.TET10}[mesh.element_type]
    rp, cv, ref = orc.mass_csr(kind, mesh.coords, mesh.conn, nf, fec.density(p.physics), d2u, len(unknown))
    assert np.array_equal(M.rowptr.cpu().numpy() + 1, rp) and np.array_equal(M.colval.cpu().numpy() + 1, cv)
    got = M.values.cpu().numpy()
    assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref) and np.abs(got - ref).max() <= 1e-6 * np.abs(ref).max()
    row = np.repeat(np.arange(len(unknown)), np.diff(rp))
    comp = (unknown - 1) % nf
    assert np.all(got[comp[row] != comp[cv - 1]] == 0.0)
    A = M.to_scipy()
    assert (A != A.T).nnz == 0
