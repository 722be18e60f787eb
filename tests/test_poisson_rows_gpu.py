"""Structured scalar hex8 assembly with one lane per element and per row: meshes whose node counts, element counts and rows end
inside a wavefront, the smallest that takes it, both work-group sizes of the row kernel, and fixed nodes inside, around and
on one side. Every CSR value and residual entry is a sum of at most 8 FP32 contributions in FP64, the same contributions as the
fused kernel's in another order: equal to FP64 rounding, 2e-15 relative in the max norm. The Jacobian alone has the same bits."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
FUSED, AUTO = 0, 4


def _brick(fec, nx, ny, nz):
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    g = np.random.default_rng(nx)
    coords = np.stack([i.ravel() / (nx - 1), j.ravel() / (ny - 1), k.ravel() / (nz - 1)], axis=1)
    coords += 0.2 / max(nx, ny, nz) * g.uniform(-1, 1, coords.shape)
    ex, ey, ez = (a.ravel() for a in np.meshgrid(np.arange(nx - 1), np.arange(ny - 1), np.arange(nz - 1), indexing="ij"))
    node = lambda a, b, c: a + nx * (b + ny * c) + 1  # noqa: E731
    conn = np.stack([node(ex, ey, ez), node(ex + 1, ey, ez), node(ex + 1, ey + 1, ez), node(ex, ey + 1, ez),
                     node(ex, ey, ez + 1), node(ex + 1, ey, ez + 1), node(ex + 1, ey + 1, ez + 1),
                     node(ex, ey + 1, ez + 1)], axis=1).astype(np.int64)
    return fec.BlockMesh(coords, [("block_1", conn)], "HEX8")


@pytest.mark.parametrize("counts,fixed,source", [((33, 34, 33), "none", "constant"), ((36, 28, 38), "all", "sines"),
                                                 ((3, 129, 131), "random", "constant"), ((1201, 30, 2), "face", "constant"),
                                                 ((2, 190, 180), "random", "sines"), ((81, 82, 79), "all", "constant"),
                                                 ((70, 90, 85), "random", "constant")])
def test_rows_match_the_fused_kernel(fec, gpu, counts, fixed, source):
    print(f"[poisson rows] {counts} {fixed} {source}", flush=True)
    mesh = _brick(fec, *counts)
    assert mesh.num_elements > 1 << 15
    g = np.random.default_rng(5)
    i = np.arange(mesh.num_nodes)
    x, y, z = i % counts[0], i // counts[0] % counts[1], i // (counts[0] * counts[1])
    nodes = {"none": i[:0], "face": i[x == 0], "random": i[g.random(i.size) < 0.3],
             "all": i[(x == 0) | (x == counts[0] - 1) | (y == 0) | (y == counts[1] - 1) | (z == 0) | (z == counts[2] - 1)]}[fixed]
    V = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    asm = fec.SparseMatrixAssembler(fec.ScalarFunction(V, "u"), sparse_matrix_type="csr", device=gpu.index or 0)
    bcs = []
    if nodes.size:
        mesh.nodeset_nodes["_bc"] = nodes + 1
        bcs = [fec.DirichletBC("u", lambda X, t: 0.25, nset_name="_bc")]
    p = fec.create_parameters(mesh, asm, fec.Poisson(source, 1.5), dirichlet_bcs=bcs)
    Uu = torch.from_numpy(np.cos(0.37 * np.arange(asm.dof.unknown_dofs.size))).to(gpu)
    out = {}
    for design in (FUSED, AUTO):
        asm.ctx.call("fecx_set_scatter", ctypes.c_int(design))
        fec.assemble_vector_and_stiffness_(asm, Uu, p)
        out[design] = fec.residual(asm).clone(), asm.stiffness_storage.clone()
    for a, b in zip(out[AUTO], out[FUSED]):
        assert (a - b).abs().max().item() <= 2e-15 * b.abs().max().item()
    asm.stiffness_storage.fill_(float("nan"))  # every value is written
    fec.assemble_stiffness_(asm, fec.stiffness, Uu, p)
    assert torch.equal(asm.stiffness_storage, out[AUTO][1])


@pytest.mark.parametrize("counts", [(33, 34, 33), (61, 72, 66)])
def test_allocation_free_call_gives_the_same_bits(fec, gpu, counts):
    """The allocation-free entry point takes the same kernels, its elements padded to 64 in its own scratch."""
    print(f"[poisson rows] allocation-free {counts}", flush=True)
    mesh = _brick(fec, *counts)
    V = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    asm = fec.SparseMatrixAssembler(fec.ScalarFunction(V, "u"), sparse_matrix_type="csr", device=gpu.index or 0)
    p = fec.create_parameters(mesh, asm, fec.Poisson("sines", 1.5))
    Uu = torch.from_numpy(np.cos(0.37 * np.arange(asm.dof.unknown_dofs.size))).to(gpu)
    fec.assemble_vector_and_stiffness_(asm, Uu, p)
    R, K = torch.full_like(asm.residual_storage, float("nan")), torch.full_like(asm.stiffness_storage, float("nan"))
    P = fec.assembler._ptr
    asm.ctx.call("fecx_assemble_vector_matrix_noalloc", P(p.field), P(R), P(K))
    assert torch.equal(R, asm.residual_storage) and torch.equal(K, asm.stiffness_storage)


@pytest.mark.parametrize("counts,fixed,source", [((33, 34, 33), "none", "constant"), ((36, 28, 38), "random", "sines"),
                                                 ((2, 190, 180), "none", "sines"), ((81, 82, 79), "random", "sines")])
def test_bits_of_the_other_two_phase_kernels(fec, gpu, counts, fixed, source):
    """The kernels with one lane per element and per row sum in the order of those with 8 lanes each, which an assembly in two
    pieces and a residual alone still take: the same bits."""
    print(f"[poisson rows] bits {counts} {fixed} {source}", flush=True)
    mesh = _brick(fec, *counts)
    V = fec.FunctionSpace(mesh, "H1Field", "Lagrange")
    asm = fec.SparseMatrixAssembler(fec.ScalarFunction(V, "u"), sparse_matrix_type="csr", device=gpu.index or 0)
    bcs = []
    if fixed == "random":
        mesh.nodeset_nodes["_bc"] = np.flatnonzero(np.random.default_rng(5).random(mesh.num_nodes) < 0.3) + 1
        bcs = [fec.DirichletBC("u", lambda X, t: 0.25, nset_name="_bc")]
    p = fec.create_parameters(mesh, asm, fec.Poisson(source, 1.5), dirichlet_bcs=bcs)
    Uu = torch.from_numpy(np.cos(0.37 * np.arange(asm.dof.unknown_dofs.size))).to(gpu)
    fec.assemble_vector_and_stiffness_(asm, Uu, p)
    R, K = asm.residual_storage.clone(), asm.stiffness_storage.clone()
    asm.ctx.call("fecx_set_chunks", ctypes.c_int(2))
    asm.stiffness_storage.fill_(float("nan"))
    fec.assemble_vector_and_stiffness_(asm, Uu, p)
    assert torch.equal(asm.residual_storage, R) and torch.equal(asm.stiffness_storage, K)
    fec.assemble_vector_(asm, fec.residual, Uu, p)
    assert torch.equal(asm.residual_storage, R)
