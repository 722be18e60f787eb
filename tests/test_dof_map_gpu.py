"""The DOF plumbing by mask words (fixed and unknown dofs written in one launch, unknowns extracted) against numpy indexing:
field sizes around the 64-dof words and the work-groups, both launch forms, empty and full Dirichlet sets, single components,
condensed mode, with and without the action's direction field. Copies, so equality is exact."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nf", [(1, 1, 1), (7, 7, 1), (8, 6, 1), (20, 12, 2), (31, 7, 2), (255, 255, 1), (1200, 900, 1),
                                      (900, 700, 2)])
@pytest.mark.parametrize("share", [0.0, 0.1, 0.97, 1.0])
@pytest.mark.parametrize("condensed", [False, True])
def test_update_and_extract(fec, gpu, nx, ny, nf, share, condensed):
    if condensed and nx > 300:
        pytest.skip("one size of the large launch form is enough")
    mesh = fec.BlockMesh(np.stack(np.meshgrid(np.arange(nx + 1.0), np.arange(ny + 1.0), indexing="ij"), -1).reshape(-1, 2),
                         [("b", np.array([[1, 2 + ny, 3 + ny, 2]]))], "QUAD4")  # one element: the plumbing needs no others
    N = nf * mesh.num_nodes
    fixed = np.flatnonzero(np.random.default_rng(7).random(N) < share)
    c = fec._lib.Context(0)
    c.call("fecx_set_stream", ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream))
    fec.assembler._set_mesh(c, mesh, fec._lib.QUAD4)
    if condensed:
        c.call("fecx_set_condensed", ctypes.c_int(1))
    one = np.ascontiguousarray(fixed + 1)
    c.call("fecx_set_dofs", ctypes.c_int(nf), fec.assembler._host_ptr(one) if len(one) else None, ctypes.c_int64(len(one)))
    free = np.setdiff1d(np.arange(N), fixed)
    g = np.random.default_rng(8)
    P = fec.assembler._ptr
    host = {k: g.standard_normal(n) for k, n in dict(U=N, V=N, bc=len(fixed), Uu=N if condensed else len(free),
                                                     Vu=N if condensed else len(free)).items()}
    d = {k: torch.from_numpy(v.copy()).to(gpu) for k, v in host.items()}
    exp_u, exp_v = host["U"].copy(), host["V"].copy()
    exp_u[free] = host["Uu"][free] if condensed else host["Uu"]
    no_bc = exp_u.copy()
    exp_u[fixed] = host["bc"]
    exp_v[free] = host["Vu"][free] if condensed else host["Vu"]
    for with_bc, with_v in ((True, True), (False, False), (True, False), (False, True)):
        U, V = d["U"].clone(), d["V"].clone()
        c.call("fecx_update_fields", P(d["bc"]) if with_bc else None, P(d["Uu"]), P(U), P(d["Vu"]) if with_v else None,
               P(V) if with_v else None)
        assert np.array_equal(U.cpu().numpy(), exp_u if with_bc else no_bc)
        assert np.array_equal(V.cpu().numpy(), exp_v if with_v else host["V"])
    U = d["U"].clone()
    c.call("fecx_update_field_unknowns", P(d["Uu"]), P(U))
    assert np.array_equal(U.cpu().numpy(), no_bc)
    out = torch.full((len(free),), float("nan"), dtype=torch.float64, device=gpu)
    c.call("fecx_extract_field_unknowns", P(d["U"]), P(out))
    assert np.array_equal(out.cpu().numpy(), host["U"][free])


@pytest.mark.parametrize("fixed", ["none", "some", "all"])
def test_null_arrays_are_refused(fec, gpu, fixed):
    """A field call refuses NULL (code -1) in the place of an array that it would read or write; arrays that the dofs leave
    untouched may be NULL."""
    mesh = fec.StructuredMesh("hex", (0, 0, 0), (1, 1, 1), (2, 2, 2))
    dirichlet = np.arange(1, {"none": 1, "some": 4, "all": 9}[fixed], dtype=np.int64)
    c = fec._lib.Context(0)
    fec.assembler._set_mesh(c, mesh, fec._lib.HEX8)
    c.call("fecx_set_dofs", ctypes.c_int(1), fec.assembler._host_ptr(dirichlet) if len(dirichlet) else None,
           ctypes.c_int64(len(dirichlet)))
    arrays = torch.zeros((5, 8), dtype=torch.float64, device=gpu)
    x = [fec.assembler._ptr(t) for t in arrays.unbind()]
    free, bc = fixed != "all", fixed != "none"
    calls = [("fecx_update_fields", (x[0], x[1], x[2], x[3], x[4]), False), ("fecx_update_fields", (None, x[1], x[2], None, None), False),
             ("fecx_update_fields", (None, x[1], x[2], x[3], None), False), ("fecx_update_fields", (x[0], None, x[2], x[3], x[4]), free),
             ("fecx_update_fields", (x[0], x[1], None, x[3], x[4]), True), ("fecx_update_fields", (None, x[1], None, x[3], x[4]), free),
             ("fecx_update_fields", (x[0], x[1], x[2], None, x[4]), free), ("fecx_update_field_unknowns", (x[0], x[1]), False),
             ("fecx_update_field_unknowns", (None, x[1]), free), ("fecx_update_field_unknowns", (x[0], None), free),
             ("fecx_update_field_dirichlet", (None, x[1]), bc), ("fecx_update_field_dirichlet", (x[0], None), bc),
             ("fecx_extract_field_unknowns", (None, x[1]), free), ("fecx_extract_field_unknowns", (x[0], None), free)]
    for name, args, refused in calls:
        if not refused:
            c.call(name, *args)
            continue
        with pytest.raises(fec.FECXError) as ei:
            c.call(name, *args)
        assert ei.value.code == -1, name
    torch.cuda.synchronize()
