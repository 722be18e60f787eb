"""The HIP library is the only compute path: without libfecx.so, or without a HIP device, the assembler refuses to run
instead of falling back to a CPU implementation."""
import numpy as np
import pytest
import torch


def test_missing_library_raises(fec, monkeypatch):
    import sys
    L = sys.modules[fec.__name__ + "._lib"]
    monkeypatch.setattr(L, "LIB_PATH", L.LIB_PATH + ".missing")
    monkeypatch.setattr(L, "_lib", None)
    with pytest.raises(fec.FECXError) as ei:
        L.Context(-1)
    assert ei.value.code == -3 and "not built" in str(ei.value)


@pytest.mark.skipif(torch.cuda.is_available(), reason="checks the refusal on a host without a HIP device")
def test_assembler_without_gpu_raises(fec):
    mesh = fec.StructuredMesh("hex", (0, 0, 0), (1, 1, 1), (3, 3, 3))
    var = fec.ScalarFunction(fec.FunctionSpace(mesh, "H1Field", "Lagrange"), "u")
    with pytest.raises(fec.FECXError) as ei:
        fec.SparseMatrixAssembler(var, sparse_matrix_type="csr")
    assert ei.value.code == -3


def test_host_context_refuses_kernels(fec):
    """A host-only context (device -1) builds patterns but refuses every assembly call."""
    mesh = fec.StructuredMesh("hex", (0, 0, 0), (1, 1, 1), (3, 3, 3))
    hp = fec.HostPattern(mesh, 1, np.zeros(0, np.int64))
    U, R = np.zeros(27), np.zeros(27)  # host arrays: the call is refused before any pointer is used
    with pytest.raises(fec.FECXError) as ei:
        hp.ctx.call("fecx_assemble_vector", U.ctypes.data_as(__import__("ctypes").c_void_p),
                    R.ctypes.data_as(__import__("ctypes").c_void_p))
    assert "host-only" in str(ei.value)


@pytest.mark.parametrize("fixed", ["none", "some", "all"])
def test_field_calls_refuse_null_arrays(fec, fixed):
    """A field call that would read or write an array refuses NULL in its place (code -1) before anything runs; arrays that the
    dofs leave untouched may be NULL, and such calls get as far as the host-only context's own refusal (code -2)."""
    import ctypes
    mesh = fec.StructuredMesh("hex", (0, 0, 0), (1, 1, 1), (2, 2, 2))
    dirichlet = np.arange(1, {"none": 1, "some": 4, "all": 9}[fixed])
    ctx = fec.HostPattern(mesh, 1, dirichlet.astype(np.int64)).ctx
    a = np.zeros(8)
    x = a.ctypes.data_as(ctypes.c_void_p)
    free, bc = fixed != "all", fixed != "none"
    calls = [("fecx_update_fields", (x, x, x, x, x), False), ("fecx_update_fields", (None, x, x, None, None), False),
             ("fecx_update_fields", (None, x, x, x, None), False), ("fecx_update_fields", (x, None, x, x, x), free),
             ("fecx_update_fields", (x, x, None, x, x), True), ("fecx_update_fields", (None, x, None, x, x), free),
             ("fecx_update_fields", (x, x, x, None, x), free), ("fecx_update_field_unknowns", (x, x), False),
             ("fecx_update_field_unknowns", (None, x), free), ("fecx_update_field_unknowns", (x, None), free),
             ("fecx_update_field_dirichlet", (None, x), bc), ("fecx_update_field_dirichlet", (x, None), bc),
             ("fecx_extract_field_unknowns", (None, x), free), ("fecx_extract_field_unknowns", (x, None), free)]
    for name, args, refused in calls:
        with pytest.raises(fec.FECXError) as ei:
            ctx.call(name, *args)
        assert ei.value.code == (-1 if refused else -2), (name, args)
