"""Network inference, 64 samples per wavefront as two 32-sample matrix tiles: sizes around the edges of a tile, a wavefront
and a work-group. A sample's outputs depend on its own inputs alone, so a shorter batch gives the same bits as the start of a
longer one; the longest is compared with the BF16-emulating reference (max |dy| <= 1e-2 of the output scale, since another
accumulation order may flip the rounding of a hidden activation). With every sample sent to the fallback (tolerance 1e-12),
the update counts each sample once and is the plain model's (FP32 in another kernel: 1e-6 of the largest output)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [1, 31, 32, 33, 63, 64, 65, 255, 256, 257, 300]


@pytest.mark.parametrize("arch", [0, 1])
def test_inference_at_tile_edges(fec, mlpref, gpu, arch):
    print(f"[network tiles] arch {arch}", flush=True)
    physics = fec.J2Surrogate(200.0, 0.3, 0.25, 2.0) if arch == 0 else fec.NeoHookeanSurrogate(1.0, 0.5)
    wl = fec.workloads.j2_hex8(2)
    V = fec.FunctionSpace(wl.mesh, "H1Field", "Lagrange")
    asm = fec.SparseMatrixAssembler(fec.VectorFunction(V, "displ"), sparse_matrix_type="csr", device=gpu.index or 0)
    p = fec.create_parameters(wl.mesh, asm, physics)  # noqa: F841 (creates the blocks)
    net = fec.Surrogate(asm, arch, seed=11)
    g = np.random.default_rng(13)
    d = net.shape
    sc = (g.uniform(-0.1, 0.1, d[0]).astype(np.float32), g.uniform(0.5, 2.0, d[0]).astype(np.float32),
          g.uniform(-0.1, 0.1, d[-1]).astype(np.float32), g.uniform(0.5, 2.0, d[-1]).astype(np.float32))
    net.set_scaling(*sc)
    raw = g.normal(0, 1, (SIZES[-1], 16 if arch == 0 else 9)).astype(np.float32)
    X = torch.from_numpy(raw).to(gpu)
    full = net.forward(X)
    ref, _ = mlpref.forward(arch, net.params(), sc, raw, emulate=True)
    ref = ref * sc[3] + sc[2]
    assert np.max(np.abs(full.cpu().numpy().astype(np.float64) - ref)) <= 1e-2 * np.max(np.abs(ref))
    net.set_tolerance(1e-12)
    Xs = 0.01 * X
    Xs[:, -1].abs_()
    plain_kind, kind = ((fec._lib.J2, fec._lib.J2_SURROGATE), (fec._lib.NEOHOOKEAN, fec._lib.NH_SURROGATE))[arch]
    plain = fec.surrogate.material_update(asm, plain_kind, Xs)
    update = fec.surrogate.material_update(asm, kind, Xs)
    assert (update - plain).abs().max().item() <= 1e-6 * plain.abs().max().item()
    for n in SIZES:
        assert torch.equal(net.forward(X[:n].contiguous()), full[:n]), n
        assert torch.equal(fec.surrogate.material_update(asm, kind, Xs[:n].contiguous()), update[:n]), n
        assert net.fallbacks() == (n, n)
    # the longest batch that runs with one tile per wavefront and the shortest with two: the same bits per sample
    big = X.repeat((1 << 18) // len(X) + 2, 1)
    for n in ((1 << 18) - 3, (1 << 18) + 1):
        assert torch.equal(net.forward(big[:n].contiguous()), full.repeat(len(big) // len(X), 1)[:n]), n
