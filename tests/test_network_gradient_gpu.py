"""The training gradient at the edges of its split: 32-sample tiles (one or two per work-group), samples padded to 64, chunks of
the weight-gradient sums (one chunk, whole chunks, a shorter last one), against the BF16-emulating reference. Tolerances of the
networks' other tests: relative 2-norm error of the gradient 2e-2 and of the loss 1e-3 (accumulation order may flip the BF16
rounding of an activation)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arch,n", [(0, 1), (0, 33), (0, 64), (0, 65), (0, 4160), (0, 8200), (1, 1), (1, 32), (1, 95), (1, 4097),
                                    (1, 8192), (1, 8193)])
def test_gradient_at_the_edges(fec, mlpref, gpu, arch, n):
    print(f"[network gradient] arch {arch} n {n}", flush=True)
    physics = fec.J2Surrogate(200.0, 0.3, 0.25, 2.0) if arch == 0 else fec.NeoHookeanSurrogate(1.0, 0.5)
    wl = fec.workloads.j2_hex8(2)
    V = fec.FunctionSpace(wl.mesh, "H1Field", "Lagrange")
    asm = fec.SparseMatrixAssembler(fec.VectorFunction(V, "displ"), sparse_matrix_type="csr", device=gpu.index or 0)
    p = fec.create_parameters(wl.mesh, asm, physics)  # noqa: F841 (creates the blocks)
    net = fec.Surrogate(asm, arch, seed=17)
    g = np.random.default_rng(n)
    d = net.shape
    sc = (g.uniform(-0.1, 0.1, d[0]).astype(np.float32), g.uniform(0.5, 2.0, d[0]).astype(np.float32),
          g.uniform(-0.1, 0.1, d[-1]).astype(np.float32), g.uniform(0.5, 2.0, d[-1]).astype(np.float32))
    net.set_scaling(*sc)
    raw = g.normal(0, 1, (n, 16 if arch == 0 else 9)).astype(np.float32)
    tgt = g.normal(0, 1, (n, d[-1])).astype(np.float32)
    X, T = torch.from_numpy(raw).to(gpu), torch.from_numpy(tgt).to(gpu)
    loss, grad = net.gradient(X, T)
    lref, gref = mlpref.loss_and_grad(arch, net.params(), sc, raw, tgt, emulate=True)
    err = np.linalg.norm(grad.cpu().numpy().astype(np.float64) - gref) / np.linalg.norm(gref)
    assert abs(loss - lref) <= 1e-3 * lref, (loss, lref)
    assert err <= 2e-2, err
    loss2, grad2 = net.gradient(X, T)  # the same bits again
    assert loss2 == loss and torch.equal(grad2, grad)


@pytest.mark.parametrize("arch", [0, 1])
@pytest.mark.parametrize("n", [1024, 4096])
def test_sums_over_chunks(fec, gpu, arch, n):
    """The gradient of n samples, whose chunks have 64 samples each, against the FP64 mean of the gradients of those 64: their
    products are the same (n and 64 are powers of two, so the scaling of dz is exact). m additions one after the other of random
    terms are off by 0.41 sqrt(m / 2) roundings of 2^-24; the sum by eights has 8 of them at most and trees of three levels, 0.41
    sqrt(3): 1.1 together, and 1.5 roundings, 9e-8 of the gradient's 2-norm, are asked for (64 additions: 2.3)."""
    print(f"[network gradient] sums of {n} samples, arch {arch}", flush=True)
    physics = fec.J2Surrogate(200.0, 0.3, 0.25, 2.0) if arch == 0 else fec.NeoHookeanSurrogate(1.0, 0.5)
    wl = fec.workloads.j2_hex8(2)
    var = fec.VectorFunction(fec.FunctionSpace(wl.mesh, "H1Field", "Lagrange"), "displ")
    asm = fec.SparseMatrixAssembler(var, sparse_matrix_type="csr", device=gpu.index or 0)
    fec.create_parameters(wl.mesh, asm, physics)
    net = fec.Surrogate(asm, arch, seed=3)
    g = np.random.default_rng(6)
    X = torch.from_numpy(g.standard_normal((n, 16 if arch == 0 else 9)).astype(np.float32)).to(gpu)
    T = torch.from_numpy(g.standard_normal((n, net.shape[-1])).astype(np.float32)).to(gpu)
    whole = net.gradient(X, T)[1].double()
    pieces = torch.zeros_like(whole)
    for k in range(0, n, 64):
        pieces += net.gradient(X[k:k + 64], T[k:k + 64])[1].double()
    pieces /= n // 64
    assert (whole - pieces).norm().item() <= 1.5 * 2.0 ** -24 * pieces.norm().item()
