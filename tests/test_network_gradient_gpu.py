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
