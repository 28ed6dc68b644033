"""The FP32 products of the learned preconditioner at every block size (the inputs of the encoders and decoders are
b^2 and b^2 + 1 wide, so their 16-wide chunks are ragged or unaligned) and at row counts around the 64-row tiles and
the parts of the weight gradient: outputs, loss and gradient against the FP64 oracle.

Bound of the gradient: FP32 sums of up to a few thousand terms through eight layers; 2e-4 of each tensor's norm is
about 1700 eps, the largest seen with one-by-one sums is 3e-5."""
import numpy as np
import pytest

import hyperfox_amd as hf
import hyperfox_amd.problems as pr
from hyperfox_amd.lpc import LearnedPreconditioner
import lpc_oracle as lo
from test_lpc_oracle import random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dim,p,n', [(2, 1, 3), (2, 2, 6), (2, 3, 1), (2, 3, 7), (2, 3, 12), (2, 4, 4), (2, 5, 3),
                                     (3, 2, 1), (3, 3, 1), (3, 3, 2)])
def test_outputs_loss_and_gradient(dim, p, n):
    print('lpc', dim, p, n, flush=True)
    w = pr.diffusion_source_2d(n, p) if dim == 2 else pr.convection_diffusion_3d(n, p)
    prob = hf.HDGProblem(dim, p)
    pr.setup_gpu(w, prob)
    prob.assemble()
    prob.set_krylov(hf.KRYLOV_BICGSTAB)
    assert prob.solve(pc=hf.PC_BJACOBI, rtol=1e-12, maxits=20000)[1] == 2
    b = prob.sizes['nNf']
    net = LearnedPreconditioner(b)
    net.add_sample(prob)
    rowptr, cols, vals, _ = prob.trace_csr()
    dirf = np.zeros(w.mesh.n_faces, dtype=bool)
    dirf[w.mesh.arrays()['boundary']] = True
    g = lo.graph_from_scalar_csr(rowptr, cols, b, dirf)
    A = lo.blocks_from_scalar_csr(g, rowptr, cols, vals, b)
    P = random_params(b, 40 + n).astype(np.float32)
    net.set_params(P)
    cn, ce = net.outputs(0)
    sinv, ahat, dinv = lo.normalise(g, A)
    acts = lo.forward(lo.unpack(P.astype(np.float64), b), g, ahat)
    scale = max(np.abs(acts['cn']).max(), np.abs(acts['ce']).max())
    assert np.abs(cn - acts['cn']).max() <= 1e-4 * scale
    assert np.abs(ce - acts['ce']).max() <= 1e-4 * scale
    loss, grad = net.loss_grad(0, n_random=1, seed=5)
    loss_o, grad_o, _ = lo.loss_grad(P.astype(np.float64), b, g, A, prob.solution()[2], 1, 5)
    assert loss == pytest.approx(loss_o, rel=1e-4)
    for k, (o, m) in ((k, v) for k, v in lo.layout(b).items() if k != 'total'):
        go, gg = grad_o[o:o + m], grad[o:o + m].astype(np.float64)
        assert np.linalg.norm(gg - go) <= 2e-4 * np.linalg.norm(go) + 1e-9, k
