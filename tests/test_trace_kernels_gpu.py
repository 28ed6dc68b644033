"""Kernels of the trace solve at the sizes where their tiling can go wrong.

* the block-Jacobi inverse (several blocks per wavefront) against numpy's
  inverse of the assembled diagonal blocks, for every block size of the 2-D
  and 3-D orders and block counts that do not fill the last wavefront;
* the reconstruction u = U lambda + U0, q = Q lambda + Q0 against numpy on the
  same condensed blocks, for odd and even row lengths.

Bounds: an inverse by Gauss-Jordan with partial pivoting is off by at most a
few n eps cond(D) (n <= 21, cond(D) computed), a dot product of NL + 1 terms by
(NL + 1) eps times the sum of the terms' magnitudes."""
import numpy as np
import pytest

import hyperfox_amd as hf
import hyperfox_amd.problems as pr

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def problem(dim, p, n):
    w = pr.diffusion_source_2d(n, p) if dim == 2 else pr.convection_diffusion_3d(n, p)
    prob = hf.HDGProblem(dim, p)
    pr.setup_gpu(w, prob)
    prob.assemble()
    return w, prob


def diagonal_blocks(w, prob):
    bs = prob.sizes['nNf']
    rowptr, cols, vals, _ = prob.trace_csr()
    nb = w.mesh.n_faces
    D = np.zeros((nb, bs, bs))
    for F in range(nb):
        for r in range(bs):
            k0, k1 = rowptr[F * bs + r], rowptr[F * bs + r + 1]
            k = k0 + int(np.where(cols[k0:k1] == F * bs)[0][0])
            D[F, r] = vals[k:k + bs]
    return D


@pytest.mark.parametrize('dim,p,n', [(2, 1, 3), (2, 2, 2), (2, 3, 5), (2, 4, 3), (2, 5, 2), (2, 6, 1), (2, 7, 2),
                                     (2, 8, 1), (2, 9, 2), (2, 10, 1), (3, 1, 2), (3, 2, 1), (3, 3, 2), (3, 4, 1),
                                     (3, 5, 1)])
def test_block_jacobi_inverse(dim, p, n):
    print('block jacobi', dim, p, n, flush=True)
    w, prob = problem(dim, p, n)
    D = diagonal_blocks(w, prob)
    bs = D.shape[1]
    rng = np.random.default_rng(p)
    x = rng.standard_normal((w.mesh.n_faces, bs))
    y = prob.pc_apply(hf.PC_BJACOBI, x.reshape(-1)).reshape(-1, bs)
    inv = np.linalg.inv(D)
    ref = np.einsum('fij,fj->fi', inv, x)
    cond = np.linalg.cond(D)
    bound = 16 * bs * EPS * cond * np.linalg.norm(inv, axis=(1, 2)) * np.linalg.norm(x, axis=1)
    assert (np.linalg.norm(y - ref, axis=1) <= bound).all()


@pytest.mark.parametrize('dim,p,n', [(2, 1, 1), (2, 2, 3), (2, 3, 2), (2, 4, 3), (2, 5, 1), (2, 8, 1), (3, 1, 1),
                                     (3, 2, 1), (3, 3, 1), (3, 4, 1), (3, 5, 1)])
def test_reconstruction(dim, p, n):
    print('reconstruct', dim, p, n, flush=True)
    w, prob = problem(dim, p, n)
    prob.set_krylov(hf.KRYLOV_BICGSTAB)
    prob.solve(pc=hf.PC_BJACOBI, rtol=1e-8, maxits=5000)
    u, q, lam = prob.solution()
    c = prob.condensed()
    a = w.mesh.arrays()
    nNf = prob.sizes['nNf']
    lc = lam.reshape(-1, nNf)[a['cell2face'][:, :, None], a['face_perm'].astype(int)].reshape(w.mesh.n_cells, -1)
    for got, M, M0 in ((u, c['U'], c['U0']), (q, c['Q'], c['Q0'])):
        ref = np.einsum('eij,ej->ei', M, lc) + M0
        mag = np.einsum('eij,ej->ei', np.abs(M), np.abs(lc)) + np.abs(M0)
        assert (np.abs(got - ref) <= 2 * (lc.shape[1] + 1) * EPS * mag).all()


@pytest.mark.parametrize('restart', [1, 2, 8, 9, 17, 33, 63])
@pytest.mark.parametrize('n', [1, 7, 19])
def test_gmres_against_a_dense_solve(n, restart):
    """Restart lengths below and above the 4 to 15 steps that these systems need (longer cycles are in the tests below),
    one and several row blocks, an iteration budget inside a cycle, and convergence inside a cycle.  At rtol the residual is at most rtol ||b||, so the error is at
    most cond(A) rtol ||x||."""
    print('gmres', n, restart, flush=True)
    rng = np.random.default_rng(n)
    N = n * n + 3
    A = 4.0 * np.eye(N) + 0.5 * (np.eye(N, k=1) + np.eye(N, k=-1)) + 0.2 * np.eye(N, k=3)
    A += np.diag(rng.random(N))
    b = rng.standard_normal(N)
    la = hf.HipLinAlgebra(hf.HipOpts(rtol=1e-11, maxits=2000, restart=restart))
    la.initialize()
    la.configure()
    la.allocate(N)
    for i in range(N):
        cols = np.nonzero(A[i])[0]
        la.setValsMatrix([i], cols, A[i, cols])
    la.setValsRHS(np.arange(N), b)
    la.assemble()
    x = np.array(la.solve())
    its, reason, rel = la.last_info
    assert reason == 2 and rel <= 1e-11
    ref = np.linalg.solve(A, b)
    assert np.linalg.norm(x - ref) <= np.linalg.cond(A) * 1e-11 * np.linalg.norm(ref)
    # a second solve of the same handle repeats the first bit for bit
    assert np.array_equal(np.array(la.solve()), x) and la.last_info[0] == its
    if its > 3:
        la.options.maxits = its - 1
        la.configure()
        la.solve()
        assert la.last_info[:2] == (its - 1, -3) and la.last_info[2] > 1e-11


@pytest.mark.parametrize('restart', [8, 9, 16, 17, 24, 33, 63])
def test_gmres_cycles_longer_than_a_chunk(restart):
    """Cycles that end on either side of a chunk of basis rows (8 in the product, 8 or 16 in the orthogonalisation) and
    run through several of them, on a five-point Laplacian that needs more steps than a cycle has."""
    print('gmres long', restart, flush=True)
    n = 40
    T = 2.0 * np.eye(n) - np.eye(n, k=1) - np.eye(n, k=-1)
    A = np.kron(T, np.eye(n)) + np.kron(np.eye(n), T) + np.diag(1e-5 * np.arange(n * n))
    b = np.random.default_rng(5).standard_normal(n * n)
    la = hf.HipLinAlgebra(hf.HipOpts(rtol=1e-10, maxits=5000, restart=restart))
    la.initialize()
    la.configure()
    la.allocate(n * n)
    for i in range(n * n):
        cols = np.nonzero(A[i])[0]
        la.setValsMatrix([i], cols, A[i, cols])
    la.setValsRHS(np.arange(n * n), b)
    la.assemble()
    x = np.array(la.solve())
    its, reason, rel = la.last_info
    assert its > restart  # a whole cycle ran
    assert reason == 2 and rel <= 1e-10
    ref = np.linalg.solve(A, b)
    assert np.linalg.norm(x - ref) <= np.linalg.cond(A) * 1e-10 * np.linalg.norm(ref)


def host_gmres(A, dinv, b, m, steps):
    """Right-preconditioned GMRES(m) from zero for `steps` steps, Gram-Schmidt twice; the iterate."""
    x, done = np.zeros_like(b), 0
    while done < steps:
        k = min(m, steps - done)
        r = b - A @ x
        beta = np.linalg.norm(r)
        V, H = np.zeros((k + 1, b.size)), np.zeros((k + 1, k))
        V[0] = r / beta
        for j in range(k):
            w = A @ (dinv * V[j])
            for _ in range(2):
                h = V[:j + 1] @ w
                w -= h @ V[:j + 1]
                H[:j + 1, j] += h
            H[j + 1, j] = np.linalg.norm(w)
            V[j + 1] = w / H[j + 1, j]
        y = np.linalg.lstsq(H, beta * np.eye(k + 1)[0], rcond=None)[0]
        x += dinv * (y @ V[:k])
        done += k
    return x


@pytest.mark.parametrize('n,restart,steps', [(73, 30, 34), (75, 30, 34), (75, 63, 45), (294, 12, 14), (298, 30, 34),
                                             (298, 63, 45)])
def test_gmres_on_long_vectors(n, restart, steps):
    """Row blocks (256 rows) on both sides of the sizes where the sums over the blocks are reduced by a kernel of their
    own: V^T w above 128 (n = 73: 127, 75: 134), ||w||^2 too above 2,048 (n = 294: 2,031, 298: 2,086); cycles of more
    than 32 columns, and a step budget that ends inside a cycle.  The residual that the solver reports is the one of
    the solution it returns, and is the least that so many steps can reach, as found on the host: the residual of a
    GMRES iterate is within a small multiple of k^(3/2) eps (|| |A| |x| || + ||b||) of that."""
    print('gmres long vectors', n, restart, steps, flush=True)
    import scipy.sparse as sp
    w, prob = problem(2, 1, n)
    prob.set_krylov(hf.KRYLOV_FGMRES)
    its, reason, rel = prob.solve(pc=hf.PC_JACOBI, rtol=1e-14, maxits=steps, restart=restart)
    assert (its, reason) == (steps, -3)
    rowptr, cols, vals, b = prob.trace_csr()
    A = sp.csr_matrix((vals, cols, rowptr))
    x = prob.solution()[2]
    nb = np.linalg.norm(b)
    eps = EPS * (np.linalg.norm(abs(A) @ np.abs(x)) + nb) / nb
    assert abs(np.linalg.norm(b - A @ x) / nb - rel) <= 8 * eps
    ref = host_gmres(A, 1.0 / A.diagonal(), b, restart, steps)
    assert abs(np.linalg.norm(b - A @ ref) / nb - rel) <= 8 * steps ** 1.5 * eps


@pytest.mark.parametrize('ordering', [hf.linalg.PC_ILU0, hf.linalg.PC_ILU0_NATURAL], ids=['multicolour', 'natural'])
@pytest.mark.parametrize('pattern', ['diagonal', 'one-way', 'lower', 'chain', 'dense'])
def test_ilu_sweeps_on_odd_patterns(pattern, ordering):
    """Patterns whose levels are degenerate: no off-diagonal entry at all (one level each way), entries without their
    mirror image (a row that no row follows but a later row reads), a triangular matrix, a tridiagonal one and a dense
    one.  No fill is dropped on any of them, so the preconditioner is the inverse and the solver stops within a few
    steps (checked every 8) at the dense solution."""
    print('ilu sweeps', pattern, ordering, flush=True)
    rng = np.random.default_rng(3)
    N = 41
    A = np.diag(2.0 + rng.random(N))
    if pattern == 'one-way':
        A[1::3, 0] = 0.3
        A[2::3, 1] = 0.2
    elif pattern == 'lower':
        A += 0.02 * np.tril(rng.random((N, N)), -1)
    elif pattern == 'chain':
        A += 0.4 * np.eye(N, k=1) + 0.3 * np.eye(N, k=-1)
    elif pattern == 'dense':
        A += 0.02 * rng.random((N, N))
    b = rng.standard_normal(N)
    la = hf.HipLinAlgebra(hf.HipOpts(solverType=hf.linalg.BCGS, preconditionnerType=ordering, rtol=1e-12, maxits=64))
    la.initialize()
    la.configure()
    la.allocate(N)
    for i in range(N):
        cols = np.nonzero(A[i])[0]
        la.setValsMatrix([i], cols, A[i, cols])
    la.setValsRHS(np.arange(N), b)
    la.assemble()
    x = np.array(la.solve())
    its, reason, rel = la.last_info
    ref = np.linalg.solve(A, b)
    assert reason == 2 and rel <= 1e-12
    if pattern != 'chain' or ordering == hf.linalg.PC_ILU0_NATURAL:  # a recoloured chain drops fill
        assert its <= 8
    assert np.linalg.norm(x - ref) <= np.linalg.cond(A) * 1e-12 * np.linalg.norm(ref)
