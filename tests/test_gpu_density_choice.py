"""The two ways to a density: purify = 0 is the eigensolver in every iteration,
purify = 1 products where F' has a gap, each against an extended-precision
projector; and the products' routes that other tests are too small for."""
import numpy as np
import pytest

from rchem_amd import basis as rb
from rchem_amd._lib import default_opts
from rchem_amd.inputs import nocc_of, water_cluster

pytestmark = pytest.mark.gpu

LD = np.longdouble


def _projector(H, S, nocc):
    """C_occ C_occ^T of H C = S C eps in extended precision, and the same from
    numpy's eigenvectors: of C orthonormalised, the occupied-virtual block of
    C^T H C removed to first order, three times."""
    n = len(H)
    w, U = np.linalg.eigh(S)
    X = (U / np.sqrt(w)) @ U.T
    C = X @ np.linalg.eigh(X.T @ H @ X)[1]
    D0 = C[:, :nocc] @ C[:, :nocc].T
    Hl, Sl, one, Q = H.astype(LD), S.astype(LD), np.eye(n, dtype=LD), C.astype(LD)
    for last in (False, False, False, True):
        for _ in range(2):
            Q = Q @ (LD(1.5) * one - LD(0.5) * (Q.T @ (Sl @ Q)))
        if last:
            break
        A = Q.T @ (Hl @ Q)
        e = np.diag(A)
        R = np.zeros((n, n), dtype=LD)
        R[nocc:, :nocc] = A[nocc:, :nocc] / (e[None, :nocc] - e[nocc:, None])
        R[:nocc, nocc:] = -R[nocc:, :nocc].T
        Q = Q + Q @ R
    return Q[:, :nocc] @ Q[:, :nocc].T, D0


@pytest.mark.parametrize("dims, basis", [((1, 1, 1), "STO-3G"), ((1, 1, 1), "6-31G"),
                                         ((1, 2, 2), "STO-3G"), ((2, 2, 2), "6-31G"),
                                         ((2, 2, 3), "6-31G")])
def test_both_ways_against_extended_precision(gpu_ctx, dims, basis):
    """The density of a core guess (nuclei screened to 5.2 and 0.75, which gives a
    gap of a molecule's size): n = 7 to 156, the one-launch kernel and the step
    kernels.  Bar: 16 times what numpy's eigenvectors are off on the same matrices.
    All of them err by roundings of S^(-1/2) and F' amplified by 1 / gap, and the
    squarings by eps / gap_k, the gap after step k growing by 1.2 or more a step:
    six such terms at most; the factor leaves two for the rest.  And the two ways
    are two: their last bits differ."""
    Z, xyz = water_cluster(dims=dims, seed=2)
    Zs = np.where(np.array(Z) == 8, 5.2, 0.75)
    B = rb.Basis.new(Z, xyz, basis, ctx=gpu_ctx)
    S, T, V = rb.one_electron(B, xyz, Zs)
    exact, D0 = _projector(T + V, S, nocc_of(Z))
    bar = 16 * max(float(np.abs(D0 - exact).max()), 16 * np.finfo(float).eps)
    D = {}
    for purify in (False, True):
        print(f"case: core guess, n = {B.nbf}, purify {purify}", flush=True)
        _, D[purify] = rb.scf(B, xyz, Zs, nocc=nocc_of(Z), max_iter=0, opts=default_opts(),
                              purify=purify)
        assert float(np.abs(D[purify] - exact).max()) <= bar
    assert np.any(D[False] != D[True])


def _row(n):
    """H2 molecules in a row, a He in front where n is odd: n s functions, a gap of 0.5."""
    Z, x = ([2.0], [-6.0]) if n % 2 else ([], [])
    for k in range(n // 2):
        Z += [1.0, 1.0]
        x += [5.0 * k, 5.0 * k + 1.4]
    xyz = np.zeros((n, 3))
    xyz[:, 0] = x
    return np.array(Z), xyz, int(sum(Z)) // 2


def _row_basis(ctx, Z, xyz):
    n, one = len(Z), np.ones(len(Z))
    return rb.Basis.from_shells(xyz, np.zeros(n, dtype=np.int32), one.astype(np.int32),
                                np.where(Z > 1, 1.3, 0.45), one, ctx=ctx)


@pytest.mark.parametrize("n", [831, 832, 833, 1025])
def test_the_step_kernels_end_and_beyond(gpu_ctx, n):
    """The largest matrices of the step kernels, and the library's products above
    them.  Bar: 1e-11 (n eps ||F'|| / gap is 2e-12, ||F'|| ~ 5, gap ~ 0.5)."""
    Z, xyz, nocc = _row(n)
    B = _row_basis(gpu_ctx, Z, xyz)
    print(f"case: core guess of {n} functions by products", flush=True)
    _, D = rb.scf(B, xyz, Z, nocc=nocc, max_iter=0, opts=default_opts(), purify=True)
    S, T, V = rb.one_electron(B, xyz, Z)
    w, U = np.linalg.eigh(S)
    X = (U / np.sqrt(w)) @ U.T
    C = X @ np.linalg.eigh(X @ (T + V) @ X)[1][:, :nocc]
    assert np.abs(D - C @ C.T).max() < 1e-11


@pytest.mark.parametrize("n", [128, 130, 257, 834])
def test_whole_iteration_graph(gpu_ctx, n):
    """DIIS with purified densities replayed as one graph against the same kernel by
    kernel: one launch, the step kernels, and the library's products (n = 834) in
    the captured iteration.  Both stop at |dE| < 1e-10 and a commutator below 1e-8,
    after which energies agree to 1e-9 and densities to 1e-7."""
    Z, xyz, nocc = _row(n)
    B = _row_basis(gpu_ctx, Z, xyz)
    out = []
    for graph in (False, True):
        print(f"case: {n} functions, DIIS(6), purified, graph {graph}", flush=True)
        out.append(rb.scf(B, xyz, Z, nocc=nocc, thresh_e=1e-10, max_iter=40, diis=6,
                          opts=default_opts(), purify=True, graph=graph))
    (r0, D0), (r1, D1) = out
    assert r0.converged and r1.converged and r1.graph_iterations > 0
    assert abs(r0.e_total - r1.e_total) < 1e-9 and np.abs(D0 - D1).max() < 1e-7


@pytest.mark.parametrize("purify", [False, True])
@pytest.mark.parametrize("reps", [1, 50])
def test_no_gap_over_iterations(gpu_ctx, purify, reps):
    """Three H atoms on a triangle (50 of them far apart), two orbitals occupied of
    which one is of a degenerate pair: the eigensolver forms the densities for
    either option, in the first iteration and in those after it.  Tr(D S) = 2 and
    idempotent, bar 1e-10 (the eigensolver's C^T S C = 1, n = 150)."""
    xyz = np.concatenate([np.array([[0, 0, 0], [2, 0, 0], [1, 3 ** 0.5, 0]]) + [0, 0, 40.0 * k]
                          for k in range(reps)])
    n = len(xyz)
    one = np.ones(n)
    B = rb.Basis.from_shells(xyz, np.zeros(n, dtype=np.int32), one.astype(np.int32), 0.5 * one,
                             one, ctx=gpu_ctx)
    S = rb.S(B)
    for it in (0, 1, 3):
        print(f"case: no gap, {n} functions, {it} iterations, purify {purify}", flush=True)
        _, D = rb.scf(B, xyz, one, nocc=2 * reps, max_iter=it, opts=default_opts(), purify=purify)
        assert abs(np.trace(D @ S) - 2 * reps) < 1e-10 * reps
        assert np.abs(D @ S @ D - D).max() < 1e-10
