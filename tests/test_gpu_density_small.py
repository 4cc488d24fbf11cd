"""The densities formed by products (scf_density.hip) against numpy's eigenvectors."""
import numpy as np
import pytest

from rchem_amd import basis as rb
from rchem_amd._lib import default_opts

pytestmark = pytest.mark.gpu


def _system(n):
    """n one-function atoms: H2 molecules in a row, a He in front where n is odd."""
    rng = np.random.default_rng(n)
    Z, x = ([2], [-6.0]) if n % 2 else ([], [])
    for k in range(n // 2):
        Z += [1, 1]
        x += [5.0 * k, 5.0 * k + 1.4]
    xyz = np.zeros((n, 3))
    xyz[:, 0] = x
    xyz[:, 1:] = rng.uniform(-0.1, 0.1, (n, 2))
    return np.array(Z, dtype=float), xyz, (sum(Z)) // 2


@pytest.mark.parametrize("purify", [False, True])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 48, 49, 127, 128, 129, 160, 161, 255, 257])
def test_density_vs_eigenvectors(gpu_ctx, n, purify):
    """One plain iteration: D = the density of F(D_0), D_0 the core guess, at the
    edges of the kernel's 16-wide tiles and of its range (128), and above it at
    those of the step kernels' 32-wide tiles and 64-wide rows.  Bar: 1e-11 -- both ways leave the
    projector ~ n eps ||F'|| / gap off, ||F'|| ~ 5, gap ~ 0.5."""
    Z, xyz, nocc = _system(n)
    one = np.ones(n)
    B = rb.Basis.from_shells(xyz, np.zeros(n, dtype=np.int32), one.astype(np.int32),
                             np.where(Z > 1, 1.3, 0.45), one, ctx=gpu_ctx)
    print(f"case: density of {n} functions, purify {purify}", flush=True)
    o = default_opts()
    _, D = rb.scf(B, xyz, Z, nocc=nocc, max_iter=1, opts=o, purify=purify)
    S, T, V = rb.one_electron(B, xyz, Z)
    w, U = np.linalg.eigh(S)
    X = (U / np.sqrt(w)) @ U.T

    def density(F):
        C = X @ np.linalg.eigh(X.T @ F @ X)[1][:, :nocc]
        return C @ C.T

    J, K = np.zeros((n, n)), np.zeros((n, n))
    rb.JK_direct(J, K, B, density(T + V), o)
    assert np.abs(D - density(T + V + 2 * J - K)).max() < 1e-11


def test_batch_of_uneven_sizes(gpu_ctx):
    """The batched SCF's densities (one workgroup a molecule, sizes 7 to 63 in
    one launch) lead to the single molecules' energies: 1e-9 Eh, two SCFs that
    both stop at |dE| < 1e-11."""
    from rchem_amd.inputs import water_cluster
    mols = []
    for k, dims in enumerate([(1, 1, 1), (1, 1, 2), (1, 1, 3), (1, 2, 2), (3, 3, 1)]):
        mols.append(water_cluster(dims=dims, seed=k))
    res = rb.batch_scf(mols, "STO-3G", thresh_e=1e-11, diis=8, ctx=gpu_ctx)
    for (Z, xyz), r in zip(mols, res):
        B = rb.Basis.new(Z, xyz, "STO-3G", ctx=gpu_ctx)
        one, _ = rb.scf(B, xyz, Z, nocc=sum(Z) // 2, diis=8)
        assert r.converged and one.converged and abs(r.e_total - one.e_total) < 1e-9


def test_no_gap_takes_the_eigensolver(gpu_ctx):
    """Three H atoms on an equilateral triangle, two orbitals occupied: the
    second and third orbitals are degenerate, no projector of rank 2 is singled
    out and the eigensolver picks one: Tr(D S) = 2, idempotent.  Bar 1e-10."""
    for reps in (1, 50):  # 3 functions and 150 (far apart: 50-fold the same)
        xyz = np.concatenate([np.array([[0, 0, 0], [2, 0, 0], [1, 3 ** 0.5, 0]]) + [0, 0, 40.0 * k]
                              for k in range(reps)])
        n = len(xyz)
        one = np.ones(n)
        B = rb.Basis.from_shells(xyz, np.zeros(n, dtype=np.int32), one.astype(np.int32),
                                 0.5 * one, one, ctx=gpu_ctx)
        print(f"case: no gap, {n} functions", flush=True)
        _, D = rb.scf(B, xyz, one, nocc=2 * reps, max_iter=1, opts=default_opts())
        S = rb.S(B)
        assert abs(np.trace(D @ S) - 2 * reps) < 1e-10 * reps
        assert np.abs(D @ S @ D - D).max() < 1e-10
