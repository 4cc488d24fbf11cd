"""Sizes at which a call takes another path than the small ones other tests run."""
import numpy as np
import pytest

from rchem_amd import basis as rb
from rchem_amd.inputs import WATER_CRAWFORD, WATER_Z, water_cluster

pytestmark = pytest.mark.gpu


def _water_among(ctx, nuclei):
    """The gradient of water among `nuclei` nuclei in all: 97 small charges around it,
    the rest of charge 0."""
    rng = np.random.default_rng(9)
    v = rng.standard_normal((2500, 3))  # the same for every count
    v *= (rng.uniform(6.0, 40.0, 2500) / np.linalg.norm(v, axis=1))[:, None]
    xyz = np.concatenate([np.array(WATER_CRAWFORD, dtype=float).reshape(-1, 3), v[:nuclei - 3]])
    Z = np.zeros(nuclei)
    Z[:3] = WATER_Z
    Z[3:100] = 1e-3 * np.random.default_rng(4).uniform(-1.0, 1.0, 97)
    B = rb.Basis.new(WATER_Z, xyz[:3], "STO-3G", ctx=ctx)
    res, g = rb.rhf_gradient(B, xyz, Z, nocc=5, thresh_e=1e-12, diis=8)
    assert res.converged
    return np.asarray(g).reshape(-1, 3)


@pytest.mark.parametrize("nuclei", [1000, 1800, 2048, 2049, 2500])
def test_gradient_among_many_nuclei(gpu_ctx, nuclei):
    """One-electron gradients whose workgroup sums take up to 48 KB of LDS, with the
    Boys table more than 64 KB (from 1800 nuclei), and beyond 2048 nuclei go to
    memory.  Nuclei without charge change nothing: the other forces are those
    among 100 nuclei, to 1e-8 (two SCFs stopped at a commutator of 1e-8 or less)."""
    print(f"case: water among {nuclei} nuclei", flush=True)
    few, many = _water_among(gpu_ctx, 100), _water_among(gpu_ctx, nuclei)
    assert np.abs(few[3:]).max() > 1e-6
    assert np.abs(many[:100] - few).max() <= 1e-8
    assert np.abs(many[100:]).max() == 0.0


def test_batch_beyond_the_one_launch_densities(gpu_ctx):
    """A molecule of 143 functions: the whole batch by the eigensolver, until only
    the small ones are left.  Bar 1e-9 Eh: two SCFs that both stop at |dE| < 1e-11."""
    mols = []
    for k, (dims, count) in enumerate([((1, 1, 1), 1), ((2, 2, 3), 11), ((1, 1, 2), 2)]):
        Z, xyz = water_cluster(dims=dims, seed=k)
        mols.append((list(Z[:3 * count]), xyz[:3 * count]))
    print("case: batch of 13, 143 and 26 functions", flush=True)
    res = rb.batch_scf(mols, "6-31G", thresh_e=1e-11, diis=8, ctx=gpu_ctx)
    for (Z, xyz), r in zip(mols, res):
        B = rb.Basis.new(Z, xyz, "6-31G", ctx=gpu_ctx)
        one, _ = rb.scf(B, xyz, Z, nocc=sum(Z) // 2, diis=8)
        assert r.converged and one.converged and abs(r.e_total - one.e_total) < 1e-9
