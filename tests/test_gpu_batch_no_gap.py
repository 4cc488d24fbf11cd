"""Batched SCFs with molecules whose F' has no gap (square H4: four electrons, its
second and third orbitals degenerate at the core guess): those alone go to the
eigensolver, and the others' results are their own."""
import numpy as np
import pytest

from rchem_amd import basis as rb
from rchem_amd.inputs import water_cluster

pytestmark = pytest.mark.gpu

SQUARE = ([1, 1, 1, 1], np.array([[0, 0, 0], [2.0, 0, 0], [2.0, 2.0, 0], [0, 2.0, 0]]))


def _waters(count, seed):
    Z, xyz = water_cluster(dims=(1, 1, count), seed=seed)
    return list(Z), xyz


@pytest.mark.parametrize("diis", [0, 8])
@pytest.mark.parametrize("order", ["first", "last", "between", "alone"])
def test_others_keep_their_results(gpu_ctx, order, diis):
    """Bar 1e-9 Eh: two SCFs that both stop at |dE| < 1e-11."""
    waters = [_waters(k, k) for k in (1, 2, 1, 3)]
    mols = {"first": [SQUARE, SQUARE] + waters, "last": waters + [SQUARE],
            "between": [waters[0], SQUARE, waters[1], SQUARE, waters[3]], "alone": [SQUARE] * 3}[order]
    print(f"case: {len(mols)} molecules, no gap {order}, DIIS {diis}", flush=True)
    res = rb.batch_scf(mols, "STO-3G", thresh_e=1e-11, max_iter=60, diis=diis, ctx=gpu_ctx)
    for (Z, xyz), r in zip(mols, res):
        assert np.isfinite(r.e_total)
        if len(Z) == 4:
            continue  # which of the degenerate orbitals is taken is not determined
        B = rb.Basis.new(Z, xyz, "STO-3G", ctx=gpu_ctx)
        one, _ = rb.scf(B, xyz, Z, nocc=sum(Z) // 2, thresh_e=1e-11, max_iter=60, diis=diis)
        assert r.converged and one.converged and abs(r.e_total - one.e_total) < 1e-9
