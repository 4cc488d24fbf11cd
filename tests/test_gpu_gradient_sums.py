"""The one-electron gradient's workgroup sums: several passes of the grid."""
import numpy as np
import pytest

from rchem_amd import basis as rb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 50])
def test_gradient_of_far_molecules(gpu_ctx, count):
    """count H2 molecules 60 bohr apart (50: 505 000 pairs x nuclei, twice what the
    grid holds): each has the gradient of one, to 1e-7 (quadrupoles at 60 bohr act
    below 1e-9, the SCF's threshold of 1e-12 leaves about 1e-7)."""
    def run(k):
        xyz = np.array([[60.0 * (i // 2), 0.1 * (i % 2), 0.6 + 1.5 * (i % 2)] for i in range(2 * k)])
        Z = np.ones(2 * k, dtype=int)
        B = rb.Basis.new(Z, xyz, "STO-3G", ctx=gpu_ctx)
        print(f"case: {k} molecules", flush=True)
        res, g = rb.rhf_gradient(B, xyz, Z, nocc=k, thresh_e=1e-12, diis=8)
        assert res.converged
        return np.asarray(g).reshape(-1, 3)
    one = run(1)
    assert np.abs(one.sum(axis=0)).max() <= 1e-9
    assert np.abs(run(count).reshape(count, 2, 3) - one).max() <= 1e-7
