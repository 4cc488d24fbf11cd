"""Fock builds whose bra density rows are in LDS, in memory, or not digested in
LDS at all, against the digestion by global atomics."""
import numpy as np
import pytest

from rchem_amd import basis as rb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, lp", [(1, 0), (63, 0), (65, 0), (1700, 0), (2700, 0), (5000, 0),
                                   (30, 1), (1205, 1)])
def test_density_rows_vs_global_atomics(monkeypatch, n, lp):
    """A chain of one-primitive s shells 3 bohr apart (lp = 1: every fifth a p
    shell): n functions or so, few significant pairs.  The K and density rows of a
    bra take (NA + NB) n doubles each: both fit the LDS up to n ~ 2500 for
    (ss|ss), the K rows alone up to ~ 8700 (1205 shells with p: both for (ps|ss)
    only).  Bar: 1e-13 of the largest element, times the ~100 terms that an
    element sums in another order."""
    rng = np.random.default_rng(n)
    ls = np.array([lp if i % 5 == 0 else 0 for i in range(n)], dtype=np.int32)
    xyz = np.zeros((n, 3))
    xyz[:, 0] = 3.0 * np.arange(n) + rng.uniform(-0.2, 0.2, n)
    xyz[:, 1] = rng.uniform(-0.5, 0.5, n)
    one = np.ones(n)
    args = (xyz, ls, one.astype(np.int32), rng.uniform(0.4, 0.9, n), one)
    out = []
    for lds in ("1", "0"):
        monkeypatch.setenv("RCHEM_LDS_DIGESTION", lds)
        print(f"case: chain of {n} shells, LDS digestion {lds}", flush=True)
        ctx = rb.Context(0)
        B = rb.Basis.from_shells(*args, ctx=ctx)
        D = np.random.default_rng(7).standard_normal((B.nbf, B.nbf))
        D = D + D.T
        J, K = np.zeros_like(D), np.zeros_like(D)
        rb.JK_direct(J, K, B, D)
        out.append((J, K))
        ctx.close()
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()
