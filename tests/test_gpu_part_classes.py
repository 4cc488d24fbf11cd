"""Fock builds of the classes whose targets are formed in parts ((dp|pp) ...
(dd|dd)) against the in-memory digestion of the integral tensor and against the
build without those kernels."""
import numpy as np
import pytest

from rchem_amd import basis as rb
from rchem_amd._lib import default_opts

pytestmark = pytest.mark.gpu


def _basis(ctx, ls, nmax, spread, seed):
    rng = np.random.default_rng(seed)
    ls = np.array(ls, dtype=np.int32)
    npr = rng.integers(1, nmax + 1, len(ls)).astype(np.int32)
    xyz = rng.uniform(-spread, spread, (len(ls), 3))
    ex = np.exp(rng.uniform(np.log(0.2), np.log(5.0), npr.sum()))
    return rb.Basis.from_shells(xyz, ls, npr, ex, rng.uniform(0.1, 1.0, npr.sum()), ctx=ctx)


def _build(B, D):
    J, K = np.zeros_like(D), np.zeros_like(D)
    rb.JK_direct(J, K, B, D, default_opts(schwarz_thresh=0.0))
    return J, K


def _density(n):
    D = np.random.default_rng(5).standard_normal((n, n))
    return D + D.T


@pytest.mark.parametrize("lds", ["1", "0"])
@pytest.mark.parametrize("ls", [
    [2],                       # one quartet
    [2, 1],                    # every class once or twice
    [2, 2, 1, 1, 1],           # a few lanes of each tile
    [2] * 7 + [1] * 4,         # 28 (dd| and (dp| kets, 10 (pp|: a tile that is short
    [2] * 4 + [1] * 10 + [0],  # 55 (pp|, 40 (dp|
    [2] * 5 + [1] * 13,        # 91 (pp| and 65 (dp|: a tile and a few
])
def test_vs_tensor(monkeypatch, ls, lds):
    """K rows in LDS (lds = 1) or by atomics in memory, every pair kept.  Bar: the
    two sum the same integrals, each good to 1e-12 of the Schwarz bound that holds
    for it (the d-class recurrences lose up to two digits of it), in another order."""
    monkeypatch.setenv("RCHEM_LDS_DIGESTION", lds)
    print(f"case: l {ls}, LDS digestion {lds}", flush=True)
    ctx = rb.Context(0)
    B = _basis(ctx, ls, 3, 1.5, len(ls))
    D = _density(B.nbf)
    I = rb.build_I(B)
    Q = np.sqrt(np.abs(np.einsum("ijij->ij", I.reshape((B.nbf,) * 4))))
    J, K = _build(B, D)
    Jo, Ko = rb.JK_inmem(I, D)
    A = np.abs(D)
    assert np.all(np.abs(J - Jo) <= 1e-12 * (Q * (Q * A).sum() + 1e-3))
    assert np.all(np.abs(K - Ko) <= 1e-12 * (Q @ A @ Q + 1e-3))
    ctx.close()


@pytest.mark.parametrize("ns", [300, 700, 1500])
def test_rows_beyond_lds(monkeypatch, ns):
    """Many far s functions: the K and D rows of a bra, then the K rows alone, then
    neither fit the LDS.  Bar: 1e-11 of the largest element (100 terms at 1e-13)."""
    out = []
    for stream in ("1", "0"):
        monkeypatch.setenv("RCHEM_ERI_STREAM", stream)
        print(f"case: {ns} s shells, {stream}", flush=True)
        ctx = rb.Context(0)
        rng = np.random.default_rng(ns)
        ls = np.array([2, 2, 2, 1, 1, 1] + [0] * ns, dtype=np.int32)
        xyz = rng.uniform(-1.0, 1.0, (len(ls), 3))
        xyz[6:, 0] = 12.0 * (1 + np.arange(ns))  # no pair of them overlaps
        one = np.ones(len(ls))
        B = rb.Basis.from_shells(xyz, ls, one.astype(np.int32), rng.uniform(0.4, 0.9, len(ls)),
                                 one, ctx=ctx)
        D = _density(B.nbf)
        J, K = np.zeros_like(D), np.zeros_like(D)
        rb.JK_direct(J, K, B, D)
        out.append((J, K))
        ctx.close()
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()
