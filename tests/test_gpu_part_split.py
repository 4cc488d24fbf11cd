"""Partwise Fock builds ((dp|pp) ... (dd|dd)) of so few quartets that their tiles
are split over the primitives, against the digested integral tensor."""
import numpy as np
import pytest

from rchem_amd import basis as rb
from rchem_amd._lib import PREC_MIXED, default_opts

pytestmark = pytest.mark.gpu


def _basis(ctx, ls, npr):
    rng = np.random.default_rng(sum(npr) + len(ls))
    ls, npr = np.array(ls, dtype=np.int32), np.array(npr, dtype=np.int32)
    ex = np.exp(rng.uniform(np.log(0.2), np.log(5.0), npr.sum()))
    return rb.Basis.from_shells(rng.uniform(-1.0, 1.0, (len(ls), 3)), ls, npr, ex,
                                rng.uniform(0.1, 1.0, npr.sum()), ctx=ctx)


@pytest.mark.parametrize("ls, npr", [
    ([2], [8]),                       # 64 primitive pairs a side, one quartet
    ([2, 1], [8, 7]),                 # 64, 56 and 49 against limits of 8 to 32
    ([2, 1, 1], [3, 1, 5]),           # 9, 3, 15, 1, 5 and 25: remainders on both sides
    ([2, 2, 1, 1], [6, 1, 2, 3]),     # split and whole quartets in one class
    ([2, 2, 2, 1, 1, 1], [5] * 6),    # tiles of several quartets
    ([2, 1], [1, 1]),                 # nothing to split
])
@pytest.mark.parametrize("mixed", [False, True])
def test_split_vs_tensor(gpu_ctx, ls, npr, mixed):
    """FP64 bar: the two sum the same integrals, each good to 1e-12 of the Schwarz
    bound that holds for it (the d-class recurrences lose up to two digits), in
    another order.  Mixed, every quartet in FP32: 2e-5 of the largest element (FP32
    integrals at ~1e-6 relative, some tens summed)."""
    B = _basis(gpu_ctx, ls, npr)
    n = B.nbf
    D = np.random.default_rng(5).standard_normal((n, n))
    D = D + D.T
    I = rb.build_I(B)
    Jo, Ko = rb.JK_inmem(I, D)
    o = default_opts(schwarz_thresh=0.0)
    if mixed:
        o.precision, o.mixed_thresh = PREC_MIXED, 1e30
    J, K = np.zeros_like(D), np.zeros_like(D)
    print(f"case: l {ls}, {npr} primitives, mixed {mixed}", flush=True)
    rb.JK_direct(J, K, B, D, o)
    if mixed:
        for a, b in ((J, Jo), (K, Ko)):
            assert np.abs(a - b).max() <= 2e-5 * np.abs(b).max()
        return
    Q = np.sqrt(np.abs(np.einsum("ijij->ij", I.reshape((n,) * 4))))
    A = np.abs(D)
    assert np.all(np.abs(J - Jo) <= 1e-12 * (Q * (Q * A).sum() + 1e-3))
    assert np.all(np.abs(K - Ko) <= 1e-12 * (Q @ A @ Q + 1e-3))
    if ls == [2]:  # one quartet's 4096 primitive quartets, twice a compute unit's share a part
        st = rb.jk_last_stats(B)
        assert st.quartets == 1 and st.tiles == 128
