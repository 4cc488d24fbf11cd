"""Fock builds whose tiles are split over the primitives, against the oracle."""
import numpy as np
import pytest

import oracle as O
from rchem_amd import basis as rb
from rchem_amd._lib import BOYS_EXACT, PREC_MIXED, default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ls, npr", [
    ([0, 0, 0], [8, 8, 8]),     # 64 primitive pairs a side: the most a record holds
    ([0, 0, 1], [1, 7, 7]),     # 1, 7 and 49: remainders on both sides
    ([1, 1], [5, 3]),           # 25, 15 and 9 against a limit of 4
    ([2, 0], [4, 6]),           # d classes: per-lane kernels and the engines that take no part
    ([1, 0], [1, 1]),           # one primitive quartet: nothing to split
])
@pytest.mark.parametrize("mixed", [False, True])
def test_split_builds_vs_oracle(gpu_ctx, ls, npr, mixed):
    """So little work that every class is cut to its shortest parts.  Bars: FP64
    1e-11 (the d-class parity bar); mixed, every quartet in FP32, 2e-5 of the
    largest element (FP32 integrals at ~1e-6 relative, some tens summed)."""
    rng = np.random.default_rng(sum(npr))
    ls, npr = np.array(ls, dtype=np.int32), np.array(npr, dtype=np.int32)
    centres = rng.uniform(-1.0, 1.0, (len(ls), 3))
    ex = np.exp(rng.uniform(np.log(0.2), np.log(20.0), npr.sum()))
    cf = rng.uniform(0.1, 1.0, npr.sum())
    B = rb.Basis.from_shells(centres, ls, npr, ex, cf, ctx=gpu_ctx)
    D = rng.standard_normal((B.nbf, B.nbf))
    D = D + D.T
    J, K = np.zeros_like(D), np.zeros_like(D)
    o = default_opts(schwarz_thresh=0.0)
    if mixed:
        o.precision, o.mixed_thresh = PREC_MIXED, 1e30
    print(f"case: l {ls.tolist()}, {npr.tolist()} primitives, mixed {mixed}", flush=True)
    rb.JK_direct(J, K, B, D, o)
    Jo, Ko = O.jk_inmem(O.eri_tensor(O.cgtos_from_shells(centres, ls, npr, ex, cf),
                                     boys=O.BOYS_EXACT), D)
    for a, b in ((J, Jo), (K, Ko)):
        bar = 2e-5 * np.abs(b).max() if mixed else 1e-11 * max(1.0, np.abs(b).max())
        assert np.abs(a - b).max() <= bar
