"""Fock builds small enough to be planned in one launch, against the digestion
of the integral tensor."""
import numpy as np
import pytest

from rchem_amd import basis as rb
from rchem_amd._lib import PREC_MIXED, default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ls, npr", [
    ([0], [1]),                                  # one unit, one task
    ([0] * 5, [2] * 5),                          # 15 units: a block's 16 groups but one
    ([0] * 5 + [1], [1] * 6),                    # 15, 5 and 1: a block across classes
    ([0] * 6, [1, 2, 3, 4, 5, 6]),               # 18 buckets: more than a group's 16 lanes
    ([0] * 16 + [1] * 2, [3] * 8 + [1] * 10),    # 136 kets: three tiles to a bucket
])
@pytest.mark.parametrize("mixed", [None, 1e30, 1e-2, 1e-300])
def test_direct_plan_vs_tensor(gpu_ctx, ls, npr, mixed):
    """FP64, and mixed builds with every, some and no quartet in FP32.  Bars: 1e-12
    of the largest element (some hundred terms at 1e-14) in FP64, 2e-5 of it with
    FP32 quartets (integrals at ~1e-6 relative, some tens summed)."""
    rng = np.random.default_rng(len(ls))
    ls, npr = np.array(ls, dtype=np.int32), np.array(npr, dtype=np.int32)
    B = rb.Basis.from_shells(rng.uniform(-2.0, 2.0, (len(ls), 3)), ls, npr,
                             np.exp(rng.uniform(np.log(0.2), np.log(9.0), npr.sum())),
                             rng.uniform(0.1, 1.0, npr.sum()), ctx=gpu_ctx)
    D = rng.standard_normal((B.nbf, B.nbf))
    D = D + D.T
    Jo, Ko = rb.JK_inmem(rb.build_I(B), D)
    o = default_opts(schwarz_thresh=0.0)
    if mixed is not None:
        o.precision, o.mixed_thresh = PREC_MIXED, mixed
    for _ in range(2):  # the counters start anew
        J, K = np.zeros_like(D), np.zeros_like(D)
        print(f"case: l {ls.tolist()}, {npr.tolist()} primitives, mixed {mixed}", flush=True)
        rb.JK_direct(J, K, B, D, o)
        for a, b in ((J, Jo), (K, Ko)):
            bar = 1e-12 if mixed in (None, 1e-300) else 2e-5
            assert np.abs(a - b).max() <= bar * max(1.0, np.abs(b).max())
