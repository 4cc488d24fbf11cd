"""The exact Boys function at the edges of the octave grid of orders 0 and 1."""
import numpy as np
import pytest

import oracle as O
from rchem_amd import basis as rb
from rchem_amd._lib import BOYS_EXACT, default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edge", [0.0625, 1.0, 3.9375, 4.0, 8.0, 12.0, 12.25, 27.75, 28.0, 35.5])
def test_cell_edges_through_eris_vs_oracle(gpu_ctx, edge):
    """Cells double in width at T = 4, 12 and 28; T on an edge, an ulp or so to
    either side (the row and the offset must change together), and at the two
    neighbouring cells' centres.  One-primitive shells (exponent 1/2) give
    (s s|s s) at T and (p s|s s), whose order-1 pass takes F_0 and F_1 from one
    polynomial.  Bar: 1e-12 relative to the oracle's exact mode, the bar of the
    uniform grid's edges (T itself carries a few ulps, F_m ~ T^-(m + 1/2))."""
    width = 0.0625 if edge < 4 else 0.125 if edge < 12 else 0.25 if edge < 28 else 0.5
    T = np.array([edge * (1 - 4e-16), edge, edge * (1 + 4e-16), edge + width / 2,
                  edge - width / 4])
    xs = np.sqrt(2.0 * T)
    centres, ls = [[0.0, 0.0, 0.0]], [0]
    for x in xs:
        centres += [[x, 0.0, 0.0], [x, 0.0, 0.0]]
        ls += [0, 1]
    centres, ls = np.array(centres), np.array(ls, dtype=np.int32)
    npr, ex, cf = np.ones(len(ls), dtype=np.int32), np.full(len(ls), 0.5), np.ones(len(ls))
    print(f"case: Boys cell edge T = {edge}", flush=True)
    B = rb.Basis.from_shells(centres, ls, npr, ex, cf, ctx=gpu_ctx)
    q = [r for k in range(len(T)) for r in ((1 + 2 * k, 1 + 2 * k, 0, 0), (2 + 2 * k, 1 + 2 * k, 0, 0))]
    blocks = rb.eri_shell_quartets(B, np.array(q, dtype=np.int32),
                                   default_opts(boys_mode=BOYS_EXACT, schwarz_thresh=0.0))
    Bo = O.cgtos_from_shells(centres, ls, npr, ex, cf)
    f0 = np.concatenate([[0], np.cumsum((ls + 1) * (ls + 2) // 2)])
    for r, blk in zip(q, blocks):
        ref = np.array([O.contracted_eri(Bo, f0[r[0]] + a, f0[r[1]], f0[r[2]], f0[r[3]],
                                         boys=O.BOYS_EXACT) for a in range(blk.shape[0])])
        assert np.abs(blk.reshape(-1) - ref).max() <= 1e-12 * np.abs(ref).max()
