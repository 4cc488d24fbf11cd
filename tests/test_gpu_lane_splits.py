"""Tensor quartets on several lanes, nuclei over a pair's lanes, and the DIIS
solve for small and large subspaces, against the oracle."""
import numpy as np
import pytest

import oracle as O
from rchem_amd import basis as rb
from rchem_amd._lib import BOYS_EXACT, default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ls, npr", [
    ([0], [1]),                         # one lane: one ket primitive pair
    ([0, 0, 1], [1, 2, 3]),             # 1 .. 9 pairs: 1, 2, 4 and 8 lanes, remainders
    ([0, 1, 1, 0, 0], [1, 1, 3, 7, 2]),  # 15, 10 and 21 kets: tiles of 8 and a few
    ([2, 1, 0], [2, 1, 3]),             # d classes: per-lane and wave engines
])
def test_tensor_lanes_vs_oracle(gpu_ctx, ls, npr):
    """Bar: 1e-11 of the largest integral, the parity bar of the d classes."""
    rng = np.random.default_rng(len(ls))
    ls, npr = np.array(ls, dtype=np.int32), np.array(npr, dtype=np.int32)
    c = rng.uniform(-1.0, 1.0, (len(ls), 3))
    ex = np.exp(rng.uniform(np.log(0.2), np.log(20.0), npr.sum()))
    cf = rng.uniform(0.1, 1.0, npr.sum())
    B = rb.Basis.from_shells(c, ls, npr, ex, cf, ctx=gpu_ctx)
    print(f"case: l {ls.tolist()}, {npr.tolist()} primitives", flush=True)
    I = rb.build_I(B, default_opts(boys_mode=BOYS_EXACT))
    Io = O.eri_tensor(O.cgtos_from_shells(c, ls, npr, ex, cf), boys=O.BOYS_EXACT)
    assert np.abs(I - Io).max() <= 1e-11 * max(1.0, np.abs(Io).max())


@pytest.mark.parametrize("ls, npr", [
    ([0], [1]),
    ([0, 0, 1], [1, 2, 7]),              # 1 .. 49 pairs of primitives
    ([2, 1, 0, 0, 0, 0], [2, 1, 3, 3, 3, 3]),  # 10 (ss| pairs of one bucket: a tile and a few
])
def test_schwarz_lanes_vs_oracle(gpu_ctx, ls, npr):
    """Bar: 1e-11 of the largest integral on the squares of the bounds."""
    rng = np.random.default_rng(len(ls))
    ls, npr = np.array(ls, dtype=np.int32), np.array(npr, dtype=np.int32)
    c = rng.uniform(-1.0, 1.0, (len(ls), 3))
    ex = np.exp(rng.uniform(np.log(0.2), np.log(20.0), npr.sum()))
    cf = rng.uniform(0.1, 1.0, npr.sum())
    B = rb.Basis.from_shells(c, ls, npr, ex, cf, ctx=gpu_ctx)
    print(f"case: l {ls.tolist()}, {npr.tolist()} primitives", flush=True)
    Q = rb.schwarz(B)
    n = B.nbf
    I = np.asarray(O.eri_tensor(O.cgtos_from_shells(c, ls, npr, ex, cf),
                                boys=O.BOYS_EXACT)).reshape(n, n, n, n)
    d = np.abs(np.einsum("ijij->ij", I))
    f = np.concatenate([[0], np.cumsum((ls + 1) * (ls + 2) // 2)])
    for a in range(len(ls)):
        for b in range(a + 1):  # the lower triangle
            ref = d[f[a]:f[a + 1], f[b]:f[b + 1]].max()
            assert abs(Q[a, b] ** 2 - ref) <= 1e-11 * max(1.0, np.abs(I).max())


@pytest.mark.parametrize("nuclei", [0, 1, 7, 8, 9, 33])
def test_nuclei_over_lanes_vs_oracle(gpu_ctx, nuclei):
    """Bar: 1e-12 per nucleus of unit charge and a few of rounding in S and T."""
    rng = np.random.default_rng(nuclei)
    ls = np.array([0, 1, 2, 1, 0], dtype=np.int32)
    npr = np.array([3, 2, 1, 3, 1], dtype=np.int32)
    c = rng.uniform(-1.5, 1.5, (5, 3))
    ex = np.exp(rng.uniform(np.log(0.2), np.log(20.0), npr.sum()))
    cf = rng.uniform(0.1, 1.0, npr.sum())
    xyz, Z = rng.uniform(-3.0, 3.0, (nuclei, 3)), rng.integers(1, 9, nuclei).astype(float)
    B = rb.Basis.from_shells(c, ls, npr, ex, cf, ctx=gpu_ctx)
    print(f"case: {nuclei} nuclei", flush=True)
    got = rb.one_electron(B, xyz, Z)
    ref = O.one_electron(O.cgtos_from_shells(c, ls, npr, ex, cf), Z, xyz)
    for a, b in zip(got, ref):
        assert np.abs(a - b).max() <= 1e-12 * (1 + Z.sum()) * max(1.0, np.abs(ref[0]).max())


@pytest.mark.parametrize("k", [1, 2, 5, 31, 32])
def test_diis_subspaces(gpu_ctx, k):
    """The energy does not depend on the subspace: 1e-9 hartree at a threshold of 1e-11."""
    Z = np.array([8, 1, 1])
    xyz = np.array([[0.0, -0.1432, 0.0], [1.638, 1.1365, 0.0], [-1.638, 1.1365, 0.0]])
    B = rb.Basis.new(Z, xyz, "6-31G", ctx=gpu_ctx)
    ref, _ = rb.scf(B, xyz, Z, nocc=5, thresh_e=1e-11, diis=8)
    print(f"case: {k} vectors", flush=True)
    res, _ = rb.scf(B, xyz, Z, nocc=5, thresh_e=1e-11, diis=k)
    assert res.converged and abs(res.e_total - ref.e_total) <= 1e-9
