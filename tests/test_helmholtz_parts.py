"""The Helmholtz translations of the FP32 engine: one real operator for both
parts of a split expansion (CPU: the operators are block diagonal), and the
mixed engine against the FP64 engine, whose translations stay (2 p^2)^2."""
import numpy as np
import pytest

import old_fmm_bem_amd as F
from conftest import rel_l2


@pytest.mark.parametrize("p", [4, 8, 12])
@pytest.mark.parametrize("kappa", [0.01, 0.6, 2.45])
def test_translations_are_one_real_operator(p, kappa):
    P2 = p * p
    for kind in (6, 7):
        for o in range(8):
            A = F.operator(p, "exact", kind, o, rb=kappa)
            # the projections' rounding: 1e-12 of the largest element
            tol = 1e-12 * np.abs(A).max()
            assert np.abs(A[:P2, :P2] - A[P2:, P2:]).max() <= tol
            assert np.abs(A[:P2, P2:]).max() <= tol and np.abs(A[P2:, :P2]).max() <= tol


# one box, leaf levels above and at the deepest translation chains, a surface
# (empty octants), every order built
@pytest.mark.gpu
@pytest.mark.parametrize("p,lmax,n,surface", [(4, 3, 1, False), (6, 3, 500, False), (8, 5, 6000, False),
                                              (10, 4, 20000, False), (12, 5, 20000, True)])
def test_mixed_matches_fp64(p, lmax, n, surface):
    rng = np.random.default_rng(p)
    x = rng.random((n, 3))
    if surface:
        x = x - 0.5
        x = 0.5 + 0.45 * x / np.linalg.norm(x, axis=1, keepdims=True)
    x = x.astype(np.float32)
    xj = x if n > 1 else rng.random((300, 3)).astype(np.float32)
    q = (rng.uniform(-1, 1, len(xj)) + 1j * rng.uniform(-1, 1, len(xj))).astype(np.complex64)
    out, pairs = [], []
    for prec in ("mixed", "fp64"):
        f = F.FMM(p=p, lmax=lmax, precision=prec, convention="exact", box=(0, 0, 0, 1), k=7.0)
        f.set_points(x, xj)
        out.append(f.evaluate(q, neq=F.HELMHOLTZ)[0])
        pairs.append(f.stats()["m2l_pairs"])
        f.close()
    print(p, lmax, n, pairs, flush=True)
    assert pairs[0] == pairs[1]
    # FP32 rounding of harmonics, radial weights, translations and near field
    # (hardware sine and cosine): a few times 1e-6 of the potential's norm
    assert rel_l2(out[0], out[1]) < 5e-6
