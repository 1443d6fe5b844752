"""The near field's work items: leaves of many targets split over workgroups,
fewer targets per item in large leaves and in small problems.  The mixed and
FP64 engines against the FP64 direct sum of the near field's own pairs: all
points in few leaves, where the near field is the whole sum."""
import numpy as np
import pytest

import old_fmm_bem_amd as F
from conftest import rel_l2

pytestmark = pytest.mark.gpu


# one leaf level-2 neighbourhood holds every point: targets per leaf below, at
# and above the item sizes (4, 8, 16, 32, 128, 256) and the 512-target rule
@pytest.mark.parametrize("n", [1, 5, 33, 129, 513, 3000])
@pytest.mark.parametrize("prec", ["mixed", "fp64"])
def test_one_leaf(n, prec):
    rng = np.random.default_rng(n)
    x = (0.30 + 0.15 * rng.random((n, 3))).astype(np.float32)  # inside one level-2 box
    q = rng.uniform(-1, 1, n).astype(np.float32)
    xj = x if n > 1 else (0.30 + 0.15 * rng.random((7, 3))).astype(np.float32)
    qj = q if n > 1 else rng.uniform(-1, 1, 7).astype(np.float32)
    f = F.FMM(p=6, lmax=2, precision=prec, convention="exact", box=(0, 0, 0, 1))
    f.set_points(x, xj)
    v, g = f.evaluate(qj)
    d, dg = f.direct(x, xj, qj)
    f.close()
    tol = 2e-6 if prec == "mixed" else 1e-13
    print(n, prec, rel_l2(v, d), rel_l2(g, dg), flush=True)
    assert rel_l2(v, d) < tol and rel_l2(g, dg) < tol


# a crowded leaf beside sparse ones, twice on one handle (the item counter is
# cleared between trees), every kernel form of the near field
@pytest.mark.parametrize("neq", [F.G, F.GNI, F.GNJ])
def test_uneven_leaves(neq):
    rng = np.random.default_rng(3)
    f = F.FMM(p=10, lmax=4, precision="mixed", convention="exact", box=(0, 0, 0, 1))
    for m in (700, 90):
        x = np.concatenate([0.52 + 0.05 * rng.random((m, 3)), rng.random((4000, 3))]).astype(np.float32)
        nrm = rng.standard_normal(x.shape).astype(np.float32)
        q = rng.uniform(-1, 1, len(x)).astype(np.float32)
        f.set_points(x, ni_normals=nrm, nj_normals=nrm)
        v, _ = f.evaluate(q, neq=neq)
        d, _ = f.direct(x, x, q, neq=neq, ni_normals=nrm, nj_normals=nrm)
        # the truncation of p = 10 over all boxes
        assert rel_l2(v, d) < 5e-4
    f.close()
