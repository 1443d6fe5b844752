"""FMMX_M2L_FUSED=0 (one M2L launch per level) against the one launch of all
levels: the same products and reductions, so equal sums, for the engines and
kernels that take the switch, where the leaf level has several splits and the
near field runs on a stream of its own."""
import numpy as np
import pytest

import old_fmm_bem_amd as F
from conftest import rel_l2, uniform_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,p,neq", [("mixed", 8, F.G), ("mixed", 10, F.GNI), ("mixed", 12, F.G),
                                        ("mixed", 8, F.YUKAWA), ("mixed", 8, F.HELMHOLTZ), ("fp64", 10, F.G),
                                        ("fp64", 6, F.GNJ), ("fp64", 8, F.YUKAWA), ("fp64", 5, F.G)])
def test_level_by_level_equals_one_launch(monkeypatch, prec, p, neq):
    x, q = uniform_cube(30000, 40 + p)
    nrm = np.random.default_rng(p).standard_normal(x.shape).astype(np.float32)
    if neq == F.HELMHOLTZ:
        q = (q + 1j * q[::-1]).astype(np.complex64)
    kw = {F.YUKAWA: {"lam": 2.0}, F.HELMHOLTZ: {"k": 6.0}}.get(neq, {})
    f = F.FMM(p=p, lmax=4, precision=prec, convention="exact", box=(0, 0, 0, 1), **kw)
    f.set_points(x, ni_normals=nrm, nj_normals=nrm)
    out = []
    for fused in ("1", "0"):
        monkeypatch.setenv("FMMX_M2L_FUSED", fused)
        print(prec, p, neq, "fused", fused, f.m2l_variant(4), flush=True)
        assert f.m2l_variant(4)[3] > 1
        out.append(f.evaluate(q, neq=neq)[0])
        assert f.stats()["m2l_all_levels"] == int(fused == "1" and not (prec == "fp64" and (neq == F.YUKAWA or p < 6)))
    f.close()
    # the locals of a level: M2L added to the parent's instead of the other way
    # round, in the engine's own arithmetic
    assert rel_l2(out[1], out[0]) < (1e-6 if prec == "mixed" else 1e-13)
