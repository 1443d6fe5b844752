"""Every shape of the near field: 64, 128 and 256 lanes with one target each
(the bound FMMX_P2P_SMALL set low), and the one-wave form with 4, 8, 16 and 32
targets per item and with a leaf over four times the mean, whose items are
cut finer.  All points lie in eight mutually adjacent leaves, so that the near
field is the whole sum, which the direct sum gives."""
import numpy as np
import pytest

import old_fmm_bem_amd as F
from conftest import rel_l2

pytestmark = pytest.mark.gpu

LANES64 = (1, 63, 64, 65, 2, 40, 33, 20)  # mean 36
LANES128 = (127, 128, 129, 1, 64, 2, 120, 30)  # mean 75
LANES256 = (255, 256, 257, 513, 1, 300, 64, 2)  # mean 206
HEAVY = (0.6, 0.1, 0.1, 0.05, 0.05, 0.05, 0.04, 0.01)  # the first over four times the mean


def _points(counts, seed):
    rng = np.random.default_rng(seed)
    x = [0.25 + 0.25 * (np.array([b & 1, b >> 1 & 1, b >> 2]) + 0.02 + 0.96 * rng.random((c, 3)))
         for b, c in enumerate(counts)]
    x = np.concatenate(x).astype(np.float32)
    return x[rng.permutation(len(x))], rng


def _counts(case):
    if isinstance(case, int):
        c = [int(w * case) for w in HEAVY]
        c[1] += case - sum(c)
        return c
    return case


def _engine(prec):
    return F.FMM(p=6, lmax=2, precision=prec, convention="exact", box=(0, 0, 0, 1), lam=2.0, k=3.0)


# 2,000 points: 4 targets per item, 20,000: 8, 40,000: 16, 70,000: 32
@pytest.mark.parametrize("case", [LANES64, LANES128, LANES256, 2000, 20000, 40000, 70000],
                         ids=["64", "128", "256", "4", "8", "16", "32"])
@pytest.mark.parametrize("prec", ["mixed", "fp64"])
def test_shapes(monkeypatch, prec, case):
    counts = _counts(case)
    if not isinstance(case, int):
        monkeypatch.setenv("FMMX_P2P_SMALL", "1")
    x, rng = _points(counts, 5)
    q = rng.uniform(-1, 1, len(x)).astype(np.float32)
    nrm = rng.standard_normal(x.shape).astype(np.float32)
    f = _engine(prec)
    f.set_points(x, ni_normals=nrm, nj_normals=nrm)
    assert f.nboxes("i", 2) == 8
    tol = 2e-6 if prec == "mixed" else 1e-13
    for neq in (F.G, F.GNI, F.GNJ, F.YUKAWA) if len(x) < 3000 else (F.G,):
        print(prec, case, neq, flush=True)
        v, g = f.evaluate(q, neq=neq)
        d, dg = f.direct(x, x, q, neq=neq, ni_normals=nrm, nj_normals=nrm)
        # dipole kernels of random normals cancel more: a few times the rounding
        assert rel_l2(v, d) < (tol if neq in (F.G, F.YUKAWA) else 4 * tol)
        if g is not None:
            assert rel_l2(g, dg) < 4 * tol
    f.close()


@pytest.mark.parametrize("prec", ["mixed", "fp64"])
def test_the_bound_changes_between_evaluations(monkeypatch, prec):
    x, rng = _points(LANES256, 6)
    q = rng.uniform(-1, 1, len(x)).astype(np.float32)
    f = _engine(prec)
    f.set_points(x)
    d, _ = f.direct(x, x, q)
    for small in (None, "1", "1000", "1", None):
        if small is None:
            monkeypatch.delenv("FMMX_P2P_SMALL", raising=False)
        else:
            monkeypatch.setenv("FMMX_P2P_SMALL", small)
        print(prec, small, flush=True)
        assert rel_l2(f.evaluate(q)[0], d) < (2e-6 if prec == "mixed" else 1e-13)
    f.close()


def test_a_captured_evaluation_keeps_its_items(monkeypatch):
    torch = pytest.importorskip("torch")
    x, rng = _points(LANES256, 7)
    xd = torch.from_numpy(x).cuda()
    qd = torch.from_numpy(rng.uniform(-1, 1, len(x)).astype(np.float32)).cuda()
    f = _engine("mixed")
    f.set_points(xd)
    want = f.evaluate(qd)[0].clone()
    v, _ = f.capture(qd)
    for rep, small in enumerate(("1", "1000", "1")):
        monkeypatch.setenv("FMMX_P2P_SMALL", small)
        f.evaluate(qd)
        v.zero_()
        torch.cuda.synchronize()
        f.replay()
        f.synchronize()
        assert torch.equal(v, want), rep
    f.close()
