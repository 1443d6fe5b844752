"""The FP16 operands of the orbit M2L carry power-of-two scales: independent
groups of very different strengths, and strengths near the ends of FP32's range,
keep the FP32 engine's accuracy (against the FP64 engine, group by group)."""
import numpy as np
import pytest

import old_fmm_bem_amd as F
from conftest import rel_l2, uniform_cube

pytestmark = pytest.mark.gpu


def _run(prec, p, x, q, neq, groups=0, staging=None, lmax=4):
    f = F.FMM(p=p, lmax=lmax, precision=prec, convention="exact", box=(0, 0, 0, 1), k=6.0)
    if groups:
        f.set_groups(groups)
    f.set_points(x)
    if staging is not None:
        for lev in range(2, lmax + 1):
            f.set_m2l_variant(lev, 0, staging)
    v = f.evaluate(q, neq=neq)[0]
    f.close()
    return v


def _complex(n, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)


@pytest.mark.parametrize("groups,lmax", [(1, 4), (2, 3), (3, 4)])
@pytest.mark.parametrize("p", [4, 12])
def test_helmholtz_groups_of_any_strength(p, groups, lmax):
    x, _ = uniform_cube(12000, 61)
    box = (x * 2 ** groups).astype(int).sum(1)
    for s in (1e-6, 1e-12):
        # every other group (checkerboard) weaker by s
        q = (_complex(len(x), 7) * np.where(box % 2, s, 1.0)).astype(np.complex64)
        print(p, groups, s, flush=True)
        vm = _run("mixed", p, x, q, F.HELMHOLTZ, groups, lmax=lmax)
        vd = _run("fp64", p, x, q, F.HELMHOLTZ, groups, lmax=lmax)
        for part in (0, 1):
            t = box % 2 == part
            # the FP32 engine's own bound (test_mixed_matches_fp64)
            assert rel_l2(vm[t] / vd[t].std(), vd[t] / vd[t].std()) < 5e-6


@pytest.mark.parametrize("scale", [1e-35, 1e-31, 1e31, 1e34])
def test_helmholtz_strengths_near_the_ends_of_fp32(scale):
    x, _ = uniform_cube(12000, 62)
    q = _complex(len(x), 8).astype(np.complex64)
    vm = _run("mixed", 10, x, (q.astype(np.complex128) * scale).astype(np.complex64), F.HELMHOLTZ)
    vd = _run("fp64", 10, x, (q.astype(np.complex128) * scale).astype(np.complex64), F.HELMHOLTZ)
    print(scale, rel_l2(vm / scale, vd / scale), flush=True)
    assert rel_l2(vm / scale, vd / scale) < 5e-6


@pytest.mark.parametrize("p", [8, 10])
def test_laplace_orbits_resolve_as_much_as_the_dense_form(p):
    """Where FP16's smallest steps are the error (a group 1e-6 weaker than the
    rest), the orbit form is no further off than the form that multiplies every
    offset: the same steps, once per sum of up to four sources and not once per
    source.  A quarter for the scatter of two roundings."""
    x, q = uniform_cube(20000, 63)
    weak = x[:, 0] <= 0.5
    q = np.where(weak, 1e-6 * q, q).astype(np.float32)
    ref = _run("fp64", p, x, q, F.G, groups=1)[weak]
    e6, e5 = (rel_l2(_run("mixed", p, x, q, F.G, groups=1, staging=s)[weak], ref) for s in (6, 5))
    print(p, e6, e5, flush=True)
    assert e6 < 1.25 * e5


@pytest.mark.parametrize("top", [0.99, 0.9995, 0.99999, 1.0])
def test_sums_at_the_top_of_fp16(top):
    """Every box alike and its largest multipole at the end of a binade: sums of
    four sources stay finite in FP16 and keep the engine's accuracy."""
    k = (np.arange(16) + 0.5) / 16
    x = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3).astype(np.float32)
    q = np.full(len(x), np.float32(top), np.float32)  # one charge per leaf: M_00 = q
    vm, vd = (_run(prec, 8, x, q, F.G) for prec in ("mixed", "fp64"))
    print(top, rel_l2(vm, vd), flush=True)
    assert rel_l2(vm, vd) < 2e-6
