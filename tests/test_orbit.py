"""The reflection-orbit M2L: its identity on the CPU (operators of reflected
offsets as sign changes of one, the sources of an orbit combined by a
Walsh-Hadamard transform before one product), and the kernel against the FP64
engine at the sizes where it can go wrong."""
import itertools

import numpy as np
import pytest

import old_fmm_bem_amd as F
from conftest import rel_l2, uniform_cube


def _classes(p):
    """sign class of every real slot: bits of the x, y, z reflections that negate it"""
    out = []
    for im in (0, 1):
        for n in range(p):
            for m in range(im, n + 1):
                out.append(((m ^ im) & 1) | im << 1 | ((n + m) & 1) << 2)
    return np.array(out)


def _char(a, b):
    return np.array([1 - 2 * (bin(int(x) & b).count("1") & 1) for x in np.atleast_1d(a)])


@pytest.mark.parametrize("p", [6, 7, 8, 9, 10])
def test_orbit_identity(p):
    cls = _classes(p)
    assert np.bincount(cls, minlength=8).max() <= 16  # one 16-row tile per class
    rng = np.random.default_rng(p)
    for d in [(2, 1, 0), (0, 2, 3), (1, 2, 2), (3, 0, 1), (3, 3, 3), (2, 0, 0)]:
        A = F.operator(p, "exact", 2, *d)
        axes = [a for a in range(3) if d[a] in (1, 2)]
        D = sum(1 << a for a in axes)
        refl = [sum(1 << a for a, b in zip(axes, bits) if b) for bits in itertools.product((0, 1), repeat=len(axes))]
        src = {r: rng.standard_normal(p * p) for r in refl}
        direct = np.zeros(p * p)
        for r in refl:
            dr = [-v if (r >> a) & 1 else v for a, v in enumerate(d)]
            T = _char(cls, r)
            Ar = F.operator(p, "exact", 2, *dr)
            # 1e-13: FP64 operators built from rotations at both offsets
            assert np.abs(Ar - T[:, None] * A * T[None, :]).max() <= 1e-13 * np.abs(A).max()
            direct += Ar @ src[r]
        spec = {psi: sum(_char(psi, r)[0] * src[r] for r in refl) for psi in refl}
        orbit = np.zeros(p * p)
        for c in range(8):
            cols = np.array([spec[(c ^ k) & D][i] for i, k in enumerate(cls)])
            orbit[cls == c] = (A @ cols)[cls == c]
        assert rel_l2(orbit, direct) < 1e-12


def _evaluate(prec, x, q, p, lmax, groups=0, splits=0, xj=None):
    f = F.FMM(p=p, lmax=lmax, precision=prec, convention="exact", box=(0, 0, 0, 1))
    if groups:
        f.set_groups(groups)
    f.set_points(x, xj)
    if prec == "mixed":
        for lev in range(2, lmax + 1):
            f.set_m2l_variant(lev, 1, 6, 8, splits)
        assert f.m2l_variant(lmax)[1] == 6
    v, g = f.evaluate(q)
    pairs = f.stats()["m2l_pairs"]
    f.close()
    return v, g, pairs


# boxes per parity class below, at and above the tile of 128 targets, one
# target, more splits than products of a mask, empty classes, separate sources
@pytest.mark.gpu
@pytest.mark.parametrize("p,lmax,n,splits", [(6, 2, 2000, 16), (7, 3, 1, 1), (8, 4, 3000, 1), (8, 5, 40, 7),
                                             (9, 5, 9000, 3), (10, 4, 60000, 5), (10, 5, 60, 16)])
def test_orbit_kernel_sizes(p, lmax, n, splits):
    x, q = uniform_cube(max(n, 2), 900 + n)
    x, q = x[:n], q[:n]
    xj, qj = uniform_cube(2500, 17) if n < 100 else (None, q)
    print(p, lmax, n, splits, flush=True)
    vm, gm, nm = _evaluate("mixed", x, qj, p, lmax, splits=splits, xj=xj)
    vd, gd, nd = _evaluate("fp64", x, qj, p, lmax, xj=xj)
    assert nm == nd  # the pairs of the interaction lists, counted by the kernels
    # the FP32 engine's own bound against FP64 (rounding of P2M, M2M, L2L and
    # P2P included); the gradient of a lone target has no sum to average over
    assert rel_l2(vm, vd) < 2e-6 and rel_l2(gm, gd) < 4e-6


@pytest.mark.gpu
def test_orbit_kernel_groups_and_scale():
    x, q = uniform_cube(40000, 5)
    vm, gm, nm = _evaluate("mixed", x, q, 8, 5, groups=2)
    vd, gd, nd = _evaluate("fp64", x, q, 8, 5, groups=2)
    assert nm == nd and rel_l2(vm, vd) < 2e-6 and rel_l2(gm, gd) < 2e-6
    # powers of two far outside FP16's range: the per-level scales carry them
    for s in (2.0 ** -40, 2.0 ** 40):
        vs, _, _ = _evaluate("mixed", x, (q * np.float32(s)).astype(np.float32), 8, 5, groups=2)
        assert rel_l2(vs / s, vm) < 1e-12
    # every box alike: sums of the largest magnitude over the reflected sources
    k = (np.arange(32) + 0.5) / 32
    xs = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3).astype(np.float32)
    qs = np.ones(len(xs), np.float32)
    vm, gm, _ = _evaluate("mixed", xs, qs, 10, 5)
    vd, gd, _ = _evaluate("fp64", xs, qs, 10, 5)
    assert np.isfinite(vm).all() and rel_l2(vm, vd) < 2e-6
