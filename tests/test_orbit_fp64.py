"""The FP64 engine's M2L by reflection orbits and its translations on the FP64
matrix cores, against the dense operators applied on the host."""
import numpy as np
import pytest

import old_fmm_bem_amd as F
from conftest import uniform_cube


def _real(c, p, scale):
    """real slots of complex expansions: re (n, m), then im (n, m > 0); scale[n] undone"""
    s = np.concatenate([[scale[n]] * (n + 1) for n in range(p)])
    c = c / s
    im = np.concatenate([[m > 0 for m in range(n + 1)] for n in range(p)])
    return np.concatenate([c.real, c.imag[:, im]], axis=1)


def _xyz(key, lev):
    b = [(key[:, None] >> (3 * np.arange(lev) + s)) & 1 for s in (1, 0, 2)]  # y | x << 1 | z << 2
    return np.stack([(v << np.arange(lev)).sum(1) for v in b], 1)


# every order built; one target, boxes per parity class below, at and above a
# tile of 128, empty octants, more targets than one XCD's block of tiles
@pytest.mark.gpu
@pytest.mark.parametrize("p,lmax,n,surface", [(6, 2, 1, False), (7, 3, 2000, False), (8, 4, 12000, False),
                                              (9, 3, 60, False), (10, 4, 3000, True), (11, 3, 700, True),
                                              (12, 3, 4000, False), (6, 5, 40000, False)])
def test_locals_against_dense_operators(p, lmax, n, surface):
    x, _ = uniform_cube(max(n, 300), 70 + n)
    if surface:
        d = x - 0.5
        x = (0.5 + 0.45 * d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    q = np.random.default_rng(n).uniform(-1, 1, len(x)).astype(np.float32)
    print(p, lmax, n, flush=True)
    f = F.FMM(p=p, lmax=lmax, precision="fp64", convention="exact", box=(0, 0, 0, 1))
    f.set_points(x[:n], x)
    f.evaluate(q)
    M, row = {}, 0
    allm = f.multipoles()
    for lev in range(lmax, 1, -1):
        nb = f.nboxes("j", lev)
        M[lev] = _real(allm[row:row + nb], p, [2.0 ** (-lev * k) for k in range(p)])
        row += nb
    L = {lev: _real(f.locals(lev), p, [2.0 ** (lev * (k + 1)) for k in range(p)]) for lev in range(2, lmax + 1)}
    box = {(s, lev): f.boxes(s, lev)[0] for s in "ij" for lev in range(2, lmax + 1)}
    pairs = f.stats()["m2l_pairs"]
    f.close()
    m2m = [F.operator(p, "exact", 0, o) for o in range(8)]
    l2l = [F.operator(p, "exact", 1, o) for o in range(8)]
    seen = 0
    for lev in range(2, lmax + 1):
        ki, kj = box["i", lev], box["j", lev]
        xi, xj = _xyz(ki, lev), _xyz(kj, lev)
        at = {k: r for r, k in enumerate(kj)}
        index = {tuple(v): r for r, v in enumerate(xj)}
        want = np.zeros_like(L[lev])
        size = np.zeros_like(want)
        if lev > 2:
            parent = {k: r for r, k in enumerate(box["i", lev - 1])}
            src = np.array([parent[k >> 3] for k in ki])
            for o in range(8):
                t = (ki & 7) == o
                want[t] += L[lev - 1][src[t]] @ l2l[o].T
                size[t] += np.abs(L[lev - 1][src[t]]) @ np.abs(l2l[o]).T
        for d in np.ndindex(7, 7, 7):
            d = np.array(d) - 3
            if np.abs(d).max() < 2:
                continue
            # source at the target minus d, a child of a neighbour of its parent
            s = np.array([index.get(tuple(v), -1) for v in xi - d])
            s[np.abs((xi - d >> 1) - (xi >> 1)).max(1) > 1] = -1
            t = np.flatnonzero(s >= 0)
            if len(t) == 0:
                continue
            A = F.operator(p, "exact", 2, *map(int, d))
            want[t] += M[lev][s[t]] @ A.T
            size[t] += np.abs(M[lev][s[t]]) @ np.abs(A).T
            seen += len(t)
        # FP64 sums of at most 189 p^2 products in any order, and the four-source
        # transform: 189 p^2 + 8 roundings of the terms' magnitudes bound it
        assert (np.abs(L[lev] - want) <= (189 * p * p + 8) * 2.3e-16 * size + 1e-300).all(), lev
        # in practice far below: the norm to 1e-13
        assert np.linalg.norm(L[lev] - want) <= 1e-13 * np.linalg.norm(size), lev
        if lev < lmax:
            mw = np.zeros_like(M[lev])
            for r, k in enumerate(box["j", lev + 1]):
                mw[at[k >> 3]] += m2m[k & 7] @ M[lev + 1][r]
            assert np.abs(M[lev] - mw).max() <= 1e-13 * np.abs(mw).max(), lev
    assert pairs == seen
