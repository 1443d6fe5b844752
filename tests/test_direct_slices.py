"""The direct sum's split of the sources over workgroups: one source, slices of
64 and of 256 sources, more targets than workgroups, against FP64 on the host."""
import numpy as np
import pytest

import old_fmm_bem_amd as F


@pytest.mark.gpu
@pytest.mark.parametrize("ni,nj", [(1, 1), (63, 5000), (1, 300000), (65, 262145), (2000, 16385), (70000, 300)])
def test_direct_sum(ni, nj):
    rng = np.random.default_rng(ni + nj)
    xi, xj = rng.random((ni, 3)).astype(np.float32), rng.random((nj, 3)).astype(np.float32)
    q = rng.uniform(-1, 1, nj).astype(np.float32)
    print(ni, nj, flush=True)
    f = F.FMM(p=6, lmax=2, precision="fp64", convention="exact", box=(0, 0, 0, 1))
    v, g = f.direct(xi, xj, q)
    f.close()
    t = rng.choice(ni, min(ni, 50), replace=False)
    d = xi[t, None].astype(np.float64) - xj[None]
    r = np.sqrt((d ** 2).sum(-1))
    w = q / r / (4 * np.pi)
    gw = -(d * (w / r ** 2)[..., None])
    # FP64: a few roundings per pair and one per addition, against the terms' sum of magnitudes
    tol = (nj + 16) * 2.3e-16
    assert (np.abs(v[t] - w.sum(1)) <= tol * np.abs(w).sum(1)).all()
    assert (np.abs(g[t] - gw.sum(1)) <= tol * np.abs(gw).sum(1)).all()
