"""A captured evaluation stays good while the handle evaluates other things:
the blocks its launches refer to outlive the growth of the handle's buffers."""
import numpy as np
import pytest

from conftest import uniform_cube

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no HIP device", allow_module_level=True)

import old_fmm_bem_amd as F  # noqa: E402


def _check_replays(f, qd, v, want, between):
    for rep in range(3):
        print("replay", rep, flush=True)
        between()
        # whatever was freed is somebody else's now
        junk = [torch.full((1 << 22,), float("nan"), device="cuda") for _ in range(8)]
        v.zero_()
        torch.cuda.synchronize()
        f.replay()
        f.synchronize()
        assert torch.equal(v, want), rep
        del junk


# 30,000 points at lmax 4: Yukawa's partial sums take more than the Laplace
# orbit form's; Helmholtz's expansions twice as much
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("other", [F.YUKAWA, F.HELMHOLTZ])
def test_replay_after_another_kernel_grew_the_buffers(precision, other):
    x, q = uniform_cube(30000, 120)
    xd, qd = torch.from_numpy(x).cuda(), torch.from_numpy(q).cuda()
    qc = torch.complex(qd, -qd)
    f = F.FMM(p=10, lmax=4, precision=precision, convention="exact", box=(0, 0, 0, 1), lam=2.0, k=5.0)
    f.set_points(xd)
    want = f.evaluate(qd)[0].clone()
    v, _ = f.capture(qd)
    _check_replays(f, qd, v, want, lambda: f.evaluate(qc if other == F.HELMHOLTZ else qd, neq=other))
    assert torch.equal(f.evaluate(qd)[0], want)
    f.set_points(xd)  # frees what the graph kept
    assert torch.equal(f.evaluate(qd)[0], want)
    f.close()
