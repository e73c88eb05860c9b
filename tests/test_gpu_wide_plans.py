"""Plans that have made wide tables only: whole ticks are the FFT form's alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE = (40, 44, 72)
RECORD = 512   # the last bytes of an FP32 separable plan's work array


def _s2(radius):
    return ((radius - 0.5) / 6.0) ** 2


def _tick(plan, u, table, work):
    import torch
    out = torch.zeros_like(u)
    plan.diffuse([{"in": u, "out": out, "work": work, "kspec": table}])
    torch.cuda.synchronize()
    return out.cpu().numpy()


def test_wide_plans_skip_the_direct_form(vfd, orc):
    """No record is made while the plan's own tables are all beyond radius 31, and
    one is as soon as it has made a short table.  A short table of another plan is
    done by the FFT passes then, and right.  Tolerance: FP32 ticks, rel-L2 1e-5."""
    import torch
    print("case wide plan", flush=True)
    plan, other = (vfd.Plan(SHAPE, kspec_format=vfd.KSPEC_SEPARABLE) for _ in range(2))
    u = orc.synth_field(SHAPE, 17, nsrc=5)
    ud = torch.from_numpy(u).cuda()
    wide, short = plan.gauss_spectrum(_s2(36), 0.97), other.gauss_spectrum(_s2(6), 0.97)
    work = plan.new_work()
    work.fill_(0xA5)
    for r, t in ((36, wide), (6, short)):
        ref = orc.direct_separable(u, _s2(r), 0.97)
        got = _tick(plan, ud, t, work)
        assert float(np.linalg.norm(got - ref) / np.linalg.norm(ref)) <= 1e-5, r
        assert bool((work[-RECORD:] == 0xA5).all()), r
    plan.gauss_spectrum(_s2(6), 0.97)
    got = _tick(plan, ud, wide, work)
    assert not bool((work[-RECORD:] == 0xA5).all())
    assert float(np.linalg.norm(got - orc.direct_separable(u, _s2(36), 0.97)) / np.linalg.norm(got)) <= 1e-5
