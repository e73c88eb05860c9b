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


@pytest.mark.parametrize("radii", [(36,) * 8, (36, 6) * 4], ids=["wide", "both"])
def test_fused_epilogues_of_wide_windows(vfd, radii):
    """The chem update and the downsample in the last pass against the separate
    calls on the same inputs: the same bits, for plans of wide tables (FFT passes
    without records) and of both kinds (with)."""
    import torch
    print(f"case epilogues {radii}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(11)
    plan = vfd.Plan(SHAPE, kspec_format=vfd.KSPEC_SEPARABLE)
    rand = lambda: torch.rand(SHAPE, generator=g, device="cuda")
    u, d, col, ela, decay = [rand() for _ in radii], [rand() for _ in radii], rand(), rand(), [0.3] * 8
    ks = [plan.gauss_spectrum(_s2(r), 0.97) for r in radii]
    entries = lambda out: [{"in": a, "out": o, "work": plan.new_work(), "kspec": k} for a, o, k in zip(u, out, ks)]
    new = lambda: [torch.empty_like(x) for x in u]
    t, levels, fused = new(), new(), new()
    grads, fused_grads = [torch.empty_like(col) for _ in range(3)], [torch.empty_like(col) for _ in range(3)]
    plan.diffuse(entries(t))
    vfd.chem_update(t, [x.clone() for x in d], levels, decay, col, ela, grads)
    plan.diffuse_update(entries(fused), d, decay, col, ela, fused_grads)
    out, want = new(), [vfd.sample_chem(x, c, 3) for c, x in enumerate(t)]
    vis = [torch.full_like(w, -1.0) for w in want]
    plan.diffuse_sample(entries(out), list(range(8)), 3, vis)
    torch.cuda.synchronize()
    for i in range(8):
        assert torch.equal(fused[i], levels[i]) and not d[i].any(), i
        assert torch.equal(out[i], t[i]) and torch.equal(vis[i], want[i]), i
    assert all(torch.equal(a, b) for a, b in zip(fused_grads, grads))
