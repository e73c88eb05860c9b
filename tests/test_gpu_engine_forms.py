"""Runs whose fields take both forms of a separable FP32 tick (windows within the
direct form's radius, 31, and beyond), and runs used right after admission.

A field goes through the same kernels whatever batch it is in, so comparisons
between engines are bit-exact; accuracy is the FP64 oracle's rel-L2 <= 1e-5 per
tick."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE = (44, 50, 52)
RADII = (36, 5, 40, 8, 31)   # FFT, direct, FFT, direct, direct
DECAY = 0.97


def _s2(radius):
    return ((radius - 0.5) / 6.0) ** 2


def _run(eng, orc, shape, radii):
    import torch
    rid = eng.create_run(shape, [_s2(r) for r in radii], [DECAY] * len(radii))
    us = [orc.synth_field(shape, 61 + f, nsrc=5) for f in range(len(radii))]
    for f, u in enumerate(us):
        eng.write_field(rid, f, torch.from_numpy(u.astype(np.float32)).cuda())
    torch.cuda.synchronize()
    return rid, us


def _fields(eng, rid, n):
    import torch
    out = [eng.read_field(rid, f) for f in range(n)]
    torch.cuda.synchronize()
    return [o.cpu().numpy() for o in out]


@pytest.mark.parametrize("how", ["step", "graph", "plain", "serve"])
def test_both_forms_share_the_one_work_buffer_of_a_tight_budget(vfd, orc, how):
    """A budget of the run and one work buffer, the least that admits the run, has
    to be enough to tick it, whatever forms its fields take."""
    import torch
    import vfd.engine as em
    print(f"case both forms, one work buffer: {how}", flush=True)
    n = len(RADII)
    work = vfd.Plan(SHAPE, kspec_format=vfd.KSPEC_SEPARABLE).info.work_bytes
    with em.Engine(1 << 30) as roomy:
        rid, us = _run(roomy, orc, SHAPE, RADII)
        roomy.step([rid], ticks=2)
        torch.cuda.synchronize()
        want = _fields(roomy, rid, n)
    with em.Engine(em.run_bytes(SHAPE, n) + work) as eng:
        rid, _ = _run(eng, orc, SHAPE, RADII)
        if how == "step":
            eng.step([rid])
            eng.step([rid])
        elif how == "graph":
            eng.step([rid], graph=True)
            torch.cuda.synchronize()
            eng.step([rid], graph=True)
        elif how == "plain":
            eng.step_plain([rid], ticks=2)
        else:
            eng.serve_start(slots=2)
            try:
                for _ in range(2):
                    eng.wait(eng.submit(rid))
            finally:
                eng.serve_stop()
        torch.cuda.synchronize()
        got = _fields(eng, rid, n)
        st = eng.stats()
        assert st["used_bytes"] == st["budget_bytes"] == st["peak_used_bytes"]
    for f, r in enumerate(RADII):
        assert np.array_equal(got[f], want[f]), (f, r)
        ref = orc.direct_separable(orc.direct_separable(us[f], _s2(r), DECAY), _s2(r), DECAY)
        assert orc.rel_l2(got[f], ref) <= 2e-5, (f, r)


def test_two_shapes_with_both_forms_in_one_batch(vfd, orc):
    """Shapes on parallel branches, each with fields of both forms: the bits of the
    runs ticked one at a time, eager and by graph."""
    import torch
    import vfd.engine as em
    print("case two shapes, both forms", flush=True)
    other = (40, 45, 70)
    with em.Engine(2 << 30) as eng:
        a1, _ = _run(eng, orc, SHAPE, RADII)
        b1, _ = _run(eng, orc, other, RADII[::-1])
        a2, _ = _run(eng, orc, SHAPE, RADII)
        b2, _ = _run(eng, orc, other, RADII[::-1])
        for rep in range(3):
            eng.step([a1])
            eng.step([b1])
            eng.step([a2, b2], graph=rep > 0)
            torch.cuda.synchronize()
        for x, y in ((a1, a2), (b1, b2)):
            for f, (p, q) in enumerate(zip(_fields(eng, x, len(RADII)), _fields(eng, y, len(RADII)))):
                assert np.array_equal(p, q), f


def test_run_is_whole_when_its_id_is_returned(vfd, orc):
    """A run is written and ticked at once on a stream that does not wait for the
    null stream: its fields and the last field's record have to be there already
    (an admission leaves no work queued)."""
    import torch
    import vfd.engine as em
    shape, radii = (64, 128, 128), (31, 5, 36, 12, 8)   # ends in a field of the direct form
    print("case run used at once on a side stream", flush=True)
    s2, dec = [_s2(r) for r in radii], [DECAY] * len(radii)
    us = [torch.from_numpy(orc.synth_field(shape, 71 + f, nsrc=5)).cuda() for f in range(len(radii))]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    got = []
    with em.Engine(4 << 30) as eng:
        for rep in range(4):
            rid = eng.create_run(shape, s2, dec)
            assert torch.cuda.default_stream().query()
            for f in reversed(range(len(radii))):
                eng.write_field(rid, f, us[f], stream=side)
            eng.step([rid], stream=side)
            side.synchronize()
            out = [eng.read_field(rid, f, stream=side) for f in range(len(radii))]
            side.synchronize()
            got.append([o.cpu().numpy() for o in out])
    for f, r in enumerate(radii):
        ref = orc.direct_separable(us[f].cpu().numpy(), s2[f], DECAY)
        assert orc.rel_l2(got[0][f], ref) <= 1e-5, r
        for g in got[1:]:
            assert np.array_equal(g[f], got[0][f]), r
