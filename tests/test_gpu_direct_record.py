"""The record that the device makes of a separable table (dir_classify_kernel):
each axis' window radius, or -1, its FP32 taps, and the factors that go with them.
It is the last bytes of the field's work array after the first pass."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

AXIS = np.dtype([("gain", "f8"), ("radius", "i4"), ("tap", "f4", 32), ("pad", "i4")])
RECORD = np.dtype([("scale", "f8"), ("ax", AXIS, 3)])   # x, y, z
RECORD_BYTES = 512
DECAY = 0.97


def _s2(radius):
    return ((radius - 0.5) / 6.0) ** 2


def _window(radius):
    j = np.arange(radius + 1)
    g = np.exp(-j * j / (2.0 * _s2(radius)))
    return g / (g[0] + 2.0 * g[1:].sum())


def _plan(vfd, shape):
    plan = vfd.Plan(shape, kspec_format=vfd.KSPEC_SEPARABLE)
    plan.gauss_spectrum(_s2(1), DECAY)   # a plan of wide tables only makes no records
    return plan


def _records(vfd, plan, tables):
    import torch
    i = plan.info
    u = torch.ones((i.nz, i.ny, i.nx), device="cuda")
    works = [plan.new_work() for _ in tables]
    plan.diffuse_pass([{"in": u, "out": u, "work": w, "kspec": t} for w, t in zip(works, tables)], vfd.PASS_XFWD)
    torch.cuda.synchronize()
    return [w[-RECORD_BYTES:].cpu().numpy()[:RECORD.itemsize].view(RECORD)[0] for w in works]


# data of 1024 and 1536 along one axis, odd lengths, boxes that are no power of two
@pytest.mark.parametrize("shape", [(32, 34, 1024), (33, 1536, 40), (301, 31, 36), (40, 75, 187), (48, 36, 560)])
def test_windows_are_recognized(vfd, shape):
    """Taps: the window's values, rounded once (the FP64 inverse errs by some 1e-16).
    Gain times the taps' sum is the window's, 1; the scale is the decay."""
    radii = (1, 2, 6, 13, 19, 30, 31)
    plan = _plan(vfd, shape)
    print(f"case records {shape}", flush=True)
    for r, rec in zip(radii, _records(vfd, plan, [plan.gauss_spectrum(_s2(r), DECAY) for r in radii])):
        g = _window(r)
        want = int(np.nonzero(g > 1e-13 * g[0])[0].max())   # the narrowest windows end before their radius
        assert abs(rec["scale"] - DECAY) <= 1e-15
        for ax in rec["ax"]:
            assert ax["radius"] == want, (r, ax["radius"])
            taps = ax["tap"].astype(np.float64)
            assert (np.abs(taps[:want + 1] - g[:want + 1]) <= 1.01 * 2.0 ** -24 * g[:want + 1] + 1e-15).all()
            assert (taps[want + 1:] == 0.0).all()
            assert abs(ax["gain"] * (taps[0] + 2.0 * taps[1:].sum()) - 1.0) <= 1e-12


def test_other_tables_are_not(vfd):
    """Windows past radius 31, an entry off by 1e-11, an uneven table, NaN and infinity:
    -1 on that axis and on no other."""
    import torch
    shape = (40, 44, 72)
    plan = _plan(vfd, shape)
    i = plan.info
    ox, oy, oz = 1, 1 + i.hx, 1 + i.hx + i.py
    short = plan.gauss_spectrum(_s2(8), DECAY).view(torch.float64)
    cases = [("wide", plan.gauss_spectrum(_s2(32), DECAY).view(torch.float64), (-1, -1, -1)),
             ("wider", plan.gauss_spectrum(_s2(40), DECAY).view(torch.float64), (-1, -1, -1))]
    for name, at, value, ax in (("x off", ox + 7, 1e-11, 0), ("y uneven", oy + 3, 1e-9, 1), ("z uneven", oz + i.pz - 2, 1e-9, 2),
                                ("x NaN", ox + i.hx - 1, float("nan"), 0), ("y NaN", oy, float("nan"), 1),
                                ("z infinite", oz + 5, float("inf"), 2)):
        t = short.clone()
        t[at] += value
        cases.append((name, t, tuple(-1 if a == ax else 8 for a in range(3))))
    for (name, _, want), rec in zip(cases, _records(vfd, plan, [t for _, t, _ in cases])):
        print(f"case {name}: {[int(a['radius']) for a in rec['ax']]}", flush=True)
        assert tuple(int(a["radius"]) for a in rec["ax"]) == want, name


def test_boxes_without_room_for_the_window(vfd):
    """A window that the padding does not hold would wrap; the table of a wide box is
    put on a plan whose data leaves less room."""
    box, radius = (128, 128, 128), 8
    full = vfd.Plan((64, 64, 64), box, kspec_format=vfd.KSPEC_SEPARABLE)
    table = full.gauss_spectrum(_s2(radius), DECAY)
    plan = vfd.Plan((124, 120, 121), box, kspec_format=vfd.KSPEC_SEPARABLE)
    (rec,) = _records(vfd, plan, [table])
    print(f"case no room: {[int(a['radius']) for a in rec['ax']]}", flush=True)
    assert [int(a["radius"]) for a in rec["ax"]] == [-1, 8, -1]   # x leaves 7, y 8, z 4
