"""Batches of 32 fields of both forms at the lengths whose work-groups end in a
partial wave: the mask of the FFT form's fields has to be whole there too.

Rows of 576 (24 lanes in the last wave) and 1152 (24, 16, 16 and 8 in schedules
0 to 3), columns of 72 (16), in both launch shapes of the FFT passes.  The FFT
form's fields sit at indexes below and past each of those lane counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WIDE = (3, 9, 17, 25, 31)   # fields of the FFT form
SHORT_R, WIDE_R = 6, 33


def _s2(radius):
    return ((radius - 0.5) / 6.0) ** 2


@pytest.mark.parametrize("few", [False, True], ids=["many", "few"])
@pytest.mark.parametrize("shape,half,schedule",
                         [((34, 35, 560), ("px", 1152), 0)] +
                         [((34, 35, 1100), ("px", 2304), v) for v in range(4)] +
                         [((34, 70, 40), ("py", 144), 0), ((70, 34, 40), ("pz", 144), 0)])
def test_mask_is_whole_in_partial_waves(vfd, orc, monkeypatch, shape, half, schedule, few):
    """Tolerance: FP32 ticks against the FP64 oracle, rel-L2 1e-5 as everywhere;
    fields with one input and one table have the same bits."""
    import torch
    print(f"case field mask shape={shape} schedule={schedule} few={few}", flush=True)
    monkeypatch.setenv("VFD_SCHEDULE", ",".join([str(schedule)] * 5))
    maker = vfd.Plan(shape, kspec_format=vfd.KSPEC_SEPARABLE)
    plan = vfd.Plan(shape, kspec_format=vfd.KSPEC_SEPARABLE) if few else maker
    assert getattr(plan.info, half[0]) == half[1]
    if few:
        plan.gauss_spectrum(_s2(5), 0.97)   # tables of the direct form only: persistent launches
    u = orc.synth_field(shape, 41, nsrc=5)
    ud = torch.from_numpy(u).cuda()
    tables = {r: maker.gauss_spectrum(_s2(r), 0.97) for r in (SHORT_R, WIDE_R)}
    radii = [WIDE_R if f in WIDE else SHORT_R for f in range(32)]
    outs = [torch.zeros_like(ud) for _ in radii]
    plan.diffuse([{"in": ud, "out": o, "work": plan.new_work(), "kspec": tables[r]} for o, r in zip(outs, radii)])
    torch.cuda.synchronize()
    got = [o.cpu().numpy() for o in outs]
    for r in (SHORT_R, WIDE_R):
        ref = orc.direct_separable(u, _s2(r), 0.97)
        fields = [f for f in range(32) if radii[f] == r]
        first = got[fields[0]]
        assert float(np.linalg.norm(first - ref) / np.linalg.norm(ref)) <= 1e-5, r
        for f in fields[1:]:
            assert np.array_equal(got[f], first), (r, f)
