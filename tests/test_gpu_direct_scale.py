"""Separable tables whose factors share the kernel's magnitude unevenly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE = (40, 44, 72)


# powers of two on (scale, gx, gy); they cancel, so the kernel is the same (gz is
# the DFT of the normalized window that the table holds beside it)
@pytest.mark.parametrize("powers", [(140, -140, 0), (160, 0, -160), (200, -100, -100), (-180, 90, 90), (-1, 1, 0),
                                    (80, -40, -40), (0, 90, -90)])
@pytest.mark.parametrize("radius", [3, 12])
def test_direct_form_of_scaled_factors(vfd, orc, powers, radius):
    """Scaling by powers of two is exact, so the outputs have the unscaled table's bits."""
    import torch
    print(f"case scaled factors {powers} radius {radius}", flush=True)
    plan = vfd.Plan(SHAPE, kspec_format=vfd.KSPEC_SEPARABLE)
    i = plan.info
    s2 = ((radius - 0.5) / 6.0) ** 2
    table = plan.gauss_spectrum(s2, 0.97)
    t = table.view(torch.float64).cpu().numpy().copy()
    ends = np.cumsum([0, 1, i.hx, i.py])
    for p, a, b in zip(powers, ends, ends[1:]):
        t[a:b] = np.ldexp(t[a:b], p)
    u = orc.synth_field(SHAPE, 23, nsrc=5)
    ud = torch.from_numpy(u).cuda()
    outs = [torch.zeros_like(ud) for _ in range(2)]
    plan.diffuse([{"in": ud, "out": o, "work": plan.new_work(), "kspec": k}
                  for o, k in zip(outs, (table, torch.from_numpy(t).cuda()))])
    torch.cuda.synchronize()
    want, got = (o.cpu().numpy() for o in outs)
    ref = orc.direct_separable(u, s2, 0.97)
    assert float(np.linalg.norm(want - ref) / np.linalg.norm(ref)) <= 1e-6
    assert bool((got == want).all())
