"""The direct-convolution form of a separable FP32 tick (vfd_direct.hpp) at the
edges of its tiles, batches, radius bounds and of the rule that selects it,
against the FP64 oracle.

Tolerance.  The fields and windows are non-negative, so an output is a sum of
non-negative terms and rounding errors are relative to it element by element:
per axis at most R + 2 roundings of the running sums, one of the tap and one of
the stored result, plus two for the decay: |err| <= (3 (R + 4) + 2) 2^-24 v.
Radius bounds of 8 and more form outputs in pairs, half the products with a
shared sum: two thirds of the roundings, and terms that exceed the output's own
only by tap differences, which for these windows (sigma >= 1.25) are below their
taps near the centre and, further out, small against the fields' background.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _s2(radius):
    """sigma^2 whose window has this radius, ceil(6 sigma)."""
    return ((radius - 0.5) / 6.0) ** 2


def _tick(vfd, plan, u, tables, passes=None):
    import torch
    ud = torch.from_numpy(u).cuda()
    outs = [torch.zeros_like(ud) for _ in tables]
    arr = plan.field_array([{"in": ud, "out": o, "work": plan.new_work(), "kspec": t} for o, t in zip(outs, tables)])
    if passes is None:
        plan.diffuse(arr)
    else:
        for p in passes:
            plan.diffuse_pass(arr, p)
    torch.cuda.synchronize()
    return [o.cpu().numpy() for o in outs]


# (radius, shape): columns 63..65 and 127..129 (strips of 64), rows and planes
# around the batches of 32, rows not a multiple of 4 floats, radii at and after
# each compiled bound, one-voxel axes, and the largest radius of the form
CASES = [(1, (2, 3, 4)), (2, (31, 33, 63)), (3, (32, 31, 65)), (4, (33, 32, 64)), (5, (9, 65, 127)),
         (8, (40, 17, 129)), (9, (17, 64, 128)), (12, (30, 97, 66)), (13, (64, 33, 130)), (16, (33, 63, 61)),
         (17, (48, 96, 192)), (19, (95, 34, 70)), (20, (21, 129, 67)), (21, (65, 40, 96)), (24, (25, 25, 301)),
         (25, (96, 31, 62)), (28, (29, 160, 36)), (29, (63, 64, 65)), (31, (32, 70, 100)), (31, (97, 33, 259)),
         (32, (40, 44, 72)), (40, (48, 41, 90))]


@pytest.mark.parametrize("radius,shape", CASES)
def test_direct_form_matches_oracle(vfd, orc, radius, shape):
    print(f"case direct radius={radius} shape={shape}", flush=True)
    plan = vfd.Plan(shape, kspec_format=vfd.KSPEC_SEPARABLE)
    s2, dec = _s2(radius), 0.97
    assert orc.gauss_radius(s2) == radius
    u = orc.synth_field(shape, 31 * radius + shape[2], nsrc=5)
    table = plan.gauss_spectrum(s2, dec)
    ref = orc.direct_separable(u, s2, dec)
    (got,) = _tick(vfd, plan, u, [table])
    rel = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    worst = float(np.max(np.abs(got - ref) / ref))
    print(f"  rel-L2 {rel:.3e} worst relative error {worst:.3e}", flush=True)
    direct = radius <= 31
    assert rel <= 1e-5
    if direct:
        assert worst <= (3 * (radius + 4) + 2) * U
    # the x-y pass goes with the first pass and the z pass with the last; the
    # passes between are the FFT form's alone
    (ends,) = _tick(vfd, plan, u, [table], passes=[vfd.PASS_XFWD, vfd.PASS_XINV])
    assert np.array_equal(ends, got) == direct
    (five,) = _tick(vfd, plan, u, [table], passes=range(5))
    assert np.array_equal(five, got)


def _axis_conv(u, windows, dec):
    v = u.astype(np.float64)
    for ax, g in zip((2, 1, 0), windows):
        R = (len(g) - 1) // 2
        n = v.shape[ax]
        a = g[R] * v
        for j in range(1, min(R, n - 1) + 1):
            lo, hi = [slice(None)] * 3, [slice(None)] * 3
            lo[ax], hi[ax] = slice(0, n - j), slice(j, n)
            a[tuple(hi)] += g[R + j] * v[tuple(lo)]
            a[tuple(lo)] += g[R - j] * v[tuple(hi)]
        v = a
    return dec * v


def test_tables_of_other_kernels(vfd, orc):
    """One batch of tables that are not vfd_gauss_spectrum's: another window per
    axis (direct), a signed window (direct), one wide axis (FFT form with the
    direct z pass), an entry off by 1e-9 (no window: FFT form)."""
    import torch
    shape = (40, 44, 72)
    plan = vfd.Plan(shape, kspec_format=vfd.KSPEC_SEPARABLE)
    i = plan.info
    ox, oy, oz = 1, 1 + i.hx, 1 + i.hx + i.py
    dec = 0.9
    u = orc.synth_field(shape, 5, nsrc=4)

    def table(s2):
        return plan.gauss_spectrum(s2, dec).view(torch.float64).cpu().numpy().copy()

    def dft(w, p, n):
        R = (len(w) - 1) // 2
        k = np.arange(n)
        return sum(w[R + j] * np.cos(2 * np.pi * j * k / p) for j in range(-R, R + 1))

    g = {r: orc.gauss_window1d(_s2(r)) for r in (3, 7, 12, 36)}
    signed = np.array([-0.1, 0.3, 0.6, 0.3, -0.1])
    cases = []
    t = table(_s2(12))
    t[ox:oy] = dft(g[3], i.px, i.hx)
    t[oy:oz] = dft(g[7], i.py, i.py)
    cases.append(("three windows", t, (g[3], g[7], g[12]), True))
    t = table(_s2(7))
    t[ox:oy] = dft(signed, i.px, i.hx)
    cases.append(("signed window", t, (signed, g[7], g[7]), True))
    t = table(_s2(7))
    t[oy:oz] = dft(g[36], i.py, i.py)
    cases.append(("wide y", t, (g[7], g[36], g[7]), False))
    t = table(_s2(7))
    t[ox + 5] += 1e-9
    cases.append(("perturbed", t, (g[7], g[7], g[7]), False))
    tabs = [torch.from_numpy(c[1]).cuda() for c in cases]
    got = _tick(vfd, plan, u, tabs)
    ends = _tick(vfd, plan, u, tabs, passes=[vfd.PASS_XFWD, vfd.PASS_XINV])
    for (name, _, win, direct), a, e in zip(cases, got, ends):
        ref = _axis_conv(u, win, dec)
        rel = float(np.linalg.norm(a - ref) / np.linalg.norm(ref))
        print(f"case {name}: rel-L2 {rel:.3e}", flush=True)
        assert rel <= 1e-6, name     # FP32 transforms of this box: 1.3e-7 (test_separable_spectrum_matches_real)
        assert np.array_equal(a, e) == direct, name


@pytest.mark.parametrize("shape,radii", [((40, 150, 330), (9, 36, 17, 33, 38)), ((48, 600, 70), (40, 6, 33)),
                                         ((64, 96, 120), (32,) * 9 + (31,))])
def test_mixed_batches_leave_the_fft_passes_their_fields(vfd, orc, shape, radii):
    """Batches of both forms, through both launch shapes of the FFT passes: one
    work-group per tile, and -- a plan that has itself made tables of the direct
    form only -- persistent launches walking the tiles of the fields that are
    theirs (more tiles than work-groups at the first two shapes; y columns long
    enough for narrow tiles at the second).  Every field has the bits it has
    alone, and both shapes match the oracle."""
    print(f"case mixed shape={shape} radii={radii}", flush=True)
    plan = vfd.Plan(shape, kspec_format=vfd.KSPEC_SEPARABLE)
    few = vfd.Plan(shape, kspec_format=vfd.KSPEC_SEPARABLE)
    few.gauss_spectrum(_s2(5), 0.97)
    u = orc.synth_field(shape, 77, nsrc=4)
    tables = [plan.gauss_spectrum(_s2(r), 0.97) for r in radii]
    refs = {r: orc.direct_separable(u, _s2(r), 0.97) for r in set(radii)}
    for p in (plan, few):
        got = _tick(vfd, p, u, tables)
        for r, t, g in zip(radii, tables, got):
            (alone,) = _tick(vfd, p, u, [t])
            assert np.array_equal(alone, g), r
            assert float(np.linalg.norm(g - refs[r]) / np.linalg.norm(refs[r])) <= 1e-5, r
