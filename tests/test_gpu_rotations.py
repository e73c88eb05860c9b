"""Gains of the transforms: the part of their error that has one sign.

The constants of a butterfly are the same on every path through it, so their
rounding scales the data by a factor of its own, the same on every call, where
all other roundings are as often up as down and vanish in the projection
<error, exact> / <exact, exact> over some 1e5 values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 64, 64), (128, 128, 128), (16, 512, 16)])
def test_double_round_trip_has_no_gain(vfd, shape):
    """R2C and back against long double.  1/sqrt(2) in one FP64 value is off by
    6.8e-17 of itself; its rotations take part in a quarter of each radix-8
    butterfly's outputs and more where stages follow each other, about 5e-17 an
    axis of 64 for the pair of transforms, 1.5e-16 over three.  Twiddle tables
    have no common sign.  Bound: half a unit roundoff, 5.6e-17."""
    import torch
    print(f"case double round trip {shape}", flush=True)
    plan = vfd.Plan(shape, shape, vfd.F64)
    u = np.random.default_rng(5).lognormal(-2.0, 1.0, shape)
    x = torch.from_numpy(u).cuda()
    spec = torch.empty(shape[:2] + (shape[2] // 2 + 1,), dtype=torch.complex128, device="cuda")
    back = torch.empty_like(x)
    plan.r2c(x, spec)
    plan.c2r(spec, back)
    torch.cuda.synchronize()
    ref = u.astype(np.longdouble) * np.longdouble(u.size)
    gain = float(((back.cpu().numpy().astype(np.longdouble) - ref) * ref).sum() / (ref * ref).sum())
    print(f"  gain {gain:.2e}", flush=True)
    assert abs(gain) <= 2.0 ** -54


def test_single_tick_gain_of_one_radix_16_lengths(vfd, orc):
    """Lengths whose power of two is 16 do it in one radix-16 butterfly, whose W16
    pair is picked for its magnitude; as radix 8 and 2 the same rotations come from
    the table, each rounded by itself.  The mean gain of streamed-spectrum ticks of
    48x48x48 is -3.9e-8 with the one and -6.5e-8 with the other: the bound lies
    halfway."""
    import torch
    n = 48
    print(f"case single gain {n}", flush=True)
    plan = vfd.Plan((n, n, n), kspec_format=vfd.KSPEC_REAL)
    gains = []
    for seed in range(6):
        u = orc.synth_field((n, n, n), 900 + seed)
        s2, dec = 2.0 * np.random.default_rng(seed).uniform(0.5, 5.0), 0.97
        ref = orc.direct_separable(u, s2, dec).astype(np.float64)
        out = torch.empty((n, n, n), device="cuda")
        plan.diffuse([{"in": torch.from_numpy(u).cuda(), "out": out, "work": plan.new_work(),
                       "kspec": plan.gauss_spectrum(s2, dec)}])
        torch.cuda.synchronize()
        gains.append(float(((out.cpu().numpy() - ref) * ref).sum() / (ref * ref).sum()))
    print(f"  gain {np.mean(gains):.2e}", flush=True)
    assert abs(np.mean(gains)) <= 5.2e-8


def test_double_tick_has_no_gain(vfd):
    """FP64 ticks against long double.  A window that is normalized to 1 in more than
    FP64 has a DFT of exactly 1 at zero frequency, where most of the field is; in FP64
    its sum and quotients miss 1 by up to some 5e-16 over three axes, by another
    amount for every sigma.  Left are the product of the tables and the decay, a few
    roundings of either sign at each frequency: bound, two roundings, 2.2e-16."""
    import torch
    shape, L = (64, 64, 64), np.longdouble
    print("case double tick gain", flush=True)
    plan = vfd.Plan(shape, precision=vfd.F64, kspec_format=vfd.KSPEC_SEPARABLE)
    rng = np.random.default_rng(8)
    worst = 0.0
    for s2 in (1.1, 1.7, 2.9, 3.7, 5.3, 7.1, 8.3, 9.7):
        u = rng.lognormal(-2.0, 1.0, shape)
        radius = int(np.ceil(6.0 * np.sqrt(s2)))
        j = np.arange(-radius, radius + 1).astype(L)
        g = np.exp(-j * j / (2 * L(s2)))
        g /= g.sum()
        ref = u.astype(L)
        for ax in range(3):
            n = shape[ax]
            m = np.zeros((n, n), dtype=L)
            for d in range(-radius, radius + 1):
                m += np.diag(np.full(n - abs(d), g[d + radius], dtype=L), d)
            ref = np.moveaxis(np.tensordot(m, np.moveaxis(ref, ax, 0), 1), 0, ax)
        out = torch.empty(shape, dtype=torch.float64, device="cuda")
        plan.diffuse([{"in": torch.from_numpy(u).cuda(), "out": out, "work": plan.new_work(),
                       "kspec": plan.gauss_spectrum(s2, 1.0)}])
        torch.cuda.synchronize()
        gain = float(((out.cpu().numpy().astype(L) - ref) * ref).sum() / (ref * ref).sum())
        print(f"  sigma^2 {s2}: gain {gain:.2e}", flush=True)
        worst = max(worst, abs(gain))
    assert worst <= 2.0 ** -52


@pytest.mark.parametrize("q", [16, 48, 80])
def test_one_radix_16_lengths_on_every_axis(vfd, orc, q):
    """FP32 rows of q, columns of q whole and split from 2 q, fused and not, in
    batches whose last tile is partial (q + 1 columns), with the streamed spectrum,
    wide separable tables (q of room for a radius of 36) and as plain transforms.
    Tolerance: rel-L2 1e-5 against the FP64 oracle, the transforms' eps log2 N."""
    import torch
    print(f"case lengths of {q}", flush=True)
    cases = [((q - 8, q, q), (q, 2 * q, 2 * q), vfd.KSPEC_REAL, 1.2), ((q, q - 8, q), (2 * q, q, 2 * q), vfd.KSPEC_REAL, 1.2)]
    if q > 36:
        cases.append(((q, q, q), (2 * q,) * 3, vfd.KSPEC_SEPARABLE, (35.5 / 6.0) ** 2))
    for shape, box, fmt, s2 in cases:
        plan = vfd.Plan(shape, box, vfd.F32, kspec_format=fmt)
        us = [orc.synth_field(shape, 40 + f, nsrc=5) for f in range(3)]
        outs = [torch.empty(shape, device="cuda") for _ in us]
        table = plan.gauss_spectrum(s2, 0.97)
        plan.diffuse([{"in": torch.from_numpy(u).cuda(), "out": o, "work": plan.new_work(), "kspec": table}
                      for u, o in zip(us, outs)])
        torch.cuda.synchronize()
        for u, o in zip(us, outs):
            assert orc.rel_l2(o.cpu().numpy(), orc.direct_separable(u, s2, 0.97)) <= 1e-5, (shape, box)
    box = (q, q, 2 * q)
    plan = vfd.Plan(box, box, vfd.F32)
    a = np.random.default_rng(q).standard_normal(box).astype(np.float32)
    spec = torch.empty(box[:2] + (q + 1,), dtype=torch.complex64, device="cuda")
    back = torch.empty(box, device="cuda")
    plan.r2c(torch.from_numpy(a).cuda(), spec)
    got = spec.cpu().numpy()
    plan.c2r(spec, back)
    ref = np.fft.rfftn(a.astype(np.float64))
    tol = 2.0 ** -23 * np.log2(a.size)
    assert np.abs(got - ref).max() <= tol * np.abs(ref).max()
    assert np.abs(back.cpu().numpy().astype(np.float64) / a.size - a).max() <= 2 * tol * np.abs(a).max()
