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
