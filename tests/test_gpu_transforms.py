"""R2C and C2R over the R2C layout (px/2 + 1 elements a row), whose rows start on
128-byte lines: rows of less than a tile, of a tile plus one element, and columns
long enough for narrow tiles, against numpy's FP64 transform."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (pz, py, px); px/2 + 1 = 3, 9, 33, 65, 17, 10
BOXES = [(2, 2, 4), (6, 10, 16), (5, 9, 64), (16, 36, 128), (640, 6, 32), (4, 1536, 18)]


@pytest.mark.parametrize("box", BOXES, ids=lambda b: "x".join(map(str, b)))
@pytest.mark.parametrize("precision", [4, 8])
def test_transforms_row_alignments(vfd, box, precision):
    """Tolerance: a radix transform of N points in precision eps errs by at most
    about eps log2 N of its largest value; the round trip by twice that."""
    import torch
    print(f"case transforms box={box} precision={precision}", flush=True)
    rdt, cdt = (torch.float32, torch.complex64) if precision == 4 else (torch.float64, torch.complex128)
    n = int(np.prod(box))
    tol = float(torch.finfo(rdt).eps) * max(np.log2(n), 1.0)
    a = torch.from_numpy(np.random.default_rng(n).standard_normal(box)).to(rdt)
    plan = vfd.Plan(box, box, vfd.F32 if precision == 4 else vfd.F64)
    ad = a.cuda()
    # elements past the layout stay as they are
    hx = box[2] // 2 + 1
    room = torch.full((box[0] * box[1] * hx + 64,), 7.0, dtype=cdt, device="cuda")
    c = room[:box[0] * box[1] * hx].view(box[0], box[1], hx)
    plan.r2c(ad, c)
    torch.cuda.synchronize()
    ref = np.fft.rfftn(a.numpy().astype(np.float64))
    assert np.abs(c.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()
    back = torch.empty_like(ad)
    plan.c2r(c, back)
    torch.cuda.synchronize()
    assert (room[box[0] * box[1] * hx:] == 7.0).all()
    err = np.abs(back.cpu().numpy().astype(np.float64) / n - a.numpy()).max()
    assert err <= 2 * tol * np.abs(a.numpy()).max()
