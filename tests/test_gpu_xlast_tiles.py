"""The z passes of the x-last order over batches of fields (each XCD takes a
contiguous run of tiles of all of them), in every schedule, against the FP64
oracle: short and long columns, odd and even row widths, tile counts that are no
multiple of 8, last tiles of one pair and full ones, both pads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL_F32 = 1e-5


@pytest.mark.parametrize("shape,box,pad,epi,base", [
    ((1100, 3, 11), (1152, 32, 32), 3, 8, 0.3),     # odd rows: the last pair has one column
    ((577, 8, 16), (1152, 32, 32), 100, 0, 0.0),    # whole tiles
    ((1152, 1, 30), (1152, 32, 32), 100, 0, 0.0),   # columns that fill the box
    ((1300, 5, 6), (1536, 32, 32), 3, 4, 0.4),      # a last tile of one pair
    ((3, 3, 3), (1536, 32, 32), 100, 0, 0.0),       # mostly padding, one tile a field
    ((40, 33, 25), (64, 64, 32), 3, 20, 0.2),       # short columns
    ((20, 17, 33), (32, 32, 64), 100, 0, 0.0),
    ((201, 100, 71), (256, 128, 128), 3, 60, 0.2),  # more than the L2s hold: no rows streamed
])
def test_z_tiles_of_a_batch_every_schedule(vfd, orc, monkeypatch, shape, box, pad, epi, base):
    """FP32 tolerance of the x-last order's other tests."""
    import torch
    print(f"case xlast long z shape={shape} box={box} pad={pad}", flush=True)
    us = [orc.synth_field(shape, 91 + f, nsrc=4) for f in range(3)]
    rng = np.random.default_rng(sum(shape))
    win = rng.random((5, 5, 5))
    spec = orc.kernel_spectrum(win / win.sum(), (2, 2, 2), box)
    refs = [orc.fft_diffuse3d(u, spec, box, pad, epi, base) for u in us]
    ks = torch.from_numpy(spec.astype(np.complex64)).cuda()
    uds = [torch.from_numpy(u).cuda() for u in us]
    monkeypatch.setenv("VFD_ORDER", str(vfd.ORDER_XLAST))
    plan = vfd.Plan(shape, box, vfd.F32, pad, vfd.KSPEC_COMPLEX_STD)
    assert plan.info.order == vfd.ORDER_XLAST
    for v in range(4):
        plan.schedule = [v] * 5
        outs = [torch.full_like(ud, float("nan")) for ud in uds]
        plan.diffuse([{"in": ud, "out": out, "work": plan.new_work(), "kspec": ks, "base": base, "epi": epi}
                      for ud, out in zip(uds, outs)])
        torch.cuda.synchronize()
        for f, (out, ref) in enumerate(zip(outs, refs)):
            got = out.cpu().numpy().astype(np.float64)
            rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
            print(f"schedule {v} field {f}: rel-L2 {rel:.3e}", flush=True)
            assert rel <= REL_F32
