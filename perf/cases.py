"""The work that users of the diffusion layer have it do, as measurable cases.

listed() names the cases and draw() gives more of the same ranges; prepare()
makes what a program holds before a tick (fields, plans, spectra, an engine
with resident runs), run() is one pass through the public entry points,
exact() the same pass in 64 bits without this package, and work() the bytes
and operations a pass cannot do without.

Fields follow the workloads of bench.py: lognormal(-2, 1) background plus 50
point sources of U[1, 100], sigma^2 = 2 D with D ~ U[0.5, 5], decay
exp(-lambda) with lambda ~ U[0.001, 0.05], drawn from the seed.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vf-version_7_3_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import vfd  # noqa: E402
from vfd import engine, legacy  # noqa: E402

DEV = "cuda:0"
CHEM_DECAY = [0.319, 0.00003052, 0.67, 0.2, 0.2, 0.7937, 0.9284, 0.2]
IL1B, TNF, TGF, FGF, IL6, IL8 = 4, 0, 1, 2, 5, 6  # chem indices of the gradient sums


def listed():
    return [
        # The tissue-scale tick of the benchmark: 8 cytokine fields of one large
        # world, a Gaussian kernel per field, all fields in one batched call.
        _field("tissue_1024x512x128_8f", 128, 512, 1024, 8),
        # The smallest world: a tick of a few tens of microseconds, where
        # launches and latency count.
        _field("patch_64x64x32_8f", 32, 64, 64, 8),
        # An ordinary world with odd extents on every axis (no row aligned, no
        # box a power of two).
        _field("odd_301x187x75_8f", 75, 187, 301, 8),
        # The full-precision path, used where 100-tick mass conservation matters.
        _field("double_256x128x64_4f", 64, 128, 256, 4, f64=True),
        # A kernel that is streamed as a 3D real spectrum (the form any even
        # kernel takes, separable or not).
        _field("spectrum_512x256x64_8f", 64, 256, 512, 8, spectrum="real"),
        # The ABM's own production tick: fftDiffuse3D of its 8 chems (constant-VF
        # pad, complex spectra) on the HUMAN_VF grid and FFT box.
        _abm("abm_human_1006x1390x110_8f", 1006, 1390, 110, 1152, 1536, 256, 8, 73),
        # The same entry point on a small world: box by the snapTransformSize rule.
        _abm("abm_small_60x100x142_8f", 142, 100, 60, 256, 128, 128, 8, 14),
        # The resident chem tick over PCIe (vfdTickChems): deltas and fragments in,
        # diffusion and update, levels and gradients out, pinned host arrays.
        {"name": "abm_hosttick_192x128x96", "kind": "hosttick", "nz": 96, "ny": 128, "nx": 192,
         "pz": 128, "py": 256, "px": 256, "radius": 15},
        # The device-resident chem tick: diffusion with the chem update, gradients
        # and totals fused, in place.
        {"name": "chemtick_512x256x64", "kind": "chemtick", "nz": 64, "ny": 256, "nx": 512},
        # A sensitivity-analysis ensemble: runs of uneven grids advanced one tick by
        # one graph launch.
        {"name": "ensemble_7runs_8f", "kind": "ensemble", "fields": 8,
         "runs": "32x64x64,32x64x64,64x128x128,64x128x128,64x128x256,64x256x256,64x256x512"},
        # Requests of concurrent small runs through the server: submit all, wait for all.
        {"name": "serve_6runs_8f", "kind": "serve", "fields": 8,
         "runs": "32x64x64,32x64x64,32x64x64,64x128x128,64x128x128,64x128x256"},
        # Standalone transforms (the kernel-spectrum precompute): R2C of a real box
        # and C2R back.
        {"name": "transform_256x256x192", "kind": "transform", "nz": 192, "ny": 256, "nx": 256, "f64": False},
    ]


def _field(name, nz, ny, nx, fields, f64=False, spectrum="separable"):
    return {"name": name, "kind": "field", "nz": nz, "ny": ny, "nx": nx, "fields": fields, "f64": f64,
            "spectrum": spectrum}


def _abm(name, nz, ny, nx, pz, py, px, fields, radius):
    return {"name": name, "kind": "abm", "nz": nz, "ny": ny, "nx": nx, "pz": pz, "py": py, "px": px,
            "fields": fields, "radius": radius}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _snap(n):
    """snapTransformSize: the multiple of 16 if it is a power of two, else the next power of two."""
    return 1 << (max(16, n) - 1).bit_length()


def draw(rng):
    kind = rng.choice(["field", "field", "field", "field", "double", "real", "abm", "abm", "hosttick", "chemtick",
                       "ensemble", "transform"])
    if kind in ("field", "double", "real", "chemtick"):
        while True:
            nz, ny, nx = _log(rng, 20, 160), _log(rng, 24, 640), _log(rng, 32, 1200)
            nf = 8 if kind == "chemtick" else rng.randint(1, 8)
            n = nz * ny * nx * nf
            if n <= (6e7 if kind != "field" else 3e8):
                break
        if kind == "chemtick":
            return {"kind": "chemtick", "nz": nz, "ny": ny, "nx": nx}
        c = _field("", nz, ny, nx, nf, kind == "double", "real" if kind == "real" else "separable")
        del c["name"]
        return c
    if kind in ("abm", "hosttick"):
        while True:
            nz, ny, nx, r = _log(rng, 30, 500), _log(rng, 30, 500), _log(rng, 30, 300), rng.randint(5, 20)
            box = [_snap(n + 2 * r) for n in (nz, ny, nx)]
            if box[0] * box[1] * box[2] <= (1 << 27 if kind == "abm" else 1 << 24):
                break
        if kind == "hosttick":
            return {"kind": "hosttick", "nz": nz, "ny": ny, "nx": nx, "pz": box[0], "py": box[1], "px": box[2],
                    "radius": r}
        c = _abm("", nz, ny, nx, *box, rng.randint(1, 8), r)
        del c["name"]
        return c
    if kind == "ensemble":
        grids = ["x".join(str(_log(rng, lo, hi)) for lo, hi in ((24, 96), (48, 256), (48, 512)))
                 for _ in range(rng.randint(2, 3))]
        return {"kind": "ensemble", "fields": rng.randint(2, 8),
                "runs": ",".join(rng.choice(grids) for _ in range(rng.randint(3, 7)))}
    n = [rng.choice([32, 48, 64, 96, 128, 192, 256, 320]) for _ in range(3)]
    return {"kind": "transform", "nz": n[0], "ny": n[1], "nx": n[2], "f64": rng.random() < 0.5}


# ------------------------------------------------------------------- inputs
def _shape(c):
    return c["nz"], c["ny"], c["nx"]


def _box(c):
    return c["pz"], c["py"], c["px"]


def _runs(c):
    return [tuple(int(v) for v in r.split("x")) for r in c["runs"].split(",")]


def _fields(shape, n, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) % (1 << 62))
    vox = shape[0] * shape[1] * shape[2]
    out = []
    for _ in range(n):
        f = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).add_(-2.0).exp_()
        at = torch.randint(0, vox, (50,), generator=g, device=DEV).unique()
        amp = torch.rand(at.numel(), generator=g, device=DEV) * 99.0 + 1.0
        f.view(-1)[at] += amp
        out.append(f)
    return out


def _params(shape, n, seed):
    """(sigma^2, decay) per field; D is bounded where a short axis leaves less zero padding than its window."""
    rng = np.random.default_rng(int(seed) % (1 << 62))
    dmax = min(5.0, 0.98 * ((min(shape) - 1) / 6.0) ** 2 / 2.0)
    D, lam = rng.uniform(0.5, dmax, n), rng.uniform(0.001, 0.05, n)
    return [(2.0 * float(d), float(np.exp(-v))) for d, v in zip(D, lam)]


def _chem_inputs(shape, seed):
    """Agents' deltas of the 8 chems and the two ECM fragment fields."""
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 7 + 3) % (1 << 62))
    deltas = [torch.rand(shape, generator=g, device=DEV) * 0.01 for _ in range(8)]
    return deltas, torch.rand(shape, generator=g, device=DEV), torch.rand(shape, generator=g, device=DEV)


def _window(sigma2, radius=None):
    """The normalized sampled Gaussian g[j + R], |j| <= R = ceil(6 sigma)."""
    R = int(math.ceil(6.0 * math.sqrt(sigma2))) if radius is None else radius
    j = np.arange(-R, R + 1, dtype=np.float64)
    g = np.exp(-j * j / (2.0 * sigma2))
    return g / g.sum()


def _abm_spectra(c, n, seed):
    """Complex R2C-layout spectra of n chems' kernels: a Gaussian window of the case's radius, times a decay."""
    pz, py, px = _box(c)
    rng = np.random.default_rng(int(seed) % (1 << 62))
    out = []
    for _ in range(n):
        g = _window((c["radius"] * rng.uniform(0.12, 0.2)) ** 2, c["radius"])
        R, ax = c["radius"], []
        for p, half in ((pz, False), (py, False), (px, True)):
            w = np.zeros(p)
            for i, v in enumerate(g):
                w[(i - R) % p] += v
            ax.append(torch.from_numpy((np.fft.rfft(w) if half else np.fft.fft(w)).real.copy()).to(DEV))
        ax[0] = ax[0] * math.exp(-rng.uniform(0.001, 0.05))
        k = (ax[0][:, None] * ax[1][None, :]).to(torch.float32)[:, :, None] * ax[2].to(torch.float32)[None, None, :]
        out.append(torch.complex(k, torch.zeros_like(k)))
        del k
    return out


def _abm_context(c, data, spectra):
    cc = legacy.CCtx()
    cc.DD, cc.DH, cc.DW = _shape(c)
    cc.FFTD, cc.FFTH, cc.FFTW = _box(c)
    cc.KD = cc.KH = cc.KW = 2 * c["radius"] + 1
    cc.KZ = cc.KY = cc.KX = c["radius"]
    for i in range(len(data)):
        cc.d_data[i] = data[i].data_ptr()
        cc.d_kernelspectrum_h[i] = spectra[i].data_ptr()
    return cc


def _base(n):
    return [0.01 * (i + 1) for i in range(n)]


class _Resident:
    """A run's resident field as the array that field_ptr names (kept with its engine)."""

    def __init__(self, eng, rid, f, shape):
        self.eng = eng
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (eng.field_ptr(rid, f), False),
                                         "version": 2}


_tuned = set()


def _plan(shape, precision, fmt, nfields):
    """A plan with its schedule autotuned, once per shape in the process (later plans of the shape take it up)."""
    p = vfd.Plan(shape, precision=precision, kspec_format=fmt)
    key = (shape, precision, fmt)
    if key not in _tuned and precision == vfd.F32:
        p.autotune(nfields)
        _tuned.add(key)
    return p


def prepare(case, seed):
    k = case["kind"]
    st = {"case": case}
    if k == "field":
        shape, n = _shape(case), case["fields"]
        fmt = vfd.KSPEC_REAL if case["spectrum"] == "real" else vfd.KSPEC_SEPARABLE
        plan = _plan(shape, vfd.F64 if case["f64"] else vfd.F32, fmt, n)
        u = _fields(shape, n, seed)
        if case["f64"]:
            u = [x.double() for x in u]
        out = [torch.empty_like(x) for x in u]
        work = [plan.new_work() for _ in u]
        ks = [plan.gauss_spectrum(s2, dec) for s2, dec in _params(shape, n, seed)]
        st.update(plan=plan, out=out, arr=plan.field_array(
            [{"in": u[i], "out": out[i], "work": work[i], "kspec": ks[i]} for i in range(n)]))
    elif k == "abm":
        data = _fields(_shape(case), case["fields"], seed)
        spectra = _abm_spectra(case, case["fields"], seed)
        st.update(data=data, spectra=spectra, cc=_abm_context(case, data, spectra), base=_base(case["fields"]))
    elif k == "hosttick":
        shape = _shape(case)
        data, spectra = _fields(shape, 8, seed), _abm_spectra(case, 8, seed)
        deltas, col, ela = _chem_inputs(shape, seed)
        cc = _abm_context(case, data, spectra)
        levels = [x.cpu().pin_memory() for x in data]
        deltas = [x.cpu().pin_memory() for x in deltas]
        col, ela = col.cpu().pin_memory(), ela.cpu().pin_memory()
        grads = [torch.empty(shape, dtype=torch.float32, pin_memory=True) for _ in range(3)]
        for i in range(8):
            cc.h_ibuffs[i] = levels[i].data_ptr()
        st.update(data=data, spectra=spectra, cc=cc, levels=levels, deltas=deltas, col=col, ela=ela, grads=grads,
                  base=(ctypes.c_float * 8)(*_base(8)), decay=(ctypes.c_float * 8)(*CHEM_DECAY),
                  dptr=(ctypes.c_void_p * 8)(*[x.data_ptr() for x in deltas]),
                  gptr=(ctypes.c_void_p * 3)(*[x.data_ptr() for x in grads]))
    elif k == "chemtick":
        shape = _shape(case)
        plan = _plan(shape, vfd.F32, vfd.KSPEC_SEPARABLE, 8)
        u = _fields(shape, 8, seed)
        deltas, col, ela = _chem_inputs(shape, seed)
        work = [plan.new_work() for _ in u]
        ks = [plan.gauss_spectrum(s2, dec) for s2, dec in _params(shape, 8, seed)]
        st.update(plan=plan, levels=u, deltas=deltas, col=col, ela=ela, grads=[torch.empty_like(col) for _ in range(3)],
                  arr=plan.field_array([{"in": u[i], "out": u[i], "work": work[i], "kspec": ks[i]} for i in range(8)]))
    elif k in ("ensemble", "serve"):
        eng = engine.Engine(64 << 30)
        ids, views = [], []
        for r, shape in enumerate(_runs(case)):
            par = _params(shape, case["fields"], seed * 64 + r)
            rid = eng.create_run(shape, [p[0] for p in par], [p[1] for p in par])
            for f, u in enumerate(_fields(shape, case["fields"], seed * 64 + r)):
                eng.write_field(rid, f, u)
            torch.cuda.synchronize()
            ids.append(rid)
            views += [torch.as_tensor(_Resident(eng, rid, f, shape), device=DEV) for f in range(case["fields"])]
        if k == "serve":
            eng.serve_start(slots=4)
        st.update(eng=eng, ids=ids, views=views)
    else:
        shape = _shape(case)
        plan = vfd.Plan(shape, shape, vfd.F64 if case["f64"] else vfd.F32)
        u = _fields(shape, 1, seed)[0]
        if case["f64"]:
            u = u.double()
        half = shape[:2] + (shape[2] // 2 + 1,)
        ct = torch.complex128 if case["f64"] else torch.complex64
        st.update(plan=plan, u=u, spec=torch.empty(half, dtype=ct, device=DEV), back=torch.empty_like(u))
    return st


# --------------------------------------------------------------------- passes
def run(st):
    k = st["case"]["kind"]
    if k == "field":
        st["plan"].diffuse(st["arr"])
        return st["out"]
    if k == "abm":
        cc, lib = st["cc"], legacy.lib
        epi = st["case"]["nx"] - 4
        for i in range(len(st["data"])):
            if not lib.fftDiffuse3D(cc.d_data[i], cc.d_kernelspectrum_h[i], 0, 0, cc, epi, st["base"][i], i, 0):
                raise RuntimeError(vfd.last_error())
        return st["data"]
    if k == "hosttick":
        totals = (ctypes.c_double * 8)()
        if not legacy.lib.vfdTickChems(st["cc"], st["case"]["nx"] - 4, st["base"], st["dptr"], st["decay"],
                                       st["col"].data_ptr(), st["ela"].data_ptr(), st["gptr"], totals):
            raise RuntimeError(vfd.last_error())
        return {"levels": st["levels"], "grads": st["grads"], "deltas": st["deltas"], "totals": list(totals)}
    if k == "chemtick":
        totals = st["plan"].diffuse_update(st["arr"], st["deltas"], CHEM_DECAY, st["col"], st["ela"], st["grads"])
        return {"levels": st["levels"], "grads": st["grads"], "deltas": st["deltas"], "totals": totals}
    if k == "ensemble":
        st["eng"].step(st["ids"], graph=True)
        return st["views"]
    if k == "serve":
        eng = st["eng"]
        for t in [eng.submit(r) for r in st["ids"]]:
            eng.wait(t)
        return st["views"]
    st["plan"].r2c(st["u"], st["spec"])
    st["plan"].c2r(st["spec"], st["back"])
    return st["back"]


# ---------------------------------------------------------------- 64-bit truth
def _exact_gauss(u, sigma2, decay):
    """The linear convolution with the window along each axis (zero outside), times the decay."""
    g = _window(sigma2)
    R = (len(g) - 1) // 2
    v = u.double()
    for ax in range(3):
        n = v.shape[ax]
        acc = v * float(g[R])
        for j in range(1, min(R, n - 1) + 1):
            w = float(g[R + j])
            acc.narrow(ax, j, n - j).add_(v.narrow(ax, 0, n - j), alpha=w)
            acc.narrow(ax, 0, n - j).add_(v.narrow(ax, j, n - j), alpha=w)
        v = acc
    return v * decay


def _exact_abm(c, u, spec, base, epi):
    """fftDiffuse3D in 64 bits: constant-VF pad, product with the spectrum, crop."""
    (nz, ny, nx), (pz, py, px) = _shape(c), _box(c)
    box = torch.full((pz, py, px), base, dtype=torch.float64, device=DEV)
    e = min(epi, nx)
    box[1:nz - 1, 1:ny - 1, 1:e] = u[1:nz - 1, 1:ny - 1, 1:e].double()
    f = torch.fft.rfftn(box)
    del box
    f.mul_(spec)
    return torch.fft.irfftn(f, s=(pz, py, px))[:nz, :ny, :nx].clone()


def _exact_update(t, deltas, col, ela):
    lv = [d.double() + x * np.float64(np.float32(w)) for d, x, w in zip(deltas, t, CHEM_DECAY)]
    g = lv[IL1B] + lv[TNF] + lv[TGF] + lv[FGF] + col.double()
    return {"levels": lv, "grads": [g + lv[IL6] + lv[IL8], g + ela.double(), lv[TGF]],
            "deltas": [torch.zeros_like(x) for x in lv], "totals": [float(x.sum()) for x in lv]}


def exact(case, seed):
    k = case["kind"]
    if k == "field":
        shape, n = _shape(case), case["fields"]
        return [_exact_gauss(u, *p) for u, p in zip(_fields(shape, n, seed), _params(shape, n, seed))]
    if k == "abm":
        n = case["fields"]
        us, spectra = _fields(_shape(case), n, seed), _abm_spectra(case, n, seed)
        return [_exact_abm(case, us[i], spectra[i], float(np.float32(b)), case["nx"] - 4)
                for i, b in enumerate(_base(n))]
    if k == "hosttick":
        us, spectra = _fields(_shape(case), 8, seed), _abm_spectra(case, 8, seed)
        t = [_exact_abm(case, us[i], spectra[i], float(np.float32(b)), case["nx"] - 4) for i, b in enumerate(_base(8))]
        return _exact_update(t, *_chem_inputs(_shape(case), seed))
    if k == "chemtick":
        shape = _shape(case)
        t = [_exact_gauss(u, *p) for u, p in zip(_fields(shape, 8, seed), _params(shape, 8, seed))]
        return _exact_update(t, *_chem_inputs(shape, seed))
    if k in ("ensemble", "serve"):
        out = []
        for r, shape in enumerate(_runs(case)):
            us = _fields(shape, case["fields"], seed * 64 + r)
            out += [_exact_gauss(u, *p) for u, p in zip(us, _params(shape, case["fields"], seed * 64 + r))]
        return out
    return _fields(_shape(case), 1, seed)[0].double() * float(np.prod(_shape(case)))


# ------------------------------------------------------------- necessary work
def work(case):
    k = case["kind"]
    # a separable window of the mean D = 2.75: radius 15, three axes
    window = 3 * 2 * 31
    if k in ("ensemble", "serve"):
        n = sum(a * b * c for a, b, c in _runs(case)) * case["fields"]
        return {"bytes": 8.0 * n, "flops": float(window * n)}
    n = float(case["nz"] * case["ny"] * case["nx"])
    if k == "transform":
        s = 8 if case["f64"] else 4
        return {"bytes": 4 * s * n, "flops": 2 * 2.5 * n * math.log2(n)}
    if k == "chemtick":
        # levels and deltas read and written, fragments read, gradients written
        return {"bytes": 4 * (4 * 8 + 2 + 3) * n, "flops": 8 * (window + 4.0) * n}
    if k == "field":
        s = 8 if case["f64"] else 4
        if case["spectrum"] == "real":
            # the field's data and its real half spectrum on the doubled box
            box = 8 * n
            return {"bytes": case["fields"] * (2 * s * n + s * box / 2),
                    "flops": case["fields"] * 5.0 * n * math.log2(box)}
        return {"bytes": 2 * s * n * case["fields"], "flops": window * n * case["fields"]}
    nf = case.get("fields", 8)
    box = float(case["pz"] * case["py"] * case["px"])
    bytes_ = nf * (8 * n + 8 * case["pz"] * case["py"] * (case["px"] // 2 + 1))
    if k == "hosttick":
        bytes_ += 4 * (8 + 2 + 8 + 3) * n  # the host arrays, each read or written once
    return {"bytes": float(bytes_), "flops": nf * 5.0 * n * math.log2(box)}
