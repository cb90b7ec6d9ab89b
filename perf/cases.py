"""The work that users of this package have it do, as measurable cases.

A case is one call through a public entry point on a tilt series:

- ``plan``: a device-resident volume plan (``VolumePlan.run``), the path of a
  program that keeps its data on the GPU: projections, CTF-corrected
  projections or sinograms in, the volume out, in one of three slab storages;
- ``volume``: ``reconstruct_projections`` on host arrays, the fused path of a
  Python program;
- ``correct``: ``correct_projections`` on host arrays, the first half of the
  two-step route;
- ``slice``: ``recon``, one slice at a time from host memory, as per-slice
  workers call it.

Images are electron counts: 40 e-/px Poisson noise over the projections of a
phantom of random ellipsoids. The microscope is the one the package's
workloads use (300 kV, Cs 2.7 mm, 0.1 amplitude contrast).
"""
import math

import numpy
import torch

import guanaco_amd as G
from guanaco_amd import _capi as C

DEFOCUS = 30000.0    # A, at the tilt axis
CS = 2.7             # mm
PHI = math.asin(0.1)  # rad
DOSE = 40.0          # electrons per pixel


def listed():
    return [
        # One slice, one defocus: the smallest call there is.
        dict(name="slice_256", kind="slice", X=256, T=61, ndf=1, Z=256,
             pixel=2.0),
        # One slice of an odd-sized detector with eight defocus slabs.
        dict(name="slice_1500_df8", kind="slice", X=1500, T=90, ndf=8, Z=300,
             pixel=1.0),
        # Phase flipping alone, a few tilts at a time, from host memory.
        dict(name="correct_512_df8", kind="correct", X=512, Y=512, T=9,
             ndf=8, pixel=2.0),
        # A whole small reconstruction from a Python program's host arrays.
        dict(name="volume_512_df4_f16", kind="volume", X=512, Y=512, T=41,
             ndf=4, Z=128, pixel=2.0, storage="f16"),
        # Plain filtered backprojection of a small series, no CTF.
        dict(name="plan_256_f32", kind="plan", X=256, Y=256, T=61, ndf=1,
             Z=256, pixel=2.0, storage="f32", layout="projections",
             ctf=False, drift=0.0),
        # An ordinary series, one defocus, in the fast storage ...
        dict(name="plan_1024_ctf_f16", kind="plan", X=1024, Y=1024, T=121,
             ndf=1, Z=256, pixel=2.0, storage="f16", layout="projections",
             ctf=True, drift=0.0),
        # ... and several defoci in the exact one.
        dict(name="plan_1024_df8_f32", kind="plan", X=1024, Y=1024, T=61,
             ndf=8, Z=256, pixel=2.0, storage="f32", layout="projections",
             ctf=True, drift=0.0),
        # Already corrected stacks in the third storage.
        dict(name="plan_1024_corrected_bf16", kind="plan", X=1024, Y=512,
             T=41, ndf=4, Z=256, pixel=2.0, storage="bf16",
             layout="corrected", ctf=False, drift=0.0),
        # Detectors that are no power of two: the sizes of the reference's
        # own test data, and a binned camera frame.
        dict(name="plan_1500x200_df8_f32", kind="plan", X=1500, Y=200, T=90,
             ndf=8, Z=300, pixel=1.0, storage="f32", layout="projections",
             ctf=True, drift=0.0),
        dict(name="plan_960x928_df4_f16", kind="plan", X=960, Y=928, T=41,
             ndf=4, Z=200, pixel=3.0, storage="f16", layout="projections",
             ctf=True, drift=0.0),
        # One rotation centre per slice: a tilt axis that is not quite
        # parallel to the detector's columns.
        dict(name="plan_512_centres_f32", kind="plan", X=512, Y=512, T=61,
             ndf=1, Z=128, pixel=2.0, storage="f32", layout="sinograms",
             ctf=False, drift=3.0),
        # The largest that fits: full defocus-range correction.
        dict(name="plan_2048_df16_f16", kind="plan", X=2048, Y=2048, T=61,
             ndf=16, Z=512, pixel=1.5, storage="f16", layout="projections",
             ctf=True, drift=0.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A detector length: a power of two, a multiple of 16 or any number."""
    n = _log_int(rng, lo, hi)
    how = rng.random()
    if how < 0.45:
        return 1 << int(round(math.log2(n)))
    return max(16, n // 16 * 16) if how < 0.75 else n


def draw(rng):
    pixel = round(rng.uniform(1.0, 4.0), 2)
    T = rng.randrange(21, 122)
    ndf = rng.choice([1, 1, 2, 3, 4, 6, 8, 12, 16])
    kind = rng.choice(["slice", "correct", "volume", "plan", "plan", "plan",
                       "plan"])
    if kind == "slice":
        X = _size(rng, 128, 2048)
        return dict(kind=kind, X=X, T=T, ndf=ndf,
                    Z=_log_int(rng, 64, min(X, 1024)), pixel=pixel)
    if kind == "correct":
        return dict(kind=kind, X=_size(rng, 128, 1024),
                    Y=_size(rng, 128, 1024), T=rng.randrange(2, 12),
                    ndf=min(ndf, 8), pixel=pixel)
    storage = rng.choice(["f32", "f16", "f16", "bf16"])
    top = 768 if kind == "volume" else 2048
    X, Y = _size(rng, 128, top), _size(rng, 64, top)
    Z = _log_int(rng, 32, max(33, X // 3))
    case = dict(kind=kind, X=X, Y=Y, T=T, ndf=ndf, Z=Z, pixel=pixel,
                storage=storage)
    if kind == "plan":
        layout = rng.choice(["projections", "projections", "corrected",
                             "sinograms"])
        ctf = layout == "projections" and (ndf > 1 or rng.random() < 0.6)
        drift = round(rng.uniform(0.5, 4.0), 2) if rng.random() < 0.12 else 0.0
        case.update(layout=layout, ctf=ctf, drift=drift)
    # no more than the largest listed one: voxels times tilts, and images
    while X * case["Y"] * case["Z"] * case["T"] > 4e10 or \
            X * case["Y"] * case["T"] * ndf > 1e9:
        case["Y"] = max(48, case["Y"] // 2)
        case["Z"] = max(24, case["Z"] * 3 // 4)
        case["T"] = max(15, case["T"] * 3 // 4)
    return case


# ------------------------------------------------------------------ inputs --

def _angles(T):
    return numpy.deg2rad(numpy.linspace(-60.0, 60.0, T)).astype(numpy.float32)


def _phantom(seed, T, Y, X, Z, device):
    """(T, Y, X) line integrals of random ellipsoids, largest value 1."""
    rng = numpy.random.default_rng(seed)
    a = torch.tensor(_angles(T), dtype=torch.float32, device=device)
    u = torch.arange(X, dtype=torch.float32, device=device) + 0.5 - X / 2
    v = torch.arange(Y, dtype=torch.float32, device=device) + 0.5
    out = torch.zeros((T, Y, X), dtype=torch.float32, device=device)
    for _ in range(8):
        x, z = rng.uniform(-0.4, 0.4) * X, rng.uniform(-0.4, 0.4) * Z
        y, d = rng.uniform(0, 1) * Y, rng.uniform(0.1, 1.0)
        r = rng.uniform(0.03, 0.12, 3) * (X, Y, X)
        cos, sin = torch.cos(a), torch.sin(a)
        w2 = (r[0] * cos) ** 2 + (r[2] * sin) ** 2
        p = (u[None, :] - (x * cos - z * sin)[:, None]) ** 2 / w2[:, None]
        q = ((v - y) / r[1]) ** 2
        height = d * 2 * r[0] * r[2] / torch.sqrt(w2)
        out += height[:, None, None] * torch.sqrt(
            (1 - p[:, None, :] - q[None, :, None]).clamp_(min=0))
    return out / out.max().clamp(min=1e-6)


def _counts(seed, T, Y, X, Z):
    """(T, Y, X) electron counts, on the GPU."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    mean = _phantom(seed, T, Y, X, Z, "cuda").mul_(0.2 * DOSE).add_(DOSE)
    return torch.poisson(mean, generator=gen)


def _defoci(case):
    """Absolute defoci of the slabs and the range relative to the axis."""
    ndf = case["ndf"]
    if ndf == 1:
        return numpy.array([DEFOCUS]), 0.0, 0.0
    half = case["X"] / 2.0 * case["pixel"]
    step = 2 * half / (ndf - 1)
    return (DEFOCUS - half) + step * numpy.arange(ndf), -half, half


def _wavelength():
    """A, relativistic, 300 kV."""
    m, c, e, h = 9.10938356e-31, 299792458.0, 1.60217662e-19, 6.62607004e-34
    V = 300000.0
    return h / math.sqrt(2 * m * e * V * (1 + e * V / (2 * m * c * c))) * 1e10


def _series(case, seed):
    """What the entry point reads, as a float32 tensor on the GPU."""
    X, T, ndf = case["X"], case["T"], case["ndf"]
    if case["kind"] == "slice":  # (ndf, T, X): counts, one row per defocus
        s = _counts(seed, T, ndf, X, case["Z"])
        return s.permute(1, 0, 2).contiguous()
    if case["kind"] == "plan" and case["layout"] != "projections":
        # a row's defocus slabs differ by noise, as corrected ones do
        s = torch.stack([_counts(seed + 7919 * k, T, case["Y"], X, case["Z"])
                         for k in range(ndf)], 1)          # (T, ndf, Y, X)
        if case["layout"] == "sinograms":
            s = s.permute(2, 1, 0, 3)                      # (Y, ndf, T, X)
        return s.contiguous()
    return _counts(seed, T, case["Y"], X, case.get("Z", X))


def _centres(case):
    """One rotation centre, or one per row."""
    mid = case["X"] / 2.0
    if not case.get("drift"):
        return mid
    return (mid + numpy.linspace(-1, 1, case["Y"]) * case["drift"]).astype(
        numpy.float32)


def prepare(case, seed):
    state = dict(case=case, angles=_angles(case["T"]))
    series = _series(case, seed)
    if case["kind"] != "plan":
        state["series"] = series.cpu().numpy()
        if case["kind"] == "slice":
            if case["ndf"] == 1:
                state["series"] = state["series"][0]
            state["out"] = numpy.zeros((case["Z"], case["X"]), numpy.float32)
        elif case["kind"] == "correct":
            state["out"] = numpy.zeros(
                (case["T"], case["ndf"], case["Y"], case["X"]), numpy.float32)
        else:
            state["out"] = numpy.zeros((case["Y"], case["Z"], case["X"]),
                                       numpy.float32)
        return state
    defoci, mn, mx = _defoci(case)
    kw = dict(num_defocus=case["ndf"], pixel_size=case["pixel"],
              centre=_centres(case), min_defocus=mn, max_defocus=mx,
              storage=case["storage"],
              input_layout={"projections": C.INPUT_PROJECTIONS,
                            "corrected": C.INPUT_CORRECTED,
                            "sinograms": C.INPUT_SINOGRAMS}[case["layout"]])
    if case["ctf"]:
        kw.update(defocus=defoci, wavelength=_wavelength(), Cs=CS * 1e7,
                  phi=PHI)
    state["plan"] = C.VolumePlan(case["X"], case["Y"], state["angles"],
                                 case["Z"], **kw)
    vol = torch.empty((case["Y"], case["Z"], case["X"]), device="cuda")
    state.update(series=series, volume=vol,
                 d_in=C.DeviceView(series.data_ptr(), series.shape),
                 d_vol=C.DeviceView(vol.data_ptr(), vol.shape))
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "plan":
        state["plan"].run(state["d_in"], state["d_vol"])
        return state["volume"]
    _, mn, mx = _defoci(case)
    if case["kind"] == "slice":
        G.recon(state["series"], state["out"], state["angles"],
                case["X"] / 2.0, case["pixel"], mn, mx, "gpu", 0)
        return state["out"]
    if case["kind"] == "correct":
        out, lo, hi = G.correct_projections(
            state["series"], None, case["pixel"], 300, DEFOCUS, case["ndf"],
            None, CS, 0, 0, math.degrees(PHI), state["out"], "gpu")
        return {"corrected": out, "range": [float(lo), float(hi)]}
    return G.reconstruct_projections(
        state["series"], state["angles"], pixel_size=case["pixel"],
        energy=300, defocus=DEFOCUS, num_defocus=case["ndf"],
        spherical_aberration=CS, phase_shift=math.degrees(PHI),
        depth=case["Z"], storage=case["storage"],
        reconstruction=state["out"])


# -------------------------------------------------------------- least work --

def work(case):
    X, T, ndf = case["X"], case["T"], case["ndf"]
    Y = case.get("Y", 1)
    corrects = case["kind"] in ("correct", "volume") or case.get("ctf", False)
    images = T * Y * X * (1 if corrects else ndf)
    nbytes, flops = 4.0 * images, 0.0
    if corrects:
        # a real 2D transform of each image, one inverse for each defocus
        flops += 2.5 * T * (1 + ndf) * X * Y * math.log2(X * Y)
    if case["kind"] == "correct":
        nbytes += 4.0 * T * ndf * Y * X
    else:
        # filtering of zero-padded real rows, two taps for each voxel and tilt
        flops += T * ndf * Y * 2 * 2.5 * 2 * X * math.log2(2 * X)
        flops += 4.0 * T * Y * case["Z"] * X
        nbytes += 4.0 * Y * case["Z"] * X
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------- the exact results --

def _flips(case):
    """-sign of the CTF of each defocus on the FFT grid, (ndf, Y, X)."""
    X, Y = case["X"], case["Y"]
    fx = torch.fft.fftfreq(X, case["pixel"], dtype=torch.float64)
    fy = torch.fft.fftfreq(Y, case["pixel"], dtype=torch.float64)
    q2 = (fx[None, :] ** 2 + fy[:, None] ** 2).cuda()
    l = _wavelength()
    cs = CS * 1e7
    defoci = _defoci(case)[0]
    return [-torch.sign(torch.sin(-(math.pi * (
        cs * l ** 3 * q2 * q2 / 2 - l * float(d) * q2) - PHI)))
        for d in defoci]


def _filtered(rows):
    """Ramp-filtered rows (last axis), zero-padded to twice their length."""
    N = rows.shape[-1]
    ramp = torch.arange(N + 1, dtype=torch.float64, device=rows.device) / N
    return torch.fft.irfft(torch.fft.rfft(rows, 2 * N) * ramp,
                           2 * N)[..., :N]


def _geometry(T, centre):
    """Per tilt: cos, sin, offset and scale in the float32 arithmetic that
    defines them."""
    f = numpy.float32
    out = []
    for a in _angles(T):
        c, s = f(math.cos(float(a))), f(math.sin(float(a)))
        x0, y0 = f(-f(centre) * c), f(-f(centre) * s)
        d = f(f(c * c) + f(s * s))
        off = f(f(f(y0 * -s) - f(x0 * c)) / d)
        scale = f(math.pi / (2 * T) * float(numpy.sqrt(d)) / float(abs(d)))
        out.append((float(f(c / d)), float(f(s / d)), float(off),
                    float(scale)))
    return out


def _position32(x, z, c, s, off, fused):
    """Detector positions less 1/2 as float32 arithmetic gives them, step by
    step or (reduced storages) as two fused multiply-adds."""
    if fused:
        inner = (-z * s + (off - 0.5).float().double()[:, :, None]).float()
        return (x * c + inner.double()).float().reshape(off.shape[0], -1)
    xc = (x.float() * torch.tensor(c, dtype=torch.float32, device="cuda")
          - z.float() * torch.tensor(s, dtype=torch.float32, device="cuda"))
    return xc.reshape(1, -1) + off.float() - 0.5


def exact(case, seed):
    """The same results in 64 bits; each voxel takes its defocus slab, and
    whether it falls on the detector, by the float32 rules that define them."""
    series = _series(case, seed)
    X, T, ndf = case["X"], case["T"], case["ndf"]
    corrects = case["kind"] in ("correct", "volume") or case.get("ctf", False)
    flips = _flips(case) if corrects else None

    def corrected(t):  # (ndf, Y, X)
        F = torch.fft.fft2(series[t].double())
        n = X * case["Y"]
        return torch.stack([torch.fft.ifft2(F * m).real for m in flips]) * n

    if case["kind"] == "correct":
        _, mn, mx = _defoci(case)
        out = torch.stack([corrected(t) for t in range(T)])
        if ndf == 1:
            out = out[:, 0]
        return {"corrected": out.cpu().numpy(), "range": [mn, mx]}

    def rows(t):  # filtered, (Y, ndf, X)
        if corrects:
            s = corrected(t).permute(1, 0, 2)
        elif case["kind"] == "slice":
            s = series[None, :, t]
        elif case["layout"] == "sinograms":
            s = series[:, :, t]
        else:
            s = series[t].reshape(ndf, case["Y"], X).permute(1, 0, 2)
        return _filtered(s.double())

    Y, Z = case.get("Y", 1), case["Z"]
    _, mn, mx = _defoci(case)
    f = numpy.float32
    ps = f(case["pixel"])
    dscale = f(f(f(ndf) * ps) / f(f(mx) - f(mn))) if ndf > 1 else f(0)
    doffset = f(-dscale * f(f(mn) / ps))
    x = (torch.arange(X, dtype=torch.float64, device="cuda") + 0.5
         - 0.5 * X)[None, :]
    z = (torch.arange(Z, dtype=torch.float64, device="cuda") + 0.5
         - 0.5 * Z)[:, None]
    drift = bool(case.get("drift"))
    fused = case.get("storage", "f32") != "f32"
    centres = _centres(case)
    tables = [_geometry(T, c) for c in centres] if drift else [
        _geometry(T, X / 2.0)]
    vol = torch.zeros((Y, Z * X), dtype=torch.float64, device="cuda")
    for t in range(T):
        c, s, off, scale = tables[0][t]
        if ndf > 1:
            cf, sf = (torch.tensor(v, dtype=torch.float32, device="cuda")
                      for v in (c, s))
            h = -x.float() * sf - z.float() * cf
            d = h * float(dscale) + float(doffset)
            k = torch.floor(d.double() + 0.5).clamp(0, ndf - 1).long()
        else:
            k = torch.zeros((1, 1), dtype=torch.int64, device="cuda")
        R = rows(t).reshape(Y, ndf * X)
        offs = torch.tensor([g[t][2] for g in tables], device="cuda",
                            dtype=torch.float64)[:, None]
        step = max(1, (1 << (25 if drift else 27)) // (Z * X))
        for y in range(0, Y, step):
            r = R[y:y + step]
            # one line of positions for all rows, or one for each
            off = offs[y:y + step] if drift else offs
            p = (x * c - z * s).reshape(1, -1) + (off - 0.5)
            edge = torch.floor(_position32(x, z, c, s, off, fused))
            ok = (edge >= 0) & (edge < X - 1)
            i = torch.floor(p).clamp(0, X - 2)
            w, i = p - i, i.long()
            at = (k * X).expand(Z, X).reshape(1, -1) + i
            if drift:
                lo, hi = r.gather(1, at), r.gather(1, at + 1)
            else:
                lo, hi = r[:, at[0]], r[:, at[0] + 1]
            vol[y:y + step] += scale * torch.where(
                ok, lo + w * (hi - lo), torch.zeros_like(lo))
    if case["kind"] == "slice":
        return vol.reshape(Z, X).cpu().numpy()
    vol = vol.reshape(Y, Z, X)
    return vol if case["kind"] == "plan" else vol.cpu().numpy()
