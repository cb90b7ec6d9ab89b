"""The backprojectors of 16-bit slabs at the edges of their tiles: the
matrix-core kernel, and the kernel for one rotation centre per row.

Each plan's own decoded slabs (times the per-tilt normalisation the filter
divided out) are backprojected in FP64 with the taps and slabs that the
storage's FP32 arithmetic gives (two fused multiply-adds for the position, as
tests/test_bp_window.py emulates them; their rounding, an ulp of a position,
is the storage's and not a kernel's). What is left is the FP32 rounding of
the kernel and the weights' split into two FP16 parts: at most 2^-22 per
weight, and about (T + 8) 2^-24 of the sum of the terms' magnitudes in the
accumulation, below 5e-6 for the 64 tilts used here at most; 1e-5 with room
for cancellation in the sums.
"""
import numpy
import pytest

from guanaco_amd import _capi as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# X, Y, T, ndf, Z, W, last tilt (deg), (min_df, max_df), weights
CASES = [
    # one voxel, one row, one tilt
    (8, 1, 1, 1, 1, 1, 0.0, (0.0, 0.0), None),
    # partial 4 x 4 blocks and tiles, odd width, one 32-row block
    (70, 31, 3, 1, 17, 67, 60.0, (0.0, 0.0), None),
    # two row blocks, the second partial; whole batches of four tilts
    (64, 33, 8, 1, 16, 64, 60.0, (0.0, 0.0), None),
    # four row blocks, and one row into the next workgroup
    (48, 129, 5, 1, 33, 50, 80.0, (0.0, 0.0), None),
    # every quadrant, a detector narrower than a staged run
    (20, 65, 64, 1, 40, 36, 175.0, (0.0, 0.0), None),
    # several slabs, small: the staged kernel
    (96, 40, 21, 6, 50, 96, 65.0, (-100.0, 100.0), None),
    (80, 97, 30, 4, 80, 80, 70.0, (-25.0, 25.0), None),
    # several wide slabs over a large volume: extra runs, batches that close
    # early, a last workgroup with one row block; partial tiles
    (260, 385, 9, 4, 130, 260, 70.0, (-130.0, 130.0), None),
    (200, 450, 6, 3, 131, 268, 85.0, (-100.0, 100.0), None),
    # tilts of very different weight
    (64, 34, 12, 2, 20, 64, 60.0, (-90.0, 90.0), 1e-3),
]


f32 = numpy.float32


def fma32(a, b, c):
    return (numpy.asarray(a, numpy.float64) * numpy.asarray(b, numpy.float64)
            + numpy.asarray(c, numpy.float64)).astype(f32)


def backproject(slabs, Z, W, angles, centre, mn, mx):
    """(ndf, T, X) slab rows to a (Z, W) slice, FP64 sums of FP32 decisions
    (1 pixel is 1 A)."""
    ndf, T, X = slabs.shape
    x = (numpy.arange(W) - 0.5 * W + 0.5).astype(f32)[None, :]
    z = (numpy.arange(Z) - 0.5 * Z + 0.5).astype(f32)[:, None]
    out = numpy.zeros((Z, W))
    ds = f32(f32(ndf) / (f32(mx) - f32(mn))) if ndf > 1 else f32(0)
    do = f32(-ds * f32(mn))
    for t, (c, s, off, scale) in enumerate(O.tilt_coefficients(angles,
                                                               centre)):
        p = fma32(x, c, fma32(-z, s, f32(off) - f32(0.5)))
        i = numpy.floor(p).astype(numpy.int64)
        w = p.astype(numpy.float64) - i
        d = (-x * f32(s) - z * f32(c)) * ds + do
        k = numpy.clip(numpy.floor(d.astype(numpy.float64) + 0.5), 0,
                       ndf - 1).astype(numpy.int64)
        ok = (i >= 0) & (i < X - 1)
        i = numpy.clip(i, 0, max(X - 2, 0))
        r = slabs[:, t].astype(numpy.float64)
        v = (1 - w) * r[k, i] + w * r[k, numpy.minimum(i + 1, X - 1)]
        out += numpy.where(ok, float(scale) * v, 0.0)
    return out


def plan_of(case, storage):
    X, Y, T, ndf, Z, W, last, (mn, mx), weights = case
    angles = numpy.deg2rad(numpy.linspace(-last, last, T)).astype(
        numpy.float32)
    rng = numpy.random.default_rng(X + Y + T + ndf)
    sino = rng.standard_normal((Y, ndf, T, X)).astype(numpy.float32)
    w = numpy.ones(T, numpy.float32)
    if weights is not None:
        w = numpy.geomspace(1.0, weights, T).astype(numpy.float32)
    plan = C.VolumePlan(X, Y, angles, Z, width=W, num_defocus=ndf,
                        centre=X / 2.0 - 0.3, min_defocus=mn, max_defocus=mx,
                        weights=w, storage=storage,
                        input_layout=C.INPUT_SINOGRAMS)
    assert plan.backprojector()[1] > 0
    return plan, sino, angles


def run(plan, case, sino):
    X, Y, T, ndf, Z, W = case[:6]
    d_in = C.DeviceArray.from_host(sino)
    d_vol = C.DeviceArray((Y, Z, W))
    C.call("gx_fill_u32", d_vol.ptr, 0x7fc00000, Y * Z * W, None)
    plan.run(d_in, d_vol)
    C.call("gx_device_synchronize")
    return d_vol.to_host()


def decoded(plan, case, storage):
    """(ndf, T, Y, X) slab values as float32."""
    X, Y, T, ndf = case[:4]
    p, n, yb = plan.slabs()
    nyb = (Y + yb - 1) // yb
    a = numpy.empty(ndf * T * nyb * X * yb, numpy.uint16)
    C.call("gx_memcpy_dtoh", a.ctypes.data, p, a.nbytes, None)
    if storage == "f16":
        f = a.view(numpy.float16).astype(numpy.float32)
    else:
        f = (a.astype(numpy.uint32) << 16).view(numpy.float32)
    f = f.reshape(ndf, T, nyb, X, yb)
    return numpy.moveaxis(f, 4, 3).reshape(ndf, T, nyb * yb, X)[:, :, :Y]


@pytest.mark.parametrize("rows", [32, 16])
@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("case", CASES)
def test_matches_oracle_on_its_own_slabs(capi, case, storage, rows):
    X, Y, T, ndf, Z, W, _, (mn, mx), _ = case
    plan, sino, angles = plan_of(case, storage)
    plan.set_tile(rows, "staged")
    vol = run(plan, case, sino)
    nrm = numpy.abs(sino).max(axis=(0, 1, 3)).astype(numpy.float32)
    slabs = decoded(plan, case, storage) * nrm[None, :, None, None]
    first, last = plan.slab_range()
    for t in range(T):  # slabs no voxel reads hold anything
        slabs[:first[t], t] = slabs[last[t] + 1:, t] = 0
    for y in sorted({0, Y // 3, Y // 2, Y - 1}):
        expect = backproject(slabs[:, :, y], Z, W, angles, X / 2.0 - 0.3, mn,
                             mx)
        err = numpy.linalg.norm(vol[y] - expect)
        assert err <= 1e-5 * numpy.linalg.norm(expect), (y, err)
    plan.destroy()


# depths about the tile order's limits: one strip of 16 tiles, then strips of
# 8 with a last one of 1 (its one voxel deep), 2 and 8 tiles; two workgroups
# of rows; several slabs
@pytest.mark.parametrize("case", [
    (60, 40, 5, 1, 256, 40, 60.0, (0.0, 0.0), None),
    (60, 40, 5, 1, 257, 40, 60.0, (0.0, 0.0), None),
    (60, 150, 5, 1, 277, 35, 80.0, (0.0, 0.0), None),
    (60, 33, 5, 1, 384, 16, 60.0, (0.0, 0.0), None),
    (300, 513, 5, 3, 281, 132, 70.0, (-180.0, 180.0), None),
])
def test_deep_volumes(capi, case):
    test_matches_oracle_on_its_own_slabs(capi, case, "f16", 32)


@pytest.mark.parametrize("case", [CASES[1], CASES[4], CASES[6], CASES[7]])
def test_exceptional_values_reach_only_their_voxels(capi, case):
    # A NaN in one row of one tilt makes that filtered row NaN, and the row
    # it is transformed with (rows 2i and 2i + 1 travel as one complex row):
    # so are exactly the voxels of the two rows that the tilt sees (an oracle
    # run of an indicator sinogram shows which); every other voxel keeps its
    # value.
    X, Y, T, ndf, Z, W, _, (mn, mx), _ = case
    plan, sino, angles = plan_of(case, "f16")
    clean = run(plan, case, sino)
    assert numpy.isfinite(clean).all()
    y, t = Y // 2, T // 3
    broken = sino.copy()
    broken[y, :, t, X // 2] = numpy.nan
    vol = run(plan, case, broken)
    plan.destroy()
    ones = numpy.zeros((ndf, T, X), numpy.float32)
    ones[:, t] = 1.0
    seen = O.project(ones if ndf > 1 else ones[0], (Z, W), angles,
                     X / 2.0 - 0.3, 1.0, mn, mx) != 0
    for r in {y, min(y ^ 1, Y - 1)}:
        numpy.testing.assert_array_equal(numpy.isnan(vol[r]), seen)
        vol[r][seen] = clean[r][seen]
    assert numpy.isfinite(vol).all()
    # the tilt's normalisation may differ (its largest value may have gone)
    err = numpy.linalg.norm(vol - clean) / numpy.linalg.norm(clean)
    assert err < 1e-3, err


# X, Y, T, ndf, Z, W, (min_df, max_df), drift of the centres (pixels)
CENTRE_CASES = [
    # one row; rows past the last block; W no multiple of four
    (16, 1, 3, 1, 5, 18, (0.0, 0.0), 0.0),
    (61, 21, 9, 1, 19, 47, (0.0, 0.0), 2.5),
    # tiles in one slab and across two, centres far off the detector
    (64, 40, 13, 4, 24, 64, (-64.0, 64.0), 40.0),
    # more slabs in a tile than the staged kernels hold
    (64, 33, 7, 16, 16, 36, (-32.0, 32.0), 1.0),
]


@pytest.mark.parametrize("rows", [32, 16])
@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("case", CENTRE_CASES)
def test_centre_per_row_matches_oracle_on_its_own_slabs(capi, case, storage,
                                                        rows):
    X, Y, T, ndf, Z, W, (mn, mx), drift = case
    angles = numpy.deg2rad(numpy.linspace(-60, 60, T)).astype(numpy.float32)
    rng = numpy.random.default_rng(X + Y)
    sino = rng.standard_normal((Y, ndf, T, X)).astype(numpy.float32)
    centres = (X / 2.0 + drift * numpy.linspace(-1, 1, Y)
               + rng.uniform(-0.5, 0.5, Y)).astype(numpy.float32)
    if Y == 1:  # (one centre would be a plan without centres)
        centres = numpy.repeat(centres, 2)
        sino = numpy.repeat(sino, 2, axis=0)
        Y = 2
        case = (X, Y) + case[2:]
    plan = C.VolumePlan(X, Y, angles, Z, width=W, num_defocus=ndf,
                        centre=centres, min_defocus=mn, max_defocus=mx,
                        storage=storage, input_layout=C.INPUT_SINOGRAMS)
    plan.set_tile(rows, "direct")
    vol = run(plan, (X, Y, T, ndf, Z, W), sino)
    nrm = numpy.abs(sino).max(axis=(0, 1, 3)).astype(numpy.float32)
    slabs = decoded(plan, (X, Y, T, ndf), storage) * nrm[None, :, None, None]
    first, last = plan.slab_range()
    for t in range(T):
        slabs[:first[t], t] = slabs[last[t] + 1:, t] = 0
    plan.destroy()
    for y in sorted({0, Y // 2, Y - 1}):
        expect = backproject(slabs[:, :, y], Z, W, angles,
                             float(centres[y]), mn, mx)
        err = numpy.linalg.norm(vol[y] - expect)
        assert err <= 1e-5 * numpy.linalg.norm(expect) + 1e-30, (y, err)
