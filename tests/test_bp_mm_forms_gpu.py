"""Every form of the matrix-core backprojector: 32, 64 and 128 rows per
workgroup, one slab and several, each with a last workgroup of every number of
row blocks, and values that are not finite in each.

The forms are chosen by size: with one slab, more than 256 tiles of 16 x 16
voxels times row groups take 128 or 64 rows; several slabs need 512, and rows
that fill groups of 128 (so that 64 and 32 rows are left to calls for a band).
"""
import numpy
import pytest

from guanaco_amd import _capi as C
from oracle import oracle as O
from test_bp_mm_gpu import backproject, decoded, f32
from test_bp_mm_precision_gpu import both

pytestmark = pytest.mark.gpu

T = 5
ANGLES = numpy.deg2rad(numpy.linspace(-60, 60, T)).astype(f32)

# X, Y, ndf, Z, W, (min_df, max_df)
ONE = [(300, Y, 1, 256, 272, (0.0, 0.0))
       for Y in (32, 33, 64, 129, 161, 193, 225)]
MULTI = [(520, Y, 3, 256, 512, (-130.0, 130.0)) for Y in (97, 225, 320, 321)]


def run_plan(shape, storage, rows, sino, weights=None):
    X, Y, ndf, Z, W, (mn, mx) = shape
    plan = C.VolumePlan(X, Y, ANGLES, Z, width=W, num_defocus=ndf,
                        centre=X / 2.0 - 0.3, min_defocus=mn, max_defocus=mx,
                        weights=weights, storage=storage,
                        input_layout=C.INPUT_SINOGRAMS)
    assert plan.matrix_cores()
    plan.set_tile(rows, "staged")
    d_in = C.DeviceArray.from_host(sino)
    d_vol = C.DeviceArray((Y, Z, W))
    plan.run(d_in, d_vol)
    C.call("gx_device_synchronize")
    taps = decoded(plan, (X, Y, T, ndf), storage)
    first, last = plan.slab_range()
    plan.destroy()
    for t in range(T):  # slabs no voxel reads hold anything
        taps[:first[t], t] = taps[last[t] + 1:, t] = 0
    return d_vol.to_host(), taps


def sinograms(shape):
    X, Y, ndf = shape[:3]
    rng = numpy.random.default_rng(X + Y + ndf)
    return rng.standard_normal((Y, ndf, T, X)).astype(f32)


@pytest.mark.parametrize("storage,rows", [("f16", 32), ("bf16", 16)])
@pytest.mark.parametrize("shape", ONE + MULTI)
def test_row_groups(capi, shape, storage, rows):
    # (the bound of tests/test_bp_mm_gpu.py)
    X, Y, ndf, Z, W, (mn, mx) = shape
    sino = sinograms(shape)
    vol, taps = run_plan(shape, storage, rows, sino)
    nrm = numpy.abs(sino).max(axis=(0, 1, 3))
    slabs = taps * nrm[None, :, None, None]
    for y in sorted({0, Y // 2, max(Y // 32 * 32, 1) - 1, Y - 1}):
        expect = backproject(slabs[:, :, y], Z, W, ANGLES, X / 2.0 - 0.3, mn,
                             mx)
        err = numpy.linalg.norm(vol[y] - expect)
        assert err <= 1e-5 * numpy.linalg.norm(expect), (y, err)


# depths and widths about the limits of the tile order (32 tiles deep and 96
# wide): columns, strips of 8 tiles, a last strip of 1 and of 6, two row groups
@pytest.mark.parametrize("shape", [
    (60, 2, 1, 496, 1540, (0.0, 0.0)), (60, 2, 1, 513, 1520, (0.0, 0.0)),
    (60, 2, 1, 512, 1521, (0.0, 0.0)), (60, 2, 1, 521, 1540, (0.0, 0.0)),
    (60, 129, 1, 600, 1540, (0.0, 0.0)), (700, 97, 3, 513, 1536, (-300., 300.)),
])
def test_tile_orders(capi, shape):
    test_row_groups(capi, shape, "f16", 32)


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("nan", [False, True])
@pytest.mark.parametrize("shape", [ONE[6], MULTI[1]])
def test_bands_of_rows_keep_the_bits(capi, shape, nan, storage):
    # 32, 64 and 128 rows per workgroup, and a last row by itself
    X, Y, ndf, Z, W, (mn, mx) = shape
    sino = sinograms(shape)
    if nan:
        sino[[3, 70, 140], 0, 1, X // 2] = numpy.nan
    plan = C.VolumePlan(X, Y, ANGLES, Z, width=W, num_defocus=ndf,
                        centre=X / 2.0 - 0.3, min_defocus=mn, max_defocus=mx,
                        storage=storage, input_layout=C.INPUT_SINOGRAMS)
    assert plan.matrix_cores()
    d_in = C.DeviceArray.from_host(sino)
    d_vol = C.DeviceArray((Y, Z, W))
    plan.run(d_in, d_vol)
    C.call("gx_device_synchronize")
    whole = d_vol.to_host()
    for y0, y1 in ((0, 32), (32, 96), (96, 224), (224, Y)):
        d_band = C.DeviceArray((y1 - y0, Z, W))
        plan.backproject_rows(y0, y1, d_band)
        C.call("gx_device_synchronize")
        numpy.testing.assert_array_equal(d_band.to_host(), whole[y0:y1])
    plan.destroy()


@pytest.mark.parametrize("storage,rows", [("f16", 16), ("bf16", 32)])
@pytest.mark.parametrize("shape", [ONE[0], ONE[1], ONE[4], MULTI[1],
                                   MULTI[3]])
def test_a_nan_changes_only_its_rows(capi, shape, storage, rows):
    # rows 2 i and 2 i + 1 are filtered as one complex row; the tilt's
    # normalisation stays, as its largest value lies in another row
    X, Y, ndf = shape[:3]
    sino = sinograms(shape)
    sino[0, 0, :, X // 2] = 8.0
    clean, _ = run_plan(shape, storage, rows, sino)
    y, t = Y - Y // 4, 2
    sino[y, :, t, X // 3] = numpy.nan
    vol, _ = run_plan(shape, storage, rows, sino)
    pair = {y, min(y ^ 1, Y - 1)}
    seen = numpy.zeros((ndf, T, X), f32)
    seen[:, t] = 1.0
    Z, W, (mn, mx) = shape[3:]
    seen = O.project(seen if ndf > 1 else seen[0], (Z, W), ANGLES,
                     X / 2.0 - 0.3, 1.0, mn, mx) != 0
    others = [r for r in range(Y) if r not in pair]
    numpy.testing.assert_array_equal(vol[others], clean[others])
    for r in pair:
        numpy.testing.assert_array_equal(numpy.isnan(vol[r]), seen)
        # (two roundings of the same sums: tests/test_bp_mm_gpu.py's 1e-5)
        err = numpy.linalg.norm(vol[r][~seen] - clean[r][~seen])
        assert err <= 1e-5 * numpy.linalg.norm(clean[r]), err


@pytest.mark.parametrize("storage,rows", [("f16", 32), ("bf16", 16)])
@pytest.mark.parametrize("shape", [ONE[0], ONE[2], ONE[5], MULTI[0],
                                   MULTI[2]])
def test_infinities_reach_the_voxels_that_read_them(capi, shape, storage,
                                                    rows):
    # a tilt's weight multiplies its filtered rows, so a large one takes some
    # values past the largest FP16 number; FP32 fused multiply-adds in tilt
    # order, as tests/test_bp_mm_precision_gpu.py emulates them, say where
    # infinities and NaNs follow. Finite rows: 1e-5 of their norm; rows with
    # infinities are such sums themselves: 1e-6 of the largest finite value.
    X, Y, ndf, Z, W, (mn, mx) = shape
    sino = sinograms(shape)
    sino[::2] *= f32(0.01)
    weights = numpy.array([1, 1, 3e5, 1, 1], f32)
    vol, taps = run_plan(shape, storage, rows, sino, weights)
    with numpy.errstate(over="ignore"):
        taps = taps.astype(numpy.float16).astype(numpy.float64)
    scale = O.tilt_coefficients(ANGLES, X / 2.0 - 0.3)[:, 3].astype(f32)
    nrm = scale * numpy.abs(sino).max(axis=(0, 1, 3)).astype(f32)
    found = 0
    for y in sorted({0, 1, Y // 2, Y - 2, Y - 1}):
        with numpy.errstate(invalid="ignore"):
            _, acc = both(taps[:, :, y], nrm, Z, W, ANGLES, X / 2.0 - 0.3, mn,
                          mx)
        finite = numpy.isfinite(acc)
        found += numpy.count_nonzero(~finite)
        numpy.testing.assert_array_equal(numpy.isnan(vol[y]), numpy.isnan(acc))
        numpy.testing.assert_array_equal(vol[y][numpy.isinf(acc)],
                                         acc[numpy.isinf(acc)])
        if finite.all():
            err = numpy.linalg.norm(vol[y] - acc)
            assert err <= 1e-5 * numpy.linalg.norm(acc), (y, err)
        else:
            err = numpy.abs(vol[y][finite] - acc[finite]).max()
            assert err <= 1e-6 * numpy.abs(acc[finite]).max(), (y, err)
    assert found > 0


@pytest.mark.parametrize("value", [numpy.nan, numpy.inf])
@pytest.mark.parametrize("X,Y", [(64, 40), (60, 37)])
def test_corrected_projections(capi, X, Y, value):
    # the correction spreads it over its projection: every voxel that the
    # tilt sees, in every storage, and no other
    rng = numpy.random.default_rng(3)
    proj = (rng.standard_normal((T, Y, X)) + 4.0).astype(f32)
    dfs = numpy.array([20000.0])
    seen = O.project(numpy.stack([numpy.full(X, t == 2, f32)
                                  for t in range(T)]), (48, X + 60), ANGLES,
                     X / 2.0, 1.0, 0.0, 0.0) != 0
    assert seen.any() and not seen.all()
    for storage, bound in (("f32", 1e-6), ("f16", 1e-3), ("bf16", 8e-3)):
        plan = C.VolumePlan(X, Y, ANGLES, 48, width=X + 60, centre=X / 2.0,
                            storage=storage, defocus=dfs,
                            wavelength=O.electron_wavelength(300000), Cs=2.7e7)
        vols = []
        for v in (proj[2, Y // 2, X // 2], value):
            p = proj.copy()
            p[2, Y // 2, X // 2] = v
            d_in = C.DeviceArray.from_host(p)
            d_vol = C.DeviceArray((Y, 48, X + 60))
            plan.run(d_in, d_vol)
            C.call("gx_device_synchronize")
            vols.append(d_vol.to_host())
        plan.destroy()
        for y in range(Y):
            numpy.testing.assert_array_equal(numpy.isnan(vols[1][y]), seen)
        err = numpy.linalg.norm((vols[1] - vols[0])[:, ~seen])
        assert err <= bound * numpy.linalg.norm(vols[0]), (storage, err)
