"""The matrix-core backprojector's rounding: no further from FP64 than FP32
weights and FP32 fused multiply-adds in tilt order, which the vector kernels
use, on the same slabs, positions and weights.

Both errors are root mean squares over n voxels of one distribution, known to
1 / sqrt(2 n): 0.4 % each for the smallest case here (32768 voxels), so that
3 % is more than five of their difference's standard errors. A weight kept as
FP16 pairs of its rounded FP32 value, high part first, was 10 to 25 % off.
"""
import numpy
import pytest

from guanaco_amd import _capi as C
from oracle import oracle as O
from test_bp_mm_gpu import decoded, f32, fma32

pytestmark = pytest.mark.gpu


def both(taps, weight, Z, W, angles, centre, mn, mx):
    """(ndf, T, X) slab values to a (Z, W) slice: in FP64, and in FP32 as the
    vector kernels add. The taps' positions are FP32 in both."""
    ndf, T, X = taps.shape
    x = (numpy.arange(W) - 0.5 * W + 0.5).astype(f32)[None, :]
    z = (numpy.arange(Z) - 0.5 * Z + 0.5).astype(f32)[:, None]
    exact, acc = numpy.zeros((Z, W)), numpy.zeros((Z, W), f32)
    ds = f32(f32(ndf) / (f32(mx) - f32(mn))) if ndf > 1 else f32(0)
    do = f32(-ds * f32(mn))
    for t, (c, s, off, _) in enumerate(O.tilt_coefficients(angles, centre)):
        p = fma32(x, c, fma32(-z, s, f32(off) - f32(0.5)))
        i = numpy.floor(p).astype(numpy.int64)
        tt = (p - numpy.floor(p)).astype(f32)
        d = (-x * f32(s) - z * f32(c)) * ds + do
        k = numpy.clip(numpy.floor(d.astype(numpy.float64) + 0.5), 0,
                       ndf - 1).astype(numpy.int64)
        ok = (i >= 0) & (i < X - 1)
        i = numpy.clip(i, 0, X - 2)
        v0, v1 = taps[k, t, i], taps[k, t, i + 1]
        q = tt.astype(numpy.float64)
        exact += numpy.where(ok, float(weight[t]) * ((1 - q) * v0 + q * v1),
                             0.0)
        w1 = weight[t] * tt
        w0 = weight[t] - w1
        acc = numpy.where(ok, fma32(w1, v1, fma32(w0, v0, acc)), acc)
    return exact, acc


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("case", [
    # X, Y, T, ndf, Z, W, (min_df, max_df): few tilts, where the weights'
    # error shows most, and an ordinary number
    (256, 3, 5, 1, 64, 256, (0.0, 0.0)),
    (256, 3, 16, 1, 64, 256, (0.0, 0.0)),
    (256, 2, 61, 1, 64, 256, (0.0, 0.0)),
    (520, 97, 6, 3, 256, 512, (-130.0, 130.0)),
])
def test_no_further_off_than_fp32(capi, case, storage):
    X, Y, T, ndf, Z, W, (mn, mx) = case
    angles = numpy.deg2rad(numpy.linspace(-60, 60, T)).astype(f32)
    rng = numpy.random.default_rng(X + T)
    sino = rng.poisson(40, (Y, ndf, T, X)).astype(f32)
    plan = C.VolumePlan(X, Y, angles, Z, width=W, num_defocus=ndf,
                        centre=X / 2.0 - 0.3, min_defocus=mn, max_defocus=mx,
                        storage=storage, input_layout=C.INPUT_SINOGRAMS)
    assert plan.matrix_cores()
    d_in = C.DeviceArray.from_host(sino)
    d_vol = C.DeviceArray((Y, Z, W))
    plan.run(d_in, d_vol)
    C.call("gx_device_synchronize")
    vol = d_vol.to_host()
    # the vector units read BF16 as FP16 too
    taps = decoded(plan, (X, Y, T, ndf), storage).astype(numpy.float16)
    taps = taps.astype(numpy.float64)
    first, last = plan.slab_range()
    plan.destroy()
    for t in range(T):  # slabs no voxel reads hold anything
        taps[:first[t], t] = taps[last[t] + 1:, t] = 0
    scale = O.tilt_coefficients(angles, X / 2.0 - 0.3)[:, 3].astype(f32)
    weight = scale * numpy.abs(sino).max(axis=(0, 1, 3)).astype(f32)
    here = fp32 = 0.0
    for y in sorted({0, Y - 1}):
        exact, acc = both(taps[:, :, y], weight, Z, W, angles, X / 2.0 - 0.3,
                          mn, mx)
        here += numpy.sum((vol[y] - exact) ** 2)
        fp32 += numpy.sum((acc - exact) ** 2)
    assert numpy.sqrt(here) <= 1.03 * numpy.sqrt(fp32), (
        numpy.sqrt(here / fp32))
