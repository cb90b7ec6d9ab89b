"""The matrix-core backprojector over the range of its inputs: tilts of very
different size, blank ones, and the units of the data.

Volumes are compared with FP64 sums over the plan's own decoded slabs, within
the bound that tests/test_bp_mm_gpu.py derives (1e-5 of each row's norm: FP32
rounding alone is below 5e-6); rows that only the weak tilts reach are
compared by themselves, so that a weak tilt's error counts as its own.
"""
import numpy
import pytest

from guanaco_amd import _capi as C
from test_bp_mm_gpu import backproject, decoded

pytestmark = pytest.mark.gpu

# X, Y, T, ndf, Z, W, (min_df, max_df): one slab; three wide ones over 512
# workgroups
SHAPES = [
    (64, 40, 16, 1, 32, 64, (0.0, 0.0)),
    (520, 97, 6, 3, 256, 512, (-130.0, 130.0)),
]


def tilts_of(kind, T):
    """The size of every tilt, and the tilts that the lower rows see."""
    size = numpy.ones(T)
    low = slice(None)
    if kind == "blank":          # a blank tilt beside very small data
        size *= 1e-12
        size[T // 2] = 0.0
    elif kind == "small":        # the smallest normal numbers
        size *= 2.0 ** -125
    elif kind.startswith("2^"):  # strong tilts first, weak ones last
        size = numpy.geomspace(1.0, 2.0 ** float(kind[2:]), T)
        low = slice(T // 2, None)
        if T > 8:
            size[3] = 0.0
    return size, low


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("kind", ["blank", "small", "2^-12", "2^-24",
                                  "2^-40", "2^-100"])
@pytest.mark.parametrize("shape", SHAPES)
def test_weak_tilts_keep_their_precision(capi, shape, kind, storage):
    X, Y, T, ndf, Z, W, (mn, mx) = shape
    angles = numpy.deg2rad(numpy.linspace(-60, 60, T)).astype(numpy.float32)
    size, low = tilts_of(kind, T)
    rng = numpy.random.default_rng(X + T)
    sino = (rng.standard_normal((Y, ndf, T, X))
            * size[None, None, :, None]).astype(numpy.float32)
    seen = numpy.zeros(T, bool)
    seen[low] = True
    sino[Y // 2:, :, ~seen] = 0.0
    plan = C.VolumePlan(X, Y, angles, Z, width=W, num_defocus=ndf,
                        centre=X / 2.0 - 0.3, min_defocus=mn, max_defocus=mx,
                        storage=storage, input_layout=C.INPUT_SINOGRAMS)
    assert plan.matrix_cores()
    d_in = C.DeviceArray.from_host(sino)
    d_vol = C.DeviceArray((Y, Z, W))
    plan.run(d_in, d_vol)
    C.call("gx_device_synchronize")
    vol = d_vol.to_host()
    nrm = numpy.abs(sino).max(axis=(0, 1, 3)).astype(numpy.float64)
    slabs = decoded(plan, (X, Y, T, ndf), storage).astype(
        numpy.float64) * nrm[None, :, None, None]
    first, last = plan.slab_range()
    plan.destroy()
    for t in range(T):  # slabs no voxel reads hold anything
        slabs[:first[t], t] = slabs[last[t] + 1:, t] = 0
    for y in (0, Y - 1):
        expect = backproject(slabs[:, :, y], Z, W, angles, X / 2.0 - 0.3, mn,
                             mx)
        assert numpy.abs(expect).max() > 0
        err = numpy.linalg.norm(vol[y].astype(numpy.float64) - expect)
        assert err <= 1e-5 * numpy.linalg.norm(expect), (y, err)
