"""recon() and the per-tilt maximum at the edges of their kernels: numbers of
tilts around a group of eight, widths around a tile, single samples, and rows
that are not whole 16-byte words."""
import numpy
import pytest

import guanaco_amd as G
from guanaco_amd import _capi as C
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,T,ndf,H,W", [
    (1, 1, 1, 1, 1), (2, 3, 1, 5, 4), (33, 7, 1, 9, 33), (64, 8, 1, 8, 32),
    (50, 9, 3, 17, 31), (40, 17, 5, 40, 65),
])
def test_project_is_bit_exact(capi, N, T, ndf, H, W):
    rng = numpy.random.default_rng(N + T)
    sino = rng.standard_normal((ndf, T, N)).astype(numpy.float32)
    angles = numpy.deg2rad(numpy.linspace(-80, 80, T)).astype(numpy.float32)
    mn, mx = (-20.0, 20.0) if ndf > 1 else (0.0, 0.0)
    cfg = C.recon_cfg(N, T, ndf, H, W, 1.0, N / 2.0 + 0.25, mn, mx, angles)
    got = numpy.zeros((H, W), numpy.float32)
    C.call("gx_project", C.ctypes.byref(cfg), C.f32p(sino), C.f32p(got))
    expect = O.project(sino if ndf > 1 else sino[0], (H, W), angles,
                       N / 2.0 + 0.25, 1.0, mn, mx)
    numpy.testing.assert_array_equal(got, expect)


@pytest.mark.parametrize("X,Y", [(8, 1), (20, 7), (37, 16), (64, 17),
                                 (1028, 25), (300, 40)])
def test_largest_value_of_a_tilt_is_found_anywhere(capi, X, Y):
    # One large value per tilt sets that tilt's scale: FP16 results are then
    # those of FP32 to FP16 rounding of values near 1 (2^-11 each, below 1e-3
    # of the volume), which a missed maximum would overflow instead.
    T, Z = 6, 8
    rng = numpy.random.default_rng(X + Y)
    proj = rng.uniform(-1, 1, (T, Y, X)).astype(numpy.float32)
    places = [(0, 0), (Y - 1, X - 1), (Y // 2, X // 3), (0, X - 1),
              (Y - 1, 0), (Y // 3, X // 2)]
    for t, (y, x) in enumerate(places):
        proj[t, y, x] = (-1) ** t * 3.0e6
    angles = numpy.deg2rad(numpy.linspace(-30, 30, T)).astype(numpy.float32)
    vols = {}
    for storage in ("f32", "f16"):
        vols[storage] = G.reconstruct(
            proj, angles, numpy.zeros((Y, Z, X), numpy.float32),
            device="gpu", storage=storage, depth=Z)
    err = numpy.linalg.norm(vols["f16"] - vols["f32"]) / numpy.linalg.norm(
        vols["f32"])
    assert err < 1e-3, err
