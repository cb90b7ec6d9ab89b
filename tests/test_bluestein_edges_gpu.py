"""Detector sizes at the edges of the any-size transforms' workgroups:
lengths just below and above a change of transform length, of the row pairs
per workgroup and of the waves that synchronise alone, row counts that leave
partial row groups, and tilts whose voxels read only some slabs.

FP32 volumes against the FP32 oracle chain, with the bound of the other
size tests (1e-5: FFT rounding of both sides, about 1e-7 per transform);
FP16 volumes against the FP32 ones (2^-11 per stored value, below 1e-3).
"""
import numpy
import pytest

import guanaco_amd as G
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [
    # X, Y, ndf: transform lengths 8, 16 (one column per thread), 64
    (3, 9, 1), (7, 5, 2), (30, 33, 2),
    # 512 and 1024 points: one-wave slots, four pairs to a workgroup
    (250, 37, 3), (500, 18, 2),
    # 2048 and 4096: two slots, one slot
    (1000, 21, 2), (1100, 35, 3),
    # power-of-two rows with other columns, and the reverse
    (64, 300, 2), (300, 64, 2),
]


@pytest.mark.parametrize("X,Y,ndf", SIZES)
def test_odd_sizes_match_the_oracle(capi, X, Y, ndf):
    rng = numpy.random.default_rng(X * 131 + Y)
    T, depth = 5, min(X, 20)
    proj = (rng.standard_normal((T, Y, X)) + 4.0).astype(numpy.float32)
    angles = numpy.deg2rad(numpy.linspace(-55, 55, T)).astype(numpy.float32)
    kw = dict(pixel_size=1.5, energy=300, defocus=20000.0, num_defocus=ndf,
              spherical_aberration=2.7, phase_shift=20.0)
    got = G.reconstruct_projections(proj, angles, depth=depth, **kw)
    centre = O.get_centre(proj.shape, None, False)
    c, mn, mx = O.correct_projections(proj, centre, 1.5, 300, 20000.0, ndf,
                                      None, 2.7, 0, 0, 20.0)
    expect = O.reconstruct(c, angles, None, 1.5, mn, mx, depth=depth)
    err = numpy.linalg.norm(got - expect) / numpy.linalg.norm(expect)
    assert err < 1e-5, err
    for storage, bound in (("f16", 1e-3), ("bf16", 8e-3)):
        r = G.reconstruct_projections(proj, angles, depth=depth,
                                      storage=storage, **kw)
        err = numpy.linalg.norm(r - got) / numpy.linalg.norm(got)
        assert err < bound, (storage, err)
