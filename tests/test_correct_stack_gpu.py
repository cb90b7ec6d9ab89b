"""correct_projections over a whole stack: outputs of every kind of memory,
batches with a remainder, astigmatism, and the same values as one corr() call
per image with the host's CTF (bit for bit: the flip mask is the same, and so
are the transforms)."""
import numpy
import pytest

import guanaco_amd as G
from guanaco_amd import _capi as C

pytestmark = pytest.mark.gpu

KW = dict(pixel_size=1.3, energy=300, defocus=25000.0,
          spherical_aberration=2.7, phase_shift=12.0)


def one_by_one(proj, ndf, astigmatism):
    T, Y, X = proj.shape
    centre = numpy.full(Y, X / 2.0, numpy.float32)
    mn, mx, step, n = G.get_defocus_steps(25000.0, ndf, None, X, centre, 1.3)
    ctf = G.get_ctf_array(X, Y, 1.3, 300, mn, n, step, 2.7, astigmatism, 30.0,
                          12.0)
    out = numpy.zeros((T, ndf, Y, X), numpy.float32)
    for t in range(T):
        G.corr(numpy.ascontiguousarray(proj[t], numpy.float32), ctf, out[t],
               "gpu")
    return out


@pytest.mark.parametrize("X,Y,T,ndf,astigmatism", [
    (64, 32, 1, 1, 0.0), (64, 32, 5, 3, 400.0), (50, 37, 3, 2, 0.0),
    # two blocks of tilts, the second smaller (256 MiB of results each)
    (1024, 1024, 18, 4, 0.0),
])
def test_equals_corr_per_image(capi, tmp_path, X, Y, T, ndf, astigmatism):
    proj = numpy.random.default_rng(X + T).poisson(40, (T, Y, X)).astype(
        numpy.float32)
    expect = one_by_one(proj, ndf, astigmatism)
    kw = dict(KW, num_defocus=ndf, astigmatism=astigmatism,
              astigmatism_angle=30.0, device="gpu")
    outs = [None, str(tmp_path / "out.dat"),
            numpy.zeros(expect.shape, numpy.float64),
            numpy.zeros(expect.shape, numpy.float32)]
    for out in outs if X < 512 else outs[3:]:
        got, _, _ = G.correct_projections(proj, corrected_output=out, **kw)
        want = expect if ndf > 1 else expect[:, 0]
        assert got.shape == want.shape
        numpy.testing.assert_array_equal(numpy.asarray(got), want)
        if isinstance(out, numpy.ndarray):  # written in place
            assert numpy.shares_memory(got, out)
    # other input types, and a view that is not contiguous
    got, _, _ = G.correct_projections(
        numpy.asfortranarray(proj.astype(numpy.uint8)),
        corrected_output=numpy.zeros(expect.shape, numpy.float32), **kw)
    numpy.testing.assert_array_equal(
        got, expect if ndf > 1 else expect[:, 0])


def test_refusals(capi):
    proj = numpy.ones((2, 8, 16), numpy.float32)
    with pytest.raises(RuntimeError):
        G.correct_projections(proj, **dict(KW, device="cpu"))
    with pytest.raises(RuntimeError, match="pixel_size"):
        G.correct_projections(proj, **dict(KW, pixel_size=0, device="gpu"))
    d = C.StackDesc(9000, 8, 1, 1, (C.ctypes.c_double * 1)(1.0), 1.0, 0.02,
                    0.0, 0.0, 0.0, 0.0, -1)
    a = numpy.zeros(8, numpy.float32)
    with pytest.raises(C.GxError, match="8192"):
        C.call("gx_correct_stack", C.ctypes.byref(d), C.f32p(a), C.f32p(a))
