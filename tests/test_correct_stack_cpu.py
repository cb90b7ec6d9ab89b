"""What correct_projections hands to the stack correction, and what it does
with outputs that are more than memory."""
import numpy
import pytest

import guanaco_amd as G
from guanaco_amd.detail import correct

KW = dict(pixel_size=1.3, energy=300, defocus=25000.0, num_defocus=2,
          spherical_aberration=2.7, device="gpu")


def test_a_masked_output_is_unmasked(monkeypatch):
    def stack(images, out, defoci, ctf, pixel_size, device):
        out[:] = images[:, None] + numpy.arange(len(defoci))[:, None, None]

    monkeypatch.setattr(correct.ext, "correct_stack", stack)
    proj = numpy.arange(24, dtype=numpy.float32).reshape(3, 2, 4)
    out = numpy.ma.masked_all((3, 2, 2, 4), numpy.float32)
    got, _, _ = G.correct_projections(proj, corrected_output=out, **KW)
    assert not numpy.ma.getmaskarray(got).any()
    numpy.testing.assert_array_equal(got.data[:, 1], proj + 1)


@pytest.mark.parametrize("shape", [(2, 4, 0), (2, 0, 4)])
def test_empty_images_are_refused(shape):
    T, Y, X = shape
    with pytest.raises(RuntimeError):
        G.correct_projections(numpy.ones(shape, numpy.float32), centre=2.0,
                              corrected_output=numpy.zeros((T, 2, Y, X)),
                              **KW)
