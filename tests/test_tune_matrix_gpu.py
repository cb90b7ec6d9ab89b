"""Tile choices of plans that differ in nothing but the width of their slabs,
and so in the kernel that they run on."""
import numpy
import pytest

from guanaco_amd import _capi as C

pytestmark = pytest.mark.gpu


def plan_of(width):
    """Three slabs `width` pixels wide; 512 workgroups."""
    angles = numpy.deg2rad(numpy.linspace(-60, 60, 5)).astype(numpy.float32)
    half = 1.5 * width
    return C.VolumePlan(520, 97, angles, 256, width=512, num_defocus=3,
                        min_defocus=-half, max_defocus=half, storage="f16",
                        input_layout=C.INPUT_SINOGRAMS)


def lines(path):
    C.tune_save(str(path))
    return [l for l in path.read_text().splitlines() if l[0] != "#"]


def test_kernels_have_their_own_choices(capi, tmp_path):
    C.tune_clear()
    d_in = C.DeviceArray.from_host(numpy.ones((97, 3, 5, 520), numpy.float32))
    d_vol = C.DeviceArray((97, 256, 512))
    # 100 pixels: the matrix cores; 40: the staged kernel, two slabs either way
    wide, narrow = plan_of(100), plan_of(40)
    assert wide.backprojector() == narrow.backprojector() == (C.BP_STAGED, 2)
    assert wide.tile() == narrow.tile() == (32, C.BP_STAGED)
    wide.autotune(d_in, d_vol)
    kept = lines(tmp_path / "a.txt")
    assert len(kept) == 1
    # a choice other than the default, for the shape of the first
    (tmp_path / "b.txt").write_text(
        " ".join(kept[0].split()[:-1] + ["16"]) + "\n")
    C.tune_load(str(tmp_path / "b.txt"))
    for width, rows in ((100, 16), (40, 32)):
        p = plan_of(width)
        assert p.tile() == (rows, C.BP_STAGED)
        p.destroy()
    # tuning the other leaves it
    narrow.autotune(d_in, d_vol)
    kept = lines(tmp_path / "c.txt")
    assert len(kept) == 2 and any(l.endswith(" 16") for l in kept)
    p = plan_of(100)
    assert p.tile() == (16, C.BP_STAGED)
    for q in (p, wide, narrow):
        q.destroy()
    C.tune_clear()


@pytest.mark.parametrize("rows,matrix", [
    (32, False), (96, False), (97, True), (128, True), (129, False),
    (192, False), (193, True), (288, False), (320, True), (928, True),
])
def test_several_slabs_need_full_row_groups(capi, rows, matrix):
    angles = numpy.zeros(1, numpy.float32)
    p = C.VolumePlan(64, rows, angles, 256, width=512, num_defocus=2,
                     min_defocus=-100.0, max_defocus=100.0, storage="f16",
                     input_layout=C.INPUT_SINOGRAMS)
    assert p.matrix_cores() == matrix
    p.destroy()
