"""One centre per row on both sides of the limit (2048 tiles times row blocks)
where a thread takes fewer voxels: the other tests' volumes lie far below it.
Float32 plans have the oracle's bits, 16-bit ones its values to the bound that
tests/test_bp_mm_gpu.py derives."""
import pytest

import test_bp_mm_gpu as mm
import test_gpu_parity as parity

pytestmark = pytest.mark.gpu


# 16 x 16 tiles by 8 and 9 blocks of 16 rows (twice as many of 8), the last
# tiles partial
@pytest.mark.parametrize("Y,ndf", [(128, 1), (141, 1), (64, 3), (141, 3)])
def test_f32(capi, Y, ndf):
    mn, mx = (-60.0, 60.0) if ndf > 1 else (0.0, 0.0)
    parity.test_per_row_centre_bp_bitexact_vs_oracle(
        capi, (75, Y, 5, ndf, 125, 509, (-60.0, 60.0), (mn, mx), 1.0))


@pytest.mark.parametrize("storage,rows", [("f16", 32), ("f16", 16),
                                          ("bf16", 32)])
@pytest.mark.parametrize("Y,ndf", [(256, 1), (270, 1), (270, 3)])
def test_reduced(capi, Y, ndf, storage, rows):
    mn, mx = (-60.0, 60.0) if ndf > 1 else (0.0, 0.0)
    mm.test_centre_per_row_matches_oracle_on_its_own_slabs(
        capi, (75, Y, 5, ndf, 125, 509, (mn, mx), 2.5), storage, rows)
