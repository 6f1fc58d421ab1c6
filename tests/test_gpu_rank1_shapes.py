"""The statistics kernels of rank-1 scaling at the sizes where their forms change or end: the
flat form up to 256 columns, or 88 where they are a multiple of 8 (a tile is 4096 / (cols | 1) rows),
the wide forms above it, and the leading statistics of tensors with several
leading dimensions, whose rows fill part of a tile, one tile or several."""
import pytest

from tests import test_gpu_rank1 as base

pytestmark = pytest.mark.gpu

# a tile's rows: 1365 for 2 and 3 columns, 240 for 16, 31 for 128 .. 131, 16 for 255, 15 for 256
MATRICES = [(1365, 3), (1366, 2), (4100, 3), (240, 16), (241, 16), (31, 128), (63, 129), (17, 255), (46, 256),
            (300, 257), (257, 263), (64, 264), (260, 511), (9, 513), (258, 1025), (70, 1031),
            # multiples of 8 on either side of the wide form's first width, fewer rows than a tile and more
            (33, 88), (1000, 88), (33, 96), (1000, 96), (260, 104)]
# where a workgroup's rows double (6144, 24576 and 98304 rows): several tiles of the flat form, more rows of the
# wide ones; the last workgroup with all of its tiles, with some, with part of one
TALL = [(6145, 50), (6144 + 63 * 5, 64), (6200, 255), (24577, 33), (24640, 88), (98305, 24), (98304 + 500, 41), (6150, 96), (24600, 104), (98310, 96), (6200, 257)]
TENSORS = [(5, 300, 3, 3), (2, 700, 3), (1400, 1, 2), (300, 2, 7), (16, 16, 16), (3, 100, 260), (2, 130, 4, 257), (64, 3, 7, 7)]


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16"), ("fp32", "fp16")])
@pytest.mark.parametrize("shape", MATRICES)
def test_statistics_of_a_matrix(cuda, shape, p_dt, g_dt):
    base.test_rank1_against_oracle(cuda, p_dt, g_dt, shape)


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16")])
@pytest.mark.parametrize("shape", TALL)
def test_statistics_of_a_tall_matrix(cuda, shape, p_dt, g_dt):
    base.test_rank1_against_oracle(cuda, p_dt, g_dt, shape)


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16")])
@pytest.mark.parametrize("shape", TENSORS)
def test_statistics_of_several_dimensions(cuda, shape, p_dt, g_dt):
    base.test_rank1_more_than_two_dimensions_against_oracle(cuda, shape, p_dt, g_dt, False)
