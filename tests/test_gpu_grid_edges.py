"""Where a grid's layout changes: runs of chunks per XCD double at 512 << k chunks (up to runs of 64),
and a tile of the leading statistics holds 32 indices of the first dimension, 16 in flight."""
import pytest

from tests import test_gpu_chunk_runs as runs
from tests import test_gpu_rank1 as rank1

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [512, 1025, 4095, 4097, 16383, 32767, 32769])
def test_chunk_runs(cuda, chunks):
    runs.test_grid_sizes(cuda, chunks)


@pytest.mark.parametrize("outer", [15, 16, 17, 31, 32, 33, 48, 49, 65])
@pytest.mark.parametrize("inner", [(40, 3, 3), (90, 5)])
def test_leading_statistics(cuda, outer, inner):
    rank1.test_rank1_more_than_two_dimensions_against_oracle(cuda, (outer, *inner), "fp32", "bf16", False)
