"""Products of few tiles, whose stages of 64 values are taken in turn by four or eight groups of waves: whole and partial turns,
remainders of rows and columns, both ends of what takes each form and the first sizes that do not, against float64."""
import pytest

from tests import test_gpu_dense_tiles as tiles
from tests.test_gpu_dense_tiles import runtime  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu
# 16 x 32 tiles: 3 stages (without), 4, 5, 8, 11, 16, 17; one tile, a row and a column more; as many as CUs and one more (32 x 32)
# 32 x 32: 4 to 19 stages, as many as CUs and one more (32 x 64, from 16 stages); 32 x 64: 15 stages (without), 16 to 19, one more tile
SIZES = [(2, 5, 192), (2, 5, 256), (16, 32, 320), (17, 33, 512), (31, 701, 704), (64, 1024, 1024), (33, 63, 1088), (64, 2048, 320),
         (64, 2049, 256), (33, 3000, 320), (60, 4000, 1152), (64, 4096, 1216), (60, 4097, 960), (60, 4097, 1024), (128, 4000, 1088),
         (127, 3001, 1152), (128, 4096, 1216), (128, 4097, 2112), (65, 300, 4096)]


@pytest.mark.parametrize("m,n,k", SIZES)
def test_sums(runtime, m, n, k):  # noqa: F811
    tiles.test_tiles(runtime, m, n, k)


@pytest.mark.parametrize("m,n,k", SIZES)
def test_rows(runtime, m, n, k):  # noqa: F811
    tiles.test_rows_split_in_two(runtime, m, n + 40, k)


@pytest.mark.parametrize("m,n,k", SIZES)
def test_pairs(runtime, m, n, k):  # noqa: F811
    tiles.test_gated_tiles(runtime, m, k, max(16, n // 2))
