"""An f32 store's prompt tiles (csrc/kr_serve_tile_f32.hip): 64, 48 and 32 rows, every number of 16-row blocks in the last one (1 - 3: each wave's rows on 4x4x1 products, 4: on
16x16x1), one row to either side of a border; one slot of k, as many as the ring holds, one more and two more; ragged columns; experts of 0 - 70 rows.
Oracle and bounds: test_serve_gemm_gpu.py."""
import pytest

from tests.test_serve_gemm_gpu import test_expert_products_sizes_f32 as expert_products
from tests.test_serve_gemm_gpu import test_vocabulary_projection_sizes_f32 as vocabulary_projection

pytestmark = pytest.mark.gpu

DENSE = [(16, 129), (17, 129), (33, 127), (64, 129),                      # tiles of 32 rows
         (112, 4100), (113, 4099), (129, 4100), (144, 4097),              # 48
         (193, 8191), (209, 8192), (225, 8191), (97, 8191), (113, 8190)]  # 64


@pytest.mark.parametrize("width", [32, 96, 128, 160])
@pytest.mark.parametrize("want,vocab", DENSE)
def test_single_matrix(want, vocab, width):
    vocabulary_projection(want, vocab, width)


@pytest.mark.parametrize("n", [15, 16, 17, 31, 33, 47, 49, 63, 65, 70])
def test_experts(n):
    expert_products(n)                                                    # every token on each of the five experts
