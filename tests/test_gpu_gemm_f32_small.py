"""float32 products of few tiles: the forms with tiles of 16 x 16 and 32 x 32, eight and sixteen waves, at the edges
of their tiles, of a K tile (128 and 256) and of the lines between them.  Whole numbers: every sum is exact
in float32."""
import pytest

from test_gpu_gemm_f32_tiles import L, product  # noqa: F401  (a fixture)

pytestmark = pytest.mark.gpu

SIZES = [(16, 16, 128), (17, 15, 129), (1, 33, 127), (128, 256, 784), (100, 3, 1000), (255, 257, 385),  # 16 x 16, eight waves
         (256, 256, 2048), (33, 47, 2049), (5, 200, 4095), (16, 16, 4096),  # sixteen
         (513, 241, 256), (600, 300, 131), (1000, 500, 384), (500, 1000, 128), (993, 481, 513),  # 32 x 32, eight
         (600, 300, 127), (1000, 500, 300)]  # four


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_few_tiles(L, M, N, K, layout):  # noqa: F811
    product(L, M, N, K, layout, odd=M % 3, epilogue=K % 2 == 1)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K,batch", [(17, 30, 200, (3, 5)), (40, 20, 2100, (2, 3)), (64, 64, 256, (8, 8)), (90, 33, 140, (5, 9))])
def test_batches_of_few_tiles(L, M, N, K, layout, batch):  # noqa: F811
    product(L, M, N, K, layout, batch=batch)
