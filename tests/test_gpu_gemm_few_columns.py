"""bf16 products with at most 32 columns and few rows, on the kernel that splits K over a workgroup's waves, on both
sides of the line where it ends (K of 4096, with more than 16 columns 2048, and where a copy of B fills the LDS)."""
import pytest

import test_gpu_kernels as kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b_layout", ["n", "t"])
@pytest.mark.parametrize("out", ["bf16", "f32"])
@pytest.mark.parametrize("shape", [(16, 8, 1024), (17, 16, 2048), (33, 32, 1024), (1000, 8, 256), (1023, 24, 320),
                                   (15, 8, 1024), (100, 16, 2112), (500, 32, 1088)])
def test_few_rows(hip, b_layout, out, shape):
    kernels.test_gemm_few_columns(hip, b_layout, out, shape)


@pytest.mark.parametrize("b_layout", ["n", "t"])
@pytest.mark.parametrize("out", ["bf16", "f32"])
@pytest.mark.parametrize("shape", [(1000, 8, 4096), (16, 8, 4032), (33, 16, 4096), (47, 16, 3072), (100, 32, 2048),
                                   (100, 24, 1984), (17, 8, 4160), (1024, 8, 6144), (8193, 8, 4096)])
def test_long_rows(hip, b_layout, out, shape):
    kernels.test_gemm_few_columns(hip, b_layout, out, shape)
