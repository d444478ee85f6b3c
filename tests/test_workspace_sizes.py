"""The workspace a trit-dot matmul reports: what its launch uses, within the 64 MiB static scratch
of the no-allocation entry wherever a launch within it exists."""

from __future__ import annotations

import pytest

from t81lib_amd import _lib

SCRATCH = 64 << 20
F32, BF16, I8 = _lib.DTYPE_F32, _lib.DTYPE_BF16, _lib.DTYPE_I8


def size(m, n, k, dtype):
    return _lib.lib().t81_hip_ternary_matmul_workspace_size(m, n, k, dtype)


@pytest.mark.parametrize("m,k,n", [(16384, 3072, 3072), (16384, 3072, 1), (4681, 14336, 14336),
                                   (9105, 25792, 2944), (17719, 16088, 1884), (4096, 28672, 512),
                                   (2048, 14336, 4096), (40000, 60000, 700)])
def test_float32_planes_fit_the_scratch(m, k, n):
    """Tokens whose planes are an uneven number of chunks, and K that is cut in parts."""
    assert 0 < size(m, n, k, F32) <= SCRATCH


@pytest.mark.parametrize("m,k,n,dtype", [(777, 3072, 9216, BF16), (1024, 3072, 9216, BF16),
                                         (1024, 4096, 6144, BF16), (1536, 4096, 6144, I8),
                                         (1024, 3072, 9216, I8), (2500, 14336, 4096, I8)])
def test_384_row_tiles_use_none(m, k, n, dtype):
    assert size(m, n, k, dtype) == 0


@pytest.mark.parametrize("m,k,n", [(512, 4096, 8448), (65, 2048, 14336), (100, 14336, 4096),
                                   (2048, 4095, 14336)])
def test_bf16_images_fit_the_scratch(m, k, n):
    """The image and its partials, not the split over K that they replace."""
    assert 0 < size(m, n, k, BF16) <= SCRATCH
