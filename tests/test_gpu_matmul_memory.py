"""A matmul on a device whose memory is nearly used up: without room for its workspace it runs as
the shapes without one do."""

from __future__ import annotations

from contextlib import contextmanager

import pytest
import torch

from conftest import accum_rtol
from t81lib_amd import _lib, ops
from test_gpu_exact_f32 import announce

pytestmark = pytest.mark.gpu


@contextmanager
def no_room_for(nbytes, device):
    """This process's allocations fail from nbytes on, by torch's own limit on it."""
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(device).total_memory
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
    held = []
    try:
        with pytest.raises(torch.OutOfMemoryError):
            while len(held) < 10000:  # what is free in the blocks that are held already
                held.append(torch.empty(nbytes, dtype=torch.uint8, device=device))
        yield
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        held.clear()


@pytest.mark.parametrize("M,K,N,dtype", [(2048, 14336, 4096, torch.float32),
                                         (512, 4096, 6144, torch.bfloat16),
                                         (700, 4095, 9000, torch.bfloat16)])
def test_without_room_for_the_workspace(gpu, M, K, N, dtype):
    announce(f"matmul near the memory limit M={M} K={K} N={N} {dtype}")
    code = _lib.DTYPE_F32 if dtype == torch.float32 else _lib.DTYPE_BF16
    need = _lib.lib().t81_hip_ternary_matmul_workspace_size(M, N, K, code)
    g = torch.Generator("cpu").manual_seed(M)
    packed = ops.quantize_pack(torch.randn((N, K), generator=g).to(gpu), 0.45, _lib.THR_CPP)
    x = torch.randn((M, K), generator=g).to(gpu, dtype)
    c = torch.zeros((M, N), device=gpu)
    t = ops.unpack(packed, N, K).double().t().contiguous()
    want, mags = x.double() @ t, x.double().abs() @ t.abs()
    del t
    assert need > 4 << 20
    with no_room_for(4 << 20, gpu):
        ops.ternary_matmul(x, packed, K, c=c)
    assert bool(((c.double() - want).abs() <= accum_rtol(K, dtype) * mags).all())
