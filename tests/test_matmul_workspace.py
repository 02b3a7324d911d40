"""The prefill matmul's workspace is its fp16 rows and their scales, whatever
kernel a size goes to: no whole-tile padding, which near the no-alloc scratch's
limit would refuse buckets that fit."""
from __future__ import annotations

import pytest

from r9v_amd import ffi


@pytest.mark.parametrize("m,k", [(9, 256), (33, 4096), (260, 28672), (577, 14336), (2048, 4096)])
def test_prefill_workspace_bytes(m, k):
    st = ffi.matmul_static(n=512, k=k, w_scheme=ffi.Q4_K, in_dtype=ffi.BF16, out_dtype=ffi.F32, m_bucket=m)
    assert ffi.matmul_workspace_bytes(st) == (2 * m * k + 255) // 256 * 256 + 4 * m
    if m in (260, 577):
        assert ffi.matmul_workspace_bytes(st) <= ffi.NOALLOC_SCRATCH_BYTES
