"""The fixed bytes a projection without an argmax is given cover what the library asks for."""

import pytest

from kernels import _native


@pytest.mark.parametrize("epilogue", [_native.EPI_STORE, _native.EPI_SWIGLU])
@pytest.mark.parametrize("flags", [0, _native.PLAN_PROLOGUE, _native.PLAN_PROLOGUE | _native.PLAN_RESIDUAL])
def test_fixed_bytes_cover_every_plan_without_an_argmax(epilogue, flags):
    configs = [None, _native.Config(_native.KIND_FLOW, 0, 0, 0, 0)]
    configs += [_native.Config(_native.KIND_MFMA, rows, unroll, 0, waves)
                for rows, unroll, waves in ((16, 1, 8), (16, 4, 4), (16, 8, 8), (32, 4, 8), (64, 2, 4))]
    for cfg in configs:
        for m in (1, 2, 4, 5, 8, 16, 17, 32):
            for n, k in ((16, 8), (4096, 1024), (24576, 4096), (4096, 12288), (151936, 4096), (1001, 777)):
                need = _native.lib().ftk_project_workspace_bytes(m, n, k, epilogue | flags, cfg)
                assert 0 <= need <= _native.PROJECT_FIXED_BYTES
