"""The static-scratch lm_head + argmax from 17 rows: taken as far as 32-entry tiles' keys fit the array,
with and without the norm, and equal to the workspace entry point bit for bit."""

import numpy as np
import pytest
import torch

from test_zz_no_alloc import _inputs, _outputs, _run

from kernels import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,v,k", [(17, 151936, 1024), (27, 151936, 512), (32, 50257, 5128)])
@pytest.mark.parametrize("norm", [False, True])
def test_static_scratch_from_17_rows(cuda, m, v, k, norm):
    assert 256 + 8 * m * ((v + 31) // 32) <= _native.STATIC_SCRATCH_BYTES
    x, w, gamma = _inputs(m, v, k, 7200 + m, cuda)
    gamma = gamma if norm else None
    flags = _native.EPI_ARGMAX | (_native.PLAN_PROLOGUE if norm else 0)
    workspace = torch.zeros(int(_native.lib().ftk_project_workspace_bytes(m, v, k, flags, None)), dtype=torch.uint8,
                            device=cuda)
    want, got = _outputs(m, v, cuda, torch.int64), _outputs(m, v, cuda, torch.int64)
    assert _run("ftk_lm_head_argmax_bf16", x, w, gamma, *want, workspace=workspace) == _native.FTK_OK
    assert _run("ftk_lm_head_argmax_static_bf16", x, w, gamma, *got) == _native.FTK_OK
    for a, b in zip(got[:2], want[:2]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert torch.equal(got[2].view(torch.int32), want[2].view(torch.int32))
    np.testing.assert_array_equal(got[1].cpu().numpy(), torch.argmax(got[0].float().cpu(), -1).numpy())
