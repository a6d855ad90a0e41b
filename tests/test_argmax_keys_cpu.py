"""Key words a vocabulary projection asks for: from 17 rows never more than one per row and 32
vocabulary entries, or per row and CU, so that calls fit the static scratch as far as 32-entry tiles
do (host only)."""

import pytest

from kernels import _native
from kernels.linear import plan


@pytest.mark.parametrize("rows", [17, 24, 25, 27, 32])
@pytest.mark.parametrize("k", [8, 1024, 4096, 5120, 5128, 8192, 12288, 32768])
@pytest.mark.parametrize("norm", [False, True])
def test_keys_from_17_rows(rows, k, norm):
    for vocab in (1, 31, 33, 8000, 50257, 151936):
        need = plan(rows, vocab, k, _native.EPI_ARGMAX, prologue=norm).workspace_bytes
        assert 0 < need <= 256 + 8 * rows * max(256, (vocab + 31) // 32)
