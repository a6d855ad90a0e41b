"""Which kind the planner takes on both sides of the lines between FLOW, the LDS-fed tiles and the kinds
before them, at 256 CUs (host only). The lines come from timing every kind of these shapes; a shape that
sits on the wrong side of its line was 4 to 60 per cent slower there."""

import pytest

from kernels import _native
from kernels.linear import plan

STORE, SWIGLU, ARGMAX = _native.EPI_STORE, _native.EPI_SWIGLU, _native.EPI_ARGMAX
GEMV, TILES, STREAM, QUAD, FLOW = (_native.KIND_GEMV, _native.KIND_MFMA, _native.KIND_STREAM, _native.KIND_QUAD,
                                   _native.KIND_FLOW)

#: (rows, N, K, epilogue, norm, kind)
LINES = [
    # the norm beside QUAD, 5..8 rows
    (5, 1024, 2048, STORE, True, QUAD), (5, 2048, 2048, STORE, True, QUAD), (8, 2048, 3072, STORE, True, QUAD),
    (6, 4096, 3072, STORE, True, QUAD), (8, 4096, 3072, STORE, True, FLOW), (5, 4096, 1024, STORE, True, FLOW),
    (5, 6144, 2048, STORE, True, FLOW), (8, 1024, 1024, STORE, True, QUAD), (9, 1024, 2048, STORE, True, FLOW),
    (5, 2560, 3072, STORE, True, FLOW), (5, 2576, 3072, STORE, True, QUAD), (6, 4112, 3072, STORE, True, FLOW),
    # gate/up beside QUAD, 3..4 rows
    (3, 2048, 2048, SWIGLU, True, QUAD), (4, 6144, 3072, SWIGLU, True, QUAD), (4, 6144, 1024, SWIGLU, True, FLOW),
    (3, 12288, 2048, SWIGLU, True, FLOW), (4, 24576, 1024, SWIGLU, True, FLOW), (4, 27648, 1024, SWIGLU, True, QUAD),
    (4, 24576, 4096, SWIGLU, True, QUAD), (4, 3072, 3072, SWIGLU, False, FLOW), (4, 2048, 3072, SWIGLU, False, QUAD),
    # vocabularies beside QUAD
    (3, 8000, 2048, ARGMAX, True, QUAD), (3, 8000, 2048, ARGMAX, False, FLOW), (3, 18992, 2048, ARGMAX, True, FLOW),
    # beside GEMV, two to four rows
    (2, 1024, 5120, STORE, True, GEMV), (3, 1024, 5120, STORE, True, GEMV), (3, 2048, 5120, STORE, True, FLOW),
    (2, 4096, 5120, SWIGLU, True, GEMV), (2, 6144, 5120, SWIGLU, True, FLOW), (2, 4096, 3584, STORE, True, GEMV),
    (2, 6144, 3584, STORE, True, FLOW), (2, 10240, 1280, SWIGLU, True, GEMV), (2, 12288, 1280, SWIGLU, True, FLOW),
    (3, 10240, 1280, SWIGLU, True, FLOW), (2, 10240, 1280, SWIGLU, False, FLOW), (4, 1024, 5120, STORE, True, FLOW),
    (4, 512, 5120, SWIGLU, False, FLOW), (4, 496, 5120, SWIGLU, False, GEMV), (4, 1024, 5120, SWIGLU, True, FLOW),
    (3, 2048, 5120, SWIGLU, True, GEMV), (2, 8192, 1152, STORE, True, FLOW), (2, 8208, 1152, STORE, True, GEMV),
    (2, 8192, 1160, STORE, True, GEMV),
    # beside GEMV, one row
    (1, 8192, 2560, STORE, True, GEMV), (1, 9216, 2560, STORE, True, FLOW), (1, 9216, 2560, SWIGLU, True, FLOW),
    # plain projections
    (1, 512, 6144, STORE, False, GEMV), (1, 2048, 6144, STORE, False, TILES), (1, 6144, 2560, STORE, False, GEMV),
    (1, 5120, 2560, STORE, False, TILES), (1, 7168, 2560, STORE, False, TILES), (1, 8192, 8192, STORE, False, GEMV),
    (2, 8192, 8192, STORE, False, GEMV), (3, 8192, 8192, STORE, False, TILES), (2, 512, 5120, STORE, False, GEMV),
    (2, 768, 5120, STORE, False, TILES), (1, 2560, 9728, STORE, False, TILES), (3, 1024, 2048, STORE, False, STREAM),
    (3, 1280, 2048, STORE, False, TILES), (4, 512, 4096, STORE, False, STREAM), (4, 768, 4096, STORE, False, TILES),
    (4, 512, 1024, STORE, False, TILES), (4, 4096, 1024, STORE, False, STREAM),
]


@pytest.mark.parametrize("m,n,k,epilogue,norm,kind", LINES)
def test_line(m, n, k, epilogue, norm, kind):
    assert plan(m, n, k, epilogue, 256, prologue=norm).kind == kind
