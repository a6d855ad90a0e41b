"""Launch choices with any fields, for every kind, at sizes with and without a default launch: the planner
answers with a status and a launch it can count, whatever it is given (host only; in a child process,
since a division by zero there would end it)."""

import subprocess
import sys

import pytest

CHILD = """
import itertools, sys
sys.path.insert(0, {package!r})
from kernels import _native
plan, call = _native.Plan(), _native.lib().ftk_plan_project
seen = set()
for m, n, k in itertools.product((1, 2, 5, 8, 16, 17, 32), (2, 768, 4096), (8, 72, 128, 640, 1024, 4096, 12288)):
    for epi, rows, unroll, groups, waves in itertools.product(
            (0, 1, 2, 0x100, 0x101, 0x102, 0x301), (-1, 0, 1, 3, 8, 16), (-1, 0, 1, 4), (0, 1), (-1, 0, 1, 3, 8)):
        status = call(m, n, k, epi, 256, _native.Config({kind}, rows, unroll, groups, waves), plan)
        seen.add(status)
        assert status in (0, 1, 2), status
        if status == 0:
            assert plan.grid > 0 and plan.tiles > 0 and plan.workspace_bytes >= 0
print("statuses", sorted(seen))
"""


@pytest.mark.parametrize("kind", range(-1, 11))
def test_any_fields(kind):
    from conftest import PKG

    child = subprocess.run([sys.executable, "-c", CHILD.format(package=str(PKG), kind=kind)], capture_output=True,
                           text=True, timeout=300)
    assert child.returncode == 0, (child.returncode, child.stderr[-400:])
    assert "statuses" in child.stdout
