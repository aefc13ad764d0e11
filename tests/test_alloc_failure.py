"""Scratch memory that could not be allocated completely is not taken as
complete by the next call (no GPU: the HIP calls of the multi-block step go to
a stand-in that counts them and fails one on request).  A call that runs out
of memory reports it and launches nothing; the next one allocates what is
missing before it launches."""
import os

import pytest

import hip_standin

BODY = r"""
case = Case(dim=3, nx=12, ny=12, nz=12)
grid, params = case.grid_struct(), case.param_struct()
lib.fcfd_blocks_create.argtypes = [vp, vp] + [C.c_int] * 6 + [vp]
lib.fcfd_blocks_level_set_rk3_solver.argtypes = [vp] * 6
lib.fcfd_blocks_destroy.argtypes = [vp]
for fail_at in range(1, 7):   # the block table, its copy, the four stacks
    h = vp()
    hip.standin_reset(fail_at)
    assert lib.fcfd_blocks_create(C.byref(grid), C.byref(params), 2, 1, 1, 0, 0, 0, C.byref(h)) == 0
    step = lambda: lib.fcfd_blocks_level_set_rk3_solver(h, 8, 8, 8, 8, None)
    assert step() != 0, fail_at
    assert hip.standin_launches() == 0, fail_at
    assert step() == 0, fail_at
    assert hip.standin_live() == 5, (fail_at, hip.standin_live())
    assert hip.standin_launches() > 0
    lib.fcfd_blocks_destroy(h)
    assert hip.standin_live() == 0, (fail_at, hip.standin_live())
print("done")
"""


@pytest.mark.skipif(not os.path.exists(hip_standin.LIB), reason="libfcfd.so not built (fortrancfd_amd/build.py)")
def test_blocks_step_after_a_failed_allocation(tmp_path):
    hip_standin.run(tmp_path, BODY)
