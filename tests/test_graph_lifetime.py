"""The captured iterations of a pressure solve are destroyed (new parameters,
the profiler, new cases) only once the stream has run them: a solve returns
with its last iteration, or one queued ahead in vain, in flight.  No GPU: the
HIP calls go to a stand-in that notes the order of graph launches, stream
synchronisations and graph destructions."""
import os

import pytest

import hip_standin

BODY = r"""
lib.fcfd_create.argtypes = [vp, vp, vp]
lib.fcfd_ppe_solve_rhs.argtypes = [vp, C.c_double, C.c_int, vp, vp]
lib.fcfd_set_params.argtypes = [vp, vp]
lib.fcfd_prof_enable.argtypes = [vp, C.c_int]
case = Case(dim=3, nx=16, ny=16, nz=16)
grid, params = case.grid_struct(), case.param_struct()
h, cyc, rel = vp(), C.c_int(), C.c_double()
hip.standin_reset(0)
assert lib.fcfd_create(C.byref(grid), C.byref(params), C.byref(h)) == 0
n = 0
for drop in (lambda: lib.fcfd_set_params(h, C.byref(params)), lambda: lib.fcfd_prof_enable(h, 0)):
    for precision in (0, 1):
        assert lib.fcfd_ppe_solve_rhs(h, 1e-10, precision, C.byref(cyc), C.byref(rel)) == 0
        assert hip.standin_graph_launches()
        assert drop() == 0
        assert hip.standin_destroyed() > n
        n = hip.standin_destroyed()
        assert hip.standin_destroyed_early() == 0, (precision, hip.standin_destroyed_early())
print("done")
"""


@pytest.mark.skipif(not os.path.exists(hip_standin.LIB), reason="libfcfd.so not built (fortrancfd_amd/build.py)")
def test_graphs_outlive_their_launches(tmp_path):
    hip_standin.run(tmp_path, BODY)
