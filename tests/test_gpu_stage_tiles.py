"""The WENO5 advection stage at the edges of its tiles and walks: rows just
below, at and above 32 and 64 cells (32- and 64-wide tiles), fewer rows than a
tile, and planes that do not fill a walk (4 planes a block on small grids),
against the oracle at the advection's tolerance (1e-12 of the field's max, as
in test_gpu_parity.py); and the multi-block launch on blocks of unequal
extents, bit for bit the whole-field step."""
import numpy as np
import pytest
import torch   # before the library: both then share one HIP runtime

from cases import bubble, max_rel, node_velocities
from fortrancfd_amd.types import Case
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

SIZES = [(31, 5, 1), (64, 4, 1), (65, 9, 1), (129, 33, 1), (32, 8, 4), (33, 9, 5), (63, 5, 17), (64, 7, 16),
         (96, 4, 9), (97, 13, 6)]


def _case(nx, ny, nz):
    h = 1.0 / 32
    return Case(dim=2 if nz == 1 else 3, nx=nx, ny=ny, nz=nz, xend=nx * h, yend=ny * h, zend=nz * h)


@pytest.mark.parametrize("size", SIZES)
def test_stage_tiles(size):
    from fortrancfd_amd import Solver
    case = _case(*size)
    s, o = Solver(case), Oracle(case)
    Oracle.threads(1)
    for n, a in {"phi": bubble(case, 0.3, 1), **node_velocities(case, 3)}.items():
        s.push(n, a)
        o.set(n, a)
    for _ in range(2):
        s.level_set_rk3_solver()
        o.call("switch")
        o.call("level_set_rk3_solver")
    r = max_rel(s.pull("phi"), o.get("phi"))
    assert r <= 1e-12, r


@pytest.mark.parametrize("size,nb", [((67, 11, 13), (2, 2, 3)), ((129, 10, 9), (2, 3, 2)), ((70, 31, 1), (3, 4, 1))])
def test_blocks_in_one_launch(size, nb):
    from fortrancfd_amd import Solver
    from fortrancfd_amd.blocks import Blocks
    from fortrancfd_amd.types import bc_copy
    case = _case(*size)
    phi = bc_copy(case, bubble(case, 0.3, 1))
    vel = [bc_copy(case, a) for a in node_velocities(case, 3).values()]
    s, B = Solver(case), Blocks(case, *nb)
    s.push("phi", phi)
    for n, a in zip(("nu", "nv", "nw"), vel):
        s.push(n, a)

    def stack(a):
        t = B.new_stack()
        B.scatter(torch.from_numpy(np.ascontiguousarray(a)).cuda(), t)
        B.sync(t)
        return t

    st, sv = stack(phi), [stack(a) for a in vel]
    for _ in range(2):
        s.level_set_rk3_solver()
        B.level_set_rk3_solver(st, *sv)
    out = torch.zeros(case.size, dtype=torch.float64, device="cuda")
    B.gather(st, out)
    torch.cuda.synchronize()
    assert np.array_equal(case.interior(out.cpu().numpy()), case.interior(s.pull("phi")))
