"""The three forms of the reduced CCD line solve at the edges of their ranges:
lines of one interface, of 20 and 21, of the 73 that fit LDS and one more, with
line counts that fill no block, and with more lines than the LDS form takes in
a round; against the oracle.  And lines that fit LDS but are too many for it,
bit for bit as where they are few."""
import numpy as np
import pytest

from fortrancfd_amd.types import Case

pytestmark = pytest.mark.gpu

# The line is solved in another order than the oracle's: each answer is off by
# up to a few eps times the condition number of the line's system in (f', h f''),
# 3544 for the upwind matrices and 2833 for CCD in the maximum norm at every
# length from 29 points on (formed and inverted in numpy).
TOL = 4.0 * 2.2e-16 * 3544

# (nx, ny, nz): n cells are n + 6 points, ceil(./16) segments, one interface less
SIZES = [(11, 70, 1), (330, 70, 1), (331, 70, 1), (70, 330, 1), (70, 331, 1), (1178, 23, 1), (1179, 23, 1),
         (23, 1178, 1), (23, 1179, 1), (190, 186, 11)]


@pytest.mark.parametrize("size", SIZES)
def test_reduced_solves(size):
    from test_gpu_parity import _cmp, _pair, bubble, node_velocities
    nx, ny, nz = size
    dim = 2 if nz == 1 else 3
    case = Case(dim=dim, nx=nx, ny=ny, nz=nz, xend=nx / 64.0, yend=ny / 64.0, zend=nz / 64.0,
                gvec=(0.0, -1.0, 0.0), name="t")
    names = ["nx", "ny", "nz"][:dim] + ["nxx", "nyy", "nzz"][:dim]
    s, o = _pair(case, {"phi": bubble(case, 0.3, 1), **node_velocities(case, 3)})
    s.curv(); o.call("curv")
    _cmp(s, o, names, TOL)
    s, o = _pair(case, {"phi": bubble(case, 0.3, 1), **node_velocities(case, 3)})
    s.uccd()
    o.call("switch"); o.call("uccd")
    _cmp(s, o, names, TOL)


def test_many_long_lines_take_the_same_bits():
    """68 interfaces, 12400 lines in two systems: more than three rounds of the
    LDS form's blocks (12288 lines on 256 CUs), so the general form takes them;
    64 lines take the LDS form.  The rows repeat every 64."""
    from fortrancfd_amd import Solver
    out = []
    for ny in (64, 12400):
        case = Case(dim=2, nx=1100, ny=ny, nz=1, xend=1100 / 64.0, yend=ny / 64.0)
        x, j = np.arange(1106)[None, :], (np.arange(-3, ny + 3) % 64)[:, None]
        rows = {"phi": np.sin(0.02 * x + 0.1 * j) + 0.01 * np.cos(0.7 * x * (1 + j)), "nu": np.cos(0.05 * x + j),
                "nv": np.zeros((ny + 6, 1106))}
        s = Solver(case)
        for n, a in rows.items():
            s.push(n, np.ascontiguousarray(a).reshape(case.shape))
        s.uccd()
        out.append([case.interior(s.pull(n)).reshape(ny, 1100).copy() for n in ("nx", "nxx")])
    for few, many in zip(*out):
        assert np.array_equal(few, many[:64]) and np.array_equal(few, many[12288:12352])
        assert np.array_equal(few[:48], many[12352:])
