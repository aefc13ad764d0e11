"""The pressure multigrid on grids with odd axes, whose last aggregates have one
child: the solve must not need more cycles than on the grid with one cell more
per odd axis (up to 3: the systems differ), for both precisions and the sizes
at which the last cells' widths end in the fused, tail and dense levels; and
the residual of the returned pressure, formed here in FP64, must meet the
tolerance it reports.  (With the last cells' equations taken as full cells' the
odd systems took up to twice the cycles, or stagnated.)"""
import numpy as np
import pytest

from fortrancfd_amd.types import Case, bc_copy

pytestmark = pytest.mark.gpu

SIZES = [(37, 64, 1), (65, 33, 1), (5, 7, 1), (131, 67, 1), (9, 11, 13), (35, 35, 70), (17, 24, 31), (33, 65, 40),
         (75, 45, 37)]
TOL = 1e-10


def _solve(size, precision):
    from fortrancfd_amd import Solver
    nx, ny, nz = size
    h = 1.0 / nx
    case = Case(dim=2 if nz == 1 else 3, nx=nx, ny=ny, nz=nz, xend=nx * h, yend=ny * h, zend=nz * h,
                ppe_precision=precision)
    n = (nx, ny) if nz == 1 else (nx, ny, nz)
    r = np.sqrt(sum((x - 0.5 * m * h) ** 2 for x, m in zip(case.coords(), n)))
    rho = np.where(r > 0.3 * min(n) * h, 1.0, 1e-3) * (1.0 + 0.1 * np.sin(7.0 * case.coords()[0]))
    f = np.random.default_rng(3).standard_normal(case.shape)
    case.interior(f)[...] -= case.interior(f).mean()
    s = Solver(case)
    s.push("rho", bc_copy(case, rho))
    s.push("ppe_src", f)
    s.push("p", np.zeros(case.shape))
    s.ppe_sor_init()
    cyc, rel = s.ppe_solve_rhs(TOL, precision)
    p, rho, f = (case.interior(a) for a in (s.pull("p"), rho, f))
    Ap = np.zeros_like(p)
    for d in range(p.ndim):
        lo, hi = ([slice(None)] * p.ndim for _ in range(2))
        lo[d], hi[d] = slice(0, -1), slice(1, None)
        lo, hi = tuple(lo), tuple(hi)
        q = 2.0 / (rho[lo] + rho[hi]) / h ** 2 * (p[hi] - p[lo])
        Ap[lo] += q
        Ap[hi] -= q
    return cyc, rel, float(np.linalg.norm(f - Ap) / np.linalg.norm(f))


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("size", SIZES)
def test_odd_axes_converge_as_even_ones(size, precision):
    even = tuple(n + n % 2 if n > 1 else 1 for n in size)
    cyc, rel, res = _solve(size, precision)
    ref, _, _ = _solve(even, precision)
    print(size, cyc, "even", ref, "rel", rel, "recomputed", res)
    assert rel <= TOL
    # the same sum in another order: each term is a difference of p times
    # 1/(rho h^2), so the two differ by eps times sum|terms| / ||f||, below
    # 1e-12 here, and 2 TOL leaves room for it
    assert res <= 2 * TOL
    assert cyc <= ref + 3, (cyc, ref)
