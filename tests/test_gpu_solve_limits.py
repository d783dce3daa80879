"""The nodal solves at the limits of what they take: a zero right-hand side behind
another solve, whose leftovers lie in the workspace; grids of a few rows or columns;
few iterations; rows without couplings; rows the preconditioners are not made for."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as sla

from fvmic2d_amd import workloads
from fvmic2d_amd.lib import Context, DeviceArray, DeviceGrid

pytestmark = pytest.mark.gpu


def _dominant(NX, NY):
    """Rows whose diagonal outweighs the couplings (their sum: 0.4)."""
    c = np.zeros((5, NY, NX))
    c[0] = 1.0
    c[1, :, :-1] = c[2, :, 1:] = -0.1
    c[3, :-1] = c[4, 1:] = -0.1
    return c


NOT_CONVERGED = 11


def _solve(ctx, NX, NY, coef, rhs, rtol=1e-12, maxit=2000, code=0):
    """(T, iterations, relative residual) of fvm_solve_thermal_system."""
    grid = DeviceGrid(ctx, workloads.thermal_box(NX, NY))
    d = [DeviceArray(ctx, np.ascontiguousarray(a).ravel()) for a in (coef, rhs, np.full(NX * NY, 7.0))]
    its, rel = C.c_int32(-1), C.c_double(-1.0)
    assert ctx.lib.fvm_solve_thermal_system(ctx.h, grid.ref, *(C.c_void_p(a.ptr) for a in d), C.c_double(rtol),
                                            C.c_int32(maxit), C.byref(its), C.byref(rel)) == code
    return d[2].get().reshape(NY, NX), its.value, rel.value


@pytest.mark.parametrize("NX,NY", [(12, 9), (33, 20), (100, 47)])
def test_zero_right_hand_side(NX, NY):
    """x = 0 without an iteration, whatever the solve before left behind."""
    print("CASE zero right-hand side", NX, NY, flush=True)
    ctx = Context()
    r = np.random.default_rng(2)
    big = 6 * NX, 6 * NY    # its right-hand side lies over the small solve's whole workspace
    _solve(ctx, *big, _dominant(*big), 1.0 + r.random(big[::-1]))
    x, its, rel = _solve(ctx, NX, NY, _dominant(NX, NY), np.zeros((NY, NX)))
    assert not np.any(x) and its == 0 and rel == 0.0


def _matrix(c):
    NY, NX = c.shape[1:]
    c = c.reshape(5, -1)
    return sp.diags([c[0], c[1, :-1], c[2, 1:], c[3, :-NX], c[4, NX:]], [0, 1, -1, NX, -NX]).tocsc()


# more tiles of 32 x 32 than blocks of 256 rows: fewer than 8 rows or columns, and more
# tiles than the 256 there is always room for; the last ones reach past the scalars
@pytest.mark.parametrize("NX,NY", [(9000, 3), (3, 9000), (8300, 7), (2, 40000), (40000, 2)])
def test_thin_grids(NX, NY):
    """Against the direct solve: couplings of 0.2 leave a condition number below 9, so
    a relative residual of 1e-12 bounds the error in the 2-norm by 9e-12."""
    print("CASE thin grid", NX, NY, flush=True)
    c, b = 2.0 * _dominant(NX, NY), np.random.default_rng(4).standard_normal((NY, NX))
    c[0] = 1.0
    x, its, rel = _solve(Context(), NX, NY, c, b)
    ref = sla.spsolve(_matrix(c), b.ravel())
    assert rel <= 1e-12 and its <= 12, (its, rel)
    assert np.linalg.norm(x.ravel() - ref) <= 9e-12 * np.linalg.norm(ref)


def _poisson(NX, NY):
    c = np.zeros((5, NY, NX))
    c[0] = 4.0
    c[1, :, :-1] = c[2, :, 1:] = c[3, :-1] = c[4, 1:] = -1.0
    return c


@pytest.mark.parametrize("maxit", [1, 3, 5])
def test_maxit_bounds_all_iterations(maxit):
    """Where maxit ends the preconditioned iteration no other one follows: x is its x,
    whose residual Jacobi's would be far from (its first iterations hardly lower it on
    a Poisson problem)."""
    print("CASE maxit", maxit, flush=True)
    NX, NY = 60, 40
    c, b = _poisson(NX, NY), np.ones((NY, NX))
    x, its, rel = _solve(Context(), NX, NY, c, b, rtol=1e-15, maxit=maxit, code=NOT_CONVERGED)
    assert its == maxit
    b = b.ravel() / 4.0
    true = np.linalg.norm(b - _matrix(c / 4.0) @ x.ravel()) / np.linalg.norm(b)
    assert rel <= 0.3 ** maxit and abs(true - rel) <= 1e-12


@pytest.mark.parametrize("coupling", [0.0, 1e-30, 1e-17, 1e-9])
def test_rows_with_next_to_no_couplings(coupling):
    """The interval of the polynomial does not close on the spectrum {1}: the first
    iteration solves the rows (an error below the couplings, which rtol exceeds)."""
    print("CASE couplings of", coupling, flush=True)
    NX, NY = 40, 33
    c, b = coupling * 10.0 * _dominant(NX, NY), np.random.default_rng(5).standard_normal((NY, NX))
    c[0] = 2.0
    x, its, rel = _solve(Context(), NX, NY, c, b, rtol=1e-8)
    assert its == 1 and rel <= 1e-8
    assert np.linalg.norm(x - b / 2.0) <= 2e-8 * np.linalg.norm(b / 2.0)


def _edges(c):
    c[1, :, -1] = c[2, :, 0] = 0.0
    c[3, -1] = c[4, 0] = 0.0
    return c


def _skew(NX, NY):
    c = np.ones((5, NY, NX))
    c[1], c[2], c[3], c[4] = 0.3, -0.3, 0.2, -0.2
    return _edges(c)


def _upwind(NX, NY):
    c = np.ones((5, NY, NX))    # cell Peclet number 10
    c[0], c[1], c[2], c[3], c[4] = 18.1, -1.0, -8.6, -1.0, -7.5
    return _edges(c)


def _random(NX, NY):
    c = np.random.default_rng(6).uniform(-0.3, 0.3, (5, NY, NX))
    c[0] = 1.0
    return _edges(c)


def _shifted(NX, NY):
    c = _poisson(NX, NY)        # a Helmholtz shift
    c[0] -= 0.05
    return c


# iterations: Jacobi's on these rows (in NumPy 23, 65, 16) and some of a preconditioned
# run that gave way, not all 60; the last is one that the preconditioner solves (327)
@pytest.mark.parametrize("rows,most", [(_skew, 40), (_upwind, 90), (_random, 30), (_shifted, 60)])
def test_rows_of_other_kinds(rows, most):
    """Against the true residual: the recurrence's may differ from it by rounding of the
    largest residual on the way, below 1e3 of b."""
    print("CASE rows of another kind", rows.__name__, flush=True)
    NX, NY = 40, 33
    c, b = rows(NX, NY), np.random.default_rng(7).standard_normal((NY, NX))
    x, its, rel = _solve(Context(), NX, NY, c, b)
    assert rel <= 1e-12 and its <= most, (its, rel)
    b = (b / c[0]).ravel()
    assert np.linalg.norm(b - _matrix(c / c[0]) @ x.ravel()) <= 1e-10 * np.linalg.norm(b)


def test_more_rows_than_the_levels_have_blocks_for():
    """1048600 rows of tiles of 16: the solve runs without the levels.  Couplings of 0.9
    and 2 x 0.03 leave a condition number of 49, so a relative residual of 1e-12 bounds
    the error in the 2-norm by 5e-11."""
    print("CASE 2 x 1048600", flush=True)
    NX, NY = 2, 1048600
    c = np.zeros((5, NY, NX))
    c[0] = 1.0
    c[1, :, :-1] = c[2, :, 1:] = -0.9
    c[3, :-1] = c[4, 1:] = -0.03
    x = np.random.default_rng(8).standard_normal((NY, NX))
    got, _, rel = _solve(Context(), NX, NY, c, (_matrix(c) @ x.ravel()).reshape(NY, NX))
    assert rel <= 1e-12 and np.linalg.norm(got - x) <= 5e-11 * np.linalg.norm(x)
