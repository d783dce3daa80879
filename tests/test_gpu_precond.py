"""The preconditioned nodal solves at the shapes where the preconditioner's
kernels change: a single level inside one workgroup, tiles with remainders, one
axis coarsened alone, the finest level alone (a diagonally dominant energy
equation).  The solution is compared with the direct solve of the oracle's
system.  Tolerance: the solves stop at a relative residual of 1e-12; the
condition numbers of these systems stay below 1e6 relative to it, and the
solution's largest value is of the order of its norm, so 1e-6 covers the
residual with room and 1e-8, the bar of the other solve tests, is kept.  The bounds on
the iterations are below what Jacobi's, which takes over where a preconditioner fails,
needs on the same system (3 and more), so a broken preconditioner does not pass."""
import numpy as np
import pytest
import scipy.sparse.linalg as sla

from fvmic2d_amd import workloads
from fvmic2d_amd.host import MarkerPath, initial_pressure_guess
from fvmic2d_amd.lib import Context, DeviceArray, DeviceGrid
from oracle import stokes as S
from oracle import thermal as TH

pytestmark = pytest.mark.gpu


class Box:
    def __init__(self, NX, NY, LX, LY, tanh):
        sx = workloads.spacing_tanh_band if tanh else workloads.spacing_uniform
        self.xp, self.xcp = workloads.pad_grid(sx(NX, LX), LX)
        self.yp, self.ycp = workloads.pad_grid(sx(NY, LY), LY)
        self.NX, self.NY, self.LX, self.LY = NX, NY, LX, LY


# smallest grid; one workgroup; its largest and the first beyond it; both axes
# with remainders; y, then x much the stronger axis; a graded grid
@pytest.mark.parametrize("NX,NY,LX,tanh,most", [
    (5, 5, 1.0, False, 7), (33, 33, 1.0, False, 10), (34, 37, 1.0, False, 10), (66, 65, 1.0, False, 10),
    (97, 131, 1.0, True, 16), (40, 150, 1.0, False, 10), (150, 40, 1.0, False, 10), (129, 65, 2.0, True, 16)])
def test_pressure_guess_shapes(NX, NY, LX, tanh, most):
    print("CASE pressure guess", NX, NY, LX, tanh, flush=True)
    ctx = Context()
    w = Box(NX, NY, LX, 1.0, tanh)
    X, Y = np.meshgrid(w.xp[2:NX + 2], w.yp[2:NY + 2])
    rho = 3300.0 + 100.0 * Y - 80.0 * np.exp(-((X - 0.4) ** 2 + (Y - 0.6) ** 2) / 0.02)
    A, b = S.pressure_guess_system(w, rho, 9.81, 0.2)
    ref = sla.spsolve(A.tocsc(), b)
    p = DeviceArray(ctx, np.zeros(NX * NY))
    its, rel = initial_pressure_guess(ctx, DeviceGrid(ctx, w), DeviceArray(ctx, rho), 9.81, gx=0.2, rtol=1e-12, p_out=p)
    assert rel <= 1e-12 and its <= most, (its, rel)
    np.testing.assert_allclose(p.get(), ref, rtol=0, atol=1e-8 * np.abs(ref).max())


# dt scales the diagonal's share: the one-level polynomial, then the V-cycle
@pytest.mark.parametrize("NX,NY,top,dt,most", [(32, 32, 0, 1.0, 2), (33, 65, 1, 1.0, 4), (100, 47, 0, 3.0, 2),
                                               (101, 90, 1, 1e4, 10), (64, 70, 0, 1e4, 10)])
def test_energy_shapes(NX, NY, top, dt, most):
    print("CASE energy", NX, NY, top, dt, flush=True)
    w = workloads.thermal_box(NX, NY, top_type=top)
    mp = MarkerPath(w)
    nn = NX * NY
    coef, rhs = DeviceArray(mp.ctx, np.zeros(5 * nn)), DeviceArray(mp.ctx, w.nodal["heating"])
    T = DeviceArray(mp.ctx, np.zeros(nn))
    mp.form_thermal_system(w.dt * dt, False, coef, rhs)
    its, rel = mp.solve_thermal_system(coef, rhs, T, rtol=1e-12)
    A, b = TH.thermal_system(w.x, w.y, w.nodal, w.materials.materialRho[0], w.options, w.dt * dt, False,
                             w.nodal["heating"])
    ref = sla.spsolve(A.tocsc(), b)
    assert rel <= 1e-12 and its <= most, (its, rel)
    assert np.abs(T.get().ravel() - ref).max() <= 1e-8 * np.abs(ref).max()


def test_rows_the_preconditioner_cannot_bound_still_solve():
    """Couplings twice the diagonal's, of opposite signs: no preconditioner is made for
    them; Jacobi's iterations solve the system."""
    print("CASE energy solve of a system that is not diagonally dominant", flush=True)
    w = workloads.thermal_box(12, 9)
    mp = MarkerPath(w)
    nn = w.NX * w.NY
    c = np.zeros((5, w.NY, w.NX))
    c[0] = 1.0
    c[1, :, :-1], c[2, :, 1:] = 1.5, -1.5
    c[3, :-1], c[4, 1:] = 0.7, -0.7
    x = np.random.default_rng(1).standard_normal((w.NY, w.NX))
    b = x.copy()
    b[:, :-1] += c[1, :, :-1] * x[:, 1:]
    b[:, 1:] += c[2, :, 1:] * x[:, :-1]
    b[:-1] += c[3, :-1] * x[1:]
    b[1:] += c[4, 1:] * x[:-1]
    T = DeviceArray(mp.ctx, np.zeros(nn))
    _, rel = mp.solve_thermal_system(DeviceArray(mp.ctx, c.ravel()), DeviceArray(mp.ctx, b.ravel()), T, rtol=1e-12,
                                     maxit=2000)
    assert rel <= 1e-12
    assert np.abs(T.get().ravel() - x.ravel()).max() <= 1e-8 * np.abs(x).max()
