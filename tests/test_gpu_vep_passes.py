"""The whole visco-elasto-plastic step against its entry points called one by one.

The step shares gathers between the strain and subgrid stress passes, keeps the
subgrid changes apart until the residual is known and updates and rotates the
stresses behind the advection; every value is formed by the same operations in
the same order, so the two ways have to leave the same bits.
"""
import ctypes as C

import numpy as np
import pytest

from fvmic2d_amd import workloads
from fvmic2d_amd.host import MarkerPath
from fvmic2d_amd.lib import FvmError
from helpers import assert_bitwise

pytestmark = pytest.mark.gpu

FIELDS = ["X", "Y", "VX", "VY", "T", "Tdot", "sxx", "syy", "sxy", "eta", "mu", "rho", "rhodot", "p", "exx", "eyy",
          "exy", "Eii", "wxy", "strainRateResidual", "cellX", "cellY"]
NODAL = ["dsxx", "dsyy", "dsxy", "proj_rho", "proj_etaN", "proj_soxy", "proj_rhodot", "proj_muS", "proj_muN"]


def _problem(kind, shape, diffusivity):
    if kind == "periodic":
        w = workloads.periodic_box("vep", NX=shape[0], NY=shape[1], NM=3)
    else:
        w = workloads.vep_subduction(NX=shape[0], NY=shape[1], NM=3)
    w.options.subgridStressDiffusivity = diffusivity
    r = np.random.default_rng(5)
    w.markers["X"][::97] = -1.0  # some markers outside
    for f in ("sxx", "syy", "sxy"):
        w.markers[f] = 1e6 * r.standard_normal(w.n_markers)
    return w


def _one_by_one(mp, w, jaumann):
    proj, _ = mp.vep_views()
    mp.find_marker_cells()
    mp.update_marker_density()
    y = mp.check_plastic_yielding(w.dt)
    mp.limit_viscosity()
    mp.project_markers_nodes_all2(proj)
    mp.update_marker_strain_pressure(w.dt)
    r = mp.strain_rate_residual()
    if w.options.subgridStressDiffusivity > 0.0:
        mp.subgrid_stress(w.dt, w.options.subgridStressDiffusivity)
    mp.update_marker_stress()
    mp.subgrid_temperature(w.dt, w.options.subgridTemperatureDiffusivity, nf=proj)
    mp.advect(w.dt, jaumann)
    return y, r


def _outcome(step, *args):
    """(yielding, residual), or (error code, 0.0): two rows of nodes have no cell
    centre between them, and the residual there is not a number."""
    try:
        return step(*args)
    except FvmError as e:
        return e.code, 0.0


def _same(a, b):
    ma, mb = a.get_markers(), b.get_markers()
    for f in FIELDS:
        assert_bitwise(ma[f], mb[f], f)
    for f in NODAL:
        assert_bitwise(a.get_nodal(f), b.get_nodal(f), f)


# the smallest grid that takes the shared passes, one that does not (two rows),
# sides that divide nothing, coordinates too many for LDS; both rotations
@pytest.mark.parametrize("kind,shape,diffusivity,jaumann", [
    ("plain", (3, 3), 1.0, 0), ("plain", (5, 2), 1.0, 0), ("plain", (61, 31), 1.0, 0), ("plain", (61, 31), 0.0, 1),
    ("plain", (2100, 7), 1.0, 0), ("periodic", (5, 4), 1.0, 0), ("periodic", (67, 33), 1.0, 1),
    ("periodic", (67, 33), 0.0, 0)])
def test_step_is_its_parts(kind, shape, diffusivity, jaumann):
    print("CASE", kind, shape, diffusivity, jaumann, flush=True)
    w = _problem(kind, shape, diffusivity)
    a, b = MarkerPath(w), MarkerPath(w)
    a.ctx.call("fvm_ctx_set_jaumann", C.c_int32(jaumann))
    for _ in range(2):
        ya, ra = _outcome(a.step_vep)
        yb, rb = _outcome(_one_by_one, b, w, jaumann)
        assert ya == yb
        assert_bitwise(np.array([ra]), np.array([rb]), "residual")
        _same(a, b)


def test_nan_residual_leaves_the_stresses():
    """A residual that is not a number ends the step before the subgrid changes,
    the temperature or the positions have been applied."""
    w = _problem("plain", (61, 31), 1.0)
    a, b = MarkerPath(w), MarkerPath(w)
    for mp in (a, b):
        e = mp.get_nodal("edotxx")
        e[7, 9] = np.nan
        mp.set_nodal("edotxx", e)
    with pytest.raises(FvmError):
        a.step_vep()
    with pytest.raises(FvmError):
        _one_by_one(b, w, 0)
    _same(a, b)
