"""RK4 stages that leave the marker's cell by several cells: the walk decides the
first step from the four coordinates around the cell and walks on from there.
Positions, velocities and spins bitwise against the oracle."""
import numpy as np
import pytest

import oracle
from fvmic2d_amd import workloads
from fvmic2d_amd.host import MarkerPath
from helpers import assert_bitwise

pytestmark = pytest.mark.gpu


# largest displacement in (smallest) cells: within one cell, into the second, far;
# a wide grid keeps its coordinates in global memory
@pytest.mark.parametrize("cells", [0.9, 2.5, 30.0])
@pytest.mark.parametrize("kind,shape", [("box", (41, 41)), ("graded", (33, 21)), ("wide", (2100, 7)),
                                        ("periodic", (24, 13)), ("narrow", (3, 3))])
def test_walk(kind, shape, cells):
    print("CASE", kind, shape, cells, flush=True)
    if kind == "box":
        w = workloads.convection_small()
    elif kind == "periodic":
        w = workloads.periodic_box("plain", NX=shape[0], NY=shape[1], NM=3)
    else:
        w = workloads.vep_subduction(NX=shape[0], NY=shape[1], NM=3)
    r = np.random.default_rng(3)
    for n in ("vx", "vy"):  # a rough field: neighbouring markers step to different sides
        w.nodal[n] = r.uniform(-1.0, 1.0, w.nodal[n].shape)
    w.nodal["wxy"] = r.uniform(-1.0, 1.0, w.nodal["wxy"].shape)
    dt = cells * min(w.LX / (w.NX - 1), w.LY / (w.NY - 1))
    st, mp = oracle.State(w), MarkerPath(w)
    for s in (st, mp):
        s.find_marker_cells()
        s.advect(dt, 0)
    g, o = mp.get_markers(), st.markers
    for f in ("X", "Y", "VX", "VY", "wxy"):
        assert_bitwise(g[f], o[f], f)
