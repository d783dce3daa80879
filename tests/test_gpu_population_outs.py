"""Population control's list of the markers without a cell, whose order decides
which slots new markers take: counted and listed by runs of 2048 markers.  Against
the oracle, every decision bitwise."""
import numpy as np
import pytest

from test_gpu_population import _compare, _pair, _population_workload

pytestmark = pytest.mark.gpu


# none outside, the ends and the edges of the runs, one whole run, every third
@pytest.mark.parametrize("case", ["none", "edges", "run", "third"])
def test_markers_without_a_cell(case):
    print("CASE", case, flush=True)
    w = _population_workload()
    X, n = w.markers["X"], w.n_markers
    X[X > w.LX] = 0.5 * w.LX  # the workload's own outside markers come back in
    idx = np.arange(n)
    sel = {"none": idx[:0], "edges": idx[(idx % 2048 < 2) | (idx % 2048 > 2045) | (idx == n - 1)],
           "run": idx[2048:4096], "third": idx[::3]}[case]
    X[sel] = 1.5 * w.LX
    st, mp = _pair(w, n + 40000)
    st.find_marker_cells()
    mp.find_marker_cells()
    assert st.check_marker_density(7) == mp.check_marker_density(7)
    _compare(st, mp, case + " ")
