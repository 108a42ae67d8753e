"""The filter kernel at its smallest and largest orders, all variables and some
of them, each weighting and geometry, against the oracle: the bar is the one of
test_gpu_filter.py."""
import numpy as np
import pytest

import nmesh_amd as nm
from test_gpu_filter import TOL, fpars, make, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("some", [False, True])
@pytest.mark.parametrize("kind,geometry,jpow", [("box", "analytic", 1), ("shell", "analytic", 1),
                                                ("shell", "analytic", -1), ("shell", "stored", -1)])
@pytest.mark.parametrize("n", [2, 9, 10])
def test_filter_sizes(n, kind, geometry, jpow, some):
    print("filter sizes", n, kind, geometry, jpow, some, flush=True)
    par = fpars(3.0, 4.0, 0, jpow, all_="no" if some else "yes", varlist="scalarwave1_cx" if some else "")
    m, om = make(kind, 1, n, dict(par, nmx_geometry=geometry))
    u = np.random.default_rng(n).standard_normal(5 * om.nnodes)
    m.upload(u)
    nm.evolve_filter_evosys_mesh(m)
    assert rel(m.download(), om.filter(u, 0b01110 if some else 31, 3.0, 4.0, 0, jpow)) <= TOL
