"""The FV stage kernel's two splits (three waves per tile up to 1024 tiles, one
above) at the smallest grid, on both sides of the line and with its periodic
images in the same block, against the FV oracle; and the primitives that steps
leave behind: those of the last stage's input, whether captured or not."""
import numpy as np
import pytest

from nmesh_amd.fv import PRIM, FvGrid, blob_initial_data
from oracle.orc import OFV

pytestmark = pytest.mark.gpu


def _grid(N, P, **pars):
    g = FvGrid(dict({"fv_n": N}, **pars), device=0)
    g.setup()
    g.upload_prim(P)
    return g


@pytest.mark.parametrize("N", [16, 80, 96])
def test_rhs_and_step_against_oracle(N):
    print("FV tiles", N, flush=True)
    P = blob_initial_data(N, seed=N, nblobs=8)
    ofv = OFV(N)
    u0 = ofv.p2c(P)
    g = _grid(N, P)
    r = g.setrhs()
    ro, _, bad = ofv.rhs(u0, P)
    assert bad == 0 and np.abs(r - ro).max() <= 1e-12 * np.abs(ro).max()
    g.upload_prim(P)
    g.evolve(1)
    u, _, bad = ofv.evolve(u0, P, g.dt, 1)
    assert bad == 0 and g.c2p_failures() == 0
    assert np.abs(g.download() - u).max() <= 1e-12 * np.abs(u).max()


@pytest.mark.parametrize("method,steps", [("Euler", 1), ("Euler", 9), ("sspRK3", 8), ("sspRK3", 9), ("RK4", 17)])
def test_primitives_after_steps(method, steps):
    print("FV primitives", method, steps, flush=True)
    P = blob_initial_data(32, seed=3, nblobs=4)
    g = _grid(32, P, evolve_method=method)
    h = _grid(32, P, evolve_method=method, nmx_graph="no")
    g.evolve(steps)
    for _ in range(steps):
        h.evolve(1)
    assert np.abs(g.download() - h.download()).max() <= 1e-12
    if method == "Euler":
        # the last stage's input is the state one step earlier
        k = _grid(32, P, evolve_method=method)
        k.evolve(steps - 1)
        k.setrhs()
        assert np.abs(g.download(PRIM) - k.download(PRIM)).max() <= 1e-12
    assert np.abs(g.download(PRIM) - h.download(PRIM)).max() <= 1e-11
