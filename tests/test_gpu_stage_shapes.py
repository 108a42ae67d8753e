"""The two shapes of the DG stage kernel against each other: one thread per
column (7 to 10 points per direction, thousands of elements in a launch) and
one per node (per-element launches), and the launch over all orders against
the per-order ones.

The shapes sum the same products in different orders: per right-hand side at
most 8 n + 40 terms per node, so 4 stages stay within 4 (8 n + 40) eps of the
largest value times the RHS's own amplification, bounded here by 1e-13."""
import numpy as np
import pytest

import nmesh_amd as nm

pytestmark = pytest.mark.gpu

K = "0.8 -0.5 0.33166247903554"


def _mesh(kind, luni, n, **extra):
    pars = {"amr_mesh_type": "BoxMesh" if kind == "box" else "Shell", "amr_luni": luni, "amr_n0": n, "amr_n1": n,
            "amr_n2": n, "amr_BoxMesh_dout": 8.0, "amr_Shell_rin": 2.0, "amr_Shell_rout": 20.0,
            "scalarwave1_k": K, "nmx_autotune": "no"}
    pars.update(extra)
    m = nm.Mesh(pars, device=0)
    nm.amr_setup_mesh(m)
    return m


@pytest.mark.parametrize("n", [7, 8, 9, 10])
@pytest.mark.parametrize("kind,luni,geometry", [("box", 4, "analytic"), ("shell", 3, "analytic"), ("shell", 3, "stored")])
def test_column_kernel_against_node_kernel(kind, luni, geometry, n):
    print("column vs node", kind, geometry, n, flush=True)
    a = _mesh(kind, luni, n, nmx_geometry=geometry)
    b = _mesh(kind, luni, n, nmx_geometry=geometry, nmx_path="perelement")
    assert a.nelem > 1024
    u = np.random.default_rng(n).standard_normal(5 * a.nnodes)
    for m in (a, b):
        m.upload(u)
    ra, rb = (nm.evolve_setrhs_mesh(m, t=0.1) for m in (a, b))
    assert np.abs(ra - rb).max() <= 1e-13 * np.abs(rb).max()
    for flux, step in (("upwind", nm.evolve_RK4_mesh), ("LLF", nm.evolve_sspRK3_mesh), ("upwind", nm.evolve_Euler_mesh)):
        for m in (a, b):
            m.set_par("scalarwave1_numflux", flux)
            m.upload(u)
            m.time = 0.0
            step(m)
        va, vb = a.download(), b.download()
        assert np.abs(va - vb).max() <= 1e-13 * np.abs(vb).max(), (flux, step)


@pytest.mark.parametrize("hi", [4, 8, 10])
@pytest.mark.parametrize("geometry", ["analytic", "stored"])
def test_one_launch_for_all_orders(hi, geometry):
    print("all orders in one launch", hi, geometry, flush=True)
    out = []
    for shape in ("persistent", "buckets"):
        m = _mesh("shell", 1, 4, nmx_path="batched", nmx_batch=shape, nmx_geometry=geometry,
                  amr_hrefine_sphere_radius=7, amr_hrefine_sphere_levels=1)
        m.set_elm_n(np.random.default_rng(5).integers(2, hi + 1, m.nelem).astype(np.int32))
        m.upload(np.random.default_rng(6).standard_normal(5 * m.nnodes))
        nm.evolve_RK4_mesh(m, 2)
        nm.evolve_sspRK3_mesh(m, 1)
        out.append(m.download())
    assert np.array_equal(*out)
