"""Stages that keep an accumulator (scored steps, which never trouble an element
here, and Euler steps) against steps without one, in the column and the node
kernels and on FV elements.

Both take the same right-hand sides; the ends of the steps are rounded
differently, a few eps of the largest value per step."""
import numpy as np
import pytest

import nmesh_amd as nm

pytestmark = pytest.mark.gpu


def _mesh(luni, n, **extra):
    m = nm.Mesh(dict({"amr_mesh_type": "Shell", "amr_luni": luni, "amr_n0": n, "amr_n1": n, "amr_n2": n,
                      "amr_Shell_rin": 2.0, "amr_Shell_rout": 20.0, "scalarwave1_k": "0.8 -0.5 0.33166247903554"},
                     **extra), device=0)
    nm.amr_setup_mesh(m)
    return m


@pytest.mark.parametrize("method", ["RK4", "sspRK3"])
@pytest.mark.parametrize("luni,n,extra", [(3, 7, {}), (3, 8, {}), (3, 8, {"nmx_geometry": "stored"}), (3, 10, {}),
                                          (1, 3, {}), (1, 7, {"nmx_path": "batched"}),
                                          (1, 6, {"amr_uniform_p": "0 1 2 3 4 5", "amr_fv_p": "0 1 2 3 4 5"})])
def test_scored_steps_equal_plain_steps(luni, n, extra, method):
    print("accumulator", luni, n, extra, method, flush=True)
    scored = {"nmx_trouble": "RDMP", "nmx_trouble_delta0": "1e30"}
    out = []
    for t in ({}, scored):
        m = _mesh(luni, n, evolve_method=method, **extra, **t)
        m.upload(np.random.default_rng(n).standard_normal(5 * m.nnodes))
        nm.evolve_myln(m, 3)
        out.append(m.download())
    assert np.abs(out[0] - out[1]).max() <= 1e-14 * np.abs(out[0]).max()


@pytest.mark.parametrize("luni,n", [(3, 7), (3, 9), (1, 4)])
def test_euler_step_is_u_plus_dt_r(luni, n):
    print("euler", luni, n, flush=True)
    m = _mesh(luni, n, evolve_method="Euler")
    u = np.random.default_rng(n).standard_normal(5 * m.nnodes)
    m.upload(u)
    r = nm.evolve_setrhs_mesh(m, t=0.0)
    nm.evolve_Euler_mesh(m)
    e = u + m.dt * r.ravel()
    assert np.abs(m.download().ravel() - e).max() <= 4 * np.finfo(float).eps * np.abs(e).max()


@pytest.mark.parametrize("hi", [4, 8, 10])
@pytest.mark.parametrize("geometry", ["analytic", "stored"])
def test_rhs_alone_in_one_launch_per_order_and_with_an_accumulator(hi, geometry):
    """the right-hand side alone, in one launch over all orders and per order, bit
    for bit; and the one that an Euler step adds, up to the step's rounding"""
    print("rhs alone", hi, geometry, flush=True)
    out = []
    for batch in ("persistent", "buckets"):
        m = _mesh(1, 4, nmx_path="batched", nmx_batch=batch, nmx_geometry=geometry, evolve_method="Euler",
                  amr_hrefine_sphere_radius=7, amr_hrefine_sphere_levels=1)
        m.set_elm_n(np.random.default_rng(5).integers(2, hi + 1, m.nelem).astype(np.int32))
        u = np.random.default_rng(6).standard_normal(5 * m.nnodes)
        m.upload(u)
        out.append(nm.evolve_setrhs_mesh(m, t=0.0).ravel().copy())
        nm.evolve_Euler_mesh(m)
        e = u + m.dt * out[-1]
        assert np.abs(m.download().ravel() - e).max() <= 4 * np.finfo(float).eps * np.abs(e).max()
    assert np.array_equal(*out)
