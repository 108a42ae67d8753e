"""The adjoint of a mixed-order mesh of more than 1024 elements: one launch per
order, forked over the stream lanes and joined, captured and replayed.

Dot-product test <J v, w> = <v, J^T w> against the device's forward RHS, at 1e-12
relative to |J v| |w|; and adjoint steps the same, bit for bit, with the orders
side by side or one after another, launched or from a graph."""
import numpy as np
import pytest

import nmesh_amd as nm

torch = pytest.importorskip("torch")
from nmesh_amd import adjoint as adj  # noqa: E402

pytestmark = pytest.mark.gpu


def _mesh(**extra):
    m = nm.Mesh(dict({"amr_mesh_type": "Shell", "amr_luni": 2, "amr_n0": 4, "amr_n1": 4, "amr_n2": 4,
                      "amr_Shell_rin": 2.0, "amr_Shell_rout": 20.0, "amr_hrefine_sphere_radius": 5,
                      "amr_hrefine_sphere_levels": 1, "scalarwave1_k": "0 0 0", "nmx_path": "batched"}, **extra), device=0)
    nm.amr_setup_mesh(m)
    m.set_elm_n(np.random.default_rng(9).integers(2, 11, m.nelem).astype(np.int32))
    assert m.nelem > 1024
    return m


@pytest.mark.parametrize("numflux", ["upwind", "LLF"])
@pytest.mark.parametrize("geometry", ["analytic", "stored"])
def test_adjoint_rhs_dot_product_many_mixed_elements(numflux, geometry):
    print("lanes rhs", numflux, geometry, flush=True)
    m = _mesh(scalarwave1_numflux=numflux, nmx_geometry=geometry)
    rng = np.random.default_rng(7)
    v, w = rng.standard_normal((2, 5 * m.nnodes))
    m.upload(v)
    Jv = nm.evolve_setrhs_mesh(m, t=0.0).ravel()
    JTw = adj.adjoint_setrhs(m, torch.from_numpy(w).cuda()).cpu().numpy()
    assert abs(float(Jv @ w) - float(v @ JTw)) <= 1e-12 * np.linalg.norm(Jv) * np.linalg.norm(w)


@pytest.mark.parametrize("method", ["RK4", "sspRK3", "Euler"])
def test_adjoint_steps_side_by_side_in_turn_and_from_graphs(method):
    print("lanes steps", method, flush=True)
    m = _mesh(evolve_method=method, nmx_graph_steps=2)
    w = torch.from_numpy(np.random.default_rng(8).standard_normal(5 * m.nnodes)).cuda()
    out = {}
    for lanes in ("yes", "no"):
        for graph in ("yes", "no"):
            m.set_par("nmx_concurrent", lanes)
            m.set_par("nmx_graph", graph)
            for rep in range(2):     # 5 steps: two replays of two steps, one launched
                out[lanes, graph, rep] = adj.adjoint_evolve(m, w, 5).cpu().numpy()
    first = out["no", "no", 0]
    assert np.abs(first).max() > 0
    for key, x in out.items():
        assert np.array_equal(x, first), key
