"""The adjoint on a mesh that was refined and coarsened back to a conforming one
equals that of a mesh that never was: nothing of the refined mesh's tables is
left."""
import numpy as np
import pytest

import nmesh_amd as nm

torch = pytest.importorskip("torch")
from nmesh_amd import adjoint as adj  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["BoxMesh", "Shell"])
@pytest.mark.parametrize("call_refined", [False, True])
def test_adjoint_after_coarsening(kind, call_refined):
    print("coarsened", kind, call_refined, flush=True)

    def mesh():
        m = nm.Mesh({"amr_mesh_type": kind, "amr_luni": 1, "amr_n0": 4, "amr_n1": 4, "amr_n2": 4,
                     "scalarwave1_k": "0 0 0"}, device=0)
        nm.amr_setup_mesh(m)
        return m

    def grad(m):
        w = np.random.default_rng(1).standard_normal(5 * m.nnodes)
        return adj.adjoint_setrhs(m, torch.from_numpy(w).cuda()).cpu().numpy()

    fresh, m = mesh(), mesh()
    ne = m.nelem
    flag = np.zeros(ne, np.int32)
    flag[3] = 1
    m.hadapt(flag)
    assert m.nelem == ne + 7
    if call_refined:
        grad(m)
    back = np.zeros(ne + 7, np.int32)
    back[3:11] = -1
    m.hadapt(back)
    assert m.nelem == ne
    assert np.array_equal(grad(m), grad(fresh))
