"""The first adjoint right-hand side of a conforming mesh allocates and copies
nothing, so a caller's graph can hold it: the replays equal the eager call."""
import numpy as np
import pytest

import nmesh_amd as nm
from nmesh_amd._lib import check, lib
from nmesh_amd.evolve import REG_ADJ

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n", [("BoxMesh", 5), ("Shell", 8)])
def test_first_adjoint_rhs_in_a_graph(kind, n):
    print("adjoint capture", kind, n, flush=True)
    m = nm.Mesh({"amr_mesh_type": kind, "amr_luni": 1, "amr_n0": n, "amr_n1": n, "amr_n2": n,
                 "scalarwave1_k": "0 0 0"}, device=0)
    nm.amr_setup_mesh(m)
    w = np.random.default_rng(2).standard_normal((2, 5 * m.nnodes))
    m.upload(w[0], REG_ADJ)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    m.set_stream(s.cuda_stream)
    try:
        with torch.cuda.graph(g, stream=s):
            check(lib().nmx_adjoint_setrhs(m.ctx, nm.REG_R, REG_ADJ))
    finally:
        m.set_stream(0)
    for x in (w[0], w[1], w[0]):
        m.upload(x, REG_ADJ)
        m.synchronize()
        g.replay()
        torch.cuda.synchronize()
        replayed = m.download(nm.REG_R).copy()
        check(lib().nmx_adjoint_setrhs(m.ctx, nm.REG_R, REG_ADJ))
        assert np.array_equal(replayed, m.download(nm.REG_R))
