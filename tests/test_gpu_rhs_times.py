"""Right-hand sides called one after another, each with its own time of the wave
in the exterior, while the stream is still busy: every call keeps the time it
was given."""
import numpy as np
import pytest

import nmesh_amd as nm
from nmesh_amd._lib import check, lib

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["plain", "batched"])
@pytest.mark.parametrize("fv", ["", "0 1 2 3 4 5"])
def test_queued_rhs_calls_keep_their_times(path, fv):
    print("queued rhs", path, fv, flush=True)
    m = nm.Mesh({"amr_mesh_type": "Shell", "amr_luni": 1, "amr_n0": 5, "amr_n1": 5, "amr_n2": 5,
                 "amr_Shell_rin": 2.0, "amr_Shell_rout": 20.0, "nmx_path": path, "amr_uniform_p": fv, "amr_fv_p": fv,
                 "scalarwave1_k": "0.8 -0.5 0.33166247903554"}, device=0)
    nm.amr_setup_mesh(m)
    m.upload(np.random.default_rng(3).standard_normal(5 * m.nnodes))
    times = {nm.REG_R: 0.3, nm.REG_P: 1.1}
    alone = {r: nm.evolve_setrhs_mesh(m, t=t, reg_out=r).copy() for r, t in times.items()}
    assert not np.array_equal(alone[nm.REG_R], alone[nm.REG_P])
    s = torch.cuda.Stream()
    a = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    m.set_stream(s.cuda_stream)
    try:
        with torch.cuda.stream(s):
            for _ in range(4):       # the calls below are queued behind these
                a = a @ a * 1e-2
        for r, t in times.items():
            check(lib().nmx_setrhs(m.ctx, r, nm.REG_U, t))
        m.synchronize()
    finally:
        m.set_stream(0)
    for r in times:
        assert np.array_equal(m.download(r), alone[r])
