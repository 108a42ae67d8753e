"""The FV element kernel at the edges of its sizes (3 points: no midpoint
between two end midpoints' neighbours; 4: no WENO5 midpoint; 8 and 10, whose
LDS rows are laid out otherwise) and in each variant: upwind, LLF, and the
s1/s2/opt limits with either flux.  Tolerance as in test_gpu_fvelm.py."""
import numpy as np
import pytest

import nmesh_amd as nm
from oracle import orc
from test_gpu_fvelm import K, TOL, make, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limit", [False, True])
@pytest.mark.parametrize("numflux", ["upwind", "LLF"])
@pytest.mark.parametrize("kind,n,rec", [("box", 3, "WENOm5_2"), ("box", 4, "WENOmT_2"), ("box", 8, "WENOmZ_2"),
                                        ("shell", 3, "WENOmZ_2"), ("shell", 4, "WENOm5_2"),
                                        ("shell", 8, "WENOmT_2"), ("shell", 10, "WENOm5_2")])
def test_fv_kernel_sizes_and_variants(kind, n, rec, numflux, limit):
    print("fvelm sizes", kind, n, rec, numflux, limit, flush=True)
    extra = {"fv_divf_extrap_s1": 0.5, "fv_divf_extrap_s2": 3.0, "fv_divf_extrap_opt": 1} if limit else {}
    m, om = make(1, n, rec, numflux, kind=kind, mid="yes", extra=extra)
    u, _ = om.profile(K, 0.2)
    u = u + 0.1 * np.random.default_rng(n).uniform(-1, 1, u.shape)
    m.upload(u)
    r = nm.evolve_setrhs_mesh(m, t=0.2)
    if limit:
        orc.set_fv_divf_extrap(0.5, 3.0, 1)
    try:
        r_o = om.rhs(u, 0.2, K, numflux)
    finally:
        orc.set_fv_divf_extrap()
        orc.set_fv_midpoint(False)
    assert rel(r, r_o) <= TOL
