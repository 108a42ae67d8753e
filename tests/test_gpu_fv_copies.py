"""Host copies of the FV grid: below, between and above the sizes from which
downloads (8 MB) and uploads (40 MB) go through pinned slots by threads, with a
last chunk that is not full, from pageable and from pinned memory: the values
that come back are the ones that went in."""
import numpy as np
import pytest
import torch

from nmesh_amd._lib import check, lib
from nmesh_amd.fv import FvGrid, _p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("n", [16, 64, 80, 112])
def test_upload_then_download(n, pinned):
    print("fv copies", n, pinned, flush=True)
    g = FvGrid({"fv_n": n})
    g.setup()
    u = np.random.default_rng(n).standard_normal(5 * n ** 3)
    v = np.zeros_like(u)
    if pinned:
        u, v = torch.from_numpy(u).pin_memory().numpy(), torch.zeros(u.size, dtype=torch.float64).pin_memory().numpy()
    for k in range(2):   # the second time with the slots in place
        g.upload(u)
        v[:] = 0
        check(lib().nmx_fv_download(g._h, 0, _p(v)))
        assert np.array_equal(u, v)
