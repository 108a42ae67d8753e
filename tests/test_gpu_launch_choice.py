"""The launch choices of a mesh (nmx_batch, nmx_inturn) outlive the switch of an
element to FV and back in the middle of a run, which rebuilds the device's tables;
nmx_block, which has no effect, leaves the autotuner on."""
import ctypes as C

import numpy as np
import pytest

import nmesh_amd as nm

pytestmark = pytest.mark.gpu


def _mesh(**extra):
    m = nm.Mesh(dict({"amr_mesh_type": "BoxMesh", "amr_luni": 1, "amr_n0": 4, "amr_n1": 4, "amr_n2": 4,
                      "scalarwave1_k": "0 0 0", "nmx_path": "batched"}, **extra), device=0)
    nm.amr_setup_mesh(m)
    m.upload(1e-3 * np.random.default_rng(1).standard_normal(5 * m.nnodes))
    return m


@pytest.mark.parametrize("batch,turn", [("persistent", "yes"), ("buckets", "yes"), ("buckets", "no"), (None, None)])
def test_launch_choice_survives_a_switch(batch, turn):
    print("launch choice", batch, turn, flush=True)
    extra = {} if batch is None else {"nmx_batch": batch, "nmx_inturn": turn}
    m = _mesh(nmx_trouble="hook", evolve_redo_troubled="step", **extra)
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpyAsync.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]
    hip.hipStreamSynchronize.argtypes = [C.c_void_p]
    calls = [0]

    def hook(u, up, tr, n, stream):
        t = np.zeros(n, np.int32)
        t[2] = calls[0] == 2
        if calls[0] > 4:
            t[:] = np.where(m.fv_flags() != 0, -1, 0)
        calls[0] += 1
        return int(hip.hipMemcpyAsync(tr, t.ctypes.data, 4 * n, 1, stream) != 0 or hip.hipStreamSynchronize(stream) != 0)

    m.set_trouble_hook(hook)
    try:
        nm.evolve_myln(m, 1)
        chosen = m.par("nmx_batch"), m.par("nmx_inturn")
        if batch is not None:
            assert chosen == (batch, turn)
        nm.evolve_myln(m, 12)
    finally:
        m.set_trouble_hook(None)
    assert m.trouble_scores()[2] > 0
    assert (m.par("nmx_batch"), m.par("nmx_inturn")) == chosen


def test_inturn_refuses_other_values():
    with pytest.raises(nm.NmxError, match="nmx_inturn"):
        _mesh().set_par("nmx_inturn", "maybe")


def test_block_parameter_leaves_the_autotuner_on():
    print("nmx_block", flush=True)
    m = _mesh()
    m.set_par("nmx_block", "full")
    assert m.par("nmx_batch") == "legacy"       # no launch shape timed yet
    nm.evolve_myln(m, 1)
    assert m.par("nmx_batch") in ("persistent", "buckets")
