"""A refused r3d_adj_set_initial between a forward run and its backward.

The call with a field missing is refused and changes nothing: the backward that
follows is that of the forward's own initial state, with one segment (which reads
the initial state itself as its checkpoint) and with three.
"""
import ctypes

import numpy as np
import pytest

from conftest import load_package

pkg = load_package()
pytestmark = pytest.mark.gpu

ARGS = ["--npx", "16", "--npy", "12", "--npz", "24", "--npey", "1", "--npez", "2", "--tp", "0"]


@pytest.mark.parametrize("every", [6, 2], ids=["one_segment", "three_segments"])
@pytest.mark.parametrize("device", [False, True], ids=["host", "device"])
def test_backward_after_a_refused_initial_state(every, device):
    print(f"[gpu] refused set_initial, every={every} device={device}", flush=True)
    run = pkg.Run(ARGS)
    state = run.state()
    adj = pkg.Adjoint(run.cfg(), run.metrics(), every)
    adj.set_initial(state)
    adj.forward(6)
    want, re, th = adj.backward()
    # other values for the first four fields, none for the last
    other = [np.ascontiguousarray(state[n] * 1.01 + 0.01) for n in adj.names[:4]]
    L = pkg.load()
    if device:
        import torch
        other = [torch.from_numpy(a).cuda() for a in other]
        torch.cuda.synchronize()
        ptrs = (ctypes.c_void_p * 5)(*[a.data_ptr() for a in other], None)
        rc = L.r3d_adj_set_initial_device(adj.h, ptrs)
    else:
        dp = ctypes.POINTER(ctypes.c_double)
        ptrs = (dp * 5)(*[a.ctypes.data_as(dp) for a in other], None)
        rc = L.r3d_adj_set_initial(adj.h, ptrs)
    assert rc != 0 and b"field 4 missing" in L.r3d_hip_last_error()
    got, re2, th2 = adj.backward()
    # two backwards of one forward differ by the order of atomic sums alone
    for n in want:
        assert np.abs(got[n] - want[n]).max() <= 1e-12 * np.abs(want[n]).max(), n
    assert abs(re2 - re) <= 1e-12 * abs(re) and abs(th2 - th) <= 1e-12 * abs(th)
    adj.close()
