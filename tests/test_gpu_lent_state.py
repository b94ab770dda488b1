"""A state written through the pointer of dsem_state_pointers: the next step
starts from the face traces of that state, whether the step before it was a
plain or a recorded one, and again after every later write (the pointer stays
with the caller).  Equal bit for bit to the same state given by
dsem_set_state."""
import ctypes as C
import os

import numpy as np
import pytest

from dsem_amd import _lib as L
from dsem_amd import cases
from dsem_amd import mesh as M
from dsem_amd.solver import DSEM

pytestmark = pytest.mark.gpu


def _device_write(s, dst, src):
    """src (a tensor on the GPU) to the device address dst, on the context's stream."""
    import torch
    hip = C.CDLL(os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so"))
    hip.hipMemcpyAsync.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]
    torch.cuda.synchronize()
    device_to_device = 3
    assert hip.hipMemcpyAsync(dst, src.data_ptr(), 8 * src.numel(), device_to_device, s.stream_handle()) == 0


@pytest.mark.parametrize("recorded", [False, True])
@pytest.mark.parametrize("p", [3, 6])
def test_steps_from_a_state_written_through_its_pointer(p, recorded):
    import torch
    print(f"\n[case] lent state p={p} recorded {recorded}", flush=True)
    with DSEM(M.rotated_box(3, p, seed=p), re=400.0) as s:
        xg, jac = s.gauss_points()
        first, second, third = (cases.tgv_state(xg, jac, "isothermal", perturb=1e-2, seed=p + i) for i in range(3))
        s.set_state(first)
        dt = 0.3 * s.dtcalc()
        want = []
        for q in (second, third):
            s.set_state(q)
            s.steps(1, dt)
            want.append(s.get_state())
        s.set_state(first)
        if recorded:
            s.tape_reserve(1)
            s.rk_step_record(dt, 0)
        else:
            s.steps(1, dt)
        ptr = C.c_void_p()
        assert L.load().dsem_state_pointers(s._h, C.byref(ptr), None) == 0
        for q, w in zip((second, third), want):
            _device_write(s, ptr, torch.from_numpy(q).to("cuda"))
            s.steps(1, dt)
            assert np.array_equal(s.get_state(), w)
