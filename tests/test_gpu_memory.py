"""Device memory: what a refused allocation leaves behind."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_operators import _Dev

pytestmark = pytest.mark.gpu


def test_refused_allocation_leaves_no_error_behind():
    """An allocation beyond any GPU's memory is refused with UST_ENOMEM; a launch after it is fine and says so (a launch
    check reads the thread's last error, which a later success does not clear)."""
    from earthbyte_underworld_amd import _lib as L
    lib = L.load()
    d, f = _Dev(lib, np.full(1000, 2.0)), _Dev(lib, np.zeros(1000, np.float32))
    p = C.c_void_p()
    assert lib.ust_dev_malloc(C.byref(p), 1 << 52) == -3 and not p.value
    assert lib.ust_k_copy_f64_to_f32(d.p, f.p, 1000, None) == 0
    assert np.all(f.get() == 2.0)
    d.free()
    f.free()
