"""A gradient that runs out of device memory halfway through its buffers
returns an error, and the same call succeeds once memory is free: nothing is
left half allocated."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _hip():
    """The HIP runtime that the library of this process has loaded."""
    with open("/proc/self/maps") as f:
        return C.CDLL(next(ln.split()[-1] for ln in f if "libamdhip64" in ln))


def test_gradient_after_running_out_of_memory(built_libs):
    from cgfd import configs, model
    sc = configs.small(ni=300, nj=300, nk=200, pml=8)
    sc.faults = []
    st = model.Setup(sc)
    core = model.Core(st)
    core.set_stations(np.array([[150, 150, 199], [40, 60, 100]], np.int32) + 3, 3)
    core.run(3)
    core.sync()
    # the four adjoint levels (36 fields) fit, the gradient terms (9 more) do
    # not; the second round takes what the first one's allocation set free
    field = 4 * ((sc.ni + 6 + 31) // 32 * 32) * (sc.nj + 6) * (sc.nk + 6)
    hip, fill, free, total = _hip(), [], C.c_size_t(), C.c_size_t()
    for _ in range(2):
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        more = free.value - 41 * field
        if more > 0:
            fill.append(C.c_void_p())
            assert hip.hipMalloc(C.byref(fill[-1]), C.c_size_t(more)) == 0
    r = np.ones((2, 3, 9), np.float32)
    r[:, :, 3:] = 1e-6
    try:
        with pytest.raises(RuntimeError, match="hipMalloc of") as error:
            core.adjoint_initial(r)
        assert f"hipMalloc of {36 * field} bytes" not in str(error.value)
    finally:
        for p in fill:
            assert hip.hipFree(p) == 0
    g = core.adjoint_initial(r)
    core.close()
    other = model.Core(st)
    other.set_stations(np.array([[150, 150, 199], [40, 60, 100]], np.int32) + 3, 3)
    other.run(3)
    assert np.array_equal(g, other.adjoint_initial(r)) and np.abs(g).max() > 0
    other.close()
    st.close()
