"""A gradient that runs out of device memory halfway through its buffers
returns an error, and the same call succeeds once memory is free: nothing is
left half allocated."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_gradient_after_running_out_of_memory(built_libs):
    import torch
    from cgfd import configs, model
    sc = configs.small(ni=300, nj=300, nk=200, pml=8)
    sc.faults = []
    st = model.Setup(sc)
    core = model.Core(st)
    core.set_stations(np.array([[150, 150, 199], [40, 60, 100]], np.int32) + 3, 3)
    core.run(3)
    core.sync()
    # the four adjoint levels (36 fields) fit, the adjoint gradient terms
    # (9 more) fit by half
    nz, ny, nx = sc.shape_ext
    plane = 4 * ((nx + 31) // 32 * 32) * ny
    field = plane * nz
    free, _ = torch.cuda.mem_get_info()
    fill = torch.empty(free - int(40.5 * field), dtype=torch.uint8, device="cuda")
    r = np.ones((2, 3, 9), np.float32)
    r[:, :, 3:] = 1e-6
    with pytest.raises(RuntimeError, match=f"hipMalloc of {9 * field + 48 * plane} bytes"):
        core.adjoint_initial(r)
    del fill
    torch.cuda.empty_cache()
    g = core.adjoint_initial(r)
    core.close()
    other = model.Core(st)
    other.set_stations(np.array([[150, 150, 199], [40, 60, 100]], np.int32) + 3, 3)
    other.run(3)
    assert np.array_equal(g, other.adjoint_initial(r)) and np.abs(g).max() > 0
    other.close()
    st.close()
