"""The tile-edge tests of the one-launch form and of the reverse kernels over
the nine-term metric kernels, which their own grids of vertical columns do not
reach: the same grids with the five-term form switched off, and grids whose
columns and planes are tilted, so that no metric term vanishes."""
import numpy as np
import pytest

import test_gpu_adjoint_sizes as sizes
import test_gpu_one_launch as one

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["off", "tilted"])
def nine(request, monkeypatch):
    """Cores of the nine-term form, or tilted grids."""
    from cgfd import configs, model
    if request.param == "off":
        class NineTermCore(model.Core):
            def __init__(self, *args, **kw):
                super().__init__(*args, **kw)
                self.set_vertical_columns(False)
                assert self.vertical_columns() == (True, False)
        monkeypatch.setattr(model, "Core", NineTermCore)
        return request.param
    small = configs.small

    def tilted(*args, **kw):
        sc = small(*args, **kw)
        k, j = np.arange(sc.nk)[:, None, None], np.arange(sc.nj)[None, :, None]
        sc.x = (sc.x + 40.0 * np.sin(k / 9.0 + 0.3) + 30.0 * np.sin(j / 11.0 + 0.2)).astype(np.float32)
        sc.y = (sc.y + 30.0 * np.sin(k / 8.0 + 0.1)).astype(np.float32)
        return sc
    monkeypatch.setattr(configs, "small", tilted)
    return request.param


@pytest.mark.parametrize("shape", one.SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_one_launch_matches_two_kernels(built_libs, nine, shape):
    one.test_one_launch_matches_two_kernels(shape, True)


@pytest.mark.parametrize("shape", sizes.SHAPES, ids=lambda s: "x".join(map(str, s[:3])))
@pytest.mark.parametrize("free", [False, True], ids=["buried", "free"])
def test_adjoint_identity_at_tile_edges(built_libs, nine, shape, free):
    sizes.test_adjoint_identity_at_tile_edges(built_libs, shape, free)


@pytest.mark.parametrize("shape", sizes.FAULT_SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_locked_fault_identity_at_tile_edges(built_libs, nine, shape):
    sizes.test_locked_fault_identity_at_tile_edges(built_libs, shape)


def test_tilted_grids_have_no_vertical_columns(built_libs, nine):
    from cgfd import configs, model
    st = model.Setup(configs.small(curvilinear=True))
    core = model.Core(st)
    assert core.vertical_columns()[1] is False
    core.close()
    st.close()
