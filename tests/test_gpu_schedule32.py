"""Schedule 32 is a batch's: on one scenario it is schedule 23, bit for bit,
where the box and the bands would be one launch on a batch and above that
size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(110, 51, 29, 8), (140, 45, 31, 12), (232, 281, 24, 5)]


@pytest.mark.parametrize("vertical", [True, False], ids=["five", "nine"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_32_is_23_on_one_scenario(built_libs, shape, vertical):
    from cgfd import configs, model
    ni, nj, nk, pml = shape
    sc = configs.small(ni=ni, nj=nj, nk=nk, pml=pml, curvilinear=True)
    st = model.Setup(sc)
    rng = np.random.default_rng(11)
    nz, ny, nx = sc.shape_ext
    w0 = np.zeros((9, nz, ny, nx), np.float32)
    w0[:3, 3:-3, 3:-3, 3:-3] = 1e-2 * rng.standard_normal((3, nk, nj, ni)).astype(np.float32)
    out = []
    for variant in (23, 32):
        core = model.Core(st, variant=variant)
        core.set_vertical_columns(vertical)
        core.write_wavefield(w0)
        core.run(9)
        out.append((core.read_wavefield(), core.read_fault(0), core.read_pg()))
        core.close()
    st.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
