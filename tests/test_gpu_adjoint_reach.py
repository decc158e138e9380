"""A NaN or an infinity in a residual reaches what the adjoint's stencils
reach and nothing else: over one reverse step, beside a split plane, exactly
points where a finite residual of the same station leaves a gradient. A tap
of weight zero (the seventh and sixth of a one-sided operator, columns beyond
a stencil, planes above the free surface) passes nothing on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# columns from the plane, planes below the surface
STATIONS = [(2, 14), (-1, 14), (3, 0), (-2, 2), (1, 3)]


@pytest.mark.parametrize("bad", [np.nan, np.inf], ids=["nan", "inf"])
@pytest.mark.parametrize("station", STATIONS, ids=lambda s: f"col{s[0]}_down{s[1]}")
@pytest.mark.parametrize("step", [0, 1])
def test_nonfinite_residual_reaches_its_stencils(built_libs, station, bad, step):
    from cgfd import configs, model
    sc = configs.small(ni=42, nj=70, nk=46, imethod=2, curvilinear=True)
    # no metric term vanishes
    k, j = np.arange(sc.nk)[:, None, None], np.arange(sc.nj)[None, :, None]
    sc.x = (sc.x + 40.0 * np.sin(k / 9.0 + 0.3) + 30.0 * np.sin(j / 11.0 + 0.2)).astype(np.float32)
    sc.y = (sc.y + 30.0 * np.sin(k / 8.0 + 0.1)).astype(np.float32)
    sc.faults[0].fields["mu_s"][:] = 1000.0
    i0 = sc.faults[0].x_index
    st = model.Setup(sc)
    rng = np.random.default_rng(5)
    w0 = np.zeros((9,) + tuple(sc.shape_ext), np.float32)
    w0[:, 3:-3, 3:-3, 3:-3] = 1e-3 * rng.standard_normal((9, sc.nk, sc.nj, sc.ni)) \
        * np.array([1.0] * 3 + [1e6] * 6)[:, None, None, None]
    core = model.Core(st)
    core.run(step)  # the operator pairs of the reversed step
    core.set_stations(np.array([[i0 + station[0], sc.nj // 2, sc.nk - 1 - station[1]]], np.int32) + 3, 2)
    core.adjoint_forward(2)
    core.write_wavefield(w0)
    core.run(2)
    r = np.zeros((1, 2, 9), np.float32)
    r[0, 1] = 1e6 * rng.uniform(0.5, 1.5, 9)
    r[0, 1, 3:] *= 1e-6
    g, _ = core.adjoint_fault(r)
    assert np.isfinite(g).all()
    r[0, 1] = bad
    h, _ = core.adjoint_fault(r)
    core.close()
    st.close()
    reach = (g != 0).any(0)
    assert not np.isfinite(h[:, reach]).all()
    out = ~np.isfinite(h).all(0) & ~reach
    assert not out.any(), np.argwhere(out)[:10]
