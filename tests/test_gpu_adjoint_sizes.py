"""Linear identity of the adjoint wave update (<T^T r, w0> = r . T w0) at the
edges of the reverse kernels' tiles: rows of 64 ghost-inclusive columns from
column 0 (the last physical column in the last lane, first lanes of a new
tile), odd and even row and plane counts of the 2 x 2 row blocks, and grids
only a few points wider than their CFS-PML layers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NT = 12
# (ni, nj, nk, curvilinear): last column 63, 64, 66 and 127
SHAPES = [(61, 22, 17, True), (62, 21, 18, False), (64, 23, 20, True), (125, 21, 21, False), (17, 19, 23, True)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s[:3])))
@pytest.mark.parametrize("free", [False, True], ids=["buried", "free"])
def test_adjoint_identity_at_tile_edges(built_libs, shape, free):
    from cgfd import configs, model
    ni, nj, nk, curvilinear = shape
    sc = configs.small(ni=ni, nj=nj, nk=nk, imethod=2, curvilinear=curvilinear)
    sc.faults = []
    sc.pml_layers = [[4, 4], [4, 4], [4, 0 if free else 4]]
    sc.free_top = free
    sc.stations = np.array([[0, 0, nk - 1], [ni - 1, nj - 1, nk - 1], [ni // 2, nj // 2, nk - 2], [ni - 3, 2, 3],
                            [3, nj - 4, nk - 4], [ni // 2, 5, nk // 2]], np.int32)
    st = model.Setup(sc)
    rng = np.random.default_rng(ni + nj + nk)
    w0 = np.zeros((9,) + tuple(sc.shape_ext), np.float32)
    body = rng.standard_normal((9, nk, nj, ni))
    for ax in (1, 2, 3):
        body = (np.roll(body, 1, ax) + 2 * body + np.roll(body, -1, ax)) / 4
    w0[:, 3:-3, 3:-3, 3:-3] = body * np.array([1.0] * 3 + [1e6] * 6)[:, None, None, None]
    core = model.Core(st)
    core.set_stations(sc.stations + 3, NT)
    core.write_wavefield(w0)
    core.run(NT)
    tr = core.read_stations()
    r = rng.standard_normal(tr.shape).astype(np.float32)
    r[:, :, 3:] *= 1e-6
    g = core.adjoint_initial(r)
    core.close()
    st.close()
    # both sums in FP64 of FP32 data, each entry off by about 4 NT roundings of
    # the largest terms it sums: 48 x 6e-8 x the terms' absolute sum
    lhs = float(np.sum(g.astype(np.float64) * w0))
    rhs = float(np.sum(r.astype(np.float64) * tr))
    size = float(np.sum(np.abs(r.astype(np.float64) * tr))) + float(np.sum(np.abs(g.astype(np.float64) * w0)))
    assert np.isfinite(g).all()
    assert abs(lhs - rhs) <= 4 * NT * 6e-8 * size
    assert not g[:, :, :3].any() and not g[..., :3].any() and not g[..., -3:].any()


# (nj, nk, imethod, nfault): rows and planes off the fault kernels' tiles of
# 10 x 4 nodes and 64 lanes, and two faults (whose columns share points)
FAULT_SHAPES = [(31, 25, 1, 1), (40, 26, 2, 1), (70, 27, 1, 1), (47, 31, 2, 2)]


@pytest.mark.parametrize("shape", FAULT_SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_locked_fault_identity_at_tile_edges(built_libs, shape):
    from cgfd import configs, model
    nj, nk, imethod, nfault = shape
    nt = 16
    sc = configs.small(ni=38, nj=nj, nk=nk, imethod=imethod, nfault=nfault, curvilinear=True)
    for f in sc.faults:
        f.fields["mu_s"][:] = 1000.0
    i0 = sc.faults[0].x_index
    j1, j2, k1, k2 = sc.faults[0].grid
    sc.stations = np.array([[i0 + d, j, k] for d, j, k in zip(
        (-6, -3, -2, -1, 1, 2, 3, 6), (j1, j2, nj // 2, j1 + 2, j2 - 2, nj // 2, j1, j2),
        (nk - 1, nk - 1, nk - 2, nk - 3, nk - 4, nk - 1, k1, k1 + 1))], np.int32)
    st = model.Setup(sc)
    rng = np.random.default_rng(nj + nk)
    w0 = np.zeros((9,) + tuple(sc.shape_ext), np.float32)
    body = rng.standard_normal((9, nk, nj, sc.ni))
    for ax in (1, 2, 3):
        body = (np.roll(body, 1, ax) + 2 * body + np.roll(body, -1, ax)) / 4
    w0[:, 3:-3, 3:-3, 3:-3] = 1e-3 * body * np.array([1.0] * 3 + [1e6] * 6)[:, None, None, None]
    core = model.Core(st)
    core.set_stations(sc.stations + 3, nt)
    core.adjoint_forward(nt)
    core.write_wavefield(w0)
    core.run(nt)
    tr = core.read_stations()
    r = rng.standard_normal(tr.shape).astype(np.float32)
    r[:, :, 3:] *= 1e-6
    g, _ = core.adjoint_fault(r)
    core.close()
    st.close()
    # as above, with two passes of sums a stage (tractions, then rates)
    lhs = float(np.sum(g.astype(np.float64) * w0))
    rhs = float(np.sum(r.astype(np.float64) * tr))
    size = float(np.sum(np.abs(r.astype(np.float64) * tr))) + float(np.sum(np.abs(g.astype(np.float64) * w0)))
    assert np.isfinite(g).all()
    assert abs(lhs - rhs) <= 8 * nt * 6e-8 * size
