"""The box split in one launch (interior box and CFS-PML bands together) is the
two-kernel form in another order: the stage fork runs the two kernels, and the
states must agree bit for bit, on boxes of whole and partial tiles, at the
size where the form changes, and without a box."""
import numpy as np
import pytest

from cgfd import configs, model

pytestmark = pytest.mark.gpu

# (ni, nj, nk, pml): box widths of 32 (one 32-wide tile), 64 and 96 columns,
# ragged rows, no box at all, and a plane just above 48000 points
SHAPES = [(84, 37, 30, 12), (110, 51, 29, 8), (140, 45, 31, 12), (40, 40, 30, 12), (232, 281, 24, 5)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("curvilinear", [False, True], ids=["flat", "topo"])
def test_one_launch_matches_two_kernels(shape, curvilinear):
    ni, nj, nk, pml = shape
    sc = configs.small(ni=ni, nj=nj, nk=nk, pml=pml, curvilinear=curvilinear)
    st = model.Setup(sc)
    rng = np.random.default_rng(11)
    nz, ny, nx = sc.shape_ext
    w0 = np.zeros((9, nz, ny, nx), np.float32)
    w0[:3, 3:-3, 3:-3, 3:-3] = 1e-2 * rng.standard_normal((3, nk, nj, ni)).astype(np.float32)
    out = []
    for fork in (False, True):
        core = model.Core(st, variant=33)
        core.set_overlap(fork)
        core.write_wavefield(w0)
        core.run(9)
        out.append((core.read_wavefield(), core.read_fault(0), core.read_pg()))
        core.close()
    st.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)


@pytest.mark.parametrize("shape", SHAPES[:3], ids=lambda s: "x".join(map(str, s)))
def test_one_launch_batch_matches_plain(shape):
    """Every scenario of a batch on vertical columns against its run alone:
    both take the one-launch form, point for point the same sums."""
    ni, nj, nk, pml = shape
    sc = configs.small(ni=ni, nj=nj, nk=nk, pml=pml, curvilinear=True)
    st = model.Setup(sc)
    f1 = {k: v.copy() for k, v in sc.faults[0].fields.items()}
    f1["Ty"] *= np.float32(0.9)
    bat = model.Batch(st, [(None, 100), ([f1], 100)])
    bat.run(9)
    got = [bat.read_wavefield(s) for s in range(2)]
    bat.close()
    for s, fields in enumerate((None, f1)):
        if fields is not None:
            sc.faults[0].fields = fields
            st.close()
            st = model.Setup(sc)
        core = model.Core(st, variant=33)
        core.run(9)
        assert np.array_equal(core.read_wavefield(), got[s])
        core.close()
    st.close()
