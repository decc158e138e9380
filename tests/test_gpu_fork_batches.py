"""The stage fork only moves kernels to other streams: a batch's states are
bit for bit those of the run without it, on every box-split schedule, in both
metric forms, while scenarios retire and on either side of the plane size up
to which the box and the bands are one launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (ni, nj, nk, pml): a 64-wide box of ragged rows, one of 96 columns, and a
# plane just above 48000 points
SHAPES = [(110, 51, 29, 8), (140, 45, 31, 12), (232, 281, 24, 5)]


@pytest.mark.parametrize("variant", [0, 23, 24, 32, 33])
@pytest.mark.parametrize("vertical", [True, False], ids=["five", "nine"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_batch_fork_matches_serial(built_libs, shape, vertical, variant):
    from cgfd import configs, model
    ni, nj, nk, pml = shape
    sc = configs.small(ni=ni, nj=nj, nk=nk, pml=pml, curvilinear=True)
    st = model.Setup(sc)
    f1 = {k: v.copy() for k, v in sc.faults[0].fields.items()}
    f1["Ty"] *= np.float32(1.2)  # above its strength over the whole fault
    out = []
    for fork in (False, True):
        bat = model.Batch(st, [(None, 24), ([f1], 20)], variant=variant)
        bat.set_overlap(fork)
        bat.set_vertical_columns(vertical)
        bat.run(24)  # one scenario alone for the last four steps
        out.append([bat.read_wavefield(s) for s in range(2)] + [bat.read_fault(s) for s in range(2)])
        bat.close()
    st.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.abs(a).max() > 0
        assert np.array_equal(a, b)
