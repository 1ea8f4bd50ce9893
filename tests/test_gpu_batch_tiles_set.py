"""Tiles set by the caller, kept by the autotuner and sized from the batch: the autotuner's outputs set
its tiles again on another batch, the tiles of sixteen by eight sum as the sized ones do, any tiles
leave the state's bits, and a segment length of zero goes back to the sized tiles."""
import numpy as np
import pytest

import lydion_amd as L
from lydion_amd.batch import M1LyaBatch
from lydion_amd.static_cloud import developed_state
from tests.helpers import small_cloud

pytestmark = pytest.mark.gpu

# one, two and four bins per lane and two cells per wavefront, alone and mixed; the last two leave one
# kind at the default length
SIZES = [[(33, 32, 64)], [(70, 33, 18)], [(31, 47, 194)], [(40, 50, 130), (24, 30, 70), (20, 30, 24)],
         [(64, 64, 32), (64, 64, 64), (40, 90, 128)], [(45, 45, 32)] + [(150, 128, 34)] * 4,
         [(200, 128, 32)] * 4 + [(24, 24, 66)]]


@pytest.fixture(scope="module")
def lut():
    return L.VoigtLUT()


def _clouds(lut, sizes):
    return [developed_state(small_cloud(n_r=r, n_z=z, n_nu=n, tau0=1e7, umax=100.0, lut=lut)) for r, z, n in sizes]


def _run(clouds, *tiles):
    b = M1LyaBatch(clouds)
    for t in tiles:
        b.set_tiles(*t)
    shape = b.tiles()
    h = [b.run_steps(5)]
    b.set_profiling(1)
    h.append(b.run_steps(2))
    names = set(b.kernel_stats())
    state = [b.download(c, k) for c in range(len(clouds)) for k in ("J", "H_r", "H_z", "f_r")]
    b.close()
    return shape, names, h, state


def _equal(x, y):
    return all(np.array_equal(a, b) for a, b in zip(x, y, strict=True))


@pytest.mark.parametrize("sizes", SIZES)
def test_sized_set_and_sized_again(lut, sizes):
    clouds = _clouds(lut, sizes)
    shape, names, h, state = _run(clouds)
    assert "k_rows" in names      # the sizes ask for shorter tiles
    shape2, names2, h2, state2 = _run(clouds, (16, 8))
    assert shape2 == (16, 8) and "k_rows" not in names2
    assert _equal(h, h2) and _equal(state, state2)
    shape3, names3, h3, state3 = _run(clouds, (3, 5))
    assert shape3 == (3, 5) and "k_rows" not in names3
    assert _equal(state, state3)
    # sums of the same compensated terms in another order
    assert all(np.allclose(x[..., :5], y[..., :5], rtol=1e-13, atol=0) for x, y in zip(h, h3))
    for again in ((0, 8), (0, 3)):
        shape4, names4, h4, state4 = _run(clouds, (3, 5), again)
        assert shape4 == shape and names4 == names
        assert _equal(h, h4) and _equal(state, state4)


@pytest.mark.parametrize("sizes", [SIZES[0], SIZES[2], SIZES[4], SIZES[6]])
def test_the_autotuners_outputs_set_its_tiles(lut, sizes):
    clouds = _clouds(lut, sizes)
    b = M1LyaBatch(clouds)
    s, w, _ = b.autotune(trial_steps=2)
    assert (s, w) == b.tiles()
    h = [b.run_steps(5)]
    b.set_profiling(1)
    h.append(b.run_steps(2))
    names = set(b.kernel_stats())
    b.close()
    shape2, names2, h2, _ = _run(clouds, (s, w))
    assert shape2 == (s, w) and names == names2 and _equal(h, h2)


def test_refused_shapes(lut):
    b = M1LyaBatch(_clouds(lut, SIZES[0]))
    for bad in ((-1, 8), (65, 8), (16, 0), (16, 9), (0, 0), (0, 9)):
        with pytest.raises(L.M1LyaError):
            b.set_tiles(*bad)
    b.close()
