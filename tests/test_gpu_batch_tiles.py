"""The tile length that the batched step takes from its clouds' sizes, against the tiles of sixteen
cells by eight rows: the state, the step scalars and the active bins are the same bits, since the
partial sums of short tiles are formed in the order of the long ones."""
import numpy as np
import pytest

import lydion_amd as L
from lydion_amd.batch import M1LyaBatch
from lydion_amd.static_cloud import developed_state
from tests.helpers import small_cloud

pytestmark = pytest.mark.gpu

STATE = ("J", "H_r", "H_z", "f_r", "f_z")


@pytest.fixture(scope="module")
def lut():
    return L.VoigtLUT()


# one, two and four bins per lane, two cells per wavefront, odd sides, and batches that mix them
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("sizes", [[(3, 3, 4)], [(17, 9, 32)], [(70, 33, 18)], [(33, 32, 64)], [(45, 70, 128)],
                                   [(31, 47, 194)], [(65, 100, 66), (20, 30, 24)], [(130, 128, 34)]])
def test_sized_tiles_keep_the_bits(lut, sizes, graph):
    clouds = [developed_state(small_cloud(n_r=r, n_z=z, n_nu=n, tau0=1e7, umax=100.0, lut=lut,
                                          bc_z_bot=L.OUTFLOW if r % 2 else L.REFLECT)) for r, z, n in sizes]
    out = []
    for tiles in (None, (16, 8)):
        b = M1LyaBatch(clouds)
        if tiles:
            b.set_tiles(*tiles)
        b.set_graph(graph)
        active = [b.active_bins()]
        hist = [b.run_steps(7), b.run_steps(6)]
        active.append(b.active_bins())
        state = [b.download(c, k) for c in range(len(clouds)) for k in STATE]
        out.append((active, hist, b.scalars(), state))
        short = b.tiles()[0] < 16
        assert short or tiles
        b.close()
    (a0, h0, s0, f0), (a1, h1, s1, f1) = out
    assert np.array_equal(a0[0], a1[0]) and np.array_equal(a0[1], a1[1])
    assert all(np.array_equal(x, y) for x, y in zip(h0, h1)) and np.array_equal(s0, s1)
    assert all(np.array_equal(x, y) for x, y in zip(f0, f1))


def test_sized_tiles_report_a_non_finite_state(lut):
    cloud = developed_state(small_cloud(n_r=20, n_z=17, n_nu=64, lut=lut))
    errors = []
    for tiles in (None, (16, 8)):
        b = M1LyaBatch([cloud])
        if tiles:
            b.set_tiles(*tiles)
        H = b.download(0, "H_r")
        H[5, 6, 7] = np.nan
        b.upload(0, "H_r", H)
        with pytest.raises(L.M1LyaError) as e:
            b.run_steps(3)
        errors.append(str(e.value))
        b.close()
    assert errors[0] == errors[1]


@pytest.mark.parametrize("shear", [False, True])
@pytest.mark.parametrize("tiles", [None, (16, 8), (5, 3)])
def test_both_kinds_of_blocks_in_one_launch(lut, tiles, shear):
    """Clouds of one and of two cells per wavefront in a batch step in one launch, or in one each when
    launches are timed; either way every cloud has the bits that it has alone."""
    sizes = [(31, 20, 32), (40, 33, 66), (7, 50, 18), (29, 17, 128)]
    clouds = [developed_state(small_cloud(n_r=r, n_z=z, n_nu=n, tau0=1e7, umax=100.0, lut=lut)) for r, z, n in sizes]
    if shear:
        for c in clouds:
            c.lya["duz_dr"] = c.lya["duz_dr"] + 0.3 * c.lya["dur_dr"]

    def run(cs, profiling, graph):
        b = M1LyaBatch(cs)
        if tiles:
            b.set_tiles(*tiles)
        b.set_graph(graph)
        b.set_profiling(profiling)
        h = b.run_steps(5)
        state = [[b.download(i, k) for k in STATE] for i in range(len(cs))]
        names = set(b.kernel_stats())
        b.close()
        return h, state, names

    h0, s0, _ = run(clouds, 0, False)
    for profiling, graph in ((1, False), (0, True)):
        h, s, names = run(clouds, profiling, graph)
        assert not profiling or {"k_step", "k_step_pair"} <= names
        assert np.array_equal(h, h0)
        assert all(np.array_equal(x, y) for a, b in zip(s, s0) for x, y in zip(a, b))
    for i, c in enumerate(clouds):
        # caller-set tiles give the row's sums their own partition; the state is free of it
        h, s, _ = run([c], 0, False)
        assert np.array_equal(h[:, 0], h0[:, i])
        assert all(np.array_equal(x, y) for x, y in zip(s[0], s0[i]))
