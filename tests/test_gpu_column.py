"""The FP64 column kernel over its launch shapes and both of its tridiagonal solves, bit for bit
against the oracle: the bins of a lane (one to nine) with every remainder at the ends, the
columns of a wavefront (one, two, four by the number of cells), cells at rest and in motion, an
empty initial field (H = 0 takes the general division), and systems outside the range of the
fast solve."""
import numpy as np
import pytest

import lydion_amd as L
from lydion_amd import m1lya as M
from lydion_amd.static_cloud import config_grid, setup_static_cloud
from oracle.oracle import OracleState
from tests.helpers import STATE, bitdiff, randomize, rel, small_cloud

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lut():
    return L.VoigtLUT()


def _assert_state(ctx, o):
    for k in STATE:
        g = ctx.download(k)
        assert bitdiff(g, o[k]) == 0, f"{k}: {bitdiff(g, o[k])} elements differ, max rel {rel(g, o[k]):.3e}"


# n_nu at the edges of 1, 2, 3, 4, 5 and 9 bins per lane; cells below, at and above the counts at
# which a wavefront takes two (4096, and 4096 above 128 bins) and four columns (8192)
@pytest.mark.parametrize("n_nu,n_r,n_z", [(3, 5, 4), (4, 6, 5), (63, 7, 5), (64, 5, 7), (65, 6, 6), (127, 5, 4),
                                          (128, 4, 5), (129, 5, 3), (191, 3, 5), (193, 4, 4), (255, 3, 4), (256, 4, 3),
                                          (257, 3, 3), (575, 3, 3), (5, 64, 64), (5, 65, 63), (4, 91, 90), (5, 128, 64),
                                          (4, 93, 91), (131, 67, 62)])
@pytest.mark.parametrize("umax", [0.0, 300.0])
def test_column_shapes_bit_exact(lut, n_nu, n_r, n_z, umax):
    grid = config_grid(n_nu + n_nu % 2, 1e7)[:n_nu + 1]
    cloud = randomize(setup_static_cloud(1e7, 1e4, tau_abs=0.5, rs=1.0, umax=umax, n_r=n_r, n_z=n_z, nu=grid, lut=lut),
                      seed=n_nu + n_r)
    ctx, o = M.M1LyaContext(cloud.lya, cloud.geometry), OracleState(cloud)
    for _ in range(2):
        so = o.step()
        sg = M.step(ctx, cloud.c_tilde, cloud.dt, cloud.Zc, bc_z_bot=cloud.bc_z_bot)
        assert (sg["kmin"], sg["kmax"]) == (so[5], so[6])
        # sums in another order than the oracle's
        assert abs(sg["M_F"] - so[0]) <= 1e-12 * max(abs(so[0]), 1e-300)
        assert abs(sg["f_esc"] - so[4]) <= 1e-12 * max(abs(so[4]), 1e-300)
    _assert_state(ctx, o)


def test_empty_field_bit_exact(lut):
    cloud = small_cloud(n_r=10, n_z=9, n_nu=66, tau0=1e7, lut=lut)
    ctx, o = M.M1LyaContext(cloud.lya, cloud.geometry), OracleState(cloud)
    for _ in range(4):
        o.step()
        M.step(ctx, cloud.c_tilde, cloud.dt, cloud.Zc, bc_z_bot=cloud.bc_z_bot)
    _assert_state(ctx, o)


@pytest.mark.parametrize("small,large", [(1e-170, 1.0), (1.0, 1e155), (0.0, 1.0)])
def test_solve_outside_the_fast_range_bit_exact(lut, small, large):
    """Stored factors with sub-diagonals below 2^-500 (or zero) and entries above 2^500 in a few
    cells: their wavefront's columns take the general solve, the others the fast one."""
    cloud = randomize(small_cloud(lut=lut, n_r=11, n_z=9, n_nu=64, tau0=1e7), seed=22)
    ctx, o = M.M1LyaContext(cloud.lya, cloud.geometry), OracleState(cloud)
    cdt = cloud.c_tilde * cloud.dt
    dw = 1.0 / cdt
    shape = cloud.lya["J"].shape
    rng = np.random.default_rng(9)
    F = {"Fkp": dw * rng.uniform(0.1, 2.0, shape), "Fk": dw * rng.uniform(0.5, 3.0, shape),
         "Fkm": dw * rng.uniform(0.1, 2.0, shape)}
    F["Fkm"][2, 3, 7:20] *= small
    F["Fkm"][5, 5, 30] *= small
    F["Fk"][7, 1, 11] *= large
    F["Fkp"][2, 8, 40] *= large
    for k, v in F.items():
        ctx.upload(k, v)
        o.set(k, v)
    o.frequency_update_all_cells(cdt, update_ff=False)
    M.frequency_update_j_lya_all_cells(cdt, ctx, update_freq_factors=False)
    _assert_state(ctx, o)
