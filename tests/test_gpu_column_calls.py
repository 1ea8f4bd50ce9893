"""The column kernel's calls one by one (emission alone, the frequency factors alone, the solve with
and without new factors) above 256 bins, where the first two have a kernel of their own, and rows
whose diffusion coefficient vanishes, which are formed again in the general form: bit for bit
against the oracle."""
import numpy as np
import pytest

import lydion_amd as L
from lydion_amd import m1lya as M
from lydion_amd.static_cloud import config_grid, setup_static_cloud
from oracle.oracle import OracleState
from tests.helpers import STATE, bitdiff, randomize

pytestmark = pytest.mark.gpu

ALL = STATE + ("J_old", "H_r_old", "H_z_old")


@pytest.fixture(scope="module")
def lut():
    return L.VoigtLUT()


def _pair(lut, n_nu, n_r, n_z, umax):
    grid = config_grid(n_nu + n_nu % 2, 1e7)[:n_nu + 1]
    cloud = randomize(setup_static_cloud(1e7, 1e4, tau_abs=0.5, rs=1.0, umax=umax, n_r=n_r, n_z=n_z, nu=grid, lut=lut),
                      seed=n_nu)
    return cloud, M.M1LyaContext(cloud.lya, cloud.geometry), OracleState(cloud)


def _same(ctx, o, keys):
    for k in keys:
        g, w = ctx.download(k), o[k]
        nan = np.isnan(w)
        assert np.array_equal(np.isnan(g), nan), k
        assert bitdiff(np.where(nan, 0.0, g), np.where(nan, 0.0, w)) == 0, k


@pytest.mark.parametrize("umax", [0.0, 300.0])
@pytest.mark.parametrize("n_nu,n_r,n_z", [(257, 4, 3), (320, 5, 3), (448, 3, 4), (511, 3, 3), (512, 5, 5), (513, 3, 3),
                                          (576, 4, 5)])
def test_calls_above_256_bins_bit_exact(lut, n_nu, n_r, n_z, umax):
    cloud, ctx, o = _pair(lut, n_nu, n_r, n_z, umax)
    cdt = cloud.c_tilde * cloud.dt
    o.emission_absorption(cloud.c_tilde, cloud.dt)
    M.lya_emission_absorption_update(ctx, cloud.c_tilde, cloud.dt)
    _same(ctx, o, ALL)
    for k in ("drhou_r", "drhou_z"):
        # sums in another order than the oracle's
        assert np.max(np.abs(ctx.download(k) - o[k])) <= 1e-12 * np.max(np.abs(o[k])), k
    o.update_freq_factors()
    M.update_freq_factors(ctx)
    _same(ctx, o, ("Fkp", "Fk", "Fkm"))
    for update_ff in (False, True):
        o.frequency_update_all_cells(cdt, update_ff=update_ff)
        M.frequency_update_j_lya_all_cells(cdt, ctx, update_freq_factors=update_ff)
        _same(ctx, o, ALL + ("Fkp", "Fk", "Fkm"))


@pytest.mark.parametrize("umax", [0.0, 300.0])
@pytest.mark.parametrize("n_nu", [3, 64, 66, 130, 194, 256, 320])
def test_vanishing_diffusion_coefficient_bit_exact(lut, n_nu, umax):
    """Hvoigt = 0 in single bins at the edges of a lane's share, and over a whole cell."""
    cloud, _, _ = _pair(lut, n_nu, 5, 4, umax)
    kpl = (n_nu + 63) // 64
    Hv = cloud.lya["Hvoigt"].copy()
    Hv[0, 0, n_nu // 2] = 0.0
    Hv[1, 1, (n_nu // 2) // kpl * kpl] = 0.0
    Hv[1, 2, min((n_nu // 2) // kpl * kpl + kpl - 1, n_nu - 1)] = 0.0
    Hv[2, 0, 0] = Hv[2, 1, n_nu - 1] = 0.0
    Hv[3, 3] = 0.0
    cloud.lya["Hvoigt"] = Hv
    ctx, o = M.M1LyaContext(cloud.lya, cloud.geometry), OracleState(cloud)
    o.update_freq_factors()
    M.update_freq_factors(ctx)
    _same(ctx, o, ("Fkp", "Fk", "Fkm"))
    o.frequency_update_all_cells(cloud.c_tilde * cloud.dt, update_ff=True)
    M.frequency_update_j_lya_all_cells(cloud.c_tilde * cloud.dt, ctx, update_freq_factors=True)
    _same(ctx, o, ("Fkp", "Fk", "Fkm"))
    # a column with infinite or NaN factors is a NaN column in both; the others are the same
    _same(ctx, o, ("J",))
