"""Values at and beyond the ends of the range in single cells of the FP64 operators: infinities, NaN,
subnormal numbers, and fluxes so far above J that their square overflows.  They take the general
divisions, and the results are the oracle's, bit for bit (a NaN's sign and payload carry nothing)."""
import numpy as np
import pytest

import lydion_amd as L
from lydion_amd import m1lya as M
from oracle.oracle import OracleState
from tests.helpers import STATE, bitdiff, randomize, small_cloud

pytestmark = pytest.mark.gpu

INF = float("inf")
# (field, value) planted in one bin of one cell each
PLANTS = {
    "infinite J": [("J", INF)],
    "infinite H_r": [("H_r", INF)],
    "infinite H_z": [("H_z", -INF)],
    "NaN J": [("J", float("nan"))],
    "NaN H_z": [("H_z", float("nan"))],
    "subnormal J": [("J", 1e-310)],
    "subnormal H": [("H_r", 1e-310), ("H_z", -1e-310)],
    "tiny H": [("H_r", 1e-280), ("H_z", 1e-275)],
    "vast J": [("J", 1e300)],
    "vast H": [("H_r", 1e300)],
    # H / J from 2^500, where its square is still finite, to beyond the largest number
    "acausal, square finite": [("J", 1e-60), ("H_r", 3e92)],
    "acausal, square overflows": [("J", 1e-60), ("H_z", -1e100)],
    "acausal, ratio overflows": [("J", 1e-60), ("H_r", 1e260)],
}


@pytest.fixture(scope="module")
def lut():
    return L.VoigtLUT()


def _planted(lut, plants, umax, hll, n_nu=66):
    cloud = randomize(small_cloud(n_r=14, n_z=11, n_nu=n_nu, tau0=1e7, umax=umax, lut=lut), seed=31)
    cloud.lya.hll = hll
    for j, i in ((0, 0), (5, 6), (10, 13)):
        for k, v in plants:
            for name in (k, k + "_old"):
                cloud.lya[name][j, i, 20 + i] = v
    return cloud, M.M1LyaContext(cloud.lya, cloud.geometry), OracleState(cloud, hll=hll)


def _same(ctx, o, keys):
    for k in keys:
        g, w = ctx.download(k), o[k]
        nan = np.isnan(w)
        assert np.array_equal(np.isnan(g), nan), (k, int(np.isnan(g).sum()), int(nan.sum()))
        g, w = np.where(nan, 0.0, g), np.where(nan, 0.0, w)
        assert bitdiff(g, w) == 0, (k, bitdiff(g, w), g[g != w][:3], w[g != w][:3])


@pytest.mark.parametrize("hll", [False, True])
@pytest.mark.parametrize("plants", PLANTS.values(), ids=PLANTS.keys())
def test_advection(lut, plants, hll):
    cloud, ctx, o = _planted(lut, plants, 150.0, hll)
    o.advect_lya(cloud.c_tilde * cloud.dt, bc_z_bot=cloud.bc_z_bot)
    M.advect_lya(cloud.c_tilde * cloud.dt, ctx, bc_z_bot=cloud.bc_z_bot)
    _same(ctx, o, STATE)


@pytest.mark.parametrize("plants", PLANTS.values(), ids=PLANTS.keys())
def test_emission_and_absorption(lut, plants):
    cloud, ctx, o = _planted(lut, plants, 0.0, False)
    o.emission_absorption(cloud.c_tilde, cloud.dt)
    M.lya_emission_absorption_update(ctx, cloud.c_tilde, cloud.dt)
    _same(ctx, o, STATE)


@pytest.mark.parametrize("n_nu", [66, 260])
@pytest.mark.parametrize("umax", [0.0, 150.0])
@pytest.mark.parametrize("plants", PLANTS.values(), ids=PLANTS.keys())
def test_frequency_factors_and_update(lut, plants, umax, n_nu):
    cloud, ctx, o = _planted(lut, plants, umax, False, n_nu)
    o.update_freq_factors()
    M.update_freq_factors(ctx)
    _same(ctx, o, ("Fkp", "Fk", "Fkm"))
    o.frequency_update_all_cells(cloud.c_tilde * cloud.dt, update_ff=True)
    M.frequency_update_j_lya_all_cells(cloud.c_tilde * cloud.dt, ctx)
    _same(ctx, o, STATE)
