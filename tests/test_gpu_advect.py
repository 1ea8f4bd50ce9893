"""The FP64 advection over its launch shapes and both kinds of divisions, bit for bit against the
oracle: segments of one cell to sixteen (chosen from the grid's size), rows and bins that do not
fill a block, and cells whose interfaces take the general divisions (no flux at all, a depth
beyond 2^400, a J near the top of the exponent range)."""
import numpy as np
import pytest

import lydion_amd as L
from lydion_amd import m1lya as M
from oracle.oracle import OracleState
from tests.helpers import STATE, bitdiff, randomize, rel, small_cloud

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lut():
    return L.VoigtLUT()


@pytest.mark.parametrize("hll", [False, True])
@pytest.mark.parametrize("n_r,n_z,n_nu,bc", [(3, 3, 4, L.REFLECT), (17, 9, 66, L.OUTFLOW), (33, 130, 64, L.REFLECT),
                                             (129, 250, 66, L.OUTFLOW), (200, 129, 128, L.REFLECT)])
def test_advection_shapes_bit_exact(lut, n_r, n_z, n_nu, bc, hll):
    cloud = randomize(small_cloud(n_r=n_r, n_z=n_z, n_nu=n_nu, tau0=1e7, umax=150.0, bc_z_bot=bc, lut=lut), seed=n_r)
    lya = cloud.lya
    lya.hll = hll
    j, i = n_z // 2, n_r // 2
    for k in ("H_r", "H_z", "H_r_old", "H_z_old"):
        lya[k][: j // 2 + 1, : i // 2 + 1] = 0.0            # no flux
    lya["alpha_F"] = lya["alpha_F"].copy()
    lya["alpha_F"][j, i, n_nu // 2] = 1e130                  # depth beyond 2^400
    for k in ("J", "J_old"):
        lya[k][n_z - 1, n_r - 1, n_nu // 3] = 1e152          # 1/J outside the short division's range
    ctx, o = M.M1LyaContext(lya, cloud.geometry), OracleState(cloud, hll=hll)
    cdt = cloud.c_tilde * cloud.dt
    for _ in range(2):
        o.advect_lya(cdt, bc_z_bot=bc)
        M.advect_lya(cdt, ctx, bc_z_bot=bc)
    for k in STATE:
        # the extreme cells overflow to NaN in both; a NaN's sign and payload carry nothing
        g, w = ctx.download(k), o[k]
        assert np.array_equal(np.isnan(g), np.isnan(w)), k
        g, w = np.where(np.isnan(g), 0.0, g), np.where(np.isnan(w), 0.0, w)
        assert bitdiff(g, w) == 0, f"{k}: {bitdiff(g, w)} elements differ, max rel {rel(g, w):.3e}"
