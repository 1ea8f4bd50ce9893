"""The reverse interfaces of the advection over their launch shapes (tiles of a line for small
grids, marches over segments for large ones, lines and segments that do not fill them) against the
dual-number passes, which evaluate every interface per cell: the same derivative in two roundings,
so the bound is that of tests/test_gpu_adjoint.py's comparison on its small grids."""
import numpy as np
import pytest

import lydion_amd as L
from lydion_amd import adjoint as A
from lydion_amd import m1lya as M
from lydion_amd.static_cloud import developed_state
from tests.helpers import small_cloud

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lut():
    return L.VoigtLUT()


@pytest.mark.parametrize("walls", ["open", "reflecting"])
@pytest.mark.parametrize("hll", [False, True])
@pytest.mark.parametrize("n_r,n_z,n_nu", [(3, 4, 4), (13, 14, 66), (40, 27, 18), (131, 127, 66), (67, 300, 130)])
def test_reverse_interfaces_over_shapes(lut, n_r, n_z, n_nu, hll, walls):
    cloud = developed_state(small_cloud(n_r=n_r, n_z=n_z, n_nu=n_nu, tau0=1e6, umax=100.0, lut=lut,
                                        bc_z_bot=L.OUTFLOW if walls == "open" else L.REFLECT))
    cloud.lya.hll = hll
    run = {"bc_z_bot": cloud.bc_z_bot}
    if walls == "reflecting":
        run.update(bc_r_right=L.REFLECT, bc_z_top=L.REFLECT)
    rng = np.random.Generator(np.random.PCG64(n_r))
    mf, sp = rng.normal(size=(2, 3)), rng.normal(size=n_nu)
    out = []
    for mode in (0, 1):
        ctx = M.M1LyaContext(cloud.lya, cloud.geometry)
        ctx.set_adjoint_mode(mode)
        out.append(A.adjoint_run(ctx, 2, cloud.c_tilde, cloud.dt, cloud.Zc, mf, sp, **run))
        ctx.close()
    rev, dual = out
    assert rev.objective == dual.objective
    for group in ("grad_state", "grad_bin", "grad_cell"):
        for k, v in getattr(dual, group).items():
            w = getattr(rev, group)[k]
            scale = np.max(np.abs(v))
            err = np.max(np.abs(w - v)) / scale if scale > 0 else np.max(np.abs(w))
            assert err <= 1e-8, (group, k, err)
