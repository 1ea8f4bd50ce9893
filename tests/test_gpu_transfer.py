"""Downloads of the FP64 state and of the batch's FP32 state, below and above the size from which
several threads share them: every value comes back, also with a last chunk of a few values and from
two threads at a time."""
import threading

import numpy as np
import pytest

import lydion_amd as L
from lydion_amd import m1lya as M
from lydion_amd.batch import M1LyaBatch
from tests.helpers import small_cloud

pytestmark = pytest.mark.gpu

SIZES = [(9, 7, 10), (64, 128, 128), (127, 131, 66), (128, 128, 64), (211, 173, 98)]


@pytest.fixture(scope="module")
def lut():
    return L.VoigtLUT()


def _fields(shape, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    return {k: np.exp(rng.normal(0.0, 3.0, shape)) for k in ("J", "H_r", "H_z")}


@pytest.mark.parametrize("n_r,n_z,n_nu", SIZES)
def test_fp64_download(lut, n_r, n_z, n_nu):
    cloud = small_cloud(n_r=n_r, n_z=n_z, n_nu=n_nu, lut=lut)
    want = _fields((n_z, n_r, n_nu), 1)
    cloud.lya.arrays.update(want)
    ctx = M.M1LyaContext(cloud.lya, cloud.geometry)
    got = {}
    threads = [threading.Thread(target=lambda k=k: got.update({k: ctx.download(k)})) for k in ("J", "H_r")]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    got["H_z"] = ctx.download("H_z")
    for k, w in want.items():
        assert np.array_equal(got[k], w), k


@pytest.mark.parametrize("n_r,n_z,n_nu", SIZES)
def test_batch_download(lut, n_r, n_z, n_nu):
    b = M1LyaBatch([small_cloud(n_r=n_r, n_z=n_z, n_nu=n_nu, lut=lut)])
    J0 = b.scale(0)
    for k, w in _fields((n_z, n_r, n_nu), 2).items():
        b.upload(0, k, w * J0)
        stored = (w * J0 * (1.0 / J0)).astype(np.float32)
        assert np.array_equal(b.download(0, k), stored.astype(np.float64) * J0), k
    b.close()
