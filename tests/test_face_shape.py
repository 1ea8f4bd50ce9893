"""The launch shape of the reverse interfaces: its bounds over all sizes, and on grids where the two
kernels were timed against each other (microseconds of both directions with the cells' own kernel, the
better segment of each) the kernel that was faster by more than a twentieth.  The rule is host
arithmetic, compiled here by itself."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lydion_amd", "csrc")
SHIM = """
#include "m1lya_shape.h"
extern "C" void shape(int nn, int n, int lines, int hll, int *out)
{
    m1::FaceShape s = m1::face_shape(nn, n, lines, hll != 0);
    out[0] = s.tile; out[1] = s.seg; out[2] = m1::kTileFaces;
}
"""


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    d = tmp_path_factory.mktemp("shape")
    (d / "shape.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "shape.so"),
                    str(d / "shape.cpp")], check=True)
    lib = C.CDLL(str(d / "shape.so"))

    def call(nn, n, lines, hll):
        out = (C.c_int * 3)()
        lib.shape(nn, n, lines, int(hll), out)
        return bool(out[0]), out[1], out[2]
    return call


@pytest.mark.parametrize("hll", [False, True])
@pytest.mark.parametrize("nn", [3, 64, 65, 128, 256])
def test_segments_within_the_kernels_bounds(shape, nn, hll):
    for n in [*range(3, 60), 127, 128, 129, 257, 512]:
        for lines in (3, 4, 5, 17, 32, 64, 100, 257, 512):
            tile, seg, faces = shape(nn, n, lines, hll)
            # a tile's interfaces are its cells and three more
            assert 1 <= seg <= (faces - 3 if tile else 32), (n, lines)


@pytest.mark.parametrize("n_r,n_z,nn,hll,tiles,marches", [
    (24, 24, 32, False, 37.0, 55.8), (24, 24, 32, True, 43.0, 71.0), (32, 32, 64, False, 39.0, 57.7),
    (32, 32, 64, True, 45.2, 77.9), (45, 61, 64, False, 64.2, 84.2), (45, 61, 64, True, 75.4, 114.8),
    (56, 56, 64, False, 78.8, 86.5), (56, 56, 64, True, 92.6, 117.4), (63, 64, 128, False, 147.0, 136.2),
    (63, 64, 128, True, 176.7, 189.5), (80, 80, 64, True, 151.6, 182.4), (100, 110, 128, False, 331.3, 283.2),
    (61, 45, 256, False, 189.9, 173.6), (61, 45, 256, True, 221.3, 240.7), (128, 96, 64, False, 202.2, 181.8),
    (128, 128, 128, False, 493.8, 391.3), (128, 128, 128, True, 580.8, 550.4)])
def test_the_faster_kernel_where_both_were_timed(shape, n_r, n_z, nn, hll, tiles, marches):
    assert max(tiles, marches) > 1.05 * min(tiles, marches)
    for n, lines in ((n_r, n_z), (n_z, n_r)):
        assert shape(nn, n, lines, hll)[0] == (tiles < marches), (n, lines)


def test_small_grids_take_one_interface_per_wavefront(shape):
    for hll in (False, True):
        tile, seg, _ = shape(32, 24, 24, hll)
        assert tile and seg <= 5
