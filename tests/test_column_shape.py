"""The launch shape of the FP64 column kernel over every number of cells and bins: no grid takes two
rounds of blocks that one round could hold, and no round leaves blocks out by giving a wavefront
more columns than it has to.  The rule is host arithmetic, compiled here by itself."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lydion_amd", "csrc")
BLOCKS = 512   # two on each of 256 CUs
SHIM = """
#include "m1lya_shape.h"
extern "C" void shape(int nn, size_t cells, int *out)
{
    m1::ColumnShape s = m1::column_shape(nn, cells);
    out[0] = s.w; out[1] = s.nw; out[2] = s.blocks;
}
"""


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    d = tmp_path_factory.mktemp("shape")
    (d / "shape.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "shape.so"),
                    str(d / "shape.cpp")], check=True)
    lib = C.CDLL(str(d / "shape.so"))

    def call(nn, cells):
        out = (C.c_int * 3)()
        lib.shape(C.c_int(nn), C.c_size_t(cells), out)
        return tuple(out)
    return call


@pytest.mark.parametrize("nn", [3, 40, 41, 64, 65, 128, 129, 256, 257, 512, 513, 576])
def test_one_round_where_one_round_holds_the_cells(shape, nn):
    w_max = 4 if nn <= 128 else 2 if nn <= 256 else 1
    for cells in list(range(9, 8400)) + [16384, 65536, 131072]:
        w, nw, blocks = shape(nn, cells)

        def groups(width):
            return -(-cells // (width * nw))
        assert w in (1, 2, 4) and w <= w_max
        assert blocks == min(groups(w), BLOCKS)
        # single columns from 41 bins on: one block per CU
        fits = [v for v in (1, 2, 4) if v <= w_max and groups(v) <= (BLOCKS // 2 if v == 1 and nn > 40 else BLOCKS)]
        assert w == (fits[0] if fits else w_max), cells


@pytest.mark.parametrize("nn", [3, 64, 128, 129, 256, 257, 512, 513, 576])
def test_two_blocks_fit_in_a_cus_lds(shape, nn):
    w, nw, _ = shape(nn, 10 ** 6)
    rows = max(nn - 2, 1) | 1
    # five arrays of rows, the read-ahead pads, a flag per column and the wavefront's slot, in
    # allocation units of 1280 bytes
    lds = 8 * (5 * rows * w * nw + 16) + 4 * (w * nw + 1)
    assert 2 * (-(-lds // 1280) * 1280) <= 160 * 1024
