// m1lya_shape.h -- launch shapes of the FP64 column kernel and of the reverse interfaces, from the
// grid's dimensions and the flux method alone (host arithmetic, no device code).
#pragma once
#include <algorithm>
#include <cstddef>

namespace m1 {

// Most cell columns per wavefront in the column kernel (lane-per-column dgtsv).
constexpr int kColumnW = 4;

// w cell columns per wavefront, nw wavefronts per block (the block shares its dgtsv phase), blocks of
// the grid.  It depends on the grid's dimensions alone, so that the partition of the fused
// reductions, and with it their bits, does not depend on the device.
//
// A column takes five arrays of N_ν-2 rows of LDS, and the w·nw columns of a block as many as leave
// room for two blocks in a CU's 160 KB: 81 KB for 16 columns of 128 bins, 82 KB for 8 of 256 and for
// 4 of 512, 69 KB for 3 of 576.  Blocks of several wavefronts above 256 bins too: a column's solve
// is a chain that takes a wavefront's issue slots however few of its lanes solve, so that eight
// one-wavefront blocks on a CU ran two chains on each SIMD (870 cycles a row, 380 for a chain alone).
// 45x61x320: 158 us, 265 by one-wavefront blocks; 128x128x542: 1.49 ms, 1.90 by one-wavefront
// blocks that spread the bins of a wavefront and shared no term between rows.
//
// The grid is at most one wave of resident blocks (two per CU at 256 VGPRs), which loop over the
// column groups: a larger one left a partial second wave starting late.  Where one round of them
// holds every cell, w is the smallest that still does, so that the columns spread over the blocks: a
// round's solve takes the same time however many columns it has, and a second round costs more than
// a wavefront saves with fewer columns.  From 41 bins on, single columns only while they are one
// block per CU: the two blocks of a CU would solve side by side what one block of two columns per
// wavefront solves at once.  Fused step's column kernel at w = 1, 2, 4, us:
//   cells         1024             1680              2070              4096              4900               8190
//   64 bins   21.0 24.0 29.5   25.6 24.1  -     39.2 27.6 29.8    42.7 29.7 30.5   56.9  46.2 35.1   74.9  49.5 36.5
//   128       33.9 37.4 46.2   42.9 38.1  -     67.7 42.5 47.7    75.9 48.2 49.2  100.1  77.7 57.6  133.4  83.7 60.2
//   194       50.7 61.4        64.2 62.4       105.3 72.2        117.0 78.0        156.8 129.4       213.0 140.7
//   24        14.1 17.4        16.4 17.3
struct ColumnShape {
    int w, nw, blocks;
};
constexpr int kColumnBlocks = 512;

inline ColumnShape column_shape(int nn, size_t ncells)
{
    ColumnShape c;
    c.nw = nn <= 512 ? 4 : 3;
    c.w = nn <= 128 ? kColumnW : (nn <= 256 ? 2 : 1);
    auto groups = [&](int w) { return (ncells + (size_t)w * c.nw - 1) / ((size_t)w * c.nw); };
    auto limit = [&](int w) { return (size_t)(w == 1 && nn > 40 ? kColumnBlocks / 2 : kColumnBlocks); };
    while (c.w > 1 && groups(c.w / 2) <= limit(c.w / 2)) c.w /= 2;
    c.blocks = (int)std::max<size_t>(1, std::min<size_t>(groups(c.w), kColumnBlocks));
    return c;
}

// Shape of the reverse interfaces along one direction (n cells on each of `lines` lines): blocks of
// kTileWaves wavefronts that take the interfaces around seg cells (k_adj_tile), or wavefronts that
// march over seg cells (k_adj_march).  The least estimated time, in units of one interface by a
// wavefront that has its SIMD to itself (4.3 us by GLF).  A march takes its segment's cells, three
// interfaces more and about one to start, on the wavefronts a SIMD gets (256 VGPRs allow two at a
// time, in 1.28 times one's time).  A tile takes 2.2 where each of its wavefronts takes one interface
// and 3.7 where it takes two, one block to a CU; its rounds of blocks count half by their number and
// half by the work in them, and its launch takes one.  HLL makes an interface of a tile 1.2 times as long and one of a march,
// which spills there, 1.47 times.
// Both directions and the cells' own kernel, us, tiles / marches (the better seg of each), GLF and HLL:
// 24x24x32 37 / 56, 43 / 71; 45x61x64 64 / 84, 75 / 115; 56x56x64 79 / 87, 93 / 117; 80x80x64 128 /
// 132, 152 / 182; 63x64x128 147 / 136, 177 / 190; 128x96x64 202 / 182, 242 / 254; 100x110x128 331 /
// 283, 391 / 396; 128x128x128 494 / 391, 581 / 550.
constexpr int kTileFaces = 16, kTileWaves = 8;

struct FaceShape {
    bool tile;
    int seg;
};

inline FaceShape face_shape(int nn, int n, int lines, bool hll)
{
    constexpr int kCUs = 256, kSimds = 4 * kCUs, kSegMax = 32;
    const int chunks = (nn + 63) / 64, groups = (lines + 3) / 4;
    FaceShape s{false, kSegMax};
    double best = 0.0;
    for (int t = kSegMax; t >= 1; --t) {
        const long per_simd = ((long)chunks * groups * 4 * ((n + t - 1) / t) + kSimds - 1) / kSimds;
        const double cost = (hll ? 1.47 : 1.0) * (1.28 * (double)(per_simd / 2) + (double)(per_simd % 2)) * (t + 4);
        if (t == kSegMax || cost < best) { best = cost; s.seg = t; }
    }
    for (int faces = kTileFaces; faces >= kTileWaves; faces -= kTileWaves) {
        const int tiles = (n + faces - 4) / (faces - 3);
        const long blocks = (long)chunks * lines * tiles;
        const double rounds = 0.5 * ((double)blocks / kCUs + (double)((blocks + kCUs - 1) / kCUs));
        const double cost = (hll ? 1.2 : 1.0) * (1.0 + (faces > kTileWaves ? 3.7 : 2.2) * rounds);
        if (cost < best) { best = cost; s = FaceShape{true, (n + tiles - 1) / tiles}; }
    }
    return s;
}

}  // namespace m1
