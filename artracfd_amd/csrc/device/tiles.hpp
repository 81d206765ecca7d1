// tiles.hpp - the tiles of the stage-by-stage sweeps: their shape for a grid
// and the place of a thread's first double.  Host and device (the shape is
// chosen on the host, the offsets are formed in the kernel).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace artra {

struct SweepTile {
    int P;                          // lines per tile
    int seg, nseg;                  // nodes per segment, segments per line
    int groups, others;             // tiles across the line axis, extent of the third axis
    int rows;                       // nodes per line in LDS: seg + 2 halo
    int perPass;                    // x: threads per line; y and z: rows of the tile the block copies at a time
    int threads;                    // of a block
    int tiles;
};

constexpr int kTileThreads = 256;
constexpr int kTileIn = 11, kTileOut = 6;            // doubles per thread of a tile's states and of its a-term

// Doubles of LDS: node states, face fluxes, with the viscous flux the
// transverse differences of every node a face touches and then, in their
// place, the viscous fluxes, and the a-term's states.
__host__ __device__ __forceinline__ int TileSpare(int P, int seg, bool visc)
{
    const int faces = P * (seg + 1), differences = (faces + P) * 4;
    return !visc ? 0 : (differences > 5 * faces) ? differences : 5 * faces;
}

__host__ __device__ __forceinline__ size_t TileDoubles(int P, int seg, int rows, bool visc)
{
    return (size_t)5 * P * (rows + (seg + 1) + seg) + TileSpare(P, seg, visc);
}

// Bytes from a tile's first double to double col of row `row`, rows being
// `stride` nodes apart (x: a row is a line).  In 32 bits: the kernel's
// accesses are then a uniform base and one register, where a 64-bit offset
// takes an addition of two words each.  TileOf takes no shape whose last row
// is 4 GiB or more from its first (TileRows).
__host__ __device__ __forceinline__ unsigned TileOffset(int row, int stride, int col)
{
    return ((unsigned)row * (unsigned)stride * 5u + (unsigned)col) * 8u;
}

// Rows of a tile that a block can copy at a time with every offset below
// 2^32: their first doubles are 40 stride bytes apart, the last row's last
// double `width` doubles behind its first.
inline int TileRows(int stride, int width)
{
    const int64_t room = (int64_t)UINT32_MAX - 8 * (int64_t)width;
    return (int)std::min<int64_t>(kTileThreads, 1 + room / (40 * (int64_t)stride));
}

// Tile of a stage sweep along s over a grid of n nodes (of these `interior`
// are swept): of the shapes that fit a block of at most kTileThreads, the
// one whose blocks cost least in all.  A wavefront's faces cost about 650
// issue slots, an element copied in or out 8 or 20 per wavefront
// (instruction counts of the kernel), a cache line moved about 6; idle lanes
// of a partly filled wavefront, the halo of a short segment and the broken
// cache lines of a narrow tile show in these counts.
// In exact arithmetic, with its divisions and roots, the faces cost 2500,
// and only eight wavefronts fit a compute unit: those a block leaves no room
// for (two blocks of three) or holds for copies alone count half.  (A step
// stage by stage on 127^3 nodes 3.10 -> 2.92 ms, on 199^3 11.50 -> 11.17, a
// viscous one on 127 x 127 x 63 2.47 -> 2.19 against 650 alone; 2500 alone
// takes 1.85 where this takes 1.60 on 511 x 511 x 3.)
// One row at a time and a segment of kTileIn - 2 halo nodes or less always
// fits, so there is a shape for every grid.
inline SweepTile TileOf(const int n[3], const int interior[3], int s, int halo, bool visc, bool fast, int longest)
{
    SweepTile best{};
    double bestCost = 0.0;
    const int line = (s == 0) ? 1 : 0, third = (s == 2) ? 1 : 2;
    const int es = interior[s], across = interior[line], others = interior[third];
    const int stride = (s == 2) ? n[0] * n[1] : n[0];                        // between rows (x: lines)
    const int extra = visc ? 2 : 1;                  // threads per line beyond its nodes
    for (int P = 1; P <= across && P <= kTileThreads / 2; ++P) {
        int seg = std::min(es, kTileThreads / P - extra);
        if (seg < 1) break;
        if (s > 0 && longest > 0) seg = std::min(seg, longest);
        const int rowsAtOnce = TileRows(stride, (s == 0) ? kTileThreads : 5 * P);
        if (s == 0 && P > rowsAtOnce) break;
        if (s > 0) seg = std::min(seg, std::min(rowsAtOnce * kTileIn - 2 * halo, rowsAtOnce * kTileOut));
        const int nseg = (es + seg - 1) / seg;
        seg = (es + nseg - 1) / nseg;
        const int rows = seg + 2 * halo;
        // x: enough threads per line for its faces and for kTileIn elements each
        const int perLine = (s == 0) ? std::max(seg + extra, (5 * rows + kTileIn - 1) / kTileIn) : seg + extra;
        const int faceWaves = (P * perLine + 63) / 64;
        if (TileDoubles(P, seg, rows, visc) * sizeof(double) > 48 * 1024) continue;
        for (int waves = faceWaves; 64 * waves <= kTileThreads; ++waves) {
            // y and z: rows of 5 P doubles per pass of the block
            if (s == 0 && waves > faceWaves) break;
            const int perPass = (s == 0) ? perLine : std::min(64 * waves / (5 * P), rowsAtOnce);
            if (perPass < 1) continue;
            const int in = (((s == 0) ? 5 * rows : rows) + perPass - 1) / perPass;
            const int out = (((s == 0) ? 5 * seg : seg) + perPass - 1) / perPass;
            if (in > kTileIn || out > kTileOut) continue;
            const double cacheLines = (s == 0) ? P * ((rows + 2 * seg) * 40.0 / 128.0 + 2.25)
                                               : (rows + 2 * seg) * (P * 40.0 / 128.0 + 0.75);
            const double tiles = (double)((across + P - 1) / P) * others * nseg;
            const double faces = fast ? 650.0 * faceWaves : 1250.0 * (faceWaves + 8.0 / (8 / waves));
            const double cost = tiles * (faces + waves * (8.0 * in + 20.0 * out) + 6.0 * cacheLines);
            if (best.P && cost >= bestCost) continue;
            best.P = P;
            best.seg = seg;
            best.nseg = nseg;
            best.groups = (across + P - 1) / P;
            best.others = others;
            best.rows = rows;
            best.perPass = perPass;
            best.threads = 64 * waves;
            best.tiles = best.groups * others * nseg;
            bestCost = cost;
        }
    }
    return best;
}

}  // namespace artra
