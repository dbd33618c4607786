// Grids of the FAS solver's kernels over one level, and the partials its norm
// kernels write: plain host arithmetic, shared by the launches and by
// pm_fas_create, which sizes the buffer of the partials.
#pragma once

#include <algorithm>

namespace pm {

// Rows per thread of the z-marching operator kernel and rows of its tile.
constexpr int FZ_RY = 2, FZ_TY = 4 * FZ_RY;

// Workgroups per box of the per-cell kernels.
inline unsigned fas_blocks(long cells) { return (unsigned)std::min<long>((cells + 255) / 256, 1024); }

// Boxes the z-marching operator kernel takes: 32..64 cells wide, at least a tile
// tall and deep.
inline bool fz_box(const int bs[3]) { return bs[0] >= 32 && bs[0] <= 64 && bs[1] >= 16 && bs[2] >= 8; }

// Its workgroups per box and planes per workgroup: 8-row tiles (16 rows of 32-wide
// boxes) x z chunks, halved while the level has fewer than 2048 workgroups.
struct FzGrid {
    int zc;
    unsigned blocks;
};
inline FzGrid fz_grid(const int bs[3], long nboxes)
{
    const int ty = bs[0] <= 32 ? 2 * FZ_TY : FZ_TY, nyt = (bs[1] + ty - 1) / ty;
    auto blocks = [&](int z) { return (long)nyt * ((bs[2] + z - 1) / z) * nboxes; };
    int z = bs[2];
    while (z > 8 && blocks(z) < 2048) { z = (z + 1) / 2; }
    // 128^3 cells: 4 planes 9.1 ms a solve, 8 planes 9.8; 192^3: 13.4 against 12.6.
    // Chunks of 3 hold no whole coarse cells, so the coarse force takes its per-cell
    // kernel, and are the faster ones all the same: 96^3 cells in 48^3 boxes 363 us a
    // cycle, 384 with 4 planes, 401 with 6
    if (z > 4 && z <= 8 && blocks(z) < 1024) { z = (z + 1) / 2; }
    return FzGrid{z, (unsigned)(nyt * ((bs[2] + z - 1) / z))};
}

// Workgroups per box of the residual norm: one partial maximum each.
inline unsigned fas_norm_blocks(const int bs[3], long nboxes)
{
    return fz_box(bs) ? fz_grid(bs, nboxes).blocks : fas_blocks((long)bs[0] * bs[1] * bs[2]);
}

}  // namespace pm
