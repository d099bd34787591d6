// The order in which the tile table walks a system's cells (cells.hip); plain
// C++ as well, so that a host program can run the same arithmetic.
#pragma once

#ifdef __HIPCC__
#define SPH_HOST_DEVICE __host__ __device__
#else
#define SPH_HOST_DEVICE
#endif

namespace sph {

// Local cell at rank lr of a grid of L1 x L2 x L3 cells in brick order: the
// grid is cut into bricks of BX x BY x BZ cells (BZ = 1 in 2D), the bricks are
// numbered x fastest, then y, then z, and the cells of a brick x fastest; the
// bricks on the far faces are cut to the grid, so the ranks are
// 0 .. L1*L2*L3 - 1.
// The tile table follows this order: each XCD walks a contiguous share of
// it, and the tiles it has in flight then cover a compact block of cells
// whose neighbour cells (the candidates) are few enough to stay in its L2,
// where a row-major order spreads them over whole rows of the grid.
constexpr int BRICK_X = 4, BRICK_Y = 4, BRICK_Z = 4, BRICK_2D = 8;

SPH_HOST_DEVICE inline int brick_cell(int L1, int L2, int L3, int lr)
{
    const auto low = [](int a, int b) { return a < b ? a : b; };
    // A brick no larger than the grid: with it every product below is at most
    // L1 * L2 * L3 <= 2^30.  (Uncut, a row of bricks of a grid one cell high
    // had eight times the grid's cells, 2^32 in the largest.)
    const int bx = low(L1, L3 > 1 ? BRICK_X : BRICK_2D);
    const int by = low(L2, L3 > 1 ? BRICK_Y : BRICK_2D);
    const int bz = low(L3, L3 > 1 ? BRICK_Z : 1);
    const int layer = bz * L1 * L2;  // a layer of bricks (the last may be thinner)
    const int kz = lr / layer;
    const int hz = low(bz, L3 - kz * bz);
    int r = lr - kz * layer;
    const int row = by * L1 * hz;    // a row of bricks
    const int ky = r / row;
    const int hy = low(by, L2 - ky * by);
    r -= ky * row;
    const int brick = bx * hy * hz;
    const int kx = r / brick;
    const int wx = low(bx, L1 - kx * bx);
    r -= kx * brick;
    const int iz = r / (wx * hy), q = r - iz * (wx * hy);
    const int iy = q / wx, ix = q - iy * wx;
    return kx * bx + ix + L1 * ((ky * by + iy) + L2 * (kz * bz + iz));
}

}  // namespace sph
