// band2_pick.hpp -- the tiles of the two-substep band kernel (k_band2.hip) and where it is
// the faster path.
#pragma once
#include <algorithm>

namespace dnsg {

// rows of a workgroup (ring included) and nodes per lane, hence output columns, for
// elements of `elem` bytes
enum Band2 {
    B2_OFF,    // two launches
    B2_LARGE,  // tiles of 10 rows
    B2_SMALL,  // tiles of 6 rows
    B2_HUGE    // tiles of 10 rows, for layers of 2 GiB and more
};
constexpr int b2_rows(int tile) { return tile == B2_SMALL ? 8 : 12; }
constexpr int b2_npl(int tile, int elem) { return tile == B2_SMALL || elem == 8 ? 1 : 2; }
constexpr int b2_cols(int tile, int elem) { return 62 * b2_npl(tile, elem); }

inline int band2_tiles(int nx, int ny, int elem, int tile) {
    const int ox = b2_cols(tile, elem), ty = b2_rows(tile) - 2;
    return ((nx + ox - 1) / ox) * ((ny + ty - 1) / ty);
}

// Which path a gratio-2 handle takes.  A tile marches nz + 1 layers, each a chain of two
// collisions, two barriers and their memory accesses, and the pass takes whole rounds of
// tiles over the CUs, so the time follows from the number of tiles:
//   large tiles  9.1 us (FP64) or 9.7 us (FP32) a layer and round, one tile to a CU
//   small tiles  5.2 us (FP64, one to a CU); FP32, two to a CU and so many that the rounds
//                run together, 1.5 us and 2.7 us a layer and tile per CU
// and not less than the time of its bytes: 2.24 lattices at 5.3 and 4.3 TB/s with large
// tiles, 2.4 with small ones, whose ring is a larger share (FP64 5.1, FP32 4.5 TB/s).  The
// two launches move 4 lattices at 5.5 TB/s.  Measured, us a step's band pass, two launches /
// large / small tiles: FP64 bands 256 x 128 x 8 73 / 59 / 44, 256 x 256 x 8 (260 large
// tiles, a second round for 4 of them) 130 / 119 / 92, 320 x 192 x 8 106 / 82 / 92, 1024 x
// 512 x 16 1650 / 1079 / 1187; FP32 512 x 128 x 8 73 / 70 / 45, 512 x 256 x 8 (260) 134 / 141
// / 86, 192 x 128 x 8 30 / 67 / 33, 2048 x 1024 x 32 6670 / 4829 / 6370.
inline int band2_pick(int nx, int ny, int nz, int elem, int cus) {
    const double lattice = 2. * nx * (double)ny * nz * 19 * elem;  // bytes of both bands
    const int nl = 2 * band2_tiles(nx, ny, elem, B2_LARGE), ns = 2 * band2_tiles(nx, ny, elem, B2_SMALL);
    auto rounds = [&](int tiles) { return (tiles + cus - 1) / cus; };
    const double two = 4. * lattice / 5.5e12;
    double large, small;
    if (elem == 8) {
        large = std::max(rounds(nl) * (nz + 1) * 9.1e-6, 2.24 * lattice / 5.3e12);
        small = std::max(rounds(ns) * (nz + 1) * 5.2e-6, 2.4 * lattice / 5.1e12);
    } else {
        large = std::max(rounds(nl) * (nz + 1) * 9.7e-6, 2.24 * lattice / 4.3e12);
        small = std::max((nz + 1) * (1.5e-6 + 2.7e-6 * ns / cus), 2.4 * lattice / 4.5e12);
    }
    if (two < std::min(large, small)) return B2_OFF;
    return small < large ? B2_SMALL : B2_LARGE;
}

}  // namespace dnsg
