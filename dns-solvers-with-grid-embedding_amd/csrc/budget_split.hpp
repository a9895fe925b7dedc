// budget_split.hpp -- how the budget's passes share the nodes of a layer out over threads.
#pragma once
#include <hip/hip_runtime.h>

namespace dnsg {

constexpr int BT = 256;  // threads per workgroup

// The threads of a layer are the columns x of its groups of `rows` rows, one after the
// other, so a workgroup of BT of them is full whatever the row length; a thread adds up the
// nodes of its column of the group before the workgroup reduction (44 values: reduced at
// every node, it costs more than the terms).
__host__ __device__ inline int bud_chunks(int X, int Y, int rows) { return (X * ((Y + rows - 1) / rows) + BT - 1) / BT; }
// thread t of chunk ch: its column and first row (y0 >= Y: none)
__host__ __device__ inline void bud_column(int X, int rows, int ch, int t, int &x, int &y0) {
    const int n = ch * BT + t;
    x = n % X;
    y0 = n / X * rows;
}

// Rows per thread for `layers` layers: the reduction and the chain of the rows make a
// workgroup's time about 1 + rows (band layers 17, 25, 40, 72 us at 1, 2, 4, 8), and a CU
// holds two of them, so the launch takes about (workgroups / (2 CUs) + 1/2) (1 + rows).
// Measured at 1, 2, 4, 8 rows, us a launch: band 96 x 64 x 9 17 24 40 80; 192 x 128 x 10
// 37 26 39 67; 320 x 160 x 16 95 70 70 88; 1024 x 512 x 17 834 590 464 428; coarse 96 x 64 x
// 36 33 25 26 42, 160 x 80 x 92 126 91 82 95, 512 x 256 x 124 1550 1071 803 716.
inline int bud_rows(int X, int Y, int layers, int cus) {
    int best = 1;
    long least = -1;
    for (int rows = 1; rows <= 8; rows *= 2) {
        const long t = ((long)layers * bud_chunks(X, Y, rows) + cus) * (1 + rows);
        if (least < 0 || t < least) {
            least = t;
            best = rows;
        }
    }
    return best;
}

}  // namespace dnsg
