// Coefficient images of the one-cluster-per-lane matrix-core kernels
// (kernels_list.hip): blocks of four coefficients, sixteen to an image
// register, 64 floats per register; element i of block b lies at 4 b + i.
#pragma once

namespace chx {

constexpr int CHX_LANE4_MAX_D = 4;  // 4-body dense dimensions the kernel takes

// 3-body: block Q D + k holds C[row][k] of rows 4 Q .. 4 Q + 3, row = a0 D + a1
template <int D>
struct lane3_shape {
    static constexpr int NQ = (D * D + 3) / 4;
    static constexpr int NV = (NQ * D + 15) / 16;
};

// 4-body, two images of D^3 x D^3 in turn (C by rows k = (a, b, c), then its
// transpose): block kk NQ + q holds M[k][4 q .. 4 q + 3], k = D^3 - 1 - kk
template <int D>
struct lane4_shape {
    static constexpr int ROWS = D * D * D;
    static constexpr int NQ = (ROWS + 3) / 4;
    static constexpr int NV = (ROWS * NQ + 15) / 16;
};

}  // namespace chx
