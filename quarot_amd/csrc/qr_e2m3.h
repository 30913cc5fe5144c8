// What the GEMM kernels on the FP6 matrix path share: slots as compile-time indexes, the place of a tile in a grid, and the
// constants that spread packed nibbles to E2M3 fields.
#pragma once
#include <type_traits>
#include <utility>
#include "qr_common.h"

namespace {

template <int V>
using IC = std::integral_constant<int, V>;
template <class F, int... I>
__device__ __forceinline__ void static_for_seq(F&& f, std::integer_sequence<int, I...>) {
    (f(IC<I>()), ...);
}
// f(0), f(1) .. f(N - 1), the argument a constant of its type: the slots of these kernels are far beyond what the compiler unrolls
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_seq(f, std::make_integer_sequence<int, N>());
}

// Row and column of tile `unit` of a grid of tiles: columns of eight row tiles in turn, so that tiles in flight together
// share rows of both operands in an XCD's L2.
struct TilePlace {
    int tm, tn;
};
__device__ __forceinline__ TilePlace tile_place(int unit, int tiles_m, int tiles_n) {
    constexpr int GROUP_M = 8;
    const int group_sz = GROUP_M * tiles_n;
    const int g = unit / group_sz;
    const int gm0 = g * GROUP_M;
    const int gh = (tiles_m - gm0) < GROUP_M ? (tiles_m - gm0) : GROUP_M;
    return TilePlace{gm0 + (unit - g * group_sz) % gh, (unit - g * group_sz) / gh};
}

// First row of A and of B of a tile
struct Origin {
    int m0, n0;
};

// Spreading: two words x, y (16 nibbles) -> 96 bits of sixteen 6-bit fields.  Fields start at bits 0, 6, 12 .. of the 96, which are bits
// {0, 12, 24 | 6, 18, 30}, {4, 16, 28 | 10, 22, (30)} and {8, 20 | 2, 14, 26} of the three words: the first of each are where x has its
// nibbles 0, 3, 6 / 1, 4, 7 / 2, 5 (kSpreadX), the others where y rotated left by 2 has its (kSpreadY).  Which k lands where is the same
// for both operands, and no sum depends on it.  kSpreadFlip: the top bits of all eight nibbles' places, where code + 8 differs from the code.
constexpr u32 kSpreadX[3] = {0x0F00F00Fu, 0xF00F00F0u, 0x00F00F00u};
constexpr u32 kSpreadY[3] = {0xC03C03C0u, 0x03C03C03u, 0x3C03C03Cu};
constexpr u32 kSpreadFlip[3] = {0x08208208u, 0x82082082u, 0x20820820u};

}  // namespace
