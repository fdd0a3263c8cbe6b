// Tile shapes of the fused stage and right-hand-side kernels (stage_kernel.inl)
// and the rule that chooses one from the number of blocks of a launch.
#pragma once

#include "fv_device.h"

namespace alpaca {

// TX x TY x TZ internal cells and NT threads per workgroup.
template <int X, int Y, int Z, int N> struct ShapeTag {
  static constexpr int TX = X, TY = Y, TZ = Z, NT = N;
};

// Calls f with the shape for a launch over n blocks on `cus` compute units.
//
// A wavefront takes about the same time for 64 faces whatever the tile (about
// 7 us for the exact 2D HLLC face alone on its SIMD), so few blocks are a chain
// of faces per wavefront, and the shape is the one with the shortest chain
// whose workgroups are on the chip at once; many blocks are bound by FP64 issue,
// and there the large tile wins, which computes the fewest shared faces twice and
// wastes the fewest lanes of its wavefronts' last faces.  Lines in multiples
// of the compute units, measured with 256 (one stage, exact HLLC, us):
//   2D blocks           6    64   100   150   225   300   529  1035  1521  9025
//     8x8   256 thr   7.9   8.3  11.7  14.7  18.0  21.1  33.5  58.5  83.9   453
//     16x16 640      14.2  14.4  14.7  15.1  15.3  27.1  39.1  65.2  90.6   486
//     16x8  192      11.6  12.0  12.1  18.7  18.7  24.3  30.8  50.0  68.7   358
//     16x16 128      25.5  26.0  26.1  25.9  26.1  40.0  42.2  58.4  59.9   328
//   3D blocks           2     8    12    24    48    64   128   512
//     4x4x4 384      12.8  24.4  35.6  67.0   130   173   344  1437
//     8x4x4 576      18.7  20.6  37.1  54.3   105   138   267  1142
//     8x8x4 512      22.2  23.4  24.7  45.4  66.9  87.8   170   714
//     8x8x8 512      34.9  35.9  37.1  38.8  72.1  75.7   153   571
//     8x8x8 256      43.1  44.3  45.2  46.4  72.1  74.9   140   530
// The Roe, FMA and mixed forms cross at the same places, but the forms whose
// face leaves registers free (wide: HLLC with FMA, HLLC mixed) also gain from
// two wavefronts per SIMD in every larger 3D launch (512 blocks, FMA: 324 us
// with 256 threads, 290 us with 512).
template <int DIM, typename F> void with_shape(long long n, long long cus, bool wide, F f) {
  if constexpr (DIM == 2) {
    (void)wide;
    if (8 * n <= 5 * cus)
      f(ShapeTag<8, 8, 1, 256>{});
    else if (n <= cus)
      f(ShapeTag<16, 16, 1, 640>{});  // one workgroup per CU, one face per thread
    else if (4 * n <= 5 * cus)
      f(ShapeTag<8, 8, 1, 256>{});
    else if (2 * n < 9 * cus)
      f(ShapeTag<16, 8, 1, 192>{});
    else
      f(ShapeTag<16, 16, 1, 128>{});
  } else {
    if (64 * n <= cus)  // one workgroup per CU, one face per thread
      f(ShapeTag<4, 4, 4, 384>{});
    else if (32 * n <= cus)
      f(ShapeTag<8, 4, 4, 576>{});
    else if (16 * n <= cus)  // ... two faces per thread
      f(ShapeTag<8, 8, 4, 512>{});
    else if (8 * n <= cus)  // ... four
      f(ShapeTag<8, 8, 8, 512>{});
    else if (16 * n <= 3 * cus)
      f(ShapeTag<8, 8, 4, 512>{});
    else if (wide && n < (1 << 20))  // a launch counts fewer than 2^32 threads
      f(ShapeTag<8, 8, 8, 512>{});
    else
      f(ShapeTag<8, 8, 8, 256>{});
  }
}

// Right-hand side of n blocks (rhs.hip): those listed of a pool of `capacity`
// blocks, or (list null) the first n; jump may be null.
void launch_rhs(const alpaca_case_desc *d, const double *avg, double *rhs, double *jump,
                const int *list, int n, int capacity, int cus, hipStream_t s);

}  // namespace alpaca
