// Per-block right-hand side (SpaceSolver::UpdateFluxes, space_solver.cpp:50-182)
// on gfx950: the launches of rhs_tile_kernel, one fused kernel per call.
//
// Bound by FP64 issue of the faces, and for few blocks by the chain of faces a
// wavefront computes one after the other.  The fluxes stay in LDS, and the kernel
// also writes the zeros of the halo cells, so a call reads the blocks once and
// writes the result once.  As separate kernels (zero fill, the faces of each
// direction through HBM, divergence) six 3D blocks, exact HLLC, took 28.9 us.
#include <hip/hip_runtime.h>

#include "fv_device.h"
#include "launch_shapes.h"

namespace alpaca {
namespace {

// Arithmetic modes as in alpaca_kernels.hip.
enum : int { kModeExact = 0, kModeFma = 1, kModeMixed = 2 };

template <int DIM, int FLUX, int MODE>
void launch(const alpaca_case_desc *d, const double *avg, double *rhs, double *jump,
            const int *list, int n, int capacity, int cus, hipStream_t s) {
  double const inv_dx = 1.0 / d->cell_size;
  constexpr bool wide = FLUX == ALPACA_FLUX_HLLC && MODE != kModeExact;
  with_shape<DIM>(n, cus, wide, [&](auto shape) {
    using S = decltype(shape);
    constexpr int tiles = exact::TileShape<DIM, S::TX, S::TY, S::TZ>::TILES;
    dim3 const grid((unsigned)((size_t)n * tiles)), block(S::NT);
    if constexpr (MODE == kModeExact)
      hipLaunchKernelGGL((exact::rhs_tile_kernel<DIM, FLUX, double, S::TX, S::TY, S::TZ, S::NT>),
                         grid, block, 0, s, avg, rhs, jump, list, n, capacity, d->gamma,
                         d->background_pressure, inv_dx);
    else
      hipLaunchKernelGGL((fast::rhs_tile_kernel<DIM, FLUX,
                                                std::conditional_t<MODE == kModeMixed, float, double>,
                                                S::TX, S::TY, S::TZ, S::NT>),
                         grid, block, 0, s, avg, rhs, jump, list, n, capacity, d->gamma,
                         d->background_pressure, inv_dx);
  });
}

template <int DIM, int FLUX>
void launch_mode(const alpaca_case_desc *d, const double *avg, double *rhs, double *jump,
                 const int *list, int n, int capacity, int cus, hipStream_t s) {
  if (d->precision == ALPACA_MIXED)
    launch<DIM, FLUX, kModeMixed>(d, avg, rhs, jump, list, n, capacity, cus, s);
  else if (d->precision == ALPACA_FP64_FMA)
    launch<DIM, FLUX, kModeFma>(d, avg, rhs, jump, list, n, capacity, cus, s);
  else
    launch<DIM, FLUX, kModeExact>(d, avg, rhs, jump, list, n, capacity, cus, s);
}

template <int DIM>
void launch_flux(const alpaca_case_desc *d, const double *avg, double *rhs, double *jump,
                 const int *list, int n, int capacity, int cus, hipStream_t s) {
  if (d->flux == ALPACA_FLUX_HLLC)
    launch_mode<DIM, ALPACA_FLUX_HLLC>(d, avg, rhs, jump, list, n, capacity, cus, s);
  else
    launch_mode<DIM, ALPACA_FLUX_ROE>(d, avg, rhs, jump, list, n, capacity, cus, s);
}

}  // namespace

void launch_rhs(const alpaca_case_desc *d, const double *avg, double *rhs, double *jump,
                const int *list, int n, int capacity, int cus, hipStream_t s) {
  if (d->dim == 2)
    launch_flux<2>(d, avg, rhs, jump, list, n, capacity, cus, s);
  else
    launch_flux<3>(d, avg, rhs, jump, list, n, capacity, cus, s);
}

}  // namespace alpaca
