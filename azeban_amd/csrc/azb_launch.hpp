// Launchers of the fused row kernels and the k-space kernel.  They live in their
// own translation unit (azb_fused.hip) so that it can be compiled with the
// instruction scheduler that suits these kernels (azeban_amd/build.py).
#pragma once

#include <hip/hip_runtime.h>

#include "azb_kernels.hpp"
#include "azb_stage.hpp"

namespace azb {

// Fused row kernel (inverse, max|u|, products, forward) over the lines of a:
// tbytes = sizeof(working real), dim 2 or 3, L the padded line length, pdiv the
// line-pair divisor of the 3D kernel.  Returns 0; 1 when no kernel is built for
// (dim, L); 2 when the line count is not a multiple of the kernel's line-pair
// tile (the caller checks the tile that pdiv selects; the FP32 kernel at
// L = 768 always takes two pairs).
int launch_row_fused(int tbytes, int dim, int L, const RowArgs& a, long nsamples, hipStream_t st, int pdiv);

// k-space kernel with the RK stage update over blocks x samples workgroups of 256.
void launch_kspace(int tbytes, int dim, const KArgs& k, unsigned blocks, unsigned samples, hipStream_t st);

// Shape of the 2D column stage (azb_stage.hpp) for nsamples grids of padded length L: the
// column blocks' width, and the threads per thread's worth of both components (F).
// Width 0: the separate passes are faster.
struct StageShape {
  int width, split;
};
StageShape stage_shape(int tbytes, int L, long nsamples);
// Launch over nsamples x ceil(nh / width) workgroups; sets a.ktiles.  Returns 0, or 1 when
// the shape is not built for L.
int launch_stage(int tbytes, int L, const StageArgs& a, long nsamples, StageShape shape, hipStream_t st);
// the stage's mode table: modes[N][nh] <- (1 / |k|^2, nu(|k|))
void launch_stage_modes(double2* modes, int N, double eps, double s2, double k0, hipStream_t st);

}  // namespace azb
