// Fused row kernels and k-space kernel launches (the kernels are in
// azb_kernels.hpp).  Compiled as a separate translation unit with the
// instruction-level-parallelism scheduler, which measured faster for these
// kernels and slower for the column passes.
#include <hip/hip_runtime.h>

#include "azb_launch.hpp"

namespace azb {
namespace {

template <typename T, int L, int P>
void launch_row4_P(const RowArgs& a, long nsamples, hipStream_t st) {
  const long blocks = a.nlines / (2 * P) * nsamples;
  hipLaunchKernelGGL((euler_row4_kernel<T, L, P>), dim3((unsigned)blocks), dim3(Row4Cfg<T, L, P>::NT), 0, st, a);
}

// pdiv in {1, 2}: where the row-4 kernel runs (3D FP32 at L = 96 and 192) it
// takes P0 = 1536/L line pairs per workgroup or half of that; every other kernel
// has one line-pair tile
template <typename T, int L, int DIM>
void launch_row_L(const RowArgs& a, long nsamples, hipStream_t st, int pdiv) {
  if constexpr (DIM == 3 && sizeof(T) == 4 && L == 768) {
    // FP32 at L = 768: the radix-24 kernel, two line pairs per workgroup, whatever
    // pdiv says (one transform plan per precision and size keeps results
    // independent of the tuning)
    const long blocks = a.nlines / (2 * Row8Cfg<T, L>::P) * nsamples;
    hipLaunchKernelGGL((euler_row8_kernel<T, L>), dim3((unsigned)blocks), dim3(Row8Cfg<T, L>::NT), 0, st, a);
    (void)pdiv;
  } else if constexpr (DIM == 3 && sizeof(T) == 8 && L == 768) {
    // FP64 at L = 768: one line pair per workgroup with a single six-sequence
    // forward round, whatever pdiv says (one plan per precision and size)
    const long blocks = a.nlines / 2 * nsamples;
    hipLaunchKernelGGL((euler_row6_kernel<T>), dim3((unsigned)blocks), dim3(Row6Cfg::NT), 0, st, a);
    (void)pdiv;
  } else if constexpr (DIM == 3 && (L == 96 || L == 192) && sizeof(T) == 4) {
    constexpr int P0 = 1536 / L, P1 = P0 / 2;
    if (pdiv == 2)
      launch_row4_P<T, L, P1>(a, nsamples, st);
    else
      launch_row4_P<T, L, P0>(a, nsamples, st);
  } else if constexpr (DIM == 3) {
    // 3D at L = 384, and FP64 at L = 192 and 96: 768/L line pairs per workgroup with a
    // single forward round, whatever pdiv says (one plan per precision and size)
    const long blocks = a.nlines / (2 * Row6pCfg<L>::P) * nsamples;
    hipLaunchKernelGGL((euler_row6p_kernel<T, L>), dim3((unsigned)blocks), dim3(Row6pCfg<L>::NT), 0, st, a);
    (void)pdiv;
  } else if constexpr (L == 1536) {
    // 2D at L = 1536: one line pair per 192-thread workgroup, 24 values per thread
    const long blocks = a.nlines / 2 * nsamples;
    hipLaunchKernelGGL((euler_row2w_kernel<T>), dim3((unsigned)blocks), dim3(Row2wCfg::NT), 0, st, a);
    (void)pdiv;
  } else if constexpr (L == 768 || L == 384) {
    // 2D at L = 768, 384: 1536/L line pairs per 192-thread workgroup, the 3D forward
    const long blocks = a.nlines / (2 * Row2pCfg<L>::P) * nsamples;
    hipLaunchKernelGGL((euler_row2p_kernel<T, L>), dim3((unsigned)blocks), dim3(Row2pCfg<L>::NT), 0, st, a);
    (void)pdiv;
  } else {
    // one shape: 768/L line pairs, 192 threads
    const long blocks = a.nlines / (2 * Row2Cfg<T, L>::P) * nsamples;
    hipLaunchKernelGGL((euler_row2_kernel<T, L>), dim3((unsigned)blocks), dim3(Row2Cfg<T, L>::NT), 0, st, a);
    (void)pdiv;
  }
}

template <typename T, int DIM>
int launch_row_T(int L, const RowArgs& a, long nsamples, hipStream_t st, int pdiv) {
  switch (L) {
    case 96:
      if (DIM == 3 && sizeof(T) == 8 && a.nlines % 16 != 0) return 2;  // eight line pairs per workgroup
      launch_row_L<T, 96, DIM>(a, nsamples, st, pdiv);
      return 0;
    case 192:
      if (DIM == 3 && sizeof(T) == 8 && a.nlines % 8 != 0) return 2;  // four line pairs per workgroup
      launch_row_L<T, 192, DIM>(a, nsamples, st, pdiv);
      return 0;
    case 384:
      if (a.nlines % (DIM == 3 ? 4 : 8) != 0) return 2;  // two (3D) or four (2D) line pairs per workgroup
      launch_row_L<T, 384, DIM>(a, nsamples, st, pdiv);
      return 0;
    case 768:
      if constexpr ((DIM == 3 && sizeof(T) == 4) || DIM == 2) {
        if (a.nlines % 4 != 0) return 2;  // two line pairs per workgroup
      }
      if (a.nlines % 2 != 0) return 2;
      launch_row_L<T, 768, DIM>(a, nsamples, st, pdiv);
      return 0;
    case 1536:
      if constexpr (DIM == 2) {
        launch_row_L<T, 1536, 2>(a, nsamples, st, pdiv);
        return 0;
      }
      return 1;
    default: return 1;
  }
}

}  // namespace

int launch_row_fused(int tbytes, int dim, int L, const RowArgs& a, long nsamples, hipStream_t st, int pdiv) {
  if (tbytes == 8) return dim == 3 ? launch_row_T<double, 3>(L, a, nsamples, st, pdiv)
                                   : launch_row_T<double, 2>(L, a, nsamples, st, pdiv);
  return dim == 3 ? launch_row_T<float, 3>(L, a, nsamples, st, pdiv)
                  : launch_row_T<float, 2>(L, a, nsamples, st, pdiv);
}

namespace {

template <typename T, int DIM>
void launch_kspace_T(const KArgs& k, dim3 grid, hipStream_t st) {
  const dim3 block(256);
  switch (k.mode) {
    case K_RK1: hipLaunchKernelGGL((kspace_kernel<T, DIM, K_RK1>), grid, block, 0, st, k); break;
    case K_RK2: hipLaunchKernelGGL((kspace_kernel<T, DIM, K_RK2>), grid, block, 0, st, k); break;
    case K_RK3: hipLaunchKernelGGL((kspace_kernel<T, DIM, K_RK3>), grid, block, 0, st, k); break;
    default: hipLaunchKernelGGL((kspace_kernel<T, DIM, K_DUDT>), grid, block, 0, st, k); break;
  }
}

}  // namespace

void launch_kspace(int tbytes, int dim, const KArgs& k, unsigned blocks, unsigned samples, hipStream_t st) {
  const dim3 grid(blocks, samples);
  if (tbytes == 8)
    dim == 3 ? launch_kspace_T<double, 3>(k, grid, st) : launch_kspace_T<double, 2>(k, grid, st);
  else
    dim == 3 ? launch_kspace_T<float, 3>(k, grid, st) : launch_kspace_T<float, 2>(k, grid, st);
}

namespace {

template <typename T, int L, int TS, int F>
int launch_stage_TS(StageArgs a, long nsamples, hipStream_t st) {
  a.ktiles = (a.nh + TS - 1) / TS;
  hipLaunchKernelGGL((col_stage_kernel<T, L, TS, F>), dim3((unsigned)(a.ktiles * nsamples)),
                     dim3(StageCfg<T, L, TS, F>::NT), 0, st, a);
  return 0;
}

// the shapes that stage_shape picks from
template <typename T, int L>
int launch_stage_L(const StageArgs& a, long nsamples, StageShape sh, hipStream_t st) {
  if constexpr (L == 96 || L == 192 || L == 768)
    if (sh.width == 4 && sh.split == 2) return launch_stage_TS<T, L, 4, 2>(a, nsamples, st);
  if constexpr (L == 384 || L == 768)
    if (sh.width == 2 && sh.split == 2) return launch_stage_TS<T, L, 2, 2>(a, nsamples, st);
  if constexpr (L == 384 || L == 1536)
    if (sh.width == 4 && sh.split == 1) return launch_stage_TS<T, L, 4, 1>(a, nsamples, st);
  if constexpr (L == 768)
    if (sh.width == 8 && sh.split == 1) return launch_stage_TS<T, L, 8, 1>(a, nsamples, st);
  return 1;
}

template <typename T>
int launch_stage_T(int L, const StageArgs& a, long nsamples, StageShape sh, hipStream_t st) {
  switch (L) {
    case 96: return launch_stage_L<T, 96>(a, nsamples, sh, st);
    case 192: return launch_stage_L<T, 192>(a, nsamples, sh, st);
    case 384: return launch_stage_L<T, 384>(a, nsamples, sh, st);
    case 768: return launch_stage_L<T, 768>(a, nsamples, sh, st);
    case 1536: return launch_stage_L<T, 1536>(a, nsamples, sh, st);
    default: return 1;
  }
}

__global__ void stage_modes_kernel(double2* modes, int N, int nh, double eps, double s2, double k0) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N * nh) return;
  const int i = idx / nh, kk = idx % nh;
  const ModeGeom<2> g(i >= nh ? i - N : i, kk, 0.0);
  modes[idx] = make_double2(1.0 / g.absk2, sv_eval(sqrt(g.absk2), eps, s2, k0));
}

}  // namespace

// The lines below were placed by timing whole steps (device loop, Fourier states of a
// shear layer; us per step against the separate passes of the same size, FP64 / FP32).
// A CU holds one workgroup of 12 waves (146-168 registers), so what counts is the number
// of rounds of 256 workgroups and how full the last one is.
//   N = 64, 128  : width 4, split 2 whatever the batch (N = 64: 57 / 51 against 86 / 101;
//                  N = 128 x 33: 115 / 84 against 160 / 149)
//   N = 256      : width 2, split 2 until the wider tiles fill the chip (one sample 78 / 70
//                  against 119 / 129), then width 4 (x 21: 204 / 140 against 274 / 215)
//   N = 512      : one sample width 2, split 2 (104 / 84 against 137 / 136); batches whole
//                  lines (width 8) unless width 4, split 2 needs less than 1.9 times the
//                  rounds (x 13: 518 / 320 against 546 / 361; x 8 FP64: 360 at width 4
//                  against 404 at width 8).  FP32 batches whose last round is less than
//                  a fifth short stay ahead of the separate passes (x 64: 1516 against
//                  1519), the others do not (x 8: 281 against 265, x 24: 653 against 624)
//   N = 1024     : one sample width 4 (207 / 162 against 234 / 194); two need two rounds for
//                  258 workgroups (415 / 320 against 390 / 298), so batches keep the
//                  separate passes
StageShape stage_shape(int tbytes, int L, long nsamples) {
  const long nh = L / 3 + 1;
  auto wgs = [&](int w) { return (nh + w - 1) / w * nsamples; };
  auto rounds = [&](int w) { return (wgs(w) + 255) / 256; };
  switch (L) {
    case 96: case 192: return {4, 2};
    case 384: return wgs(4) <= 256 ? StageShape{2, 2} : StageShape{4, 1};
    case 768: {
      if (nsamples == 1) return {2, 2};
      const bool wide = 1.9 * rounds(8) <= rounds(4);
      if (tbytes == 8) return wide ? StageShape{8, 1} : StageShape{4, 2};
      if (rounds(8) == 1) return wide ? StageShape{8, 1} : StageShape{4, 2};
      return wgs(8) >= 0.8 * 256 * rounds(8) ? StageShape{8, 1} : StageShape{0, 0};
    }
    case 1536: return nsamples == 1 ? StageShape{4, 1} : StageShape{0, 0};
    default: return {0, 0};
  }
}

int launch_stage(int tbytes, int L, const StageArgs& a, long nsamples, StageShape shape, hipStream_t st) {
  return tbytes == 8 ? launch_stage_T<double>(L, a, nsamples, shape, st) : launch_stage_T<float>(L, a, nsamples, shape, st);
}

void launch_stage_modes(double2* modes, int N, double eps, double s2, double k0, hipStream_t st) {
  const int nh = N / 2 + 1;
  hipLaunchKernelGGL(stage_modes_kernel, dim3((unsigned)((N * nh + 255) / 256)), dim3(256), 0, st, modes, N, nh, eps,
                     s2, k0);
}

}  // namespace azb
