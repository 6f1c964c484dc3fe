// 2D column stage: everything of an RK stage between two row kernels in one launch.
//
// In 2D the axis-0 transforms of one block of last-axis modes k touch nothing but that
// block, so one workgroup takes TS consecutive k and runs for them
//   forward  : the three products' axis-0 transforms (M rows in, the N kept ones used),
//   k-space  : ik.B_hat, Leray, viscosity and the RK stage update of every mode (i, k),
//   inverse  : the axis-0 transforms of the two components of the new stage value, the
//              next row kernel's input.
// B_hat never leaves the workgroup and the stage value is not read back.
#pragma once
#include "azb_kernels.hpp"

namespace azb {

// The working arrays between the row kernel and the column stage are stored in column
// blocks of TS modes, [component][k / TS][line][k % TS]: a workgroup's columns are one
// contiguous run per component, and the TS modes of the consecutive lines that a row
// workgroup holds lie next to each other, so both kernels move whole cache lines.
struct StageArgs {
  const void* s2;       // [sample][3][block][M][TS] products after the row kernel, working precision
  const double2* u_in;  // stage input u_hat
  const double2* u0;    // RK base state (stages 2, 3), in the caller's layout [sample][2][N][nh]
  double2* out;         // stage value (or du/dt)
  void* x;              // [sample][2][block][M][TS]: next row kernel's input; NULL: no inverse
  // [N][nh] of (1 / |k|^2, nu(|k|)), made once per solver: the stage's few resident waves
  // would otherwise spend a division, a square root and an exponential on every mode
  const double2* modes;
  int in_blocked, out_blocked;  // u_in / out in column blocks [sample][2][block][N][TS], else as u0
  int nh, ktiles;       // ktiles = ceil(nh / TS) blocks
  double Md, C, Nd;     // u_max = max / Md; stage 1: dt = min(C / (Nd u_max), max_dt)
  const void *tw_f, *tw_i;
  DevState* st;
  int mode, slot;       // KMode, or K_LEAD: only the inverse transforms, of u_in
  int clear;    // max|u| slot whose bins the next row kernel fills: cleared here (-1: none)
  int advance;  // last stage of a step of the device-driven loop: time += dt, ++steps
  double* dt_out;  // host-visible copy of the first sample's dt (NULL: none)
};

// First and remaining radices of a plan
template <int R0, int... Rs>
constexpr Plan<Rs...> plan_rest(Plan<R0, Rs...>) { return {}; }

// F = 1: a thread makes both components of its modes; F = 2: one, with twice the threads
// (shorter chains per wave, for launches that leave the chip idle).
template <typename T, int L, int TS, int F>
struct StageCfg {
  static constexpr int NT = F * TS * L / 8;
  static constexpr int N = 2 * L / 3;
  using P = typename LenPlan<L>::P;
  using LF = ColLayout<3 * TS, 2 * TS>;
  using LI = ColLayout<2 * TS, TS>;
  static constexpr int ELEMS = LF::elems(L);
  // real and imaginary halves in turn unless whole values leave room for four (FP32: two) workgroups
  static constexpr bool SPLIT = ELEMS * 2 * (int)sizeof(T) > (sizeof(T) == 8 ? 40960 : 81920);
  static constexpr int WORDS = ELEMS * (SPLIT ? 1 : 2);
  // a workgroup fits a CU, and 16 lanes share the max|u| bins
  static constexpr bool built = WORDS * (int)sizeof(T) <= 163840 && NT <= 1024 && NT % 16 == 0;
  static_assert(first_radix(P{}) == 8, "the k-space update hands its rows to radix-8 butterflies");
};

template <typename T, int L, int TS, int F>
__global__ __launch_bounds__((StageCfg<T, L, TS, F>::NT)) __attribute__((amdgpu_waves_per_eu(3))) void col_stage_kernel(StageArgs a) {
  using C = StageCfg<T, L, TS, F>;
  using P = typename C::P;
  constexpr int NT = C::NT, N = C::N, half = N / 2, RL = last_radix(P{}), NQ = 2 / F;
  constexpr bool SPLIT = C::SPLIT, PT = sizeof(T) == 4 && L == 768;
  using FF = ColFFT<T, L, 3 * TS, NT, -1, SPLIT, typename C::LF, PT>;
  using FI = ColFFT<T, L, 2 * TS, NT, +1, SPLIT, typename C::LI, PT>;
  using LF = typename C::LF;
  using LI = typename C::LI;
  __shared__ T lds[C::WORDS];
  const unsigned t = threadIdx.x;
  const unsigned blk = xcd_contiguous(blockIdx.x, gridDim.x);
  const unsigned kt = blk % (unsigned)a.ktiles;
  const long sample = blk / (unsigned)a.ktiles;
  DevState* st = a.st + sample;
  if (st->done) return;
  const unsigned c0 = kt * TS, cols = (unsigned)a.nh - c0;
  const unsigned cs = (unsigned)a.ktiles * (L * TS);  // component stride of the products
  const bool lead = a.mode == K_LEAD;

  cx<T> v[24];
  if (!lead) {
    const void* in = (const cx<T>*)a.s2 + sample * (3l * cs) + kt * (L * TS);
    const unsigned s = t % (3u * TS), m = s / TS, col = s % TS, j = t / (3u * TS);
    const unsigned base = m * cs + j * TS + col;
#pragma unroll
    for (int b = 0; b < FF::template rounds<8>(); ++b)
#pragma unroll
      for (int r = 0; r < 8; ++r)
        v[b * 8 + r] = FF::template on<8>(j, b) && col < cols ? gload<T>(in, base + (FF::JS * b + r * (L / 8)) * TS)
                                                              : mk(T(0), T(0));
  }
  // stage step: every wave reduces the row kernel's max|u| bins at stage 1, the first
  // workgroup of a sample at every stage (it stores u_max)
  double dt = 0.0;
  if (!lead) {
    const bool first = kt == 0;
    double um = 0.0;
    if (a.mode == K_RK1 || first) {
      // 16 lanes cover the bins (NT is a multiple of 16, not of the wave)
      const unsigned long long* bins = st->umax_bins[a.slot] + (t & 15u);
#pragma unroll
      for (int e = 0; e < kBins; e += 16) um = fmax(um, __longlong_as_double((long long)bins[e]));
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) um = fmax(um, __shfl_xor(um, o, 16));
      um /= a.Md;
    }
    dt = a.mode == K_RK1 ? fmin(a.C / (a.Nd * um), st->max_dt) : st->dt;
    if (first && t == 0) {
      st->u_max = um;
      if (a.mode == K_RK1) {
        st->dt = dt;
        if (a.dt_out && sample == 0) *a.dt_out = dt;
      }
      if (a.advance) {
        st->time += dt;
        st->steps += 1;
      }
    }
    if (first && a.clear >= 0)
      for (unsigned e = t; e < (unsigned)kBins; e += NT) st->umax_bins[a.clear][e] = 0ull;
  }

  if (!lead) {
    FF::template butterflies<1, 8>(v, t, (const cx<T>*)a.tw_f);
    FF::template after<8>([&](int c) { FF::template put<1, 8>(v, t, lds, c); }, v, t, lds, (const cx<T>*)a.tw_f,
                          plan_rest(P{}));
  }

  // The thread's modes: column `col`, rows of the radix-8 butterfly j of the inverse's
  // first pass (positions j + r L/8; r = 3, 4 and parts of r = 2, 5 are the padding),
  // components q0 .. q0 + NQ - 1
  unsigned tt = t;
  asm volatile("" : "+v"(tt));
  const unsigned col = tt % TS, j = (tt / TS) % (L / 8), q0 = F == 2 ? tt / (TS * L / 8) : 0u;
  // slot e = 0 .. 5 of the rows that can be kept: r = 0, 1, 2, 5, 6, 7
  constexpr int NE = 6;
  auto radix_row = [](int e) { return e < 3 ? e : e + 2; };
  bool keep[NE];
  unsigned at_state[NE];
  const unsigned scs = N * (unsigned)a.nh, bcs = (unsigned)a.ktiles * (N * TS);  // component strides
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const unsigned pos = j + radix_row(e) * (L / 8);
    keep[e] = col < cols && (pos <= (unsigned)half || pos >= (unsigned)(L - half + 1));
    const unsigned row = pos <= (unsigned)half ? pos : pos - (L - N);
    at_state[e] = q0 * scs + row * (unsigned)a.nh + col;
  }
  auto at_block = [&](int e) {
    const unsigned pos = j + radix_row(e) * (L / 8);
    return q0 * bcs + (pos <= (unsigned)half ? pos : pos - (L - N)) * TS + col;
  };
  const long sbase = sample * (2l * N) * a.nh + c0, bbase = sample * (2l * bcs) + kt * (N * TS);
  const double2* u_in = a.u_in + (a.in_blocked ? bbase : sbase);
  const unsigned ics = a.in_blocked ? bcs : scs, ocs = a.out_blocked ? bcs : scs;
  cx<double> u[NQ][NE];
  const bool base_state = a.mode == K_RK2 || a.mode == K_RK3;
  const double2* u0 = a.u0 + sbase;
  auto load_state = [&]() {
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        u[q][e] = keep[e] ? gload<double>(u_in, (a.in_blocked ? at_block(e) : at_state[e]) + q * ics) : mk(0.0, 0.0);
  };

  cx<T> w[NQ * 8];  // stage value at working precision: component q0 + q, butterfly input r at w[8 q + r]
#pragma unroll
  for (int e = 0; e < NQ * 8; ++e) w[e] = mk(T(0), T(0));
  if (lead) {
    load_state();
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
      for (int q = 0; q < NQ; ++q) w[8 * q + radix_row(e)] = mk(T(u[q][e].x), T(u[q][e].y));
  } else {
    double br[2][NE];  // real half of b = ik.B_hat
    const double2* modes = a.modes + c0;
    double2* out = a.out + (a.out_blocked ? bbase : sbase);
    auto put_kept = [&](int c) {  // kept rows of the forward output, half c
      const unsigned s = tt % (3u * TS), j0 = tt / (3u * TS);
#pragma unroll
      for (int b = 0; b < FF::template rounds<RL>(); ++b)
#pragma unroll
        for (int r = 0; r < RL; ++r) {
          const unsigned pos = j0 + FF::JS * b + r * (L / RL);
          if (FF::template on<RL>(j0, b) && (pos <= (unsigned)half || pos >= (unsigned)(L - half + 1))) {
            const unsigned idx = LF::at(s, pos);
            if (SPLIT) {
              lds[idx] = c == 0 ? v[b * RL + r].x : v[b * RL + r].y;
            } else {
              lds[2 * idx] = v[b * RL + r].x;
              lds[2 * idx + 1] = v[b * RL + r].y;
            }
          }
        }
    };
    auto mode_of = [&](int e, double inv) {
      const unsigned pos = j + radix_row(e) * (L / 8);
      return ModeGeom<2>(pos <= (unsigned)half ? (int)pos : (int)pos - L, (int)(c0 + col), inv);
    };
    auto real_half = [&](int e) {  // from the imaginary parts
      if (!keep[e]) return;
      double B[3], o[2];
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        const unsigned idx = LF::at(m * TS + col, j + radix_row(e) * (L / 8));
        B[m] = -(double)lds[SPLIT ? idx : 2 * idx + 1];
      }
      kspace_dot<2>(mode_of(e, 0.0), B, o);
      br[0][e] = o[0];
      br[1][e] = o[1];
    };
    __syncthreads();
    put_kept(1);
    if (SPLIT) {
      // the stage input's loads go out as the transform's registers become free, ahead
      // of the exchanges that the update waits for
      load_state();
      __syncthreads();
#pragma unroll
      for (int e = 0; e < NE; ++e) real_half(e);
      __syncthreads();
      put_kept(0);
    } else {
      load_state();
    }
    // the update in groups of rows whose loads are in flight together
    constexpr int G = F == 1 ? 2 : 6;
    cx<double> md[G], b0[NQ][G];
    auto load_group = [&](int e0) {
#pragma unroll
      for (int i = 0; i < G; ++i) {
        md[i] = keep[e0 + i] ? gload<double>(modes, at_state[e0 + i] - q0 * scs) : mk(0.0, 0.0);
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          b0[q][i] = keep[e0 + i] && base_state ? gload<double>(u0, at_state[e0 + i] + q * scs) : mk(0.0, 0.0);
      }
    };
    load_group(0);
    __syncthreads();
#pragma unroll
    for (int e0 = 0; e0 < NE; e0 += G) {
      if (e0) load_group(e0);
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const int e = e0 + i;
        if (!SPLIT) real_half(e);
        if (!keep[e]) continue;
        const ModeGeom<2> g = mode_of(e, md[i].x);
        double B[3], bi[2], Lr[2], Li[2];
        const double b2[2] = {br[0][e], br[1][e]};
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          const unsigned idx = LF::at(m * TS + col, j + radix_row(e) * (L / 8));
          B[m] = (double)lds[SPLIT ? idx : 2 * idx];
        }
        kspace_dot<2>(g, B, bi);
        kspace_project<2>(g, b2, Lr);
        kspace_project<2>(g, bi, Li);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const double lr = F == 1 ? Lr[q] : (q0 == 0 ? Lr[0] : Lr[1]);
          const double li = F == 1 ? Li[q] : (q0 == 0 ? Li[0] : Li[1]);
          const double x = stage_value(a.mode, g.absk2, lr, md[i].y, u[q][e].x, b0[q][i].x, dt);
          const double y = stage_value(a.mode, g.absk2, li, md[i].y, u[q][e].y, b0[q][i].y, dt);
          // cached store: the caller's rows are not line-aligned, and the neighbouring
          // tile completes the lines
          out[(a.out_blocked ? at_block(e) : at_state[e]) + q * ocs] = make_double2(x, y);
          w[8 * q + radix_row(e)] = mk(T(x), T(y));
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (!a.x) return;

  // inverse: first pass in registers (no twiddles)
#pragma unroll
  for (int q = 0; q < NQ; ++q) DFT<8, +1, T>::run(w + 8 * q);
  cx<T> z[24];  // an array of its own: idle lanes' slots then hold nothing across the k-space part
  FI::template after<8>(
      [&](int c) {
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
          for (int r = 0; r < 8; ++r) {
            const unsigned idx = LI::at((q0 + q) * TS + col, 8 * j + r);
            if (SPLIT) {
              lds[idx] = c == 0 ? w[8 * q + r].x : w[8 * q + r].y;
            } else {
              lds[2 * idx] = w[8 * q + r].x;
              lds[2 * idx + 1] = w[8 * q + r].y;
            }
          }
      },
      z, t, lds, (const cx<T>*)a.tw_i, plan_rest(P{}));
  {
    unsigned t3 = t;
    asm volatile("" : "+v"(t3));
    void* x = (cx<T>*)a.x + sample * (2l * cs) + kt * (L * TS);
    const unsigned s = t3 % (2u * TS), q = s / TS, cl = s % TS, j0 = t3 / (2u * TS);
#pragma unroll
    for (int b = 0; b < FI::template rounds<RL>(); ++b) {
      if (!FI::template on<RL>(j0, b)) continue;
#pragma unroll
      for (int r = 0; r < RL; ++r) {
        const unsigned pos = j0 + FI::JS * b + r * (L / RL);
        if (cl < cols) gstore<T>(x, q * cs + pos * TS + cl, z[b * RL + r].x, z[b * RL + r].y);
      }
    }
  }
}

}  // namespace azb
