// Kernels of the standalone transforms and of what is fused with them: the last-axis real
// transforms (pairs of real lines share one complex FFT) and the forward axis-0 pass with
// the Leray projection of initial data.
#pragma once
#include "azb_kernels.hpp"

namespace azb {

// ---------------------------------------------------------------------------
// Last-axis real transforms.  One wave per workgroup holds LINE_E * 64 / L sequences, so
// the exchanges need no workgroup barrier and small batches still spread over the chip.
// c2r reads the half spectra straight into the first pass (Hermitian extension in
// registers) and r2c separates the two half spectra over lane permutes and stores whole
// complex values, where the staged versions moved every spectrum through LDS once more and
// wrote the real and imaginary parts of a result at different times.  Bound by memory:
// 256^3 FP64, three components (0.81 GB): r2c 222 -> 157 us (197 with non-temporal stores:
// the N/2+1-wide rows are not line-aligned), c2r 303 -> 156 us.
// ---------------------------------------------------------------------------
struct LineArgs {
  const void* in;
  void* out;
  long nlines;
  const void* tw;
};

// the last pass leaves butterfly j of a sequence in lane j of an L/R-lane group, which has
// to lie within a wave: 1024 takes its radix 16 last
template <int L>
struct LinePlan {
  using P = typename LenPlan<L>::P;
};
template <> struct LinePlan<1024> { using P = Plan<8, 8, 16>; };

template <typename T, int L, int DIR>
struct LineCfg {
  static constexpr int NT = 64;
  static constexpr int E = LenPlan<L>::E;
  static constexpr int TS = NT * E / L;  // sequences (line pairs) per workgroup
  using P = typename LinePlan<L>::P;
  static constexpr bool SPLIT = sizeof(T) == 8;  // 8-byte slots in both precisions
  // twiddle powers from the table: bound by memory, these kernels need not chain them
  using F = BlockFFT2<T, L, TS, NT, DIR, SPLIT, 1, MAP_SEQ1, MAP_SEQ1, true, 1, 0u, 32, 0u, void, false, false>;
};

template <typename T, int L>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : 4))) void line_r2c_kernel(LineArgs a) {
  using C = LineCfg<T, L, -1>;
  using F = typename C::F;
  using P = typename C::P;
  constexpr int R0 = first_radix(P{}), RL = last_radix(P{}), NB = L / RL, NH = L / 2 + 1;
  __shared__ T lds[F::lds_words];
  const unsigned t = threadIdx.x;
  const long pair0 = (long)xcd_contiguous(blockIdx.x, gridDim.x) * C::TS;
  const T* in = (const T*)a.in;
  cx<T> v[C::E];
  F::template load<R0>(v, t, [&](unsigned s, unsigned pos) -> cx<T> {
    const long la = 2 * (pair0 + s);
    return mk(la < a.nlines ? in[la * L + pos] : T(0), la + 1 < a.nlines ? in[(la + 1) * L + pos] : T(0));
  });
  F::run(v, t, lds, (const cx<T>*)a.tw, P{});
  vec2_t<T>* out = (vec2_t<T>*)a.out;
#pragma unroll
  for (int q = 0; q < C::E / RL; ++q) {
    const unsigned u = t + 64u * q, j = u % NB;
    const long la = 2 * (pair0 + u / NB);
    row_separate_store<T, NB, RL, PlainCols, RL / 2, false>(v + q * RL, t, j, out + la * NH, out + (la + 1) * NH, PlainCols{},
                                                     la < a.nlines, la + 1 < a.nlines);
  }
}

template <typename T, int L>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : 4))) void line_c2r_kernel(LineArgs a) {
  using C = LineCfg<T, L, +1>;
  using F = typename C::F;
  using P = typename C::P;
  constexpr int R0 = first_radix(P{}), RL = last_radix(P{}), NB = L / R0, NH = L / 2 + 1;
  static_assert(R0 % 2 == 0, "mode L/2 falls on a butterfly row");
  __shared__ T lds[F::lds_words];
  const unsigned t = threadIdx.x;
  const long pair0 = (long)xcd_contiguous(blockIdx.x, gridDim.x) * C::TS;
  const cx<T>* in = (const cx<T>*)a.in;
  cx<T> v[C::E];
  // Im at k = 0 and L/2 is dropped (FFTW/cuFFT convention)
#pragma unroll
  for (int q = 0; q < C::E / R0; ++q) {
    const unsigned u = t + 64u * q, j = u % NB;
    const long la = 2 * (pair0 + u / NB);
    const bool va = la < a.nlines, vb = la + 1 < a.nlines;
    const cx<T>*px = in + la * NH, *py = px + NH;
#pragma unroll
    for (int r = 0; r < R0; ++r) {
      const bool mirror = r >= R0 / 2;  // position j + NB r holds the conjugate of mode NB (R0 - r) - j
      const unsigned k = mirror ? NB * (R0 - r) - j : j + NB * r;
      const cx<T> X = va ? px[k] : mk(T(0), T(0)), Y = vb ? py[k] : mk(T(0), T(0));
      cx<T> z = mirror ? mk(X.x + Y.y, Y.x - X.y) : mk(X.x - Y.y, X.y + Y.x);
      if ((r == 0 || r == R0 / 2) && j == 0) z = mk(X.x, Y.x);
      v[q * R0 + r] = z;
    }
    // one butterfly's 2 R0 loads at a time: those of all of them would take the registers
    // of half the waves
    DFT<R0, +1, T>::run(v + q * R0);
    __builtin_amdgcn_sched_barrier(0);
  }
  F::run_rest(v, t, lds, (const cx<T>*)a.tw, P{});
  T* out = (T*)a.out;
  F::template store<RL>(v, t, [&](unsigned s, unsigned pos, cx<T> val) {
    const long la = 2 * (pair0 + s);
    if (la < a.nlines) __builtin_nontemporal_store(val.x, out + la * L + pos);
    if (la + 1 < a.nlines) __builtin_nontemporal_store(val.y, out + (la + 1) * L + pos);
  });
}

// ---------------------------------------------------------------------------
// Forward axis-0 pass of all DIM components with the Leray projection: a workgroup owns TS
// columns of every component, so the projection of a mode needs only an exchange of the
// last pass's values through LDS (real and imaginary halves in turn, the transform's own
// buffer), not another pass over memory: 256^3 FP64 204 us against 160 + 214 us for the
// pass and the projection apart (237 us with 8 columns per workgroup, 268 with every thread
// forming the projector for its own component's values).  In place on u_hat after the other axes' passes
// (src/azeban/operations/leray.cpp:28-116 for the projection).
// ---------------------------------------------------------------------------
struct LerayArgs {
  double2* u;   // [DIM][L][inner]
  long inner;   // columns: nh (2D) or L*nh (3D)
  const void* tw;
};

template <int DIM, int L>
struct LerayCfg {
  // whole lines and more of each row where the exchange buffer leaves 12 waves a CU
  static constexpr int TS = L <= 32 ? 32 : (DIM * L <= 768 ? 16 : (DIM * L <= 1152 ? 8 : 4));
  static constexpr int E = LenPlan<L>::E;
  static constexpr int NT = DIM * TS * L / E;
  using F = BlockFFT2<double, L, DIM * TS, NT, -1, true, 1, MAP_STD, MAP_STD>;
};

template <int DIM, int L>
__global__ __launch_bounds__((LerayCfg<DIM, L>::NT)) __attribute__((amdgpu_waves_per_eu(LerayCfg<DIM, L>::E == 16 ? 4 : 2))) void col_leray_kernel(LerayArgs a) {
  using C = LerayCfg<DIM, L>;
  using F = typename C::F;
  using P = typename LenPlan<L>::P;
  constexpr int TS = C::TS, NT = C::NT, R0 = first_radix(P{}), RL = last_radix(P{}), NH = L / 2 + 1;
  __shared__ double lds[F::lds_words];
  const unsigned t = threadIdx.x;
  const long c0 = (long)xcd_contiguous(blockIdx.x, gridDim.x) * TS;
  const unsigned cols = (unsigned)(a.inner - c0 < TS ? a.inner - c0 : TS);
  cx<double>* base = (cx<double>*)a.u + c0;
  const long cs = (long)L * a.inner;
  cx<double> v[C::E];
  F::template load<R0>(v, t, [&](unsigned s, unsigned pos) -> cx<double> {
    return s % TS < cols ? gload<double>(base + (s / TS) * cs + pos * a.inner, s % TS) : mk(0.0, 0.0);
  });
  F::run(v, t, lds, (const cx<double>*)a.tw, P{});

  // Projection: a thread takes whole modes (m = t + NT e: column m % TS, row m / TS), so the
  // wavevector and its reciprocal are formed once per mode, not once per component
  constexpr int NM = (TS * L + NT - 1) / NT;
  unsigned tt = t;
  asm volatile("" : "+v"(tt));
  auto put = [&](int c) {
    F::template store<RL>(v, tt, [&](unsigned s, unsigned pos, cx<double> val) {
      lds[pos * (DIM * TS) + s] = c == 0 ? val.x : val.y;
    });
  };
  auto active = [&](int e) { return (e + 1) * NT <= TS * L || tt + NT * e < (unsigned)(TS * L); };
  double im[NM][DIM];
  __syncthreads();
  put(1);
  __syncthreads();
#pragma unroll
  for (int e = 0; e < NM; ++e)
    if (active(e)) {
      const unsigned m = tt + NT * e;
#pragma unroll
      for (int d = 0; d < DIM; ++d) im[e][d] = lds[m / TS * (DIM * TS) + d * TS + m % TS];
    }
  __syncthreads();
  put(0);
  __syncthreads();
#pragma unroll
  for (int e = 0; e < NM; ++e) {
    const unsigned m = tt + NT * e, col = m % TS, pos = m / TS;
    if (!active(e) || col >= cols) continue;
    const unsigned flat = (unsigned)(c0 + col);
    const int kk = (int)(flat % NH), jj = DIM == 3 ? (int)(flat / NH) : 0, i = (int)pos;
    double k[DIM], re[DIM];
    k[0] = kTwoPi * (i >= NH ? i - L : i);
    if (DIM == 3) k[1] = kTwoPi * (jj >= NH ? jj - L : jj);
    k[DIM - 1] = kTwoPi * kk;
    double k2 = 0.0, dr = 0.0, di = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      re[d] = lds[pos * (DIM * TS) + d * TS + col];
      k2 += k[d] * k[d];
      dr += k[d] * re[d];
      di += k[d] * im[e][d];
    }
    const double inv = 1.0 / k2;
    dr *= inv;
    di *= inv;
    const bool zero = k2 == 0.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      const double x = zero ? 0.0 : re[d] - k[d] * dr, y = zero ? 0.0 : im[e][d] - k[d] * di;
      gstore<double, false>(base + d * cs + pos * a.inner, col, x, y);
    }
  }
}

}  // namespace azb
