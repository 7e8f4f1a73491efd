// rl_kernels.hpp -- compile-time-length kernels of the fused multiview
// Richardson-Lucy iteration
//   psi <- psi * (1/V) sum_v corr(phi_v / max(conv(psi, P_v), eps), P_v)
// built on fft_static.hpp and the pass bodies of static_kernels_impl.hpp.
//
//   sk_zfan      one z tile of FFTxy(psi): FFTz once, then per view the
//                product with FFTz(P_v) and IFFTz into that view's spectrum
//   sk_xratio    per view, rows of the blurred estimate: x-C2R, ratio
//                phi / max(blur, eps) in registers, x-R2C back in place
//                (the ratio volume never reaches HBM)
//   sk_zsum      one z tile: sum over views of FFTz(ratio_v) * conj(FFTz(P_v)),
//                IFFTz (correlations add in the spectral domain)
//   sk_xupdate   x-C2R of the summed correlation with the epilogue
//                psi <- psi * acc / V
#pragma once

#include <type_traits>

#include "static_kernels_impl.hpp"

namespace fcamd {

// Waves per SIMD asked of the ratio kernel: 4, the most its LDS allows, took
// the 10-iteration, 4-view 384 x 384 x 192 run from 15.34 to 15.04 ms.
constexpr int kRatioWaves = 4;
// and of the sum over views, which holds three columns of MAXE float2 (sum,
// view, kernel) and some 30 registers more: as many as that leaves room for.
// Four at every length spilled 130 registers at 384, 127 at 80, 200 at 112 and
// 50 at 600; three views of 256 x 192 x z with 15 taps, us, before and after:
// z = 80 54.7 / 37.8, 112 84.6 / 43.2, 384 255 / 175, 600 413 (8-bin tiles; 443
// with 16-bin ones) / 244, 432 178 / 177.
template <int L, int TX>
constexpr int zsum_waves() {
  constexpr int regs = 6 * PlanOf<L, false>::MAXE() + 30;
  constexpr int wg = (TX * threads_per_transform<L>() + 63) / 64;  // its waves
  // (of 9 to 12 waves one workgroup fits either way)
  return regs <= 128 && (wg <= 8 || wg > 12) ? 4 : regs <= 168 ? 3 : 2;
}

// phi / d for d = max(blur, eps) > 0.  With eps a normal number (the
// launch-uniform case FAST) every d is one, and the hardware reciprocal (at
// most 1 ulp) times phi replaces the IEEE division sequence: one rounding
// more, some ten instructions fewer per sample.  A subnormal eps keeps the
// division.
constexpr float kMinNormal = 1.17549435e-38f;
template <bool FAST>
__device__ __forceinline__ float rl_div(float phi, float d) {
  if constexpr (FAST) return phi * __builtin_amdgcn_rcpf(d);
  return phi / d;
}

// column access at position pos through a base at position t
template <class T>
__device__ __forceinline__ T& col_at(T* base_t, int pos, int t, long stride) {
  return base_t[(long)(pos - t) * stride];
}

// H: every view's taps lie within the first and last H stage-0 slots
// (kernel_prune; 0: anywhere)
template <int L, int TX, int H>
__global__ void __launch_bounds__(TX * threads_per_transform<L>())
sk_zfan(RLZArgs a) {
  using P = PlanOf<L, false>;
  __shared__ float2 lds[L * TX];
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  long y;
  int x;
  bool ok;
  column_tile_decode(a.nbins, TX, a.ny, blockIdx.x, c, &y, &x, &ok);
  const long base = ok ? y * a.s_row + x : 0;
  auto addr = [&](int pos) { return pos * TX + c; };
  float2 X[P::MAXE()];
  const float2* src_t = a.src + base + (long)t * a.s_plane;
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) {
    float2 val = make_float2(0.f, 0.f);
    if (ok) val = col_at(src_t, pos, t, a.s_plane);
    X[slot] = val;
  });
  sfft_run<L, false, -1>(X, t, lds, addr, a.fft.stw);
  for (int v = 0; v < a.nviews; ++v) {
    float2 W[P::MAXE()];
    load_kernel_taps<L, H>(W, t, ok, a.kplanes[v] + base, a.s_plane, a.kz[v], a.cz[v]);
    sfft_run<L, false, -1>(W, t, lds, addr, a.fft.stw);
    sfft_for_outputs<L, false>(t, [&](int slot, int) { W[slot] = cscale(cmul(X[slot], W[slot]), a.scale); });
    sfft_run<L, true, +1>(W, t, lds, addr, a.fft.stw);
    float2* out_t = a.view[v] + base + (long)t * a.s_plane;
    if (ok) sfft_for_outputs<L, true>(t, [&](int slot, int pos) { col_at(out_t, pos, t, a.s_plane) = W[slot]; });
  }
}

// The taps' columns are taken whole: pruned slots (H as in sk_zfan) gain
// nothing beside two live transforms (ten iterations of four views of 384 x 384
// x 192 with 51 taps 13.05 ms pruned, 13.03 whole).
template <int L, int TX>
__global__ void __launch_bounds__(TX * threads_per_transform<L>(), (zsum_waves<L, TX>()))
sk_zsum(RLZArgs a) {
  using P = PlanOf<L, false>;
  __shared__ float2 lds[L * TX];
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  long y;
  int x;
  bool ok;
  column_tile_decode(a.nbins, TX, a.ny, blockIdx.x, c, &y, &x, &ok);
  const long base = ok ? y * a.s_row + x : 0;
  auto addr = [&](int pos) { return pos * TX + c; };
  float2 acc[P::MAXE()];
#pragma unroll
  for (int i = 0; i < P::MAXE(); ++i) acc[i] = make_float2(0.f, 0.f);
  for (int v = 0; v < a.nviews; ++v) {
    float2 X[P::MAXE()], W[P::MAXE()];
    const float2* in_t = a.view[v] + base + (long)t * a.s_plane;
    sfft_for_inputs<L, false>(t, [&](int slot, int pos) {
      float2 val = make_float2(0.f, 0.f);
      if (ok) val = col_at(in_t, pos, t, a.s_plane);
      X[slot] = val;
    });
    load_kernel_taps<L, 0>(W, t, ok, a.kplanes[v] + base, a.s_plane, a.kz[v], a.cz[v]);
    sfft_run<L, false, -1>(X, t, lds, addr, a.fft.stw);
    sfft_run<L, false, -1>(W, t, lds, addr, a.fft.stw);
    sfft_for_outputs<L, false>(t, [&](int slot, int) { acc[slot] = cadd(acc[slot], cmulc(X[slot], W[slot])); });
  }
  sfft_for_outputs<L, false>(t, [&](int slot, int) { acc[slot] = cscale(acc[slot], a.scale); });
  sfft_run<L, true, +1>(acc, t, lds, addr, a.fft.stw);
  float2* out_t = a.dst + base + (long)t * a.s_plane;
  if (ok) sfft_for_outputs<L, true>(t, [&](int slot, int pos) { col_at(out_t, pos, t, a.s_plane) = acc[slot]; });
}

// The x kernels move the workgroup's spectrum rows and real rows (phi, psi)
// between HBM and LDS staging as coalesced runs, as the flat x passes do
// (xflat_* in static_kernels_impl.hpp).  The real rows are dense.
template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>(), kRatioWaves)
sk_xratio(RLXArgs a) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP, SL = XStage<L>::SL;
  constexpr int NT = PAIRS * T, MAXR = 2 * PAIRS;
  __shared__ float2 lds[xflat_lds_floats<L>(PAIRS) / 2];
  const long groups = ((a.nrows + 1) / 2 + PAIRS - 1) / PAIRS;
  const int v = (int)(blockIdx.x / groups);
  const long r0 = 2 * (blockIdx.x - (long)v * groups) * PAIRS;
  const int nr = a.nrows - r0 < MAXR ? (int)(a.nrows - r0) : MAXR;
  float2* spec = a.spec[v];
  XBins<L, PAIRS>().load(spec + r0 * a.srow, a.srow, nr, lds);
  __syncthreads();
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  float2 z[P::MAXE()];
  // C2R on the reversed plan: its outputs sit where the forward plan reads
  const float2* in = lds + c * LP;
  sfft_for_inputs<L, true>(t, [&](int slot, int pos) { z[slot] = in[XRow<L>::at(t, pos - t)]; });
  __syncthreads();
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, true, +1>(z, t, row, addr, a.fft.stw);
  // phi rows through LDS; ratio at the transform's output positions
  float* st = reinterpret_cast<float*>(lds);
  xflat_load_rows<L, NT, MAXR>(a.phi[v] + r0 * L, st, nr);
  __syncthreads();
  const float* fa = st + 2 * c * SL;
  const float* fb = fa + (2 * c + 1 < nr ? SL : 0);  // a missing second row repeats the first
  const float eps = a.eps;
  auto ratio = [&](auto fast) {
    constexpr bool F = decltype(fast)::value;
    sfft_for_outputs<L, true>(t, [&](int slot, int pos) {
      z[slot] = make_float2(rl_div<F>(fa[pos], fmaxf(z[slot].x, eps)),
                            rl_div<F>(fb[pos], fmaxf(z[slot].y, eps)));
    });
  };
  if (eps >= kMinNormal)
    ratio(std::true_type{});
  else
    ratio(std::false_type{});
  __syncthreads();
  sfft_run<L, false, -1>(z, t, row, addr, a.fft.stw);
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) { row[addr(t, pos - t)] = z[slot]; });
  __syncthreads();
  // Hermitian split back into the view's spectrum rows
  XBins<L, PAIRS>::again().store(spec + r0 * a.srow, a.srow, nr, lds);
}

template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xupdate(RLXArgs a) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP, SL = XStage<L>::SL;
  constexpr int NT = PAIRS * T, MAXR = 2 * PAIRS;
  __shared__ float2 lds[xflat_lds_floats<L>(PAIRS) / 2];
  const long r0 = 2 * (long)blockIdx.x * PAIRS;
  const int nr = a.nrows - r0 < MAXR ? (int)(a.nrows - r0) : MAXR;
  XBins<L, PAIRS>().load(a.spec[0] + r0 * a.srow, a.srow, nr, lds);
  __syncthreads();
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  float2 z[P::MAXE()];
  const float2* in = lds + c * LP;
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) { z[slot] = in[XRow<L>::at(t, pos - t)]; });
  __syncthreads();
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, false, +1>(z, t, row, addr, a.fft.stw);
  // psi rows through LDS: psi <- psi * acc / V at the output positions
  float* st = reinterpret_cast<float*>(lds);
  float* psi = a.psi + r0 * L;
  xflat_load_rows<L, NT, MAXR>(psi, st, nr);
  __syncthreads();
  const float iv = a.inv_views;
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) {
    st[2 * c * SL + pos] *= z[slot].x * iv;  // (rows past nr are not stored)
    st[(2 * c + 1) * SL + pos] *= z[slot].y * iv;
  });
  __syncthreads();
  xflat_store_rows<L, NT, MAXR>(psi, st, nr);
}

// calls f with the pruned tap slots that hold every view's kernel
template <int L, class F>
void rl_with_slots(const RLZArgs& a, F f) {
  int n = 1;  // the widest view's; 0: some view fits neither
  for (int v = 0; v < a.nviews; ++v) {
    const int p = kernel_prune<L>(a.kz[v], a.cz[v]);
    n = p == 0 || n == 0 ? 0 : p > n ? p : n;
  }
  if (n == 1)
    f(std::integral_constant<int, kernel_slots<L>(1)>{});
  else if (n == 2)
    f(std::integral_constant<int, kernel_slots<L>(2)>{});
  else
    f(std::integral_constant<int, 0>{});
}

template <int L>
void rl_launch_zfan(const RLZArgs& a, long ny, hipStream_t st) {
  constexpr int TX = fit_tile<L, 16, kTileLdsZ>();
  RLZArgs b = a;
  b.ny = ny;
  rl_with_slots<L>(a, [&](auto h) {
    hipLaunchKernelGGL((sk_zfan<L, TX, decltype(h)::value>),
                       dim3((unsigned)column_tiles(a.nbins, TX, ny)),
                       dim3(TX * threads_per_transform<L>()), 0, st, b);
  });
}

template <int L>
void rl_launch_zsum(const RLZArgs& a, long ny, hipStream_t st) {
  constexpr int TX = fit_tile<L, 16, kTileLdsZ>();
  RLZArgs b = a;
  b.ny = ny;
  hipLaunchKernelGGL((sk_zsum<L, TX>), dim3((unsigned)column_tiles(a.nbins, TX, ny)),
                     dim3(TX * threads_per_transform<L>()), 0, st, b);
}

template <int L>
void rl_launch_xratio(const RLXArgs& a, int nviews, hipStream_t st) {
  constexpr int P = flat_fill_pairs<L>();
  const long groups = ((a.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xratio<L, P>), dim3((unsigned)(groups * nviews)),
                     dim3(P * threads_per_transform<L>()), 0, st, a);
}

template <int L>
void rl_launch_xupdate(const RLXArgs& a, hipStream_t st) {
  constexpr int P = flat_fill_pairs<L>();
  const long groups = ((a.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xupdate<L, P>), dim3((unsigned)groups),
                     dim3(P * threads_per_transform<L>()), 0, st, a);
}

}  // namespace fcamd
