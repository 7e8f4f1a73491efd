// static_kernels_impl.hpp -- compile-time-length pass kernels built on
// fft_static.hpp, in several variants per pass.  Instantiated per length by
// static_inst.hip; the driver reaches them through the registry in
// static_kernels.hip.
//
// Variants:
//   x forward  "w<N>"            about N threads (N/T row pairs) per workgroup
//              "w<N>-flat"       rows staged through LDS with workgroup-wide
//                                coalesced loads and stores
//   x inverse  "w<N>", "w<N>-flat"
//              "w256-ldsmirror"  Hermitian extension formed in LDS
//   column     "t<TX>"           one TX-bin tile per workgroup
//              "t<TX>-pipe"      persistent workgroups; the next tile's loads
//                                are issued before the current tile's FFT
//   fused z    "t<TX>-fft"       kernel column by the same FFT as the image
//              "t<TX>-dft"       kernel spectrum by direct DFT over its kz
//                                taps straight into the last-stage registers
// and one batched form per pass (sb_*) whose workgroups take their
// (argument record, tile) from a device task table.
#pragma once

#include "fft_static.hpp"
#include "kernels.hpp"
#include "static_registry.hpp"

namespace fcamd {

template <int L>
constexpr int threads_per_transform() {
  return PlanOf<L, false>::T;
}

// plan identifier and threads per column of the fused z kernels (PATH 1: the
// tap path; 0: a second column transformed like the image's, H = 0: a whole
// one, else cut to H slots)
template <int L, int PATH, int H = 0>
constexpr int zk_id() {
  return PATH == 1 ? z_id<L>() : H == 0 ? z_whole_id<L>() : z_full_id<L>();
}
template <int L, int PATH, int H = 0>
constexpr int z_threads() {
  return PlanOf<zk_id<L, PATH, H>(), false>::T;
}

// Largest tile <= want that keeps a workgroup within 1024 threads and its LDS
// (L rows of the tile).  A 16-bin tile is a 128-byte line per row and takes
// up to CAP bytes; 8-bin tiles move half lines and reach 3.0-4.1 TB/s in a
// bare copy where 16-bin tiles reach 5.1-6.4 (384 x 384 x 192 to 512 x 512 x
// 256).  Two workgroups per CU (80 KiB each) pay: y passes over L x 512 x 64
// volumes 42.8 -> 33.9 us at L = 540, 46.3 -> 43.6 at 600, the z pass at 640
// 180 -> 126 us.  One workgroup per CU still pays in the inverse y pass up to
// 768 (56.9 -> 50.2 us), not in the z pass (720: 132 -> 138, 960: 180 -> 201
// us), and the forward y pass takes 16 bins to 600 only: its launch may carry
// many kernel planes, whose tiles are arithmetic alone (48 of them at 640 x
// 640 x 48: 71 -> 77 us, at 768 x 512 x 48: 70 -> 78; without them 48 -> 47
// and 60.6 -> 57.9).
constexpr int kTileLds = 65536, kTileLdsFwd = 76800, kTileLdsZ = 81920, kTileLdsInv = 98304;
template <int L, int WANT, int CAP = kTileLds, int T = threads_per_transform<L>()>
constexpr int fit_tile() {
  int tx = WANT;
  while (tx > 1 && (tx * T > 1024 ||
                    (long)tx * L * 8 > (tx == 16 ? CAP : kTileLds)))
    tx /= 2;
  return tx;
}
// tiles of the column (y) and z passes
template <int L, int WANT, int DIR>
constexpr int col_fit() {
  return fit_tile<L, WANT, WANT != 16 ? kTileLds : DIR < 0 ? kTileLdsFwd : kTileLdsInv>();
}
template <int L, int WANT>
constexpr int z_fit() {
  constexpr int whole = z_threads<L, 0, 0>(), cut = z_threads<L, 0, 1>();
  return fit_tile<L, WANT, WANT == 16 ? kTileLdsZ : kTileLds, (whole > cut ? whole : cut)>();
}

// row pairs per x-pass workgroup for about TGT threads (T threads per row
// pair), within the LDS and thread limits of fit_pairs
template <int L, int TGT>
constexpr int pairs_for() {
  const int t = threads_per_transform<L>();
  return t >= TGT ? 1 : TGT / t;
}

template <int L, int WANT>
constexpr int fit_pairs() {
  int p = WANT;
  while (p > 1 && (p * threads_per_transform<L>() > 1024 || (long)p * (L + L / 8 + 1) * 8 > 65536))
    p /= 2;
  return p;
}


// padded LDS row of the x passes: one float2 of padding per 8 keeps the
// stride-8 and stride-Ns stores of the early stages off a single bank set
template <int L>
struct XRow {
  static constexpr int LP = L + L / 8 + 1;
  __device__ static int at(int pos) { return pos + (pos >> 3); }
  // at(base + off): an offset of whole eights moves the index by a constant
  __device__ static int at(int base, int off) {
    return off % 8 == 0 ? at(base) + off + off / 8 : at(base + off);
  }
};
struct XAddr {
  __device__ int operator()(int pos) const { return XRow<0>::at(pos); }
  __device__ int operator()(int base, int off) const { return XRow<0>::at(base, off); }
};

// ---------------------------------------------------------------------------
// x pass forward: two real rows per complex FFT (see kernels_generic.hip).
// The first k_blocks workgroups transform the compact kernel's rows, placed
// circularly so tap x lands at (x - kx/2) mod nx.
// ---------------------------------------------------------------------------
template <int L, int PAIRS>
__device__ __forceinline__ void xfwd_body(const XPassArgs& a, long blk, float2* lds) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP;
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  const long ra = 2 * (blk * PAIRS + c), rb = ra + 1;
  const bool oka = ra < a.nrows, okb = rb < a.nrows;
  const float* pa = a.src + ra * a.src_row;
  const float* pb = a.src + rb * a.src_row;
  const int kc = a.kcenter, kl = a.klen;
  float2 v[P::MAXE()];
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) {
    int x = pos + kc;
    if (x >= L) x -= L;
    float xa = 0.f, xb = 0.f;
    if (x < kl) {
      if (oka) xa = pa[x];
      if (okb) xb = pb[x];
    }
    v[slot] = make_float2(xa, xb);
  });
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, false, -1, 9>(v, t, row, addr, a.fft.stw);
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) { row[addr(t, pos - t)] = v[slot]; });
  __syncthreads();
  float2* da = a.dst + ra * a.dst_row;
  float2* db = a.dst + rb * a.dst_row;
  for (int kb = t; kb < a.nbins; kb += T) {
    const float2 Z = row[addr(kb)];
    const float2 Zm = row[addr(kb == 0 ? 0 : L - kb)];
    if (oka) da[kb] = make_float2(0.5f * (Z.x + Zm.x), 0.5f * (Z.y - Zm.y));
    if (okb) db[kb] = make_float2(0.5f * (Z.y + Zm.y), 0.5f * (Zm.x - Z.x));
  }
}

// Image rows of a virtually padded volume (VPad in kernels.hpp): row and
// element indices go through the boundary maps, zeros where undefined.
template <int L, int PAIRS>
__device__ __forceinline__ void xfwd_vpad_body(const XPassArgs& a, long blk, float2* lds) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP;
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  const long ra = 2 * (blk * PAIRS + c), rb = ra + 1;
  const VPad& vp = a.vp;
  long sa = 0, sb = 0;
  const bool oka = ra < a.nrows && vpad_row(vp, ra, &sa);
  const bool okb = rb < a.nrows && vpad_row(vp, rb, &sb);
  const float* pa = a.src + sa * vp.n[0];
  const float* pb = a.src + sb * vp.n[0];
  float2 v[P::MAXE()];
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) {
    bool okx;
    const int xs = vpad_src(vp, 0, pos, &okx);
    float xa = 0.f, xb = 0.f;
    if (okx) {
      if (oka) xa = pa[xs];
      if (okb) xb = pb[xs];
    }
    v[slot] = make_float2(xa, xb);
  });
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, false, -1, 9>(v, t, row, addr, a.fft.stw);
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) { row[addr(t, pos - t)] = v[slot]; });
  __syncthreads();
  float2* da = a.dst + ra * a.dst_row;
  float2* db = a.dst + rb * a.dst_row;
  const bool wa = ra < a.nrows, wb = rb < a.nrows;
  for (int kb = t; kb < a.nbins; kb += T) {
    const float2 Z = row[addr(kb)];
    const float2 Zm = row[addr(kb == 0 ? 0 : L - kb)];
    if (wa) da[kb] = make_float2(0.5f * (Z.x + Zm.x), 0.5f * (Z.y - Zm.y));
    if (wb) db[kb] = make_float2(0.5f * (Z.y + Zm.y), 0.5f * (Zm.x - Z.x));
  }
}

// kernel rows first (xfwd_body), then the padded image rows
template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xfwd_vpad(XPass2 a2) {
  __shared__ float2 lds[PAIRS * XRow<L>::LP];
  if ((long)blockIdx.x >= a2.k_blocks)
    xfwd_vpad_body<L, PAIRS>(a2.m, (long)blockIdx.x - a2.k_blocks, lds);
  else
    xfwd_body<L, PAIRS>(a2.k, blockIdx.x, lds);
}

template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xfwd(XPass2 a2) {
  __shared__ float2 lds[PAIRS * XRow<L>::LP];
  // the kernel's rows take the first k_blocks workgroups so they run
  // alongside the image rows instead of trailing them
  const bool main = (long)blockIdx.x >= a2.k_blocks;
  xfwd_body<L, PAIRS>(main ? a2.m : a2.k, main ? (long)blockIdx.x - a2.k_blocks : (long)blockIdx.x,
                      lds);
}


// ---------------------------------------------------------------------------
// x pass inverse (C2R), two rows per complex FFT
// ---------------------------------------------------------------------------
template <int L, int PAIRS>
__device__ __forceinline__ void xinv_body(const XPassArgs& a, long blk, float2* lds) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP;
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  const long ra = 2 * (blk * PAIRS + c), rb = ra + 1;
  const bool oka = ra < a.nrows, okb = rb < a.nrows;
  const float2* pa = a.csrc + ra * a.src_row;
  const float2* pb = a.csrc + rb * a.src_row;
  const int nb = a.nbins;
  float2 v[P::MAXE()];
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) {
    const bool mirror = pos >= nb;
    const int kb = mirror ? L - pos : pos;
    float2 A = make_float2(0.f, 0.f), B = make_float2(0.f, 0.f);
    if (oka) A = pa[kb];
    if (okb) B = pb[kb];
    if (kb == 0 || 2 * kb == L) {
      A.y = 0.f;
      B.y = 0.f;
    }
    if (mirror) {
      A.y = -A.y;
      B.y = -B.y;
    }
    v[slot] = make_float2(A.x - B.y, A.y + B.x);
  });
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, false, +1>(v, t, row, addr, a.fft.stw);
  float* oa = a.rdst + ra * a.dst_row;
  float* ob = a.rdst + rb * a.dst_row;
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) {
    if (oka) oa[pos] = v[slot].x;
    if (okb) ob[pos] = v[slot].y;
  });
}

// Same transform, but every half-spectrum bin of the two rows is read from
// HBM once (coalesced) into LDS and the Hermitian mirror is formed there.
template <int L, int PAIRS>
__device__ __forceinline__ void xinv_lds_body(const XPassArgs& a, long blk, float2* lds) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP;
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  const long ra = 2 * (blk * PAIRS + c), rb = ra + 1;
  const bool oka = ra < a.nrows, okb = rb < a.nrows;
  const float2* pa = a.csrc + ra * a.src_row;
  const float2* pb = a.csrc + rb * a.src_row;
  const int nb = a.nbins;
  float2* row = lds + c * LP;
  const XAddr addr;
  // Z = A' + iB' over all L positions, built from the nb bins of each row:
  // position kb takes A + iB, its mirror L - kb takes conj(A) + i conj(B)
  for (int kb = t; kb < nb; kb += T) {
    float2 A = make_float2(0.f, 0.f), B = make_float2(0.f, 0.f);
    if (oka) A = pa[kb];
    if (okb) B = pb[kb];
    if (kb == 0 || 2 * kb == L) {
      A.y = 0.f;
      B.y = 0.f;
    }
    // Z[kb] = A + iB and Z[L-kb] = conj(A) + i conj(B)
    row[addr(kb)] = make_float2(A.x - B.y, A.y + B.x);
    if (kb != 0 && 2 * kb != L) row[addr(L - kb)] = make_float2(A.x + B.y, B.x - A.y);
  }
  __syncthreads();
  float2 v[P::MAXE()];
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) { v[slot] = row[addr(t, pos - t)]; });
  __syncthreads();
  sfft_run<L, false, +1>(v, t, row, addr, a.fft.stw);
  float* oa = a.rdst + ra * a.dst_row;
  float* ob = a.rdst + rb * a.dst_row;
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) {
    if (oka) oa[pos] = v[slot].x;
    if (okb) ob[pos] = v[slot].y;
  });
}

template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xinv_lds(XPassArgs a) {
  __shared__ float2 lds[PAIRS * XRow<L>::LP];
  xinv_lds_body<L, PAIRS>(a, blockIdx.x, lds);
}

template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xinv(XPassArgs a) {
  __shared__ float2 lds[PAIRS * XRow<L>::LP];
  xinv_body<L, PAIRS>(a, blockIdx.x, lds);
}


// ---------------------------------------------------------------------------
// x passes with workgroup-wide ("flat") global access.  In the bodies above
// the T threads of a row pair touch T consecutive elements of each of its
// rows per instruction, so for short rows one wavefront instruction spans up
// to 64/T rows and as many cache lines.  Here the workgroup's rows, which are
// adjacent in memory, move between HBM and an LDS staging area as one run:
// consecutive lanes take consecutive 16-byte (real rows) or 8-byte
// (spectrum bins) pieces.  The staging area aliases the exchange rows.
// ---------------------------------------------------------------------------
template <int L>
struct XStage {
  static constexpr bool V4 = (L % 4) == 0;       // real rows split into float4s
  static constexpr int SL = V4 ? L + 4 : L + 1;  // staging row stride (floats)
};

// LDS floats of a flat x-pass workgroup of `pairs` row pairs: the larger of
// the exchange rows and the real staging rows
template <int L>
constexpr int xflat_lds_floats(int pairs) {
  const int ex = 2 * pairs * XRow<L>::LP;
  const int st = 2 * pairs * XStage<L>::SL;
  return ex > st ? ex : st;
}

// row pairs of a flat x-pass workgroup: about TGT threads, within 1024
// threads and 64 KiB of LDS
template <int L, int TGT>
constexpr int flat_pairs() {
  int p = pairs_for<L, TGT>();
  while (p > 1 && (p * threads_per_transform<L>() > 1024 || xflat_lds_floats<L>(p) * 4 > 65536))
    p /= 2;
  return p;
}

// Row pairs of a flat x-pass workgroup of 96 to 256 threads: the fewest whose
// threads fill their wavefronts to within 8 % of the best (T = 45 at 540: two
// pairs leave 30 % of the lanes idle, four 6 %: x inverse of 512 x 512 x 256
// with a zero boundary 124 us at two pairs, 116 at five).
template <int L>
constexpr int flat_fill_pairs() {
  constexpr int T = threads_per_transform<L>();
  auto fits = [](int p) {
    return p * T <= (T > 256 ? T : 256) && xflat_lds_floats<L>(p) * 4 <= 65536;
  };
  auto fill = [](int p) { return (double)(p * T) / ((p * T + 63) / 64 * 64); };
  double best = 0;
  for (int p = 1; fits(p); ++p)
    if (p * T >= 96 && fill(p) > best) best = fill(p);
  for (int p = 1; fits(p); ++p)
    if (p * T >= 96 && fill(p) >= best - 0.08) return p;
  return flat_pairs<L, 128>();
}

#ifndef FC_BATCH_XTGT
#define FC_BATCH_XTGT 256
#endif
#ifndef FC_BATCH_XFLAT
#define FC_BATCH_XFLAT 1
#endif
// row pairs per workgroup of the batched x passes
template <int L>
constexpr int batch_pairs() {
  return FC_BATCH_XFLAT ? flat_pairs<L, FC_BATCH_XTGT>() : fit_pairs<L, pairs_for<L, FC_BATCH_XTGT>()>();
}

// nr dense rows of L floats at g -> staging rows of stride SL.  A full
// workgroup's rows move without a bounds test per piece; only the last
// workgroup of a pass (or plane) is not full, and takes a rolled loop.
template <int L, int NT, int MAXR>
__device__ __forceinline__ void xflat_load_rows(const float* __restrict__ g, float* st, int nr) {
  constexpr int SL = XStage<L>::SL;
  if constexpr (XStage<L>::V4) {
    if ((reinterpret_cast<uintptr_t>(g) & 15) == 0) {
      constexpr int Q = L / 4, N = MAXR * Q, IT = (N + NT - 1) / NT;
      const float4* g4 = reinterpret_cast<const float4*>(g);
      auto put = [&](int i, float4 v) {
        const int row = i / Q;
        *reinterpret_cast<float4*>(st + row * SL + 4 * (i - row * Q)) = v;
      };
      if (nr == MAXR) {
        float4 r[IT];
#pragma unroll
        for (int j = 0; j < IT; ++j) {
          const int i = threadIdx.x + j * NT;
          if ((j + 1) * NT <= N || i < N) r[j] = g4[i];
        }
#pragma unroll
        for (int j = 0; j < IT; ++j) {
          const int i = threadIdx.x + j * NT;
          if ((j + 1) * NT <= N || i < N) put(i, r[j]);
        }
      } else {
#pragma unroll 1
        for (int i = threadIdx.x; i < nr * Q; i += NT) put(i, g4[i]);
      }
      return;
    }
  }
  constexpr int N = MAXR * L, IT = (N + NT - 1) / NT;
  auto put = [&](int i, float v) {
    const int row = i / L;
    st[row * SL + (i - row * L)] = v;
  };
  if (nr == MAXR) {
    float r[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      const int i = threadIdx.x + j * NT;
      if ((j + 1) * NT <= N || i < N) r[j] = g[i];
    }
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      const int i = threadIdx.x + j * NT;
      if ((j + 1) * NT <= N || i < N) put(i, r[j]);
    }
  } else {
#pragma unroll 1
    for (int i = threadIdx.x; i < nr * L; i += NT) put(i, g[i]);
  }
}

// staging rows of stride SL -> nr dense rows of L floats at g
template <int L, int NT, int MAXR>
__device__ __forceinline__ void xflat_store_rows(float* __restrict__ g, const float* st, int nr) {
  constexpr int SL = XStage<L>::SL;
  if constexpr (XStage<L>::V4) {
    if ((reinterpret_cast<uintptr_t>(g) & 15) == 0) {
      constexpr int Q = L / 4, N = MAXR * Q, IT = (N + NT - 1) / NT;
      float4* g4 = reinterpret_cast<float4*>(g);
      auto put = [&](int i) {
        const int row = i / Q;
        g4[i] = *reinterpret_cast<const float4*>(st + row * SL + 4 * (i - row * Q));
      };
      if (nr == MAXR) {
#pragma unroll
        for (int j = 0; j < IT; ++j) {
          const int i = threadIdx.x + j * NT;
          if ((j + 1) * NT <= N || i < N) put(i);
        }
      } else {
#pragma unroll 1
        for (int i = threadIdx.x; i < nr * Q; i += NT) put(i);
      }
      return;
    }
  }
  constexpr int N = MAXR * L, IT = (N + NT - 1) / NT;
  auto put = [&](int i) {
    const int row = i / L;
    g[i] = st[row * SL + (i - row * L)];
  };
  if (nr == MAXR) {
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      const int i = threadIdx.x + j * NT;
      if ((j + 1) * NT <= N || i < N) put(i);
    }
  } else {
#pragma unroll 1
    for (int i = threadIdx.x; i < nr * L; i += NT) put(i);
  }
}

// Spectrum rows of a flat x-pass workgroup.  A lane keeps one bin (two or
// more where a row is longer than the workgroup) over all row pairs, G pairs
// at a time, so that a row or pair step moves every address by a constant;
// walking the rows' bins as one run takes a division by the bin count and
// 64-bit address arithmetic per bin.  The lone Nyquist bin of even L goes
// last, one lane per pair.
template <int L, int PAIRS>
struct XBins {
  static constexpr int NT = PAIRS * PlanOf<L, false>::T;
  static constexpr int MB = (L + 1) / 2;                   // bins below Nyquist
  static constexpr int G = NT >= MB ? NT / MB : 1;         // pairs side by side
  static constexpr int KI = NT >= MB ? 1 : (MB + NT - 1) / NT;  // bins per lane
  static constexpr int PI = (PAIRS + G - 1) / G;           // pair steps
  static constexpr int LP = XRow<L>::LP;
  int tid, g, k0;
  __device__ explicit XBins(int t) : tid(t), g(t / MB), k0(t - g * MB) {
    if (G == 1 && KI > 1) {
      g = 0;
      k0 = t;
    }
  }
  __device__ XBins() : XBins((int)threadIdx.x) {}
  // for a second use far from the first: the compiler cannot tell that the
  // lane's constants are the same and does not hold them across a transform
  __device__ static XBins again() {
    int t = threadIdx.x;
    asm("" : "+v"(t));
    return XBins(t);
  }
  // does the lane hold pair step pi of bin step ki in a full workgroup?
  // (compile-time true but in the last steps)
  __device__ bool has(int pi, int ki) const {
    return ((pi + 1) * G <= PAIRS || g + pi * G < PAIRS) &&
           ((ki + 1) * NT <= MB || k0 + ki * NT < MB);
  }
  __device__ bool active() const { return G * MB >= NT || g < G; }
  // Z = A + iB of a row pair at the exchange positions of bin k, Hermitian
  // extension included (bin 0's imaginary parts dropped, as a C2R does)
  __device__ static void put(float2* lo, float2* hi, float2 a, float2 b, bool dc) {
    if (dc) a.y = b.y = 0.f;
    *lo = make_float2(a.x - b.y, a.y + b.x);
    *hi = make_float2(a.x + b.y, b.x - a.y);
  }
  __device__ static void split(float2* pa, float2* pb, float2 Z, float2 Zm, bool second) {
    *pa = make_float2(0.5f * (Z.x + Zm.x), 0.5f * (Z.y - Zm.y));
    if (second) *pb = make_float2(0.5f * (Z.y + Zm.y), 0.5f * (Zm.x - Z.x));
  }
  // the exchange rows of every row pair from nr spectrum rows at g_ (row
  // pitch `pitch`); a missing last row repeats its pair's first (its result
  // is not stored)
  __device__ void load(const float2* __restrict__ g_, long pitch, int nr, float2* rows) const {
    const int npairs = (nr + 1) >> 1;
    float2 nyq = make_float2(0.f, 0.f);
    if (L % 2 == 0 && tid < npairs) {  // the pair whose Nyquist bin the lane moves
      const float2* p = g_ + (long)(2 * tid) * pitch + L / 2;
      nyq.x = p[0].x;
      nyq.y = p[2 * tid + 1 < nr ? pitch : 0].x;
    }
    if (nr == 2 * PAIRS) {
      const float2* base = g_ + (long)(2 * g) * pitch + k0;
      float2 A[KI * PI], B[KI * PI];
      if (active()) {
#pragma unroll
        for (int ki = 0; ki < KI; ++ki)
#pragma unroll
          for (int pi = 0; pi < PI; ++pi) {
            if (!has(pi, ki)) continue;
            const float2* p = base + (long)(2 * pi * G) * pitch + ki * NT;
            A[ki * PI + pi] = p[0];
            B[ki * PI + pi] = p[pitch];
          }
#pragma unroll
        for (int ki = 0; ki < KI; ++ki) {
          const int k = k0 + ki * NT;
          float2* lo = rows + g * LP + XRow<L>::at(k);
          float2* hi = rows + g * LP + XRow<L>::at(k == 0 ? 0 : L - k);
#pragma unroll
          for (int pi = 0; pi < PI; ++pi)
            if (has(pi, ki))
              put(lo + pi * G * LP, hi + pi * G * LP, A[ki * PI + pi], B[ki * PI + pi], k == 0);
        }
      }
    } else {
#pragma unroll 1
      for (int i = tid; i < npairs * MB; i += NT) {
        const int c = i / MB, k = i - c * MB;
        const float2* p = g_ + (long)(2 * c) * pitch + k;
        put(rows + c * LP + XRow<L>::at(k), rows + c * LP + XRow<L>::at(k == 0 ? 0 : L - k), p[0],
            p[2 * c + 1 < nr ? pitch : 0], k == 0);
      }
    }
    if (L % 2 == 0 && tid < npairs) rows[tid * LP + XRow<L>::at(L / 2)] = nyq;
  }
  // the half spectra of both rows of every pair, separated from the pair's
  // complex transform in the exchange rows
  __device__ void store(float2* __restrict__ g_, long pitch, int nr, const float2* rows) const {
    const int npairs = (nr + 1) >> 1;
    if (nr == 2 * PAIRS) {
      float2* base = g_ + (long)(2 * g) * pitch + k0;
      if (active()) {
#pragma unroll
        for (int ki = 0; ki < KI; ++ki) {
          const int k = k0 + ki * NT;
          const float2* lo = rows + g * LP + XRow<L>::at(k);
          const float2* hi = rows + g * LP + XRow<L>::at(k == 0 ? 0 : L - k);
#pragma unroll
          for (int pi = 0; pi < PI; ++pi) {
            if (!has(pi, ki)) continue;
            float2* p = base + (long)(2 * pi * G) * pitch + ki * NT;
            split(p, p + pitch, lo[pi * G * LP], hi[pi * G * LP], true);
          }
        }
      }
    } else {
#pragma unroll 1
      for (int i = tid; i < npairs * MB; i += NT) {
        const int c = i / MB, k = i - c * MB;
        float2* p = g_ + (long)(2 * c) * pitch + k;
        split(p, p + pitch, rows[c * LP + XRow<L>::at(k)],
              rows[c * LP + XRow<L>::at(k == 0 ? 0 : L - k)], 2 * c + 1 < nr);
      }
    }
    if (L % 2 == 0 && tid < npairs) {
      const float2 Z = rows[tid * LP + XRow<L>::at(L / 2)];
      float2* p = g_ + (long)(2 * tid) * pitch + L / 2;
      p[0] = make_float2(Z.x, 0.f);
      if (2 * tid + 1 < nr) p[pitch] = make_float2(Z.y, 0.f);
    }
  }
};

// R2C of up to 2*PAIRS dense image rows starting at row 2*blk*PAIRS
template <int L, int PAIRS>
__device__ __forceinline__ void xfwd_flat_body(const XPassArgs& a, long blk, float2* lds) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP, SL = XStage<L>::SL;
  constexpr int NT = PAIRS * T, MAXR = 2 * PAIRS;
  const long r0 = 2 * blk * PAIRS;
  if (r0 >= a.nrows) return;  // whole workgroup
  const int nr = a.nrows - r0 < MAXR ? (int)(a.nrows - r0) : MAXR;
  float* st = reinterpret_cast<float*>(lds);
  xflat_load_rows<L, NT, MAXR>(a.src + r0 * L, st, nr);
  __syncthreads();
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  // a missing second row repeats the first (its result is not stored); pairs
  // past the last transform what the staging area holds
  const float* ra = st + 2 * c * SL;
  const float* rb = ra + (2 * c + 1 < nr ? SL : 0);
  float2 v[P::MAXE()];
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) { v[slot] = make_float2(ra[pos], rb[pos]); });
  __syncthreads();
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, false, -1, 9>(v, t, row, addr, a.fft.stw);
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) { row[addr(t, pos - t)] = v[slot]; });
  __syncthreads();
  XBins<L, PAIRS>().store(a.dst + r0 * a.dst_row, a.dst_row, nr, lds);
}

// C2R of up to 2*PAIRS spectrum rows into dense real rows
template <int L, int PAIRS>
__device__ __forceinline__ void xinv_flat_body(const XPassArgs& a, long blk, float2* lds) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP, SL = XStage<L>::SL;
  constexpr int NT = PAIRS * T, MAXR = 2 * PAIRS;
  const long r0 = 2 * blk * PAIRS;
  if (r0 >= a.nrows) return;  // whole workgroup
  const int nr = a.nrows - r0 < MAXR ? (int)(a.nrows - r0) : MAXR;
  XBins<L, PAIRS>().load(a.csrc + r0 * a.src_row, a.src_row, nr, lds);
  __syncthreads();
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  float2 v[P::MAXE()];
  const float2* in = lds + c * LP;
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) { v[slot] = in[XRow<L>::at(t, pos - t)]; });
  __syncthreads();
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, false, +1>(v, t, row, addr, a.fft.stw);
  // sfft_run ends on a barrier after its last LDS read
  float* st = reinterpret_cast<float*>(lds);
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) {
    st[2 * c * SL + pos] = v[slot].x;
    st[(2 * c + 1) * SL + pos] = v[slot].y;
  });
  __syncthreads();
  xflat_store_rows<L, NT, MAXR>(a.rdst + r0 * L, st, nr);
}

template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xfwd_flat(XPass2 a2) {
  static_assert(xflat_lds_floats<L>(PAIRS) * 4 <= 65536, "flat x pass LDS");
  __shared__ float2 lds[xflat_lds_floats<L>(PAIRS) / 2];
  if ((long)blockIdx.x >= a2.k_blocks)
    xfwd_flat_body<L, PAIRS>(a2.m, (long)blockIdx.x - a2.k_blocks, lds);
  else
    xfwd_body<L, PAIRS>(a2.k, blockIdx.x, lds);
}

template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xinv_flat(XPassArgs a) {
  static_assert(xflat_lds_floats<L>(PAIRS) * 4 <= 65536, "flat x pass LDS");
  __shared__ float2 lds[xflat_lds_floats<L>(PAIRS) / 2];
  xinv_flat_body<L, PAIRS>(a, blockIdx.x, lds);
}

// Flat form of the cropped x-C2R of a virtually padded volume (VPad in
// kernels.hpp): the workgroup's spectrum rows are staged as in the flat x
// passes, and each kept row's interior [lo, lo + m) is written with
// coalesced stores.  (A flat forward over the boundary maps, staging whole
// source rows, measured slower than the per-pair body: 258 vs 171 us at
// 600 x 600 x 288.)
template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xinv_crop_flat(XPassArgs a) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP, SL = XStage<L>::SL;
  constexpr int NT = PAIRS * T, MAXR = 2 * PAIRS;
  static_assert(xflat_lds_floats<L>(PAIRS) * 4 <= 65536, "flat x pass LDS");
  __shared__ float2 lds[xflat_lds_floats<L>(PAIRS) / 2];
  const long r0 = 2 * (long)blockIdx.x * PAIRS;
  const int nr = a.nrows - r0 < MAXR ? (int)(a.nrows - r0) : MAXR;
  XBins<L, PAIRS>().load(a.csrc + r0 * a.src_row, a.src_row, nr, lds);
  __syncthreads();
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  float2 v[P::MAXE()];
  const float2* in = lds + c * LP;
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) { v[slot] = in[XRow<L>::at(t, pos - t)]; });
  __syncthreads();
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, false, +1>(v, t, row, addr, a.fft.stw);
  float* st = reinterpret_cast<float*>(lds);
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) {
    st[2 * c * SL + pos] = v[slot].x;
    st[(2 * c + 1) * SL + pos] = v[slot].y;
  });
  __syncthreads();
  const VPad& vp = a.vp;
  const int m0 = vp.m[0], x0 = vp.lo[0];
  for (int r = 0; r < nr; ++r) {
    long orow = 0;
    if (!vpad_out_row(vp, r0 + r, &orow)) continue;  // uniform across the workgroup
    float* g = a.rdst + orow * m0;
    for (int x = threadIdx.x; x < m0; x += NT) g[x] = st[r * SL + x0 + x];
  }
}

// ---------------------------------------------------------------------------
// x passes over an extended image (AxisExt in kernels.hpp).  The workgroup's
// rows lie in one plane, so they are one run of nr * n floats in the image;
// it moves between HBM and the staging rows with consecutive lanes on
// consecutive floats (rows of any length start at any alignment), as
// 16-byte pieces where the rows are not extended.  The extension is applied
// on the way from the staging rows to the transform's registers, so a row is
// read from HBM once.
// ---------------------------------------------------------------------------
// row of element i of a run of rows of n < 4096 elements: (i + 1/2) / n is at
// least 1 / (2n) > 1.2e-4 from an integer, and its single-precision error
// stays below 2^-22 times the row count (< 2^7)
__device__ __forceinline__ int run_row(int i, float inv_n) { return (int)(((float)i + 0.5f) * inv_n); }

template <int L, int PAIRS>
__device__ __forceinline__ void xfwd_ext_body(const XExtArgs& a, long blk, float2* lds) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP, SL = XStage<L>::SL;
  constexpr int NT = PAIRS * T, MAXR = 2 * PAIRS;
  const unsigned z = (unsigned)blk / (unsigned)a.groups;
  const int r0 = 2 * PAIRS * (int)((unsigned)blk - z * (unsigned)a.groups);
  const int nr = a.ny - r0 < MAXR ? a.ny - r0 : MAXR;
  const AxisExt e = a.ext;
  const int n = e.n;
  float* st = reinterpret_cast<float*>(lds);
  const float* src = a.m.src + ((long)z * a.ny + r0) * n;
  if (n == L) {
    xflat_load_rows<L, NT, MAXR>(src, st, nr);
  } else {
    constexpr int IT = (MAXR * L + NT - 1) / NT;
    const int tot = nr * n;
    const float inv = 1.f / (float)n;
    float r[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      const int i = threadIdx.x + j * NT;
      r[j] = 0.f;
      if (i < tot) r[j] = src[i];
    }
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      const int i = threadIdx.x + j * NT;
      if (i < tot) {
        const int row = run_row(i, inv);
        st[row * SL + (i - row * n)] = r[j];
      }
    }
  }
  __syncthreads();
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  const float* ra = st + 2 * c * SL;  // missing rows as in xfwd_flat_body
  const float* rb = ra + (2 * c + 1 < nr ? SL : 0);
  float2 v[P::MAXE()];
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) {
    const int q = pos < n ? pos : axis_ext_src(e, L, pos);
    v[slot] = q >= 0 ? make_float2(ra[q], rb[q]) : make_float2(0.f, 0.f);
  });
  __syncthreads();
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, false, -1, 9>(v, t, row, addr, a.m.fft.stw);
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) { row[addr(t, pos - t)] = v[slot]; });
  __syncthreads();
  XBins<L, PAIRS>().store(a.m.dst + (long)z * a.spec_plane + (long)r0 * a.m.dst_row, a.m.dst_row, nr,
                          lds);
}

template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xfwd_ext(XExtArgs a) {
  static_assert(xflat_lds_floats<L>(PAIRS) * 4 <= 65536, "flat x pass LDS");
  __shared__ float2 lds[xflat_lds_floats<L>(PAIRS) / 2];
  if ((long)blockIdx.x >= a.k_blocks)
    xfwd_ext_body<L, PAIRS>(a, (long)blockIdx.x - a.k_blocks, lds);
  else
    xfwd_body<L, PAIRS>(a.k, blockIdx.x, lds);
}

template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sk_xinv_ext(XExtArgs a) {
  using P = PlanOf<L, false>;
  constexpr int T = P::T, LP = XRow<L>::LP, SL = XStage<L>::SL;
  constexpr int NT = PAIRS * T, MAXR = 2 * PAIRS;
  static_assert(xflat_lds_floats<L>(PAIRS) * 4 <= 65536, "flat x pass LDS");
  __shared__ float2 lds[xflat_lds_floats<L>(PAIRS) / 2];
  const unsigned z = blockIdx.x / (unsigned)a.groups;
  const int r0 = 2 * PAIRS * (int)(blockIdx.x - z * (unsigned)a.groups);
  const int nr = a.ny - r0 < MAXR ? a.ny - r0 : MAXR;
  XBins<L, PAIRS>().load(a.m.csrc + (long)z * a.spec_plane + (long)r0 * a.m.src_row, a.m.src_row, nr, lds);
  __syncthreads();
  const int t = threadIdx.x % T, c = threadIdx.x / T;
  float2 v[P::MAXE()];
  const float2* in = lds + c * LP;
  sfft_for_inputs<L, false>(t, [&](int slot, int pos) { v[slot] = in[XRow<L>::at(t, pos - t)]; });
  __syncthreads();
  float2* row = lds + c * LP;
  const XAddr addr;
  sfft_run<L, false, +1>(v, t, row, addr, a.m.fft.stw);
  // sfft_run ends on a barrier after its last LDS read
  float* st = reinterpret_cast<float*>(lds);
  const int n = a.ext.n;
  sfft_for_outputs<L, false>(t, [&](int slot, int pos) {
    st[2 * c * SL + pos] = v[slot].x;
    st[(2 * c + 1) * SL + pos] = v[slot].y;
  });
  __syncthreads();
  float* dst = a.m.rdst + ((long)z * a.ny + r0) * n;
  if (n == L) {
    xflat_store_rows<L, NT, MAXR>(dst, st, nr);
    return;
  }
  constexpr int IT = (MAXR * L + NT - 1) / NT;
  const int tot = nr * n;
  const float inv = 1.f / (float)n;
#pragma unroll
  for (int j = 0; j < IT; ++j) {
    const int i = threadIdx.x + j * NT;
    if (i < tot) {
      const int r = run_row(i, inv);
      dst[i] = st[r * SL + (i - r * n)];
    }
  }
}

// batched x passes: workgroup i serves tasks[i] = {argument record, row-pair
// group}.  Image rows (dense, unshifted) take the flat bodies; the compact
// kernel's rows the per-pair body.
template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sb_xfwd(const XPassArgs* __restrict__ args, const int2* __restrict__ tasks) {
  __shared__ float2 lds[xflat_lds_floats<L>(PAIRS) / 2];
  const int2 tk = tasks[blockIdx.x];
  const XPassArgs& a = args[tk.x];
  if (FC_BATCH_XFLAT && a.src_row == L && a.klen == L && a.kcenter == 0)
    xfwd_flat_body<L, PAIRS>(a, tk.y, lds);
  else
    xfwd_body<L, PAIRS>(a, tk.y, lds);
}

template <int L, int PAIRS>
__global__ void __launch_bounds__(PAIRS * threads_per_transform<L>())
sb_xinv(const XPassArgs* __restrict__ args, const int2* __restrict__ tasks) {
  __shared__ float2 lds[xflat_lds_floats<L>(PAIRS) / 2];
  const int2 tk = tasks[blockIdx.x];
  const XPassArgs& a = args[tk.x];
  if (FC_BATCH_XFLAT && a.dst_row == L)
    xinv_flat_body<L, PAIRS>(a, tk.y, lds);
  else
    xinv_lds_body<L, PAIRS>(a, tk.y, lds);
}

// ---------------------------------------------------------------------------
// column pass (y): tiles of TX bins x L positions, numbered by
// column_tile_decode (kernels.hpp)
// ---------------------------------------------------------------------------
template <int L, int TX, bool REV = false>
struct ColTile {
  using P = PlanOf<L, REV>;
  static constexpr int MAXE = P::MAXE();
  const ColArgs* a;
  long base_src, base_dst;
  bool ok;

  __device__ ColTile(const ColArgs& args, long tile, int c) : a(&args) {
    long o;
    int x;
    column_tile_decode(args.nbins, TX, args.nouter, tile, c, &o, &x, &ok);
    base_src = ok ? o * args.src_outer + x : 0;
    base_dst = ok ? o * args.dst_outer + x : 0;
  }
  // Positions are t + (compile-time constant) after unrolling, so the
  // accesses go through a per-thread base at position t and a uniform
  // offset (pos - t) * stride instead of a 64-bit product per element.
  __device__ void load(int t, float2 (&v)[MAXE]) const {
    const float2* src = a->src + base_src;
    const int center = a->center, nvalid = a->nvalid;
    const long es = a->src_elem;
    const bool okk = ok;
    if (center == 0 && nvalid == L) {
      const float2* st = src + (long)t * es;
      sfft_for_inputs<L, REV>(t, [&](int slot, int pos) {
        float2 val = make_float2(0.f, 0.f);
        if (okk) val = st[(long)(pos - t) * es];
        v[slot] = val;
      });
      return;
    }
    // compact support placed circularly (kernel planes): j < nvalid < 2^31 / es
    const int esi = (int)es;
    sfft_for_inputs<L, REV>(t, [&](int slot, int pos) {
      int j = pos + center;
      if (j >= L) j -= L;
      float2 val = make_float2(0.f, 0.f);
      if (okk && j < nvalid) val = src[j * esi];
      v[slot] = val;
    });
  }
  __device__ void store(int t, const float2 (&v)[MAXE]) const {
    if (!ok) return;
    const long es = a->dst_elem;
    float2* dt = a->dst + base_dst + (long)t * es;
    sfft_for_outputs<L, REV>(t, [&](int slot, int pos) { dt[(long)(pos - t) * es] = v[slot]; });
  }
  // extended columns (AxisExt): the rows at positions below n are read and
  // written through the base and uniform offset; only the waves that hold
  // positions of the extension compute the mapped row
  __device__ void load_ext(const AxisExt& e, int t, float2 (&v)[MAXE]) const {
    const float2* src = a->src + base_src;
    const long es = a->src_elem;
    const float2* st = src + (long)t * es;
    const bool okk = ok;
    sfft_for_inputs<L, REV>(t, [&](int slot, int pos) {
      float2 val = make_float2(0.f, 0.f);
      if (okk) {
        if (pos < e.n) {
          val = st[(long)(pos - t) * es];
        } else {
          const int q = axis_ext_src(e, L, pos);
          if (q >= 0) val = src[(long)q * es];
        }
      }
      v[slot] = val;
    });
  }
  __device__ void store_below(int n, int t, const float2 (&v)[MAXE]) const {
    if (!ok) return;
    const long es = a->dst_elem;
    float2* dt = a->dst + base_dst + (long)t * es;
    sfft_for_outputs<L, REV>(t, [&](int slot, int pos) {
      if (pos < n) dt[(long)(pos - t) * es] = v[slot];
    });
  }
};

// kernel-plane tiles first, then the image's
__device__ __forceinline__ const ColArgs& col2_args(const Col2& a2, long tile, long* local) {
  const long ktiles = a2.ntiles - a2.m_tiles;
  const bool main = tile >= ktiles;
  *local = main ? tile - ktiles : tile;
  return main ? a2.m : a2.k;
}

template <int L, int TX, int DIR, bool REV = false>
__device__ __forceinline__ void col_body(const ColArgs& args, long local, float2* lds) {
  using CT = ColTile<L, TX, REV>;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const CT tile(args, local, c);
  float2 v[CT::MAXE];
  tile.load(t, v);
  auto addr = [&](int pos) { return pos * TX + c; };
  sfft_run<L, REV, DIR>(v, t, lds, addr, args.fft.stw);
  tile.store(t, v);
}

// REV runs the radix plan in the opposite stage order
template <int L, int TX, int DIR, bool REV>
__global__ void __launch_bounds__(TX * threads_per_transform<L>())
sk_col(Col2 a2) {
  __shared__ float2 lds[L * TX];
  long local;
  const ColArgs& a = col2_args(a2, blockIdx.x, &local);
  col_body<L, TX, DIR, REV>(a, local, lds);
}

// y pass of an extended image: the forward reads the image's rows (mapped
// past their ends) and writes all L, the inverse reads all L and writes the
// image's
template <int L, int TX, int DIR>
__global__ void __launch_bounds__(TX * threads_per_transform<L>())
sk_col_ext(ColExtArgs b) {
  using CT = ColTile<L, TX>;
  __shared__ float2 lds[L * TX];
  long local;
  const ColArgs& a = col2_args(b.c, blockIdx.x, &local);
  if (DIR < 0 && (long)blockIdx.x < b.c.ntiles - b.c.m_tiles) {  // kernel planes
    col_body<L, TX, DIR, false>(a, local, lds);
    return;
  }
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const CT tile(a, local, c);
  float2 v[CT::MAXE];
  if (DIR < 0)
    tile.load_ext(b.ext, t, v);
  else
    tile.load(t, v);
  auto addr = [&](int pos) { return pos * TX + c; };
  sfft_run<L, false, DIR>(v, t, lds, addr, a.fft.stw);
  if (DIR < 0)
    tile.store(t, v);
  else
    tile.store_below(b.ext.n, t, v);
}

template <int L, int TX, int DIR>
__global__ void __launch_bounds__(TX * threads_per_transform<L>())
sb_col(const ColArgs* __restrict__ args, const int2* __restrict__ tasks) {
  __shared__ float2 lds[L * TX];
  const int2 tk = tasks[blockIdx.x];
  col_body<L, TX, DIR>(args[tk.x], tk.y, lds);
}

template <int L, int TX, int DIR>
__global__ void __launch_bounds__(TX * threads_per_transform<L>())
sk_col_pipe(Col2 a2) {
  using CT = ColTile<L, TX>;
  __shared__ float2 lds[L * TX];
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  auto addr = [&](int pos) { return pos * TX + c; };
  long tile = blockIdx.x;
  float2 v[CT::MAXE], nv[CT::MAXE];
  long local;
  if (tile < a2.ntiles) {
    const ColArgs& a = col2_args(a2, tile, &local);
    CT(a, local, c).load(t, v);
  }
  for (; tile < a2.ntiles; tile += gridDim.x) {
    const long next = tile + gridDim.x;
    if (next < a2.ntiles) {
      long nl;
      const ColArgs& na = col2_args(a2, next, &nl);
      CT(na, nl, c).load(t, nv);
    }
    const ColArgs& a = col2_args(a2, tile, &local);
    const CT cur(a, local, c);
    sfft_run<L, false, DIR>(v, t, lds, addr, a.fft.stw);
    cur.store(t, v);
#pragma unroll
    for (int i = 0; i < CT::MAXE; ++i) v[i] = nv[i];
  }
}

// ---------------------------------------------------------------------------
// fused z pass
// ---------------------------------------------------------------------------
// Kernel spectrum at the thread's last-stage output positions f = b + M*r
// (M = L/R, R = last radix) by direct DFT over the kz taps of the column:
//   K[f] = sum_j k_j W^(f (j - cz)),  W = exp(-2 pi i / L)
// With acc_q = sum_{j = q mod R} k_j W^(b (j - cz)) this is
//   K[b + M r] = W_R^(-r cz) * DFT_R(acc)[r].
template <int L, int MAXE>
__device__ __forceinline__ void kernel_spectrum_direct(float2 (&w)[MAXE], int t, bool ok,
                                                       const float2* __restrict__ kcol, long kplane,
                                                       int kz, int cz,
                                                       const float2* __restrict__ tw) {
  using P = PlanOf<z_full_id<L>(), false>;
  constexpr int s = P::S - 1;
  constexpr int R = P::R(s), M = P::M(s), NB = P::NB(s);
#pragma unroll
  for (int i = 0; i < NB * R; ++i) w[i] = make_float2(0.f, 0.f);
  // twiddle exponent e_i = b_i * (j - cz) mod L, advanced by b_i per tap
  int e[NB];
  int bb[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    bb[i] = t + i * P::T;
    e[i] = (int)(((long)bb[i] * (L - cz)) % L);
  }
  for (int j0 = 0; j0 < kz; j0 += R) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int j = j0 + q;
      if (j < kz) {
        float2 kv = make_float2(0.f, 0.f);
        if (ok) kv = kcol[(long)j * kplane];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          const float2 wt = tw[e[i]];
          w[i * R + q] = make_float2(w[i * R + q].x + kv.x * wt.x - kv.y * wt.y,
                                     w[i * R + q].y + kv.x * wt.y + kv.y * wt.x);
          e[i] += bb[i];
          if (e[i] >= L) e[i] -= L;
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    Dft<R, -1>::run(&w[i * R]);
    // W_R^(-r cz) = conj(tw[M * ((r cz) mod R)])
#pragma unroll
    for (int r = 1; r < R; ++r) w[i * R + r] = cmulc(w[i * R + r], tw[M * ((r * cz) % R)]);
  }
}

// Stage-0 input slots of a kernel column, from either end, that a pruned
// z kernel keeps: a quarter of the column (n = 1) or half of it (n = 2).
template <int ID>
constexpr int kernel_slots(int n) {
  return n == 1 ? (PlanOf<ID, false>::R(0) + 7) / 8 : (PlanOf<ID, false>::R(0) + 3) / 4;
}
// which of the two holds nvalid taps centred at `center` (0: neither)
template <int ID>
inline int kernel_prune(int nvalid, int center) {
  constexpr int M = PlanOf<ID, false>::M(0);
  const int far = nvalid - center > center ? nvalid - center : center;
  const int need = (far + M - 1) / M;
  return need <= kernel_slots<ID>(1) ? 1 : need <= kernel_slots<ID>(2) ? 2 : 0;
}

// w <- the kernel column's taps at the thread's stage-0 positions (ID: plan
// identifier of length L); H as in ZTile::load_kernel.  Nothing uses a value
// here: the loads stay in flight under what follows (scaling the taps as they
// arrive made the z pass 5-15 % slower)
template <int ID, int H, int MAXE>
__device__ __forceinline__ void load_kernel_taps(float2 (&w)[MAXE], int t, bool ok,
                                                 const float2* kcol, long kp, int nvalid,
                                                 int center) {
  using P = PlanOf<ID, false>;
  constexpr int L = P::L, R = P::R(0), M = P::M(0);
  // tap j = pos + center (- L when it wraps): base at tap t + center
  const float2* kt = kcol + (long)(t + center) * kp;
  const float2* kw = kt - (long)L * kp;
  if constexpr (H == 0) {
    sfft_for_inputs<ID, false>(t, [&](int slot, int pos) {
      const bool wrap = pos + center >= L;
      const int j = wrap ? pos + center - L : pos + center;
      float2 val = make_float2(0.f, 0.f);
      if (ok && j < nvalid) val = (wrap ? kw : kt)[(long)(pos - t) * kp];
      w[slot] = val;
    });
  } else {
    static_assert(2 * H <= R, "pruned slots overlap");
    const int jt = ok ? t + center : -(1 << 30);  // tap of position t, or none
    sfft_for_inputs<ID, false>(t, [&](int slot, int pos) {
      const int r = slot % R, d = slot / R * P::T + r * M;  // pos = t + d
      float2 val = make_float2(0.f, 0.f);
      if (r < H) {
        const int j = jt + d;
        if (j >= 0 && j < nvalid) val = kt[(long)d * kp];
      } else if (r >= R - H) {
        if (jt + d - L >= 0) val = kw[(long)d * kp];
      }
      w[slot] = val;
    });
  }
}

template <int L, int TX, int ID>
struct ZTile {
  using P = PlanOf<ID, false>;
  static constexpr int MAXE = P::MAXE();
  float2* col;
  const float2* kcol;
  bool ok;
  __device__ ZTile(const ZArgs& a, long tile, int c) {
    long y;
    int x;
    column_tile_decode(a.nbins, TX, a.ny, tile, c, &y, &x, &ok);
    if (!ok) {
      y = 0;
      x = 0;
    }
    col = a.s + y * a.s_row + x;
    kcol = a.k + y * a.k_row + x;
  }
  // per-thread base at position t plus a uniform offset (pos - t) * stride
  __device__ void load(const ZArgs& a, int t, float2 (&v)[MAXE]) const {
    const long sp = a.s_plane;
    const bool okk = ok;
    const float2* ct = col + (long)t * sp;
    sfft_for_inputs<ID, false>(t, [&](int slot, int pos) {
      float2 val = make_float2(0.f, 0.f);
      if (okk) val = ct[(long)(pos - t) * sp];
      v[slot] = val;
    });
  }
  // SUBSET: honour ZArgs::out_planes (compiled only where a dense operand,
  // the PSF gradient's, can reach the kernel)
  template <bool SUBSET>
  __device__ void store(const ZArgs& a, int t, const float2 (&v)[MAXE]) const {
    if (!ok) return;
    const long sp = a.s_plane;
    if (SUBSET && a.out_planes > 0) {  // rotated subset (see ZArgs)
      const int sh = a.out_shift, np = a.out_planes;
      sfft_for_outputs<ID, true>(t, [&](int slot, int pos) {
        int q = pos + sh;
        if (q >= L) q -= L;
        if (q < np) col[(long)q * sp] = v[slot];
      });
      return;
    }
    float2* ct = col + (long)t * sp;
    sfft_for_outputs<ID, true>(t, [&](int slot, int pos) { ct[(long)(pos - t) * sp] = v[slot]; });
  }
  // extended columns (AxisExt): planes mapped past the image's ends on the
  // way in, only the image's own planes written
  __device__ void load_ext(const ZArgs& a, const AxisExt& e, int t, float2 (&v)[MAXE]) const {
    load_mapped(col, a.s_plane, e, t, v);
  }
  __device__ void load_mapped(const float2* c0, long sp, const AxisExt& e, int t,
                              float2 (&v)[MAXE]) const {
    const float2* ct = c0 + (long)t * sp;
    const bool okk = ok;
    sfft_for_inputs<ID, false>(t, [&](int slot, int pos) {
      float2 val = make_float2(0.f, 0.f);
      if (okk) {
        if (pos < e.n) {
          val = ct[(long)(pos - t) * sp];
        } else {
          const int q = axis_ext_src(e, P::L, pos);
          if (q >= 0) val = c0[(long)q * sp];
        }
      }
      v[slot] = val;
    });
  }
  __device__ void load_operand(const ZArgs& a, const AxisExt& e, int t, float2 (&w)[MAXE]) const {
    load_mapped(kcol, a.k_plane, e, t, w);
  }
  __device__ void store_below(const ZArgs& a, int n, int t, const float2 (&v)[MAXE]) const {
    if (!ok) return;
    const long sp = a.s_plane;
    float2* ct = col + (long)t * sp;
    sfft_for_outputs<ID, true>(t, [&](int slot, int pos) {
      if (pos < n) ct[(long)(pos - t) * sp] = v[slot];
    });
  }
  // Kernel column: taps j < nvalid placed circularly at (j - center) mod L.
  // H > 0: the taps lie within the first and the last H stage-0 input slots
  // of every thread (kernel_slots), and the other slots are the constant zero
  // that the stage-0 butterfly folds away.
  template <int H>
  __device__ void load_kernel(const ZArgs& a, int t, float2 (&w)[MAXE]) const {
    load_kernel_taps<ID, H>(w, t, ok, kcol, a.k_plane, a.nvalid, a.center);
  }
};

// product of the forward image spectrum (v) with the kernel spectrum (w),
// conjugated for correlation, times the scale: v * (sc*w.x, +-sc*w.y)
// (ID: the plan identifier of both, see PlanOf)
template <int ID, int MAXE>
__device__ __forceinline__ void zproduct(float2 (&v)[MAXE], const float2 (&w)[MAXE], int t,
                                         bool cj, float sc) {
  const float si = cj ? -sc : sc;
  sfft_for_outputs<ID, false>(t, [&](int slot, int) {
    v[slot] = cmul(v[slot], make_float2(sc * w[slot].x, si * w[slot].y));
  });
}

// the same product with the scale already in w (the tap path scales its
// taps once as it loads them): v * (w.x, +-w.y)
template <int ID, int MAXE>
__device__ __forceinline__ void zproduct_prescaled(float2 (&v)[MAXE], const float2 (&w)[MAXE], int t,
                                                   bool cj) {
  const float si = cj ? -1.f : 1.f;
  sfft_for_outputs<ID, false>(t, [&](int slot, int) {
    v[slot] = cmul(v[slot], make_float2(w[slot].x, si * w[slot].y));
  });
}

// taps per column the two-stage fast path can hold (its stage-1 radix)
template <int L>
constexpr int ktap_slots() {
  return PlanOf<z_id<L>(), false>::S == 2 ? PlanOf<z_id<L>(), false>::R(1) : 1;
}

// Two-stage plan (L = R0*R1) with the kz taps within one stage-0 stride
// (nvalid <= R1): stage-0 butterfly r of the kernel column (positions
// r + rho*R1) meets at most one tap, rho = 0 (tap r + center) or
// rho = R0 - 1 (tap r + center - R1), so its output k is that tap times 1 or
// exp(+2 pi i k / R0).  Output k = b of butterfly r is the kernel's stage-1
// input slot (i, r) of the thread owning stage-1 butterfly b = t + i*T.
// Each thread loads at most ceil(kz / T) taps into `ktaps`; the image
// transform's stage-0 exchange barrier publishes them, and the stage-1
// inputs are read back by broadcast.  Compared with transforming the
// kernel column like the image's, this drops its stage-0 butterflies, its
// per-slot predicated loads and one LDS exchange (two per tile remain).
// (`keep`: positions written, L or the planes of an extended image)
template <int L, int TX, bool EXT = false>
__device__ __forceinline__ void zfused_sparse_body(const ZArgs& a, const ZTile<L, TX, z_id<L>()>& tile, int t,
                                                   int c, float2 (&v)[ZTile<L, TX, z_id<L>()>::MAXE],
                                                   float2* lds, float2* ktaps, int keep = L) {
  using P = PlanOf<z_id<L>(), false>;
  constexpr int R1 = P::R(1), M1 = P::M(1), NB1 = P::NB(1), T = P::T;
  constexpr int MAXE = ZTile<L, TX, z_id<L>()>::MAXE;
  auto addr = [&](int pos) { return pos * TX + c; };
  const int center = a.center, nvalid = a.nvalid;
  for (int j = t; j < nvalid; j += T)
    ktaps[j * TX + c] = tile.ok ? cscale(tile.kcol[(long)j * a.k_plane], a.scale) : make_float2(0.f, 0.f);
  // exp(+2 pi i b / R0) = conj(tw[b * R1]), tw[j] = exp(-2 pi i j / L)
  float2 e[NB1];
#pragma unroll
  for (int i = 0; i < NB1; ++i) {
    const int b = t + i * T;
    e[i] = (M1 % T) != 0 && b >= M1 ? make_float2(1.f, 0.f) : cconj(a.fft.tw[b * R1]);
  }
  // image: stage 0 and its exchange; the barrier also publishes the taps
  sfft_compute<z_id<L>(), false, -1, 0>(v, t, a.fft.stw);
  sfft_store_lds<z_id<L>(), false, 0>(v, t, lds, addr);
  StageTw<z_id<L>(), false, 1> tw1;
  sfft_load_tw<z_id<L>(), false, 1>(tw1, t, a.fft.stw);
  __syncthreads();
  sfft_load_lds<z_id<L>(), false, 1>(v, t, lds, addr);
  // every thread is done with the exchange tile before the inverse reuses it
  // (the taps live in their own array)
  __syncthreads();
  sfft_twiddle<z_id<L>(), false, -1, 1>(v, t, tw1);
  sfft_butterflies<z_id<L>(), false, -1, 1>(v, t);
  // the kernel column's stage-1 inputs, built only now to keep them out of
  // the image transform's register peak; same butterflies, same twiddles
  float2 w[MAXE];
#pragma unroll
  for (int i = 0; i < NB1; ++i) {
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      const int j0 = r + center, j1 = r + center - R1;
      float2 val = make_float2(0.f, 0.f);
      if (j0 < nvalid)
        val = ktaps[j0 * TX + c];
      else if (j1 >= 0)
        val = cmul(ktaps[j1 * TX + c], e[i]);
      w[i * R1 + r] = val;
    }
  }
  sfft_twiddle<z_id<L>(), false, -1, 1>(w, t, tw1);
  sfft_butterflies<z_id<L>(), false, -1, 1>(w, t);
  zproduct_prescaled<z_id<L>()>(v, w, t, a.conj != 0);
  sfft_run<z_id<L>(), true, +1>(v, t, lds, addr, a.fft.stw);
  if constexpr (EXT)
    tile.store_below(a, keep, t, v);
  else
    tile.template store<false>(a, t, v);
}

// whether the two-stage tap path applies to this launch
template <int L>
__host__ __device__ constexpr bool zfused_sparse_ok(int nvalid) {
  return PlanOf<z_id<L>(), false>::S == 2 && nvalid <= PlanOf<z_id<L>(), false>::R(1);
}

// Fused z pass of one tile.  PATH 0: kernel column transformed like the
// image's, its taps in the first and last H stage-0 slots (H = 0: anywhere);
// 1: the two-stage tap path (caller guarantees zfused_sparse_ok).  Separate
// instantiations: compiled into one kernel their register peaks add up (~144
// against ~105 VGPRs each).  EXT: columns of an extended image.
template <int L, int TX, int PATH, int H = 0, bool EXT = false>
__device__ __forceinline__ void zfused_body(const ZArgs& a, const AxisExt* ext, long tile_index,
                                            float2* lds, float2* ktaps) {
  constexpr int ID = zk_id<L, PATH, H>();
  using ZT = ZTile<L, TX, ID>;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const ZT tile(a, tile_index, c);
  auto addr = [&](int pos) { return pos * TX + c; };
  float2 v[ZT::MAXE];
  if constexpr (EXT)
    tile.load_ext(a, *ext, t, v);
  else
    tile.load(a, t, v);
  if constexpr (PATH == 1) {
    zfused_sparse_body<L, TX, EXT>(a, tile, t, c, v, lds, ktaps, EXT ? ext->n : L);
  } else {
    (void)ktaps;
    float2 w[ZT::MAXE];
    // a whole kernel column of a z plan is loaded after the image's transform
    // to stay out of its registers
    constexpr bool kLate = PlanOf<ID, false>::Z && H == 0;
    if (!kLate) tile.template load_kernel<H>(a, t, w);
    // every sfft_run ends with a barrier after its last LDS read, so the
    // next transform may reuse the tile
    sfft_run<ID, false, -1>(v, t, lds, addr, a.fft.stw);
    if (kLate) tile.template load_kernel<H>(a, t, w);
    sfft_run<ID, false, -1>(w, t, lds, addr, a.fft.stw);
    zproduct<ID>(v, w, t, a.conj != 0, a.scale);
    sfft_run<ID, true, +1>(v, t, lds, addr, a.fft.stw);
    if constexpr (EXT)
      tile.store_below(a, ext->n, t, v);
    else
      tile.template store<H == 0>(a, t, v);
  }
}

template <int L, int TX, int PATH, int H = 0>
__global__ void __launch_bounds__((TX * z_threads<L, PATH, H>()))
sk_zfused_fft(ZArgs a) {
  __shared__ float2 lds[L * TX];
  __shared__ float2 ktaps[TX * (PATH == 0 ? 1 : ktap_slots<L>())];
  zfused_body<L, TX, PATH, H>(a, nullptr, blockIdx.x, lds, ktaps);
}

template <int L, int TX, int PATH>
__global__ void __launch_bounds__((TX * z_threads<L, PATH>()))
sb_zfused(const ZArgs* __restrict__ args, const int2* __restrict__ tasks) {
  __shared__ float2 lds[L * TX];
  __shared__ float2 ktaps[TX * (PATH == 0 ? 1 : ktap_slots<L>())];
  const int2 tk = tasks[blockIdx.x];
  zfused_body<L, TX, PATH>(args[tk.x], nullptr, tk.y, lds, ktaps);
}

// the fused z pass of an extended image; PATH 0 and 1 as above
template <int L, int TX, int PATH, int H = 0>
__global__ void __launch_bounds__((TX * z_threads<L, PATH, H>()))
sk_zfused_ext(ZExtArgs b) {
  __shared__ float2 lds[L * TX];
  __shared__ float2 ktaps[TX * (PATH == 0 ? 1 : ktap_slots<L>())];
  zfused_body<L, TX, PATH, H, true>(b.z, &b.ext, blockIdx.x, lds, ktaps);
}

// z pass of the PSF gradient over extended volumes
template <int L, int TX>
__global__ void __launch_bounds__((TX * z_threads<L, 0>()))
sk_zcorr_ext(ZCorrArgs b) {
  constexpr int ID = zk_id<L, 0>();
  using ZT = ZTile<L, TX, ID>;
  __shared__ float2 lds[L * TX];
  const ZArgs& a = b.z;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const ZT tile(a, blockIdx.x, c);
  auto addr = [&](int pos) { return pos * TX + c; };
  float2 v[ZT::MAXE], w[ZT::MAXE];
  tile.load_ext(a, b.ext, t, v);
  sfft_run<ID, false, -1>(v, t, lds, addr, a.fft.stw);
  tile.load_operand(a, b.kext, t, w);
  sfft_run<ID, false, -1>(w, t, lds, addr, a.fft.stw);
  zproduct<ID>(v, w, t, true, a.scale);
  sfft_run<ID, true, +1>(v, t, lds, addr, a.fft.stw);
  tile.template store<true>(a, t, v);
}

template <int L, int TX>
__global__ void __launch_bounds__((TX * z_threads<L, 0, 1>()))
sk_zfused_dft(ZArgs a) {
  using ZT = ZTile<L, TX, z_full_id<L>()>;
  __shared__ float2 lds[L * TX];
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const ZT tile(a, blockIdx.x, c);
  auto addr = [&](int pos) { return pos * TX + c; };
  float2 v[ZT::MAXE];
  tile.load(a, t, v);
  sfft_run<z_full_id<L>(), false, -1>(v, t, lds, addr, a.fft.stw);
  float2 w[ZT::MAXE];
  kernel_spectrum_direct<L>(w, t, tile.ok, tile.kcol, a.k_plane, a.nvalid, a.center, a.fft.tw);
  zproduct<z_full_id<L>()>(v, w, t, a.conj != 0, a.scale);
  sfft_run<z_full_id<L>(), true, +1>(v, t, lds, addr, a.fft.stw);
  tile.template store<false>(a, t, v);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// x-pass launchers take the target thread count per workgroup (TGT)
template <int L, int TGT>
bool sk_launch_xfwd(const XPass2& a, hipStream_t st) {
  constexpr int P = fit_pairs<L, pairs_for<L, TGT>()>();
  XPass2 b = a;
  b.m_blocks = ((a.m.nrows + 1) / 2 + P - 1) / P;
  b.k_blocks = ((a.k.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xfwd<L, P>), dim3((unsigned)(b.m_blocks + b.k_blocks)),
                     dim3(P * threads_per_transform<L>()), 0, st, b);
  return true;
}

template <int L, int TGT>
bool sk_launch_xinv(const XPassArgs& a, hipStream_t st) {
  constexpr int P = fit_pairs<L, pairs_for<L, TGT>()>();
  const long blocks = ((a.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xinv<L, P>), dim3((unsigned)blocks), dim3(P * threads_per_transform<L>()),
                     0, st, a);
  return true;
}

template <int L, int TGT>
bool sk_launch_xfwd_vpad(const XPass2& a, hipStream_t st) {
  constexpr int P = fit_pairs<L, pairs_for<L, TGT>()>();
  XPass2 b = a;
  b.m_blocks = ((a.m.nrows + 1) / 2 + P - 1) / P;
  b.k_blocks = ((a.k.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xfwd_vpad<L, P>), dim3((unsigned)(b.m_blocks + b.k_blocks)),
                     dim3(P * threads_per_transform<L>()), 0, st, b);
  return true;
}

template <int L, int TGT>
bool sk_launch_xinv_crop_flat(const XPassArgs& a, hipStream_t st) {
  constexpr int P = flat_pairs<L, TGT>();
  const long blocks = ((a.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xinv_crop_flat<L, P>), dim3((unsigned)blocks),
                     dim3(P * threads_per_transform<L>()), 0, st, a);
  return true;
}

template <int L, int TGT>
bool sk_launch_xinv_lds(const XPassArgs& a, hipStream_t st) {
  constexpr int P = fit_pairs<L, pairs_for<L, TGT>()>();
  const long blocks = ((a.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xinv_lds<L, P>), dim3((unsigned)blocks),
                     dim3(P * threads_per_transform<L>()), 0, st, a);
  return true;
}

// flat variants need dense real rows (row stride L)
template <int L, int TGT>
bool sk_launch_xfwd_flat(const XPass2& a, hipStream_t st) {
  if (a.m.nrows > 0 && a.m.src_row != L) return false;
  constexpr int P = TGT == 128 ? flat_fill_pairs<L>() : flat_pairs<L, TGT>();
  XPass2 b = a;
  b.m_blocks = ((a.m.nrows + 1) / 2 + P - 1) / P;
  b.k_blocks = ((a.k.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xfwd_flat<L, P>), dim3((unsigned)(b.m_blocks + b.k_blocks)),
                     dim3(P * threads_per_transform<L>()), 0, st, b);
  return true;
}

template <int L, int TGT>
bool sk_launch_xinv_flat(const XPassArgs& a, hipStream_t st) {
  if (a.dst_row != L) return false;
  constexpr int P = TGT == 128 ? flat_fill_pairs<L>() : flat_pairs<L, TGT>();
  const long blocks = ((a.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xinv_flat<L, P>), dim3((unsigned)blocks),
                     dim3(P * threads_per_transform<L>()), 0, st, a);
  return true;
}

template <int L, int TX>
Col2 col2_tiles(const Col2& a) {
  Col2 b = a;
  b.ntx = (a.m.nbins + TX - 1) / TX;
  b.m.nouter = a.m_outer;
  b.k.nouter = a.k_outer;
  b.m_tiles = column_tiles(a.m.nbins, TX, a.m_outer);
  b.ntiles = b.m_tiles + (a.k_outer > 0 ? column_tiles(a.k.nbins, TX, a.k_outer) : 0);
  return b;
}

template <int L, int WANT, bool REV = false>
bool sk_launch_col(const Col2& a, int dir, hipStream_t st) {
  if (REV && PlanOf<L, false>::S < 2) return false;  // one stage: same as forward order
  constexpr int TF = col_fit<L, WANT, -1>(), TI = col_fit<L, WANT, +1>();
  constexpr int T = threads_per_transform<L>();
  if (dir < 0) {
    const Col2 b = col2_tiles<L, TF>(a);
    hipLaunchKernelGGL((sk_col<L, TF, -1, REV>), dim3((unsigned)b.ntiles), dim3(TF * T), 0, st, b);
  } else {
    const Col2 b = col2_tiles<L, TI>(a);
    hipLaunchKernelGGL((sk_col<L, TI, +1, REV>), dim3((unsigned)b.ntiles), dim3(TI * T), 0, st, b);
  }
  return true;
}

template <int L, int WANT>
bool sk_launch_col_pipe(const Col2& a, int dir, hipStream_t st) {
  constexpr int TX = col_fit<L, WANT, -1>();
  constexpr int threads = TX * threads_per_transform<L>();
  const Col2 b = col2_tiles<L, TX>(a);
  const void* fn = dir < 0 ? (const void*)sk_col_pipe<L, TX, -1> : (const void*)sk_col_pipe<L, TX, +1>;
  long grid = persistent_blocks(fn, threads);
  if (grid > b.ntiles) grid = b.ntiles;
  if (grid < 1) grid = 1;
  if (dir < 0)
    hipLaunchKernelGGL((sk_col_pipe<L, TX, -1>), dim3((unsigned)grid), dim3(threads), 0, st, b);
  else
    hipLaunchKernelGGL((sk_col_pipe<L, TX, +1>), dim3((unsigned)grid), dim3(threads), 0, st, b);
  return true;
}

template <int L, int WANT>
bool sk_launch_zfused_fft(const ZArgs& a, long ny, hipStream_t st) {
  constexpr int TX = z_fit<L, WANT>();
  ZArgs b = a;
  b.ny = ny;
  const dim3 grid((unsigned)column_tiles(a.nbins, TX, ny)), block(TX * z_threads<L, 0>());
  const dim3 cut(TX * z_threads<L, 0, 1>());
  if constexpr (PlanOf<z_id<L>(), false>::S == 2) {
    if (zfused_sparse_ok<L>(a.nvalid)) {
      hipLaunchKernelGGL((sk_zfused_fft<L, TX, 1>), grid, dim3(TX * z_threads<L, 1>()), 0, st, b);
      return true;
    }
  }
  if constexpr (WANT == 16) {
    constexpr int ID = z_full_id<L>();
    const int n = a.out_planes > 0 ? 0 : kernel_prune<ID>(a.nvalid, a.center);
    if (n == 1) {
      hipLaunchKernelGGL((sk_zfused_fft<L, TX, 0, kernel_slots<ID>(1)>), grid, cut, 0, st, b);
      return true;
    }
    if (n == 2) {
      hipLaunchKernelGGL((sk_zfused_fft<L, TX, 0, kernel_slots<ID>(2)>), grid, cut, 0, st, b);
      return true;
    }
  }
  hipLaunchKernelGGL((sk_zfused_fft<L, TX, 0>), grid, block, 0, st, b);
  return true;
}

// launchers over an extended image
template <int L>
void sk_launch_xfwd_ext(const XExtArgs& a, hipStream_t st) {
  constexpr int P = flat_fill_pairs<L>();
  XExtArgs b = a;
  b.groups = (a.ny + 2 * P - 1) / (2 * P);
  b.k_blocks = ((a.k.nrows + 1) / 2 + P - 1) / P;
  hipLaunchKernelGGL((sk_xfwd_ext<L, P>), dim3((unsigned)(b.groups * a.nplanes + b.k_blocks)),
                     dim3(P * threads_per_transform<L>()), 0, st, b);
}
template <int L>
void sk_launch_xinv_ext(const XExtArgs& a, hipStream_t st) {
  constexpr int P = flat_fill_pairs<L>();
  XExtArgs b = a;
  b.groups = (a.ny + 2 * P - 1) / (2 * P);
  hipLaunchKernelGGL((sk_xinv_ext<L, P>), dim3((unsigned)(b.groups * a.nplanes)),
                     dim3(P * threads_per_transform<L>()), 0, st, b);
}
template <int L>
void sk_launch_col_ext(const ColExtArgs& a, int dir, hipStream_t st) {
  constexpr int TF = col_fit<L, 16, -1>(), TI = col_fit<L, 16, +1>();
  constexpr int T = threads_per_transform<L>();
  ColExtArgs b = a;
  if (dir < 0) {
    b.c = col2_tiles<L, TF>(a.c);
    hipLaunchKernelGGL((sk_col_ext<L, TF, -1>), dim3((unsigned)b.c.ntiles), dim3(TF * T), 0, st, b);
  } else {
    b.c = col2_tiles<L, TI>(a.c);
    hipLaunchKernelGGL((sk_col_ext<L, TI, +1>), dim3((unsigned)b.c.ntiles), dim3(TI * T), 0, st, b);
  }
}
template <int L>
void sk_launch_zfused_ext(const ZExtArgs& a, long ny, hipStream_t st) {
  constexpr int TX = z_fit<L, 16>();
  ZExtArgs b = a;
  b.z.ny = ny;
  const dim3 grid((unsigned)column_tiles(a.z.nbins, TX, ny)), block(TX * z_threads<L, 0>());
  const dim3 cut(TX * z_threads<L, 0, 1>());
  if constexpr (PlanOf<z_id<L>(), false>::S == 2) {
    if (zfused_sparse_ok<L>(a.z.nvalid)) {
      hipLaunchKernelGGL((sk_zfused_ext<L, TX, 1>), grid, dim3(TX * z_threads<L, 1>()), 0, st, b);
      return;
    }
  }
  constexpr int ID = z_full_id<L>();
  const int n = kernel_prune<ID>(a.z.nvalid, a.z.center);
  if (n == 1)
    hipLaunchKernelGGL((sk_zfused_ext<L, TX, 0, kernel_slots<ID>(1)>), grid, cut, 0, st, b);
  else if (n == 2)
    hipLaunchKernelGGL((sk_zfused_ext<L, TX, 0, kernel_slots<ID>(2)>), grid, cut, 0, st, b);
  else
    hipLaunchKernelGGL((sk_zfused_ext<L, TX, 0>), grid, block, 0, st, b);
}

template <int L>
void sk_launch_zcorr_ext(const ZCorrArgs& a, long ny, hipStream_t st) {
  constexpr int TX = z_fit<L, 16>();
  ZCorrArgs b = a;
  b.z.ny = ny;
  hipLaunchKernelGGL((sk_zcorr_ext<L, TX>), dim3((unsigned)column_tiles(a.z.nbins, TX, ny)),
                     dim3(TX * z_threads<L, 0>()), 0, st, b);
}

// direct kernel DFT costs kz complex MACs per output; use it while that is
// cheaper than a transform of the mostly-zero kernel column
template <int L>
constexpr int dft_kz_limit() {
  return L / 4 > 64 ? 64 : L / 4;
}

template <int L, int WANT>
bool sk_launch_zfused_dft(const ZArgs& a, long ny, hipStream_t st) {
  if (a.nvalid > dft_kz_limit<L>()) return false;
  constexpr int TX = z_fit<L, WANT>();
  ZArgs b = a;
  b.ny = ny;
  hipLaunchKernelGGL((sk_zfused_dft<L, TX>), dim3((unsigned)column_tiles(a.nbins, TX, ny)),
                     dim3(TX * z_threads<L, 0, 1>()), 0, st, b);
  return true;
}

// batched launches over device task tables (default variants)
template <int L>
void sb_launch_xfwd(const XPassArgs* args, const int2* tasks, int ntasks, hipStream_t st) {
  constexpr int P = batch_pairs<L>();
  hipLaunchKernelGGL((sb_xfwd<L, P>), dim3((unsigned)ntasks), dim3(P * threads_per_transform<L>()),
                     0, st, args, tasks);
}
template <int L>
void sb_launch_xinv(const XPassArgs* args, const int2* tasks, int ntasks, hipStream_t st) {
  constexpr int P = batch_pairs<L>();
  hipLaunchKernelGGL((sb_xinv<L, P>), dim3((unsigned)ntasks), dim3(P * threads_per_transform<L>()),
                     0, st, args, tasks);
}
template <int L>
void sb_launch_col(const ColArgs* args, const int2* tasks, int ntasks, int dir, hipStream_t st) {
  constexpr int TX = fit_tile<L, 16>();
  const dim3 block(TX * threads_per_transform<L>());
  if (dir < 0)
    hipLaunchKernelGGL((sb_col<L, TX, -1>), dim3((unsigned)ntasks), block, 0, st, args, tasks);
  else
    hipLaunchKernelGGL((sb_col<L, TX, +1>), dim3((unsigned)ntasks), block, 0, st, args, tasks);
}
template <int L>
void sb_launch_zfused(const ZArgs* args, const int2* tasks, int ntasks, hipStream_t st) {
  constexpr int TX = fit_tile<L, 16>();
  hipLaunchKernelGGL((sb_zfused<L, TX, 0>), dim3((unsigned)ntasks),
                     dim3(TX * z_threads<L, 0>()), 0, st, args, tasks);
}
template <int L>
void sb_launch_zfused_sparse(const ZArgs* args, const int2* tasks, int ntasks, hipStream_t st) {
  constexpr int TX = fit_tile<L, 16>();
  if constexpr (PlanOf<z_id<L>(), false>::S == 2)
    hipLaunchKernelGGL((sb_zfused<L, TX, 1>), dim3((unsigned)ntasks),
                       dim3(TX * z_threads<L, 1>()), 0, st, args, tasks);
}

template <int L>
StaticEntry make_static_entry() {
  StaticEntry e;
  e.xfwd = {{"w256", &sk_launch_xfwd<L, 256>},
            {"w128", &sk_launch_xfwd<L, 128>},
            {"w64", &sk_launch_xfwd<L, 64>},
            {"w256-flat", &sk_launch_xfwd_flat<L, 256>},
            {"w128-flat", &sk_launch_xfwd_flat<L, 128>}};
  e.xinv = {{"w256", &sk_launch_xinv<L, 256>},
            {"w128", &sk_launch_xinv<L, 128>},
            {"w64", &sk_launch_xinv<L, 64>},
            {"w256-ldsmirror", &sk_launch_xinv_lds<L, 256>},
            {"w256-flat", &sk_launch_xinv_flat<L, 256>},
            {"w128-flat", &sk_launch_xinv_flat<L, 128>}};
  e.col = {{"t16", &sk_launch_col<L, 16>, col_fit<L, 16, +1>()},
           {"t16-pipe", &sk_launch_col_pipe<L, 16>},
           {"t8-pipe", &sk_launch_col_pipe<L, 8>},
           {"t16-revradix", &sk_launch_col<L, 16, true>},
           {"t8", &sk_launch_col<L, 8>, col_fit<L, 8, +1>()},
           {"t32", &sk_launch_col<L, 32>, col_fit<L, 32, +1>()},
           {"t64", &sk_launch_col<L, 64>, col_fit<L, 64, +1>()}};
  e.zfused = {{"t16-fft", &sk_launch_zfused_fft<L, 16>},
              {"t16-dft", &sk_launch_zfused_dft<L, 16>},
              {"t8-fft", &sk_launch_zfused_fft<L, 8>},
              {"t32-fft", &sk_launch_zfused_fft<L, 32>},
              {"t64-fft", &sk_launch_zfused_fft<L, 64>}};
  // defaults: the flat forms at about 128 threads (measured over L x 300 x 96
  // volumes: x forward at 384 23.0 us w256, 21.2 w256-flat, 20.4 w128-flat;
  // at 1024 53.8, 47.7, 46.4; x inverse at 384 21.3, 20.6, 19.5; at 128 to 216
  // w64 is 0.3 to 0.7 us of 15 faster forward)
  auto index_of = [](const auto& vs, const char* name) {
    for (size_t i = 0; i < vs.size(); ++i)
      if (__builtin_strcmp(vs[i].name, name) == 0) return (int)i;
    return 0;
  };
  e.selected[kSxInv] = index_of(e.xinv, "w128-flat");
  e.selected[kSxFwd] = index_of(e.xfwd, "w128-flat");
  e.xfwd_vpad = &sk_launch_xfwd_vpad<L, 64>;
  e.xinv_crop = &sk_launch_xinv_crop_flat<L, 256>;  // 171 vs 193 us at 600 x 600 x 288
  e.ext.xfwd = &sk_launch_xfwd_ext<L>;
  e.ext.xinv = &sk_launch_xinv_ext<L>;
  e.ext.col = &sk_launch_col_ext<L>;
  e.ext.zfused = &sk_launch_zfused_ext<L>;
  e.ext.zcorr = &sk_launch_zcorr_ext<L>;
  e.batch.pairs = batch_pairs<L>();
  e.batch.tx = fit_tile<L, 16>();
  e.batch.xfwd = &sb_launch_xfwd<L>;
  e.batch.xinv = &sb_launch_xinv<L>;
  e.batch.col = &sb_launch_col<L>;
  e.batch.zfused = &sb_launch_zfused<L>;
  if constexpr (PlanOf<z_id<L>(), false>::S == 2) {
    e.batch.zfused_sparse = &sb_launch_zfused_sparse<L>;
    e.batch.sparse_kz = PlanOf<z_id<L>(), false>::R(1);
  }
  return e;
}

}  // namespace fcamd
