// Spectral passes fused into FFT passes (gfx950).
//
// The reference applies every k-space multiplier and every real-space
// screening factor as a separate sweep over FP64 meshes between FFTW calls
// (src/mg.h:21-309, src/auxPM.c:450-535).  Here each multiplier rides on the
// FFT pass that touches the same data, so no mesh is read or written only to
// be scaled:
//   green x pass (inverse)   S = delta(k) [+ phi(k)] times the Green's function
//                            or smoothing window, then the x transform; the
//                            force variant writes two transforms, of i n_x G
//                            and of G (the y and z components share G);
//   dual y pass (inverse)    y transform of T and of i n_y T from one read;
//   z screen pass            c2r of the potential (or smoothed density) row,
//                            the real-space screening against the delta(x)
//                            row, and the r2c of the effective density row, in
//                            one kernel, the row handed on in registers;
//   epilogue x pass (fwd)    x transform followed by coupling n^2/(n^2 + m^2);
//   z c2r with i n_z         (fft.hip) the z force component.
// Integer wavenumbers follow the Forces convention n in (-N/2, N/2] (the
// Nyquist index counts as +N/2, src/auxPM.c:467-479); only n^2 enters the
// MG and smoothing multipliers, where the sign convention does not matter.
#include "fft_core.h"

#include <cmath>

namespace {

using namespace fftc;

// Stores of the dual y pass and of the x pass pairs: past the caches from 384 on, where a
// mesh is larger than they keep until the next pass reads it, and with full 128-byte lines
// (16 columns; half lines, as the 8 columns of the force pairs write, cost more than they
// gain).  Dual y pass / density pair: 146 / 165 -> 137 / 143 us at 384, 1.38 / 1.93 -> 1.20 /
// 1.80 ms at 768, 2.84 / 4.19 -> 2.80 / 4.15 ms at 1024; up to 256 the next pass finds the
// meshes in the caches.
template <int L, int T>
__device__ __forceinline__ void put(float2 &p, float2 v) {
  if constexpr (L >= 384 && T == 16) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    __builtin_nontemporal_store(f2{v.x, v.y}, reinterpret_cast<f2 *>(&p));
  } else {
    p = v;
  }
}

__device__ __forceinline__ int nsgn(int i, int N) { return i > N / 2 ? i - N : i; }

enum { GREEN_FORCE = FUSED_GREEN_FORCE, GREEN_LAPLACE = FUSED_GREEN_LAPLACE, GREEN_SMOOTH = FUSED_GREEN_SMOOTH };
struct GreenArgs {
  float cnorm;  // GREEN_FORCE: 1 / (N^3 2 pi / Box)
  float nf;     // GREEN_LAPLACE: 1.5 Omega / a (Box / (2 pi c/H0))^2 / N^3; GREEN_SMOOTH: 1 / N^3
  float kfac;   // GREEN_SMOOTH: 2 pi R / Box
  int filter;   // GREEN_SMOOTH: MGPU_FILTER_*
  const float *mult = nullptr;  // GREEN_FORCE: learned multiplier per n^2, or none
};

__device__ __forceinline__ float window(int filter, float kR) {
  switch (filter) {
    case MGPU_FILTER_GAUSSIAN: return expf(-0.5f * kR * kR);
    case MGPU_FILTER_TOPHAT: return kR < 1e-5f ? 1.f : 3.f / (kR * kR * kR) * (sinf(kR) - kR * cosf(kR));
    case MGPU_FILTER_SHARPK: return kR < 1.f ? 1.f : 0.f;
    default: return 1.f;
  }
}

// The x pass's Green's / smoothing multiplier of S at (n_x, n^2), valid = the
// column is a stored mode (kz <= N/2): o1 = G (or i n_x G for GREEN_FORCE,
// o2 = G), G = f S.
template <int MODE>
__device__ __forceinline__ void green_mul(float2 S, int nx, int n2, bool valid, const GreenArgs &ga, float2 &o1,
                                          float2 &o2) {
  float f = 0.f;
  if (valid) {
    if (MODE == GREEN_FORCE) {
      f = n2 > 0 ? -ga.cnorm / (float)n2 : 0.f;
      if (ga.mult) f *= ga.mult[n2];
    }
    if (MODE == GREEN_LAPLACE) f = n2 > 0 ? -ga.nf / (float)n2 : 0.f;
    if (MODE == GREEN_SMOOTH) f = window(ga.filter, sqrtf((float)n2) * ga.kfac) * ga.nf;
  }
  const float2 G = cscale(S, f);
  if (MODE == GREEN_FORCE) {
    o1 = cscale(mul_i<+1>(G), (float)nx);
    o2 = G;
  } else {
    o1 = G;
  }
}

// x pass, inverse.  Tile (bx, by) of xcd_tile: columns kz = bx*T + c, outer index ky = by,
// line index kx.  out1 is written by GREEN_FORCE only.
template <int L, int T, int MODE>
__global__ __launch_bounds__(col_threads(L, T)) void k_col_green(const float2 *__restrict__ a,
                                                                   const float2 *__restrict__ b, float2 *out0,
                                                                   float2 *out1, size_t ls, size_t os,
                                                                   const float2 *__restrict__ tw, GreenArgs ga) {
  extern __shared__ float2 lds[];
  constexpr int NT = col_threads(L, T), E = col_ept(L, T);
  constexpr int R0 = pick_radix(L, E), NB0 = E / R0, M0 = L / R0;
  constexpr int N = L;
  const int tid = threadIdx.x;
  int bx, ky;
  xcd_tile(bx, ky);
  const int kz0 = bx * T;
  const size_t tile = (size_t)ky * os + kz0;
  StageTwiddles<L, T, NT> stw(tw, tid);
  float2 p1[E], p2[E];
#pragma unroll
  for (int q = 0; q < NB0; ++q) {
    const int g = tid + q * NT, c = g % T, j = g / T;
#pragma unroll
    for (int r = 0; r < R0; ++r) {
      float2 v = col_at<L, T>(a + tile, ls, c, j, r * M0);
      if (b) v = cadd(v, col_at<L, T>(b + tile, ls, c, j, r * M0));
      p1[q * R0 + r] = v;
    }
  }
  const int ny = nsgn(ky, N);
#pragma unroll
  for (int q = 0; q < NB0; ++q) {
    const int g = tid + q * NT, c = g % T, j = g / T;
    const int kz = kz0 + c;
#pragma unroll
    for (int r = 0; r < R0; ++r) {
      const int nx = nsgn(j + r * M0, N);
      const int n2 = nx * nx + ny * ny + kz * kz;
      green_mul<MODE>(p1[q * R0 + r], nx, n2, kz <= N / 2, ga, p1[q * R0 + r], p2[q * R0 + r]);
    }
  }
  auto ld = [&](int, int, int) { return make_float2(0.f, 0.f); };
  auto st0 = [&](int c, int j, int o, float2 v) { col_at<L, T>(out0 + tile, ls, c, j, o) = v; };
  const float2 *twl = stw.to_lds(lds, tid);
  fft_stages<L, T, NT, +1, 1, T, true, false, 1, false, true>(lds, twl, 1, tid, ld, st0, p1);
  if (MODE == GREEN_FORCE) {
    __syncthreads();
    auto st1 = [&](int c, int j, int o, float2 v) { col_at<L, T>(out1 + tile, ls, c, j, o) = v; };
    fft_stages<L, T, NT, +1, 1, T, true, false, 1, false, true>(lds, twl, 1, tid, ld, st1, p2);
  }
}

// y pass, inverse, two outputs from one read: buf <- Y[buf], oy <- Y[i n_y buf].
// Tile (bx, by) of xcd_tile: columns kz, outer index kx = by, line index ky.
template <int L, int T>
__global__ __launch_bounds__(col_threads(L, T)) void k_col_dual(float2 *buf, float2 *__restrict__ oy, size_t ls,
                                                                  size_t os, const float2 *__restrict__ tw, size_t zs) {
  buf = zbuf(buf, zs);
  oy = zbuf(oy, zs);
  extern __shared__ float2 lds[];
  constexpr int NT = col_threads(L, T), E = col_ept(L, T);
  constexpr int R0 = pick_radix(L, E), NB0 = E / R0, M0 = L / R0;
  const int tid = threadIdx.x;
  int bx, by;
  xcd_tile(bx, by);
  const size_t tile = (size_t)by * os + (size_t)bx * T;
  StageTwiddles<L, T, NT> stw(tw, tid);
  float2 p1[E], p2[E];
#pragma unroll
  for (int q = 0; q < NB0; ++q) {
    const int g = tid + q * NT, c = g % T, j = g / T;
#pragma unroll
    for (int r = 0; r < R0; ++r) {
      const float2 v = col_at<L, T>((const float2 *)buf + tile, ls, c, j, r * M0);
      p2[q * R0 + r] = v;
      p1[q * R0 + r] = cscale(mul_i<+1>(v), (float)nsgn(j + r * M0, L));
    }
  }
  auto ld = [&](int, int, int) { return make_float2(0.f, 0.f); };
  auto st0 = [&](int c, int j, int o, float2 v) { put<L, T>(col_at<L, T>(oy + tile, ls, c, j, o), v); };
  const float2 *twl = stw.to_lds(lds, tid);
  fft_stages<L, T, NT, +1, 1, T, true, false, 1, false, true>(lds, twl, 1, tid, ld, st0, p1);
  __syncthreads();
  auto st1 = [&](int c, int j, int o, float2 v) { put<L, T>(col_at<L, T>(buf + tile, ls, c, j, o), v); };
  fft_stages<L, T, NT, +1, 1, T, true, false, 1, false, true>(lds, twl, 1, tid, ld, st1, p2);
}

// The y passes of the force tail in one launch, for meshes whose launches are short:
// even rows of the grid take k_col_dual's tiles, odd rows the inverse y pass of other.
// Each row of the grid is one kx (see k_col_dual).
constexpr int kForceYOne = 256;
template <int L, int T>
__global__ __launch_bounds__(col_threads(L, T)) void k_col_force_y(float2 *buf, float2 *__restrict__ oy, float2 *other,
                                                                     size_t ls, size_t os,
                                                                     const float2 *__restrict__ tw, size_t zs) {
  buf = zbuf(buf, zs);
  oy = zbuf(oy, zs);
  other = zbuf(other, zs);
  extern __shared__ float2 lds[];
  constexpr int NT = col_threads(L, T), E = col_ept(L, T);
  constexpr int R0 = pick_radix(L, E), NB0 = E / R0, M0 = L / R0;
  const int tid = threadIdx.x;
  int bx, by;
  xcd_tile(bx, by);
  const bool dual = (by & 1) == 0;  // the same for the whole workgroup
  const size_t tile = (size_t)(by >> 1) * os + (size_t)bx * T;
  const float2 *src = dual ? buf : other;
  StageTwiddles<L, T, NT> stw(tw, tid);
  float2 p1[E], p2[E];
  first_loads<L, T, NT, true>(p2, tid, [&](int c, int j, int o) { return col_at<L, T>(src + tile, ls, c, j, o); });
  const float2 *twl = stw.to_lds(lds, tid);
  auto ld = [&](int, int, int) { return make_float2(0.f, 0.f); };
  if (dual) {
#pragma unroll
    for (int q = 0; q < NB0; ++q) {
      const int j = (tid + q * NT) / T;
#pragma unroll
      for (int r = 0; r < R0; ++r)
        p1[q * R0 + r] = cscale(mul_i<+1>(p2[q * R0 + r]), (float)nsgn(j + r * M0, L));
    }
    auto st0 = [&](int c, int j, int o, float2 v) { col_at<L, T>(oy + tile, ls, c, j, o) = v; };
    fft_stages<L, T, NT, +1, 1, T, true, false, 1, false, true>(lds, twl, 1, tid, ld, st0, p1);
    __syncthreads();
  }
  float2 *dst = dual ? buf : other;
  auto st1 = [&](int c, int j, int o, float2 v) { col_at<L, T>(dst + tile, ls, c, j, o) = v; };
  fft_stages<L, T, NT, +1, 1, T, true, false, 1, false, true>(lds, twl, 1, tid, ld, st1, p2);
}

// x pass, forward, then phi = coupling n^2/(n^2 + m2) X (0 at n = 0): EffDensitykToPhiofk
// (src/mg.h:74-116) on the transform's output.  Tile: columns kz, outer ky, line kx.
template <int L, int T>
__global__ __launch_bounds__(col_threads(L, T)) void k_col_epi(float2 *buf, size_t ls, size_t os,
                                                                 const float2 *__restrict__ tw, float coupling,
                                                                 float m2) {
  extern __shared__ float2 lds[];
  constexpr int NT = col_threads(L, T);
  constexpr int N = L;
  const int tid = threadIdx.x;
  int bx, ky;
  xcd_tile(bx, ky);
  const int kz0 = bx * T;
  const size_t tile = (size_t)ky * os + kz0;
  const int ny = nsgn(ky, N);
  auto ld = [&](int c, int j, int o) { return col_at<L, T>((const float2 *)buf + tile, ls, c, j, o); };
  auto st = [&](int c, int j, int o, float2 v) {
    const int kz = kz0 + c, nx = nsgn(j + o, N);
    const int n2 = nx * nx + ny * ny + kz * kz;
    const float f = (kz <= N / 2 && n2 > 0) ? coupling * ((float)n2 / ((float)n2 + m2)) : 0.f;
    col_at<L, T>(buf + tile, ls, c, j, o) = cscale(v, f);
  };
  StageTwiddles<L, T, NT> stw(tw, tid);
  float2 pre[col_ept(L, T)];
  first_loads<L, T, NT, true>(pre, tid, ld);
  const float2 *twl = stw.to_lds(lds, tid);
  fft_stages<L, T, NT, -1, 1, T, true, false, 1, false, true>(lds, twl, 1, tid, ld, st, pre);
}

// P(k) sums of an x pass in LDS: copies sets of bin sums (lanes take them in turn, so
// fewer lanes of a wave add to one address: most of a wave's modes share a few bins),
// the per-axis window and, with EDGES, the bin edges (see fused_pofk_by).  init() goes
// behind the tile's loads, so that it costs no latency of its own, and in front of the
// twiddles' barrier (without one, a barrier of its own or the stages' barriers).
template <int L, int NT, bool EDGES>
struct PofkLds {
  double *bins;
  float *wv;
  int *edge;
  int e0, e1;
  __device__ __forceinline__ void init(void *lds, const PkBinFn &f, int copies, const float *__restrict__ winv,
                                       int tid) {
    bins = (double *)lds;
    wv = (float *)(bins + copies * f.nbins);
    edge = (int *)(wv + L / 2 + 1);
    for (int b = tid; b < copies * f.nbins; b += NT) bins[b] = 0.0;
    for (int d = tid; d <= L / 2; d += NT) wv[d] = winv[d];
    if (EDGES)
      for (int b = tid; b <= f.nbins; b += NT) edge[b] = f.edge[b];
  }
  // after a barrier
  __device__ __forceinline__ void begin(const PkBinFn &f) {
    if (!EDGES) return;
    e0 = edge[0];
    e1 = edge[f.nbins];
  }
  // mode (kx, d1 = |ky|, kz) of power |v|^2: weight 1 (kz = 0, N/2) or 2, CIC deconvolution
  __device__ __forceinline__ void add(float2 v, int kx, int d1, int kz, const PkBinFn &f, int copies, int tid) const {
    if (kz > L / 2) return;
    const int d0 = kx > L / 2 ? L - kx : kx, n2 = d0 * d0 + d1 * d1 + kz * kz;
    const int nk = EDGES ? pk_bin_of(n2, f, edge, e0, e1) : f.table[n2];
    if (nk < 0) return;
    const float w = (kz == 0 || kz == L / 2) ? 1.f : 2.f;
    atomicAdd(&bins[EDGES ? nk + f.nbins * (tid & (copies - 1)) : nk],
              (double)((v.x * v.x + v.y * v.y) * (w * wv[d0] * wv[d1] * wv[kz])));
  }
  // into the workgroup's set of MGPU_PK_SETS global sums (adds to one address are
  // serialised: with one set the 1344 workgroups of a 192 mesh cost 18 us)
  __device__ __forceinline__ void flush(double *__restrict__ pk, const PkBinFn &f, int copies, int tid) const {
    pk += ((blockIdx.x + blockIdx.y * gridDim.x) % MGPU_PK_SETS) * f.nbins;
    for (int b = tid; b < f.nbins; b += NT) {
      double s = bins[b];
      for (int c = 1; c < copies; ++c) s += bins[b + c * f.nbins];
      if (s != 0.0) atomicAdd(&pk[b], s);
    }
  }
};

// x pass, forward, accumulating compute_power_spectrum's binned power
// (src/compute_pofk.c:71-236) from the transform's output as it is stored:
// weight 1 (kz = 0, N/2) or 2, CIC deconvolution winv[d0] winv[d1] winv[d2]
// (1/N^6 folded in), |n| binned linearly (bintype 0) or logarithmically.
// Bin sums go to LDS doubles, then one global atomic per bin and block.
template <int L, int T, bool EDGES>
__global__ __launch_bounds__(col_threads(L, T)) void k_col_pofk(float2 *buf, size_t ls, size_t os,
                                                                  const float2 *__restrict__ tw,
                                                                  const float *__restrict__ winv, PkBinFn fn,
                                                                  int copies, double *__restrict__ pk) {
  extern __shared__ float2 lds[];
  constexpr int NT = col_threads(L, T);
  constexpr int N = L;
  const int tid = threadIdx.x;
  PofkLds<L, NT, EDGES> pl;
  int bx, ky;
  xcd_tile(bx, ky);
  const int kz0 = bx * T;
  const size_t tile = (size_t)ky * os + kz0;
  const int d1 = ky > N / 2 ? N - ky : ky;
  auto ld = [&](int c, int j, int o) { return col_at<L, T>((const float2 *)buf + tile, ls, c, j, o); };
  auto st = [&](int c, int j, int o, float2 v) {
    col_at<L, T>(buf + tile, ls, c, j, o) = v;
    pl.add(v, j + o, d1, kz0 + c, fn, copies, tid);
  };
  StageTwiddles<L, T, NT, EDGES && tw_in_lds(L)> stw(tw, tid);
  float2 pre[col_ept(L, T)];
  first_loads<L, T, NT, true>(pre, tid, ld);
  pl.init(lds + (EDGES ? col_lds_elems(L, T) : (size_t)L * T), fn, copies, winv, tid);
  if (!EDGES) __syncthreads();  // up to 16 points the only stage adds to the sums
  const float2 *twl = stw.to_lds(lds, tid);
  fft_stages<L, T, NT, -1, 1, T, true, false, 1, false, true>(lds, twl, 1, tid, ld, st, pre, [&]() { pl.begin(fn); });
  __syncthreads();
  pl.flush(pk, fn, copies, tid);
}

// x pass pair: a forward x transform and, from its output, an inverse x
// transform with a Green's / smoothing multiplier, so the spectrum between
// them is never written and read back.
//   FWD_DENSITY  the density's forward x pass: delta(k) stored to kout (when
//                not null) and its power binned into pk (when not null) as
//                k_col_pofk does; S = delta(k).
//   FWD_EPI      forward x pass of the screened effective density, the
//                EffDensitykToPhiofk epilogue (as k_col_epi), S = delta(k) + phi(k)
//                with delta(k) read from dk (as k_col_green adds them).
//   FWD_PLAIN    the same without the epilogue (DGP: phi(k) is the transform).
// Then S times the MODE multiplier and the inverse x transform(s), as
// k_col_green.  The forward's outputs reach the inverse in registers or through LDS
// (see kHand).
// What bounds it: with one workgroup per CU its load, transform and store phases add
// up.  At most 128 VGPRs (four waves per SIMD, two 512-thread workgroups per CU at
// 1024) let one tile's loads and stores run under another's transforms; the stage
// twiddles in LDS free the registers and the vector-memory queue for that.  Force
// pair 6.45 -> 4.55 ms at 1024 (2.7 -> 3.8 TB/s), 316 -> 239 us at 384; density pair
// with P(k) 4.81 -> 4.19 ms at 1024, with the Green's force (LCDM) 7.2 -> 5.2 ms.
enum { FWD_DENSITY = 0, FWD_EPI = 1, FWD_PLAIN = 2 };
template <int L, int T, int FWD, int MODE, bool EDGES = true>
__global__ __launch_bounds__(col_threads(L, T), tw_in_lds(L) && EDGES ? 4 : 1) void k_col_fused(
    const float2 *in, float2 *kout, const float2 *__restrict__ dk, float2 *out0, float2 *out1, size_t ls, size_t os,
    const float2 *__restrict__ tw, GreenArgs ga, float coupling, float m2, const float *__restrict__ winv,
    PkBinFn fn, int copies, double *__restrict__ pk, size_t zs) {
  in = zbuf(in, zs);
  kout = zbuf(kout, zs);
  dk = zbuf(dk, zs);
  out0 = zbuf(out0, zs);
  out1 = zbuf(out1, zs);
  pk = zbuf(pk, zs);
  extern __shared__ float2 lds[];
  constexpr int NT = col_threads(L, T), E = col_ept(L, T);
  // The forward's outputs are handed to the inverse in registers (its stages reversed);
  // with delta(k) to add at 16 elements per thread those registers spill (1024: 4.94
  // against 4.69 ms, 256: 96 against 82 us), and the outputs go through LDS instead.  24
  // elements have twice the registers, and it is the way through LDS that spills (68 and
  // more of them; 1536: 24.4 against 32.1 ms).
  constexpr bool kHand = FWD == FWD_DENSITY || E != 16;
  constexpr int RX = stage_radix(L, E, 1, kHand), MX = L / RX;  // the inverse's first stage
  constexpr int N = L;
  const int tid = threadIdx.x;
  int bx, ky;
  xcd_tile(bx, ky);
  const int kz0 = bx * T;
  const size_t tile = (size_t)ky * os + kz0;
  const int ny = nsgn(ky, N), d1 = ky > N / 2 ? N - ky : ky;
  const bool bin = FWD == FWD_DENSITY && pk != nullptr;
  PofkLds<L, NT, EDGES> pl;
  // forward transform; its outputs stay in the registers of the threads that form them
  float2 p1[E], p2[E];
  auto ld = [&](int c, int j, int o) { return col_at<L, T>(in + tile, ls, c, j, o); };
  int oi = 0;  // output index of the store (a constant of the unrolled last stage)
  auto st = [&](int c, int j, int o, float2 v) {
    const int kx = j + o, kz = kz0 + c;
    if (FWD == FWD_DENSITY) {
      if (kout) put<L, T>(col_at<L, T>(kout + tile, ls, c, j, o), v);
      if (bin) pl.add(v, kx, d1, kz, fn, copies, tid);
    }
    if (FWD == FWD_EPI) {
      const int nx = nsgn(kx, N), n2 = nx * nx + ny * ny + kz * kz;
      const float f = (kz <= N / 2 && n2 > 0) ? coupling * ((float)n2 / ((float)n2 + m2)) : 0.f;
      v = cscale(v, f);
    }
    if constexpr (kHand) p1[oi++] = v;
    else lds[c + kx * T] = v;
  };
  StageTwiddles<L, T, NT, EDGES && tw_in_lds(L)> stw(tw, tid);
  first_loads<L, T, NT, true>(p1, tid, ld);
  if (bin) pl.init(lds + (EDGES ? col_lds_elems(L, T) : (size_t)L * T), fn, copies, winv, tid);
  if (!EDGES) __syncthreads();  // as in k_col_pofk
  const float2 *twl = stw.to_lds(lds, tid);
  // delta(k) to add, in the layout of the inverse's first stage: requested before the
  // forward's last stage, or after it where the registers are short
  auto ldk = [&](int c, int j, int o) { return col_at<L, T>(dk + tile, ls, c, j, o); };
  auto hook = [&]() {
    if constexpr (FWD != FWD_DENSITY && kHand) first_loads<L, T, NT, true, kHand>(p2, tid, ldk);
    if (bin) pl.begin(fn);
  };
  fft_stages<L, T, NT, -1, 1, T, true, false, 1, !kHand, true>(lds, twl, 1, tid, ld, st, p1, hook);
  if constexpr (!kHand) {
    first_loads<L, T, NT, true, kHand>(p2, tid, ldk);
    __syncthreads();
    first_loads<L, T, NT, true, kHand>(p1, tid, [&](int c, int j, int o) { return lds[c + (j + o) * T]; });
  }
#pragma unroll
  for (int q = 0; q < E / RX; ++q) {
    const int g = tid + q * NT, c = g % T, j = g / T;
    const int kz = kz0 + c;
#pragma unroll
    for (int r = 0; r < RX; ++r) {
      const int i = q * RX + r, nx = nsgn(j + r * MX, N);
      const int n2 = nx * nx + ny * ny + kz * kz;
      const float2 S = FWD == FWD_DENSITY ? p1[i] : cadd(p2[i], p1[i]);
      green_mul<MODE>(S, nx, n2, kz <= N / 2, ga, p1[i], p2[i]);
    }
  }
  auto ldz = [&](int, int, int) { return make_float2(0.f, 0.f); };
  auto st0 = [&](int c, int j, int o, float2 v) { put<L, T>(col_at<L, T>(out0 + tile, ls, c, j, o), v); };
  fft_stages<L, T, NT, +1, 1, T, true, true, 1, false, true, kHand>(lds, twl, 1, tid, ldz, st0, p1);
  if (MODE == GREEN_FORCE) {
    auto st1 = [&](int c, int j, int o, float2 v) { put<L, T>(col_at<L, T>(out1 + tile, ls, c, j, o), v); };
    fft_stages<L, T, NT, +1, 1, T, true, true, 1, false, true, kHand>(lds, twl, 1, tid, ldz, st1, p2);
  }
  if (bin) {
    __syncthreads();
    pl.flush(pk, fn, copies, tid);
  }
}

enum { SCREEN_POTENTIAL = 0, SCREEN_DENSITY = 1 };

// z pass: c2r of the row (potential Phi_N or smoothed density delta_R), the
// screening against the delta(x) row, r2c of the effective density.  The screened row
// goes from the one's last stage to the other's first, of the same radix, in registers:
// 3.53 -> 3.02 ms at 1024 (4.3 TB/s), 213 -> 183 us at 384 with the potential.
//   SCREEN_POTENTIAL (f(R), m-beta; src/mg.h:169-171, src/user_defined_functions.h:725-752):
//       delta_eff = delta * min(1, |p0 / Phi|) where Phi < 0, else delta       (p0 = phi_crit)
//   SCREEN_DENSITY (DGP; src/mg.h:235-244, src/user_defined_functions.h:757-773):
//       delta_eff = delta * p0 * 2 (sqrt(1 + f) - 1) / f, f = p1 (1 + delta_R), 1 if f < 1e-5
//                                                                   (p0 = coupling, p1 = dgp_fac)
// Four waves per SIMD (128 registers) up to 1024; three where the row's last radix is 16
// (512: 12 to 14 registers spilled at four, 473 -> 442 us with the potential, 517 -> 485
// with the density), one beyond, where a row has a workgroup's registers.
template <int N>
constexpr int screen_waves() {
  return N > 1024 ? 1 : last_radix(N / 2, elems_per_thread(N / 2)) == 16 ? 3 : 4;
}
template <int N, int KIND>
__global__ __launch_bounds__(RowCfg<N>::NT, screen_waves<N>()) void k_z_screen(float2 *buf, const float2 *__restrict__ dx, int HP,
                                                             size_t nrows, const float2 *__restrict__ tw, float p0,
                                                             float p1, size_t zs) {
  buf = zbuf(buf, zs);
  dx = zbuf(dx, zs);
  using C = RowCfg<N>;
  constexpr int E = C::M * C::RB / C::NT, RL = last_radix(C::M, E), ML = C::M / RL;
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x;
  const size_t row0 = (size_t)blockIdx.x * C::RB;
  // the delta(x) pairs this thread screens, loaded first so they arrive during the c2r
  float2 dv[E], f[E];
#pragma unroll
  for (int q = 0; q < E / RL; ++q) {
    const int g = tid + q * C::NT, j = g % ML;
    const size_t row = row0 + g / ML < nrows ? row0 + g / ML : nrows - 1;
#pragma unroll
    for (int r = 0; r < RL; ++r) dv[q * RL + r] = dx[row * HP + j + r * ML];
  }
  z_merge<N>(lds, buf, HP, row0, nrows, tw, tid);
  __syncthreads();
  auto ldl = [&](int r, int j, int o) { return lds[r * C::LS + j + o]; };
  auto stl = [&](int r, int j, int o, float2 v) { lds[r * C::LS + j + o] = v; };
  int oi = 0;  // output index of the store (a constant of the unrolled last stage)
  auto sts = [&](int, int, int, float2 v) {
    const float2 d = dv[oi];
    float s0, s1;
    if (KIND == SCREEN_POTENTIAL) {
      s0 = v.x < 0.f ? fminf(1.f, fabsf(p0 / v.x)) : 1.f;
      s1 = v.y < 0.f ? fminf(1.f, fabsf(p0 / v.y)) : 1.f;
    } else {
      const float a0 = p1 * (1.f + v.x), a1 = p1 * (1.f + v.y);
      s0 = p0 * (a0 < 1e-5f ? 1.f : 2.f * (sqrtf(1.f + a0) - 1.f) / a0);
      s1 = p0 * (a1 < 1e-5f ? 1.f : 2.f * (sqrtf(1.f + a1) - 1.f) / a1);
    }
    f[oi++] = make_float2(d.x * s0, d.y * s1);
  };
  fft_stages<C::M, C::RB, C::NT, +1, C::LS, 1, false, true, 1>(lds, tw, 2, tid, ldl, sts);
  float2 w[ZSplit<N>::ITER];
  z_split_twiddles<N>(w, tw, tid);
  fft_stages<C::M, C::RB, C::NT, -1, C::LS, 1, false, true, 1, false, true, true>(lds, tw, 2, tid, ldl, stl, f);
  __syncthreads();
  z_split<N>(lds, w, buf, HP, row0, nrows, tid);
}

template <class K>
int set_lds(mgpu_ctx *ctx, K kern, size_t lds) {
  if (lds > 65536) MGPU_HIP(ctx, hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  return MGPU_OK;
}

template <int N, int T>
int green_launch(mgpu_ctx *ctx, int mode, const float2 *a, const float2 *b, float2 *o0, float2 *o1, GreenArgs ga) {
  const size_t HP = ctx->fft.hp, ls = (size_t)N * HP, os = HP;
  const size_t lds = col_lds_elems(N, T) * sizeof(float2);
  dim3 grid(HP / T, N), block(col_threads(N, T));
  int rc;
  if (mode == GREEN_FORCE) {
    if ((rc = set_lds(ctx, k_col_green<N, T, GREEN_FORCE>, lds))) return rc;
    hipLaunchKernelGGL((k_col_green<N, T, GREEN_FORCE>), grid, block, lds, ctx->stream, a, b, o0, o1, ls, os,
                       ctx->fft.tw, ga);
  } else if (mode == GREEN_LAPLACE) {
    if ((rc = set_lds(ctx, k_col_green<N, T, GREEN_LAPLACE>, lds))) return rc;
    hipLaunchKernelGGL((k_col_green<N, T, GREEN_LAPLACE>), grid, block, lds, ctx->stream, a, b, o0, o1, ls, os,
                       ctx->fft.tw, ga);
  } else {
    if ((rc = set_lds(ctx, k_col_green<N, T, GREEN_SMOOTH>, lds))) return rc;
    hipLaunchKernelGGL((k_col_green<N, T, GREEN_SMOOTH>), grid, block, lds, ctx->stream, a, b, o0, o1, ls, os,
                       ctx->fft.tw, ga);
  }
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

struct FusedXArgs {
  int fwd, mode;
  const float2 *in;
  float2 *kout;
  const float2 *dk;
  float2 *o0, *o1;
  GreenArgs ga;
  float coupling, m2;
  double *pk;
};

// two copies of the P(k) sums where the LDS has room for both (a third and fourth
// gained nothing more)
int pofk_copies(const mgpu_ctx *ctx, size_t tile_lds) {
  const size_t l1 = tile_lds + pofk_lds(ctx->N, ctx->p.pofk_nbins, 1), l2 = tile_lds + pofk_lds(ctx->N, ctx->p.pofk_nbins, 2);
  // not at the price of a workgroup per CU
  return l2 <= ctx->lds_max && (ctx->lds_max / l2 == ctx->lds_max / l1 || ctx->lds_max / l2 >= 4) ? 2 : 1;
}
// LDS of an x pass that bins P(k) by the table: the tile, the bin sums and the window
size_t pofk_table_lds(const mgpu_ctx *ctx, int T) {
  return (size_t)ctx->N * T * sizeof(float2) + sizeof(double) * (size_t)ctx->p.pofk_nbins + sizeof(float) * (size_t)(ctx->N / 2 + 1);
}

template <int N, int T, int FWD, int MODE, bool EDGES>
int fused_x_launch_by(mgpu_ctx *ctx, const FusedXArgs &a, size_t lds, int copies) {
  const size_t HP = ctx->fft.hp, ls = (size_t)N * HP, os = HP;
  int rc;
  auto kern = k_col_fused<N, T, FWD, MODE, EDGES>;
  if ((rc = set_lds(ctx, kern, lds))) return rc;
  hipLaunchKernelGGL(kern, dim3(HP / T, N, ctx->bz), dim3(col_threads(N, T)), lds, ctx->stream, a.in, a.kout, a.dk,
                     a.o0, a.o1, ls, os, ctx->fft.tw, a.ga, a.coupling, a.m2, ctx->winvf, ctx->pk_fn, copies, a.pk,
                     ctx->zs);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}
template <int N, int T, int FWD, int MODE>
int fused_x_launch_k(mgpu_ctx *ctx, const FusedXArgs &a) {
  const size_t tile_lds = col_lds_elems(N, T) * sizeof(float2);
  if (FWD != FWD_DENSITY || !a.pk) return fused_x_launch_by<N, T, FWD, MODE, true>(ctx, a, tile_lds, 1);
  const int by = fused_pofk_by(ctx, T);
  if (by == POFK_NONE) return mgpu_fail(ctx, MGPU_E_INVALID, "P(k) bins do not fit the LDS of the x pass");
  if constexpr (FWD == FWD_DENSITY)
    if (by == POFK_TABLE) return fused_x_launch_by<N, T, FWD, MODE, false>(ctx, a, pofk_table_lds(ctx, T), 1);
  const int copies = pofk_copies(ctx, tile_lds);
  return fused_x_launch_by<N, T, FWD, MODE, true>(ctx, a, tile_lds + pofk_lds(N, ctx->p.pofk_nbins, copies), copies);
}

template <int N, int T>
int fused_x_launch(mgpu_ctx *ctx, const FusedXArgs &a) {
  if (a.fwd == FWD_DENSITY && a.mode == GREEN_LAPLACE) return fused_x_launch_k<N, T, FWD_DENSITY, GREEN_LAPLACE>(ctx, a);
  if (a.fwd == FWD_DENSITY && a.mode == GREEN_SMOOTH) return fused_x_launch_k<N, T, FWD_DENSITY, GREEN_SMOOTH>(ctx, a);
  // the force pair keeps G and i n_x G in registers: only with 8-column tiles
  if constexpr (T == 8) {
    if (a.fwd == FWD_DENSITY && a.mode == GREEN_FORCE) return fused_x_launch_k<N, T, FWD_DENSITY, GREEN_FORCE>(ctx, a);
    if (a.fwd == FWD_EPI && a.mode == GREEN_FORCE) return fused_x_launch_k<N, T, FWD_EPI, GREEN_FORCE>(ctx, a);
    if (a.fwd == FWD_PLAIN && a.mode == GREEN_FORCE) return fused_x_launch_k<N, T, FWD_PLAIN, GREEN_FORCE>(ctx, a);
  }
  return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported fused x pass");
}

template <int N, int T>
int dual_launch(mgpu_ctx *ctx, float2 *buf, float2 *oy) {
  const size_t HP = ctx->fft.hp, ls = HP, os = (size_t)N * HP;
  const size_t lds = col_lds_elems(N, T) * sizeof(float2);
  int rc;
  if ((rc = set_lds(ctx, k_col_dual<N, T>, lds))) return rc;
  hipLaunchKernelGGL((k_col_dual<N, T>), dim3(HP / T, N, ctx->bz), dim3(col_threads(N, T)), lds, ctx->stream, buf, oy,
                     ls, os, ctx->fft.tw, ctx->zs);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

template <int N, int T>
int force_y_launch(mgpu_ctx *ctx, float2 *buf, float2 *oy, float2 *other) {
  const size_t HP = ctx->fft.hp, ls = HP, os = (size_t)N * HP;
  const size_t lds = col_lds_elems(N, T) * sizeof(float2);
  int rc;
  if ((rc = set_lds(ctx, k_col_force_y<N, T>, lds))) return rc;
  hipLaunchKernelGGL((k_col_force_y<N, T>), dim3(HP / T, 2 * N, ctx->bz), dim3(col_threads(N, T)), lds, ctx->stream, buf,
                     oy, other, ls, os, ctx->fft.tw, ctx->zs);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

template <int N, int T>
int epi_launch(mgpu_ctx *ctx, float2 *buf, float coupling, float m2) {
  const size_t HP = ctx->fft.hp, ls = (size_t)N * HP, os = HP;
  const size_t lds = col_lds_elems(N, T) * sizeof(float2);
  int rc;
  if ((rc = set_lds(ctx, k_col_epi<N, T>, lds))) return rc;
  hipLaunchKernelGGL((k_col_epi<N, T>), dim3(HP / T, N), dim3(col_threads(N, T)), lds, ctx->stream, buf, ls, os,
                     ctx->fft.tw, coupling, m2);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

template <int N, int T, bool EDGES>
int pofk_launch_by(mgpu_ctx *ctx, float2 *buf, double *pk, size_t lds, int copies) {
  const size_t HP = ctx->fft.hp, ls = (size_t)N * HP, os = HP;
  int rc;
  if ((rc = set_lds(ctx, k_col_pofk<N, T, EDGES>, lds))) return rc;
  hipLaunchKernelGGL((k_col_pofk<N, T, EDGES>), dim3(HP / T, N), dim3(col_threads(N, T)), lds, ctx->stream, buf, ls, os,
                     ctx->fft.tw, ctx->winvf, ctx->pk_fn, copies, pk);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}
template <int N, int T>
int pofk_launch(mgpu_ctx *ctx, float2 *buf, double *pk) {
  const int by = fused_pofk_by(ctx, T);
  if (by == POFK_NONE) return mgpu_fail(ctx, MGPU_E_INVALID, "P(k) bins do not fit the LDS of the x pass");
  if (by == POFK_TABLE) return pofk_launch_by<N, T, false>(ctx, buf, pk, pofk_table_lds(ctx, T), 1);
  const size_t tile_lds = col_lds_elems(N, T) * sizeof(float2);
  const int copies = pofk_copies(ctx, tile_lds);
  return pofk_launch_by<N, T, true>(ctx, buf, pk, tile_lds + pofk_lds(N, ctx->p.pofk_nbins, copies), copies);
}

template <int N>
int screen_launch(mgpu_ctx *ctx, int kind, float2 *buf, const float2 *dx, float p0, float p1) {
  using C = RowCfg<N>;
  const size_t nrows = (size_t)N * N;
  const size_t lds = (size_t)C::RB * C::LS * sizeof(float2);
  dim3 grid(cdiv(nrows, C::RB), 1, ctx->bz), block(C::NT);
  int rc;
  if (kind == SCREEN_POTENTIAL) {
    if ((rc = set_lds(ctx, k_z_screen<N, SCREEN_POTENTIAL>, lds))) return rc;
    hipLaunchKernelGGL((k_z_screen<N, SCREEN_POTENTIAL>), grid, block, lds, ctx->stream, buf, dx, (int)ctx->fft.hp,
                       nrows, ctx->fft.tw, p0, p1, ctx->zs);
  } else {
    if ((rc = set_lds(ctx, k_z_screen<N, SCREEN_DENSITY>, lds))) return rc;
    hipLaunchKernelGGL((k_z_screen<N, SCREEN_DENSITY>), grid, block, lds, ctx->stream, buf, dx, (int)ctx->fft.hp,
                       nrows, ctx->fft.tw, p0, p1, ctx->zs);
  }
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

// column kernels are instantiated for the tile width the plan chose
template <int N, template <int, int> class F, class... A>
int by_tile(mgpu_ctx *ctx, A... args) {
  if constexpr (col_threads(N, 16) <= 1024) {
    if (ctx->fft.tcols == 16) return F<N, 16>::run(ctx, args...);
  }
  return F<N, 8>::run(ctx, args...);
}
template <int N, int T>
struct GreenF {
  static int run(mgpu_ctx *c, int m, const float2 *a, const float2 *b, float2 *o0, float2 *o1, GreenArgs g) {
    return green_launch<N, T>(c, m, a, b, o0, o1, g);
  }
};
template <int N, int T>
struct DualF {
  static int run(mgpu_ctx *c, float2 *buf, float2 *oy) { return dual_launch<N, T>(c, buf, oy); }
};
template <int N, int T>
struct ForceYF {
  static int run(mgpu_ctx *c, float2 *buf, float2 *oy, float2 *other) { return force_y_launch<N, T>(c, buf, oy, other); }
};
template <int N, int T>
struct PofkF {
  static int run(mgpu_ctx *c, float2 *buf, double *pk) { return pofk_launch<N, T>(c, buf, pk); }
};
template <int N, int T>
struct FusedXF {
  static int run(mgpu_ctx *c, const FusedXArgs &a) { return fused_x_launch<N, T>(c, a); }
};
template <int N, int T>
struct EpiF {
  static int run(mgpu_ctx *c, float2 *buf, float cp, float m2) { return epi_launch<N, T>(c, buf, cp, m2); }
};


}  // namespace

// ---------------------------------------------------------------- host entry points

// The edges' and the twiddles' LDS pays while the edges are at most a sixth of the tile:
// every workgroup copies them, and they cost workgroups per CU.  By the edges / by the
// table: density and P(k) 8.87 / 9.29 ms at 1024 with 16 columns and 1024 bins (a 32nd),
// 661 / 589 us at 384, 16 columns and 2500 bins (a fifth), 1.53 / 1.51 ms at 512, 16
// columns and 4000 bins (a quarter); an LCDM step (8 columns) 28.2 / 28.5 ms at 1024 with
// 1024 bins (a 16th), 1.65 / 1.74 ms at 384 with 1024 (a sixth), 4.63 / 4.04 ms at 512 with
// 4000 (a half).
int fused_pofk_by(const mgpu_ctx *ctx, int T) {
  if (ctx->pk_fn.edge && (size_t)ctx->p.pofk_nbins <= (size_t)ctx->N * T / 3 &&
      fft_col_lds(ctx->N, T) + pofk_lds(ctx->N, ctx->p.pofk_nbins, 1) <= ctx->lds_max)
    return POFK_EDGES;
  return ctx->pk_fn.table && pofk_table_lds(ctx, T) <= ctx->lds_max ? POFK_TABLE : POFK_NONE;
}

int fused_green_x(mgpu_ctx *ctx, int mode, const float2 *a, const float2 *b, float2 *o0, float2 *o1, double p0,
                  double p1, int filter) {
  GreenArgs ga{0.f, 0.f, 0.f, filter};
  if (mode == GREEN_FORCE) ga.cnorm = (float)p0, ga.mult = ctx->mlp ? ctx->green_mult : nullptr;
  else ga.nf = (float)p0;
  ga.kfac = (float)p1;
  const double modes = (double)ctx->N * ctx->N * (ctx->N / 2 + 1);
  KScope ks(ctx, mode == GREEN_FORCE ? MGPU_K_FFT_GREEN : MGPU_K_FFT_POT,
            8.0 * modes * ((b ? 2 : 1) + (mode == GREEN_FORCE ? 2 : 1)));
  switch (ctx->N) {
#define X(S) \
  case S:    \
    return by_tile<S, GreenF>(ctx, mode, a, b, o0, o1, ga);
    MGPU_FFT_SIZES(X)
#undef X
    default:
      return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported FFT size");
  }
}

int fused_x_pair(mgpu_ctx *ctx, int fwd, int mode, const float2 *in, float2 *kout, const float2 *dk, float2 *o0,
                 float2 *o1, double p0, double p1, int filter, double coupling, double massterm2, double *pk) {
  FusedXArgs a;
  a.fwd = fwd;
  a.mode = mode;
  a.in = in;
  a.kout = kout;
  a.dk = dk;
  a.o0 = o0;
  a.o1 = o1;
  a.ga = GreenArgs{0.f, 0.f, 0.f, filter};
  if (mode == GREEN_FORCE) a.ga.cnorm = (float)p0, a.ga.mult = ctx->mlp ? ctx->green_mult : nullptr;
  else a.ga.nf = (float)p0;
  a.ga.kfac = (float)p1;
  a.coupling = (float)coupling;
  a.m2 = (float)massterm2;
  a.pk = pk;
  // compulsory: the input (and delta(k)) read, the outputs (and delta(k)) written
  const double modes = (double)ctx->N * ctx->N * (ctx->N / 2 + 1);
  const int nio = 1 + (dk ? 1 : 0) + (kout ? 1 : 0) + (mode == GREEN_FORCE ? 2 : 1);
  KScope ks(ctx, fwd == FWD_DENSITY ? MGPU_K_FFT_XDENS : MGPU_K_FFT_XFORCE, 8.0 * modes * nio);
  switch (ctx->N) {
#define X(S)                                                               \
  case S:                                                                  \
    /* the force pairs hold G through the first inverse: 8-column tiles */ \
    if (mode == GREEN_FORCE) return FusedXF<S, 8>::run(ctx, a);            \
    return by_tile<S, FusedXF>(ctx, a);
    MGPU_FFT_SIZES(X)
#undef X
    default:
      return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported FFT size");
  }
}

// inverse y pass: buf <- Y[buf], oy <- Y[i n_y buf], for the meshes beyond kForceYOne
static int fused_dual_y(mgpu_ctx *ctx, float2 *buf, float2 *oy) {
  const double modes = (double)ctx->N * ctx->N * (ctx->N / 2 + 1);
  KScope ks(ctx, MGPU_K_FFT_DUAL, 8.0 * modes * 3);
  switch (ctx->N) {
#define X(S)                                                                \
  case S:                                                                   \
    if constexpr (S > kForceYOne) return by_tile<S, DualF>(ctx, buf, oy);   \
    break;
    MGPU_FFT_SIZES(X)
#undef X
  }
  return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported FFT size");
}

int fused_force_y(mgpu_ctx *ctx, float2 *buf, float2 *oy, float2 *other) {
  // one launch up to 256, where a pass is short against a launch (128: 16.6 us for the
  // two launches); beyond, the plain pass keeps its own kernel's occupancy
  if (ctx->N <= kForceYOne) {
    const double modes = (double)ctx->N * ctx->N * (ctx->N / 2 + 1);
    KScope ks(ctx, MGPU_K_FFT_DUAL, 8.0 * modes * 5);
    switch (ctx->N) {
#define X(S)                                                                          \
  case S:                                                                             \
    if constexpr (S <= kForceYOne) return by_tile<S, ForceYF>(ctx, buf, oy, other);   \
    break;
      MGPU_FFT_SIZES(X)
#undef X
    }
    return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported FFT size");
  }
  int rc = fused_dual_y(ctx, buf, oy);
  return rc ? rc : fft_pass_col(ctx, &ctx->fft, other, 1, 0);
}

int fused_epi_phi_x(mgpu_ctx *ctx, float2 *buf, double coupling, double massterm2) {
  const double modes = (double)ctx->N * ctx->N * (ctx->N / 2 + 1);
  KScope ks(ctx, MGPU_K_FFT_EPI, 16.0 * modes);
  switch (ctx->N) {
#define X(S) \
  case S:    \
    return by_tile<S, EpiF>(ctx, buf, (float)coupling, (float)massterm2);
    MGPU_FFT_SIZES(X)
#undef X
    default:
      return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported FFT size");
  }
}

int fused_z_screen(mgpu_ctx *ctx, int density_kind, float2 *buf, const float *dx, double p0, double p1) {
  const double rows = (double)ctx->N * ctx->N;
  KScope ks(ctx, MGPU_K_FFT_SCREEN, rows * (16.0 * (ctx->N / 2 + 1) + 4.0 * ctx->N));
  const int kind = density_kind ? SCREEN_DENSITY : SCREEN_POTENTIAL;
  switch (ctx->N) {
#define X(S) \
  case S:    \
    return screen_launch<S>(ctx, kind, buf, (const float2 *)dx, (float)p0, (float)p1);
    MGPU_FFT_SIZES(X)
#undef X
    default:
      return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported FFT size");
  }
}

int fused_pofk_x(mgpu_ctx *ctx, float2 *buf, double *pk) {
  const double modes = (double)ctx->N * ctx->N * (ctx->N / 2 + 1);
  KScope ks(ctx, MGPU_K_FFT_PK, 16.0 * modes);
  switch (ctx->N) {
#define X(S) \
  case S:    \
    return by_tile<S, PofkF>(ctx, buf, pk);
    MGPU_FFT_SIZES(X)
#undef X
    default:
      return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported FFT size");
  }
}
