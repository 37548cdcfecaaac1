// Spectral passes of the initial conditions fused into their FFT passes (gfx950): the
// 2LPT source from the displacement-gradient tensor (src/2LPT.c:1247-1345).
//
//   lpt_x_pass       x pass (inverse) of up to three fields i k_a/k^2 delta(k) or
//                    -k_a k_b/k^2 delta(k) from one read of delta(k)
//   lpt_source_pass  z pass (c2r) of up to three fields of the tensor and the products
//                    that enter the source, with its r2c at the last one
//
// Each multiplier is formed in FP64 and rounded once, as a sweep of its own would.
#include "fft_core.h"

namespace {

using namespace fftc;

// Keeps a value from being taken as known: what depends on it is formed again where it is
// used.  Without it the multipliers and twiddles common to the fields are held in
// registers from one field to the next (216 instead of 128, or spills).
template <class V>
__device__ __forceinline__ void anew(V &v) {
  asm volatile("" : "+s"(v));
}

// Tile (bx, by) of xcd_tile: columns kz = bx T + c, outer index ky = by, line index kx.
// The tile is read once; each field's multiplied copy goes through the stages in turn.
// Bound by memory: one read and n writes for n fields, where a sweep for each field's
// spectrum and a plain x pass read and wrote it twice.  The six fields of the tensor at
// 384, in launches of three, two and one: 0.55 ms, where six sweeps took 0.80 ms and
// their x passes 0.58 ms.
template <int L, int T>
__global__ __launch_bounds__(col_threads(L, T), tw_in_lds(L) ? 4 : 1) void k_lpt_x(const float2 *__restrict__ cd, float2 *o0, float2 *o1,
                                                             float2 *o2, LptFields f, size_t ls, size_t os,
                                                             const float2 *__restrict__ tw, double kf, size_t zs) {
  cd = zbuf(cd, zs);
  extern __shared__ float2 lds[];
  constexpr int NT = col_threads(L, T), E = col_ept(L, T);
  constexpr int R0 = pick_radix(L, E), NB0 = E / R0, M0 = L / R0;
  const int tid = threadIdx.x;
  int bx, by;
  xcd_tile(bx, by);
  const size_t tile = (size_t)by * os + (size_t)bx * T;
  StageTwiddles<L, T, NT> stw(tw, tid);
  float2 raw[E];
  first_loads<L, T, NT, true>(raw, tid, [&](int c, int j, int o) { return col_at<L, T>(cd + tile, ls, c, j, o); });
  const float2 *twl = stw.to_lds(lds, tid);
  auto ld = [&](int, int, int) { return make_float2(0.f, 0.f); };
  for (int n = 0; n < f.n; ++n) {
    const int a = f.a[n], b = f.b[n];
    const double scale = b < 0 ? 1.0 / kf : 1.0;
    int ny = kint(by, L);
    anew(ny);
    float2 p[E];
#pragma unroll
    for (int q = 0; q < NB0; ++q) {
      const int g = tid + q * NT, c = g % T, k = bx * T + c, nz = kint(k, L);
      int j = g / T;
#pragma unroll
      for (int r = 0; r < R0; ++r) {
        // one element after the other: side by side their FP64 values take 60 registers more
        asm volatile("" : "+v"(j));
        const int nx = kint(j + r * M0, L), n2 = nx * nx + ny * ny + nz * nz;
        const int na = a == 0 ? nx : a == 1 ? ny : nz, nb = b < 0 ? 1 : b == 0 ? nx : b == 1 ? ny : nz;
        const double w = k <= L / 2 && n2 > 0 ? scale * (double)(na * nb) * recip(n2) : 0.0;
        // i k_a/k^2 d, or i k_b times that
        const float2 d = raw[q * R0 + r];
        float2 v = make_float2((float)(-w * (b < 0 ? d.y : d.x)), (float)(w * (b < 0 ? d.x : -d.y)));
        asm volatile("" : "+v"(v.x), "+v"(v.y));
        p[q * R0 + r] = v;
      }
    }
    float2 *out = zbuf(n == 0 ? o0 : n == 1 ? o1 : o2, zs) + tile;
    auto st = [&](int c, int j, int o, float2 v) { col_at<L, T>(out, ls, c, j, o) = v; };
    if (n > 0) __syncthreads();  // the last field's stages have read the LDS
    fft_stages<L, T, NT, +1, 1, T, true, false, 1, false, true>(lds, twl, 1, tid, ld, st, p);
  }
}

// c2r of one field's rows; the real pairs stay in registers, in the order of the
// last stage's stores
template <int N, class ST>
__device__ __forceinline__ void z_c2r_regs(float2 *lds, const float2 *f, int HP, size_t row0, size_t nrows,
                                           const float2 *__restrict__ tw, int tid, const ST &st) {
  using C = RowCfg<N>;
  z_merge<N>(lds, f, HP, row0, nrows, tw, tid);
  __syncthreads();
  auto ldl = [&](int r, int j, int o) { return lds[r * C::LS + j + o]; };
  fft_stages<C::M, C::RB, C::NT, +1, C::LS, 1, false, true, 1>(lds, tw, 2, tid, ldl, st);
}

// z pass of the 2LPT source (src/2LPT.c:1282-1290), source rows in s:
//   LPT_DIAG  s <- d0 (d1 + d2) + d1 d2, the rows of d0 being s's own
//   LPT_OFF2  s <- s - d1^2 - d2^2
//   LPT_OFF1  s <- r2c of (s - d1^2)
// Bound by memory: the source and the fields cross it once; the c2r of each field and
// the sweeps over real meshes that formed the products crossed it more often.  The three
// launches at 384: 0.76 ms, where six c2r, four sweeps and the r2c took 1.52 ms.
// Three waves per SIMD up to 1024: with none asked for / three / four, DIAG 82 / 73 / 114 us
// at 256, 721 / 678 / 826 at 512 and 6.33 / 6.23 / 6.88 ms at 1024, OFF2 472 / 481 / 713 us
// at 512, OFF1 411 / 415 / 409.  Beyond, rows have their workgroup's registers.
template <int N, int MODE>
__global__ __launch_bounds__(RowCfg<N>::NT, N > 1024 ? 1 : 3) void k_lpt_source(float2 *s, const float2 *d1,
                                                                                const float2 *d2, int HP, size_t nrows,
                                                                                const float2 *__restrict__ tw,
                                                                                size_t zs) {
  s = zbuf(s, zs);
  d1 = zbuf(d1, zs);
  d2 = zbuf(d2, zs);
  using C = RowCfg<N>;
  constexpr int E = C::M * C::RB / C::NT, RL = last_radix(C::M, E), ML = C::M / RL;
  extern __shared__ float2 lds[];
  int tid = threadIdx.x;
  const size_t row0 = (size_t)blockIdx.x * C::RB;
  float2 u[E], v[E];
  if (MODE != LPT_DIAG) {
#pragma unroll
    for (int q = 0; q < E / RL; ++q) {
      const int g = tid + q * C::NT, j = g % ML;
      const size_t row = row0 + g / ML < nrows ? row0 + g / ML : nrows - 1;
#pragma unroll
      for (int r = 0; r < RL; ++r) u[q * RL + r] = s[row * HP + j + r * ML];
    }
  }
  int oi = 0;  // output index of the stores (a constant of the unrolled last stage)
  auto put = [&](int r, int j, int o, float2 x) {
    if (row0 + r < nrows) s[(row0 + r) * HP + j + o] = x;
  };
  auto less = [](float a, float b) { return (float)((double)a - (double)b * (double)b); };
  if (MODE == LPT_DIAG) {
    z_c2r_regs<N>(lds, s, HP, row0, nrows, tw, tid, [&](int, int, int, float2 x) { u[oi++] = x; });
    __syncthreads();
    anew(tw);
    asm volatile("" : "+v"(tid));
    oi = 0;
    z_c2r_regs<N>(lds, d1, HP, row0, nrows, tw, tid, [&](int, int, int, float2 x) { v[oi++] = x; });
    __syncthreads();
    anew(tw);
    asm volatile("" : "+v"(tid));
    oi = 0;
    auto dia = [](double a, double b, double c) { return (float)(a * (b + c) + b * c); };
    z_c2r_regs<N>(lds, d2, HP, row0, nrows, tw, tid, [&](int r, int j, int o, float2 x) {
      put(r, j, o, make_float2(dia(u[oi].x, v[oi].x, x.x), dia(u[oi].y, v[oi].y, x.y)));
      oi++;
    });
  } else if (MODE == LPT_OFF2) {
    z_c2r_regs<N>(lds, d1, HP, row0, nrows, tw, tid, [&](int, int, int, float2 x) { v[oi++] = x; });
    __syncthreads();
    anew(tw);
    asm volatile("" : "+v"(tid));
    oi = 0;
    auto less2 = [](float a, double b, double c) { return (float)((double)a - b * b - c * c); };
    z_c2r_regs<N>(lds, d2, HP, row0, nrows, tw, tid, [&](int r, int j, int o, float2 x) {
      put(r, j, o, make_float2(less2(u[oi].x, v[oi].x, x.x), less2(u[oi].y, v[oi].y, x.y)));
      oi++;
    });
  } else {
    z_c2r_regs<N>(lds, d1, HP, row0, nrows, tw, tid, [&](int, int, int, float2 x) {
      v[oi] = make_float2(less(u[oi].x, x.x), less(u[oi].y, x.y));
      oi++;
    });
    anew(tw);
    float2 w[ZSplit<N>::ITER];
    z_split_twiddles<N>(w, tw, tid);
    auto ldl = [&](int r, int j, int o) { return lds[r * C::LS + j + o]; };
    auto stl = [&](int r, int j, int o, float2 x) { lds[r * C::LS + j + o] = x; };
    fft_stages<C::M, C::RB, C::NT, -1, C::LS, 1, false, true, 1, false, true, true>(lds, tw, 2, tid, ldl, stl, v);
    __syncthreads();
    z_split<N>(lds, w, s, HP, row0, nrows, tid);
  }
}

template <class K>
int set_lds(mgpu_ctx *ctx, K kern, size_t lds) {
  if (lds > 65536) MGPU_HIP(ctx, hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  return MGPU_OK;
}

template <int N, int T>
int launch_x(mgpu_ctx *ctx, const float2 *cd, float2 *const o[3], const LptFields &f) {
  const size_t HP = ctx->fft.hp, lds = col_lds_elems(N, T) * sizeof(float2);
  auto kern = k_lpt_x<N, T>;
  int rc = set_lds(ctx, kern, lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3(HP / T, N, ctx->bz), dim3(col_threads(N, T)), lds, ctx->stream, cd, o[0], o[1], o[2], f,
                     (size_t)N * HP, HP, ctx->fft.tw, 2 * MGPU_PI / ctx->p.box, ctx->zs);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

template <int N>
int dispatch_x(mgpu_ctx *ctx, const float2 *cd, float2 *const o[3], const LptFields &f) {
  if constexpr (col_threads(N, 16) <= 1024)
    if (ctx->fft.tcols == 16) return launch_x<N, 16>(ctx, cd, o, f);
  return launch_x<N, 8>(ctx, cd, o, f);
}

template <int N>
int launch_source(mgpu_ctx *ctx, int mode, float2 *s, const float2 *d1, const float2 *d2) {
  using C = RowCfg<N>;
  const size_t nrows = (size_t)N * N, lds = (size_t)C::RB * C::LS * sizeof(float2);
  auto kern = mode == LPT_DIAG ? k_lpt_source<N, LPT_DIAG> : mode == LPT_OFF2 ? k_lpt_source<N, LPT_OFF2> : k_lpt_source<N, LPT_OFF1>;
  int rc = set_lds(ctx, kern, lds);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3(cdiv(nrows, C::RB), 1, ctx->bz), dim3(C::NT), lds, ctx->stream, s, d1, d2, ctx->fft.hp,
                     nrows, ctx->fft.tw, ctx->zs);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

}  // namespace

int lpt_x_pass(mgpu_ctx *ctx, const float2 *cd, float2 *o0, float2 *o1, float2 *o2, const LptFields &f) {
  // compulsory traffic: the half spectrum read once and written once per field
  const double N = ctx->N;
  KScope ks(ctx, MGPU_K_LPT, ctx->bz * (1.0 + f.n) * 8.0 * N * N * (ctx->N / 2 + 1));
  float2 *const o[3] = {o0, o1 ? o1 : o0, o2 ? o2 : o0};
  switch (ctx->N) {
#define X(S) \
  case S:    \
    return dispatch_x<S>(ctx, cd, o, f);
    MGPU_FFT_SIZES(X)
#undef X
    default:
      return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported FFT size");
  }
}

int lpt_source_pass(mgpu_ctx *ctx, int mode, float2 *s, const float2 *d1, const float2 *d2) {
  const double rows = (double)ctx->N * ctx->N, re = 4.0 * ctx->N, co = 8.0 * (ctx->N / 2 + 1);
  // DIAG 3 complex in, 1 real out; OFF2 2 complex and 1 real in, 1 real out; OFF1 1 complex and 1 real in, 1 complex out
  KScope ks(ctx, MGPU_K_LPT,
            ctx->bz * rows * (mode == LPT_DIAG ? 3 * co + re : mode == LPT_OFF2 ? 2 * co + 2 * re : 2 * co + re));
  switch (ctx->N) {
#define X(S) \
  case S:    \
    return launch_source<S>(ctx, mode, s, d1, d2 ? d2 : d1);
    MGPU_FFT_SIZES(X)
#undef X
    default:
      return mgpu_fail(ctx, MGPU_E_INVALID, "unsupported FFT size");
  }
}
