// 2LPT initial conditions and scale-dependent LPT fields for gfx950.
//
//   k_ic_delta         displacement_fields' Gaussian mode loop (src/2LPT.c:337-495):
//                      one thread per (i, j) column re-seeds RANLUX from the seed
//                      table and draws (phase, amplitude) for kz < N/2 in order.
//   k_lpt_spectrum     i k_a/k^2 delta(k) g(|k|) of the scale-dependent fields
//                      (src/2LPT.c:1583-1629), 2LPT.c wavenumbers (Nyquist = -N/2);
//                      the displacements' and the gradients' spectra ride on their
//                      x passes (lpt_passes.hip).
//   k_disp_fold        the displacement spectra folded onto the particle lattice
//   k_lattice_read     trilinear read-out at the Lagrangian lattice
//                      (src/2LPT.c:1407-1476, 1657-1702) + per-block sums for the
//                      mean removal (src/2LPT.c:1493-1508, 1713-1729).
#include "mgpu_internal.h"
#include "fft_core.h"
#include "ranlux.h"
#include "ranlux_jump.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

// Seed table staging of the allocation-free IC entry point: one copy per GPU,
// held until the process ends.  Host code never passes `scratch` itself to a
// kernel or a copy (the name is only a host-side stand-in for the symbol); it
// uses the per-device address that ic_scratch_init obtains with
// hipGetSymbolAddress.
static __device__ __align__(256) unsigned scratch[MGPU_IC_SCRATCH_SEEDS];

namespace {

using fftc::kint;
using fftc::recip;

constexpr int kBlock = 256;
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned *g_scratch_ptr[kMaxDevices] = {};

// Seed table (src/2LPT.c:259-271): the N^2 values of one RANLUX stream, in the
// reference's order of shells.  Shell i holds 4 (2 i + 1) values from draw 4 i^2 on:
// for each of four sign quadrants i values along one axis and i + 1 along the other.
// Thread t generates the draws [12 adv t, 12 adv (t + 1)) from its own state of the
// stream, which the host jumped ahead to (state q of thread t at st[q n + t], the
// carry as the 13th).  The stream itself is one serial chain of 17 dependent steps per
// draw: the host took 10.5 ms for the table of a 384 mesh, the chunks take 0.3 ms
// there and 60 us here.
// With flag, st[13 n] (a realization's inversion) goes behind the table.
__global__ __launch_bounds__(64) void k_seed_table(const double *__restrict__ st, unsigned n, unsigned adv, int N,
                                                   int flag, unsigned *__restrict__ table, size_t zs) {
  st = zbuf(st, zs);
  table = zbuf(table, zs);
  const unsigned t = blockIdx.x * 64 + threadIdx.x;
  if (t >= n) return;
  Ranlxd1 r;
#pragma unroll
  for (int q = 0; q < 12; q++) r.y[q] = st[(size_t)q * n + t];
  r.carry = st[(size_t)12 * n + t];
  const unsigned total = (unsigned)N * (unsigned)N;
  if (flag && t == 0) table[total] = (unsigned)st[(size_t)13 * n];
  unsigned d = 12 * adv * t;
  for (unsigned a = 0; a < adv && d < total; a++) {
    r.advance();
#pragma unroll
    for (int q = 0; q < 12; q++, d++) {
      if (d >= total) break;
      unsigned i = (unsigned)(0.5f * sqrtf((float)d));  // the shell: 4 i^2 <= d < 4 (i + 1)^2
      while (4 * i * i > d) i--;
      while (4 * (i + 1) * (i + 1) <= d) i++;
      const unsigned e = d - 4 * i * i, g = e / (2 * i + 1), k = e % (2 * i + 1);
      unsigned x = k < i ? i : k - i, y = k < i ? k : i;
      if (g & 1) x = (unsigned)N - 1 - x;
      if (g & 2) y = (unsigned)N - 1 - y;
      table[(size_t)x * N + y] = (unsigned)(0x7fffffff * r.y[q]);
    }
  }
}

// one thread per column (i, j) of the N x N grid
__global__ __launch_bounds__(kBlock) void k_ic_delta(const unsigned *__restrict__ seedtable, int N, int Np, int HP,
                                                     double box, int sphere_mode, int amp_fixed, int inverted,
                                                     const double *__restrict__ pk_n2, float2 *__restrict__ cd,
                                                     size_t zs, const int *__restrict__ inv_z) {
  // a batch: realization blockIdx.z's seed table and inversion flag
  cd = zbuf(cd, zs);
  seedtable = zbuf(seedtable, zs);
  if (inv_z) inverted = *zbuf(inv_z, zs);
  const int col = blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= N * N) return;
  const int i = col / N, j = col % N;
  Ranlxd1 r;
  r.seed(seedtable[col]);
  const double bnorm = pow(box, -1.5);
  for (int k = 0; k < N / 2; k++) {
    const double phase = r.uniform() * 2 * MGPU_PI;
    double ampl = 0.0;
    if (!amp_fixed) {
      do {
        ampl = r.uniform();
      } while (ampl == 0);
    }
    if (i == N / 2 || j == N / 2 || k == N / 2) continue;
    if (i == 0 && j == 0 && k == 0) continue;
    // src/2LPT.c:364-386: k-vector with index < N/2 -> index, else -(N-index); cube or sphere cut
    // same double expressions as the reference so the cut rounds identically
    const int ni = i < N / 2 ? i : -(N - i), nj = j < N / 2 ? j : -(N - j), nk = k;
    const double kx = ni * 2 * MGPU_PI / box, ky = nj * 2 * MGPU_PI / box, kz = nk * 2 * MGPU_PI / box;
    if (sphere_mode == 1) {
      const double kmag = sqrt(kx * kx + ky * ky + kz * kz);
      if (kmag * box / (2 * MGPU_PI) > Np / 2) continue;
    } else {
      if (fabs(kx) * box / (2 * MGPU_PI) > Np / 2) continue;
      if (fabs(ky) * box / (2 * MGPU_PI) > Np / 2) continue;
      if (fabs(kz) * box / (2 * MGPU_PI) > Np / 2) continue;
    }
    double p_of_k = pk_n2[ni * ni + nj * nj + nk * nk];
    if (!amp_fixed) p_of_k *= -log(ampl);
    double delta = bnorm * sqrt(p_of_k);
    if (inverted) delta *= -1.0;
    const float2 v = make_float2((float)(delta * cos(phase)), (float)(delta * sin(phase)));
    const float2 vc = make_float2(v.x, -v.y);
    if (k > 0) {
      cd[((size_t)i * N + j) * HP + k] = v;
    } else if (i == 0) {
      if (j >= N / 2) continue;
      cd[((size_t)0 * N + j) * HP] = v;
      cd[((size_t)0 * N + (N - j)) * HP] = vc;
    } else {
      if (i >= N / 2) continue;
      const int jj = (N - j) == N ? 0 : N - j;
      cd[((size_t)i * N + j) * HP] = v;
      cd[((size_t)(N - i) * N + jj) * HP] = vc;
    }
  }
}

// 2LPT.c wavenumber component of index i (Nyquist -> -N/2), in h/Mpc
__device__ __forceinline__ double kc(int i, int N, double kf) { return (i < N / 2 ? i : -(N - i)) * kf; }
__device__ __forceinline__ int nabs(int i, int N) { return i < N / 2 ? i : N - i; }

enum { SPEC_FIELD = 0, SPEC_NEG = 1 };

// Spectral kernel of the scale-dependent LPT fields.  mode:
//   SPEC_FIELD  out = i k_a/k^2 (g1 cd + g2 cd2)            (from_cdisp_store_to_ZA, both orders)
//   SPEC_NEG    out = -src, 0 at k = 0                      (cdelta_cdm2, src/2LPT.c:1336-1345)
__global__ __launch_bounds__(kBlock) void k_lpt_spectrum(int mode, const float2 *__restrict__ cd,
                                                         const float2 *__restrict__ cd2, float2 *__restrict__ out,
                                                         int N, int HP, double kf, int a,
                                                         const double *__restrict__ g1,
                                                         const double *__restrict__ g2, size_t zs) {
  cd = zbuf(cd, zs);
  cd2 = zbuf(cd2, zs);
  out = zbuf(out, zs);
  size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)N * N * HP) return;
  const int k = (int)(e % HP);
  const size_t row = e / HP;
  const int j = (int)(row % N), i = (int)(row / N);
  float2 r = make_float2(0.f, 0.f);
  if (k <= N / 2) {
    const double kv[3] = {kc(i, N, kf), kc(j, N, kf), kc(k, N, kf)};
    const double k2 = kv[0] * kv[0] + kv[1] * kv[1] + kv[2] * kv[2];
    if (k2 > 0.0) {
      double re = 0, im = 0;
      if (mode == SPEC_FIELD) {
        const int n2 = nabs(i, N) * nabs(i, N) + nabs(j, N) * nabs(j, N) + nabs(k, N) * nabs(k, N);
        const float2 d = cd[e];
        double dr = d.x * g1[n2], di = d.y * g1[n2];
        if (cd2) {
          const float2 d2 = cd2[e];
          dr += d2.x * g2[n2];
          di += d2.y * g2[n2];
        }
        re = -kv[a] / k2 * di;
        im = kv[a] / k2 * dr;
      } else {  // SPEC_NEG
        const float2 s = cd[e];
        re = -s.x;
        im = -s.y;
      }
      r = make_float2((float)re, (float)im);
    }
  }
  out[e] = r;
}

// trilinear lattice read-out, src/2LPT.c:1407-1476.  out[q] = scale * value
__global__ __launch_bounds__(kBlock) void k_lattice_read(const float *__restrict__ m, int N, int Np, int HP2,
                                                         double scale, float *__restrict__ out,
                                                         double *__restrict__ partial, size_t zs) {
  m = zbuf(m, zs);
  out = zbuf(out, zs);
  partial = zbuf(partial, zs);
  __shared__ double red[kBlock];
  const size_t np = (size_t)Np * Np * Np;
  size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  double val = 0.0;
  if (q < np) {
    const int p = (int)(q % Np), mm = (int)((q / Np) % Np), n = (int)(q / ((size_t)Np * Np));
    double u = (double)(n * N) / (double)Np, v = (double)(mm * N) / (double)Np, w = (double)(p * N) / (double)Np;
    int i = (int)u, j = (int)v, k = (int)w;
    if (i >= N) i = N - 1;
    if (j >= N) j = N - 1;
    if (k >= N) k = N - 1;
    u -= i;
    v -= j;
    w -= k;
    const int ii = i + 1 >= N ? 0 : i + 1, jj = j + 1 >= N ? 0 : j + 1, kk = k + 1 >= N ? 0 : k + 1;
    auto at = [&](int x, int y, int z) { return (double)m[((size_t)x * N + y) * HP2 + z]; };
    val = at(i, j, k) * ((1 - u) * (1 - v) * (1 - w)) + at(i, j, kk) * ((1 - u) * (1 - v) * w) +
          at(i, jj, k) * ((1 - u) * v * (1 - w)) + at(i, jj, kk) * ((1 - u) * v * w) +
          at(ii, j, k) * (u * (1 - v) * (1 - w)) + at(ii, j, kk) * (u * (1 - v) * w) +
          at(ii, jj, k) * (u * v * (1 - w)) + at(ii, jj, kk) * (u * v * w);
    val *= scale;
    out[q] = (float)val;
  }
  red[threadIdx.x] = val;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[(size_t)blockIdx.x * 3] = red[0];
}

__global__ __launch_bounds__(kBlock) void k_sub_mean(float *__restrict__ v, size_t n, const double *__restrict__ sum,
                                                     double inv_n, size_t zs) {
  v = zbuf(v, zs);
  sum = zbuf(sum, zs);
  size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  v[q] = (float)((double)v[q] - sum[0] * inv_n);
}

// sum partial[b*3] over blocks in a fixed order -> out[0]
__global__ __launch_bounds__(1024) void k_reduce1(const double *__restrict__ partial, int nb, double *__restrict__ out,
                                                  size_t zs) {
  partial = zbuf(partial, zs);
  out = zbuf(out, zs);
  __shared__ double red[1024];
  double s = 0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) s += partial[(size_t)b * 3];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

// particle init, src/main.c:257-309
__global__ __launch_bounds__(kBlock) void k_init_particles(float *__restrict__ pos, float *__restrict__ vel,
                                                           const float *__restrict__ l0,
                                                           const float *__restrict__ l1, int Np, double box,
                                                           int sd, double Di, double Di2, int use_cola,
                                                           double v1, double v2) {
  const size_t np = (size_t)Np * Np * Np;
  size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= np) return;
  const int c[3] = {(int)(q / ((size_t)Np * Np)), (int)((q / Np) % Np), (int)(q % Np)};
  const float fb = (float)box;
  for (int a = 0; a < 3; a++) {
    const size_t idx = (size_t)a * np + q;
    double x = c[a] * (box / (double)Np);
    if (sd) x += (double)l0[idx];
    else x += (double)l0[idx] * Di + (double)l1[idx] * Di2;
    float f = (float)x;
    for (int it = 0; it < 4 && f >= fb; ++it) f -= fb;
    for (int it = 0; it < 4 && f < 0.f; ++it) f += fb;
    if (!(f >= 0.f && f < fb)) f = 0.f;
    pos[idx] = f;
    if (use_cola) vel[idx] = 0.f;
    else vel[idx] = sd ? l1[idx] : (float)((double)l0[idx] * v1 + (double)l1[idx] * v2);
  }
}

// ---------------------------------------------------------------- lattice fold
// LPT field components X_a = i k_a/k^2 (g1 cd1 + g2 cd2) at half-spectrum index
// (i, j, l), l in [0, N/2], 2LPT.c wavenumbers (src/2LPT.c:1583-1629), in FP32
// (the stored spectra and the output fields are FP32).  ikf = 1 / (2 pi/Box).
// Growth sources of the fold, for NS LPT slots at once: eval(n2, y, g) sets
// g[s][o] = growth of order o + 1 for slot s at |n|^2 = n2, y = ln k = ln kf +
// ln|n| (only the slice source uses y).
// From FP32 per-|n|^2 tables (one slot):
struct GTab {
  static constexpr bool kNeedsLnk = false;
  const float *t1, *t2;
  __device__ __forceinline__ void eval(int n2, float, float g[1][2]) const {
    g[0][0] = t1[n2];
    g[0][1] = t2[n2];
  }
};
// From cubic Hermite slices on one uniform ln k grid shared by all slices,
// held in LDS node-major with 1 + NS float4 per node: (den_1, dden_1, den_2,
// dden_2), shared by the slots, then per slot (num_1, dnum_1, num_2, dnum_2);
// g = norm_o num / den.  The Hermite basis is computed once per mode.
template <int NS>
struct GShared {
  static constexpr bool kNeedsLnk = true;
  const float4 *sl;
  float y0, dy, idy, ymax, norm1, norm2;
  int ny;
  __device__ __forceinline__ void eval(int, float y, float g[NS][2]) const {
    y = fminf(fmaxf(y, y0), ymax);
    int j = (int)((y - y0) * idy);
    j = min(max(j, 0), ny - 2);
    const float t = (y - (y0 + (float)j * dy)) * idy, t2 = t * t, t3 = t2 * t;
    const float h00 = 2.f * t3 - 3.f * t2 + 1.f, h10 = (t3 - 2.f * t2 + t) * dy, h01 = -2.f * t3 + 3.f * t2,
                h11 = (t3 - t2) * dy;
    const float4 *A = sl + j * (1 + NS), *B = A + (1 + NS);
    float4 a = A[0], b = B[0];
    const float r1 = norm1 * __builtin_amdgcn_rcpf(h00 * a.x + h10 * a.y + h01 * b.x + h11 * b.y);
    const float r2 = norm2 * __builtin_amdgcn_rcpf(h00 * a.z + h10 * a.w + h01 * b.z + h11 * b.w);
#pragma unroll
    for (int s = 0; s < NS; s++) {
      a = A[1 + s];
      b = B[1 + s];
      g[s][0] = r1 * (h00 * a.x + h10 * a.y + h01 * b.x + h11 * b.y);
      g[s][1] = r2 * (h00 * a.z + h10 * a.w + h01 * b.z + h11 * b.w);
    }
  }
};

// LPT field components X[s][a] = i k_a/k^2 (g1 cd1 + g2 cd2) of slot s at half-spectrum
// index (i, j, l), l in [0, N/2], 2LPT.c wavenumbers (src/2LPT.c:1583-1629), in FP32
// (the stored spectra and the output fields are FP32).  ikf = 1 / (2 pi/Box).
template <int NS, class G>
__device__ __forceinline__ void lpt_xf(int i, int j, int l, int N, int HP, int Np, float ikf, float lnkf,
                                       const float2 *__restrict__ cd1, const float2 *__restrict__ cd2, const G &gr,
                                       float X[NS][6]) {
  const int ni = i < N / 2 ? i : i - N, nj = j < N / 2 ? j : j - N, nl = l < N / 2 ? l : l - N;
  const int n2 = ni * ni + nj * nj + nl * nl;
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int q = 0; q < 6; q++) X[s][q] = 0.f;
  if (n2 == 0) return;
  const size_t e = ((size_t)i * N + j) * HP + l;
  // the 1LPT field is zero outside the initial-condition cube |n_a| <= Nsample/2
  const bool cube = abs(ni) <= Np / 2 && abs(nj) <= Np / 2 && abs(nl) <= Np / 2;
  const float2 d1 = cube ? cd1[e] : make_float2(0.f, 0.f);
  const float2 d2 = cd2 ? cd2[e] : make_float2(0.f, 0.f);
  float g[NS][2];
  gr.eval(n2, G::kNeedsLnk ? lnkf + 0.5f * __logf((float)n2) : 0.f, g);
  // k_a / k^2 = n_a / (kf n^2)
  const float sc = ikf * __builtin_amdgcn_rcpf((float)n2);
  const float nv[3] = {(float)ni * sc, (float)nj * sc, (float)nl * sc};
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const float dr = d1.x * g[s][0] + d2.x * g[s][1], di = d1.y * g[s][0] + d2.y * g[s][1];
#pragma unroll
    for (int q = 0; q < 3; q++) {
      X[s][2 * q] = -nv[q] * di;
      X[s][2 * q + 1] = nv[q] * dr;
    }
  }
}

// Sampling the c2r of a field at every m-th mesh point (the Lagrangian lattice
// when N = m * Nsample, where the read-out of src/2LPT.c:1657-1702 has weight 1
// on one node) equals an Nsample^3 c2r of the aliased spectrum
//   F_f(k') = sum_{k = k' (mod Nsample)} F(k),
// F the Hermitian extension of the half spectrum with the kz = 0, N/2 planes
// symmetrised as the c2r's real-part rule implies.  One thread per output mode;
// consecutive threads take consecutive kz, so every alias read is a coalesced
// row segment.  The folded DC mode is zeroed, which removes the lattice mean
// exactly (src/2LPT.c:1719-1729).
// One folded mode (ip, jp, lp), lp <= Np/2: the sum over its m^3 aliases, for
// NS slots.  MF > 0 is the fold factor m = N / Nsample as a compile-time
// constant, so the alias loop unrolls and all its loads are in flight
// together; MF = 0 takes m at run time.  PLANES = false is for 0 < lp < Np/2:
// then no alias lies on the kz = 0 or N/2 plane, and whether alias c lies
// below or above N/2 does not depend on lp, so the lanes of a wave take one
// path.
template <int MF, int NS, class G, bool PLANES = true>
__device__ __forceinline__ void fold_mode(int ip, int jp, int lp, int N, int HP, int Np, int m_rt, float ikf,
                                          float lnkf, const float2 *__restrict__ cd1, const float2 *__restrict__ cd2,
                                          const G &gr, float acc[NS][6]) {
  const int m = MF > 0 ? MF : m_rt;
  float X[NS][6], Y[NS][6];
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int q = 0; q < 6; q++) acc[s][q] = 0.f;
  if (ip == 0 && jp == 0 && lp == 0) return;
#pragma unroll
  for (int a = 0; a < m; a++) {
    const int i = ip + a * Np, mi = i == 0 ? 0 : N - i;
#pragma unroll
    for (int b = 0; b < m; b++) {
      const int j = jp + b * Np, mj = j == 0 ? 0 : N - j;
#pragma unroll
      for (int c = 0; c < m; c++) {
        const int l = lp + c * Np;
        if (l > 0 && l < N / 2) {
          lpt_xf<NS>(i, j, l, N, HP, Np, ikf, lnkf, cd1, cd2, gr, X);
#pragma unroll
          for (int s = 0; s < NS; s++)
#pragma unroll
            for (int q = 0; q < 6; q++) acc[s][q] += X[s][q];
        } else if (l > N / 2) {
          lpt_xf<NS>(mi, mj, N - l, N, HP, Np, ikf, lnkf, cd1, cd2, gr, X);
#pragma unroll
          for (int s = 0; s < NS; s++)
#pragma unroll
            for (int q = 0; q < 3; q++) {
              acc[s][2 * q] += X[s][2 * q];
              acc[s][2 * q + 1] -= X[s][2 * q + 1];
            }
        } else if (PLANES) {  // kz = 0 or N/2 plane: (X(k) + conj X(-k)) / 2
          lpt_xf<NS>(i, j, l, N, HP, Np, ikf, lnkf, cd1, cd2, gr, X);
          lpt_xf<NS>(mi, mj, l, N, HP, Np, ikf, lnkf, cd1, cd2, gr, Y);
#pragma unroll
          for (int s = 0; s < NS; s++)
#pragma unroll
            for (int q = 0; q < 3; q++) {
              acc[s][2 * q] += 0.5f * (X[s][2 * q] + Y[s][2 * q]);
              acc[s][2 * q + 1] += 0.5f * (X[s][2 * q + 1] - Y[s][2 * q + 1]);
            }
        }
      }
    }
  }
}

// growth from per-|n|^2 tables, one slot; grid (Nsample^2 rows, kz blocks)
template <int MF>
__global__ __launch_bounds__(kBlock) void k_lpt_fold(const float2 *__restrict__ cd1, const float2 *__restrict__ cd2,
                                                     GTab gr, int N, int HP, int Np, int HPn, int m_rt, float ikf,
                                                     float2 *__restrict__ out, size_t nl) {
  const int lp = blockIdx.y * blockDim.x + threadIdx.x;
  if (lp > Np / 2) return;
  const unsigned row = blockIdx.x;
  const int jp = (int)(row % (unsigned)Np), ip = (int)(row / (unsigned)Np);
  float acc[1][6];
  fold_mode<MF, 1>(ip, jp, lp, N, HP, Np, m_rt, ikf, 0.f, cd1, cd2, gr, acc);
  const size_t e = (size_t)row * HPn + lp;
#pragma unroll
  for (int a = 0; a < 3; a++) out[a * nl + e] = make_float2(acc[0][2 * a], acc[0][2 * a + 1]);
}

// growth from the shared-grid ln k slices of NS slots (node-major float4s,
// copied once per block into LDS).  The blocks stride over the Nsample^2 rows, lpw
// (a power of two) lanes to a row and kFoldNT/lpw rows at a time; the interior kz of
// the rows first, then the kz = 0 and Nsample/2 modes of all rows.  Output spectrum
// (slot s, component a) at out + (3 s + a) nl.
// What bounds it: the slices of 1000 nodes take 48 KB, so blocks of 256 threads left
// three waves per SIMD, and a row of a 128 lattice 63 of the 256 lanes.
constexpr int kFoldNT = 512;
template <int MF, int NS>
__global__ __launch_bounds__(kFoldNT, 4) void k_lpt_fold_gs(const float2 *__restrict__ cd1,
                                                            const float2 *__restrict__ cd2,
                                                            const float4 *__restrict__ nodes, GShared<NS> gs,
                                                            float lnkf, int N, int HP, int Np, int HPn, int m_rt,
                                                            float ikf, int lpw, float2 *__restrict__ out, size_t nl) {
  extern __shared__ float4 sl[];
  const int nn = gs.ny * (1 + NS);
  for (int e = threadIdx.x; e < nn; e += kFoldNT) sl[e] = nodes[e];
  __syncthreads();
  gs.sl = sl;
  const unsigned rows = (unsigned)Np * (unsigned)Np, rpb = kFoldNT / lpw;
  const int H = Np / 2, l0 = (int)threadIdx.x & (lpw - 1);
  for (unsigned row = blockIdx.x * rpb + threadIdx.x / lpw; row < rows; row += gridDim.x * rpb) {
    const int jp = (int)(row % (unsigned)Np), ip = (int)(row / (unsigned)Np);
    for (int lp = l0 ? l0 : lpw; lp < H; lp += lpw) {
      float acc[NS][6];
      fold_mode<MF, NS, GShared<NS>, false>(ip, jp, lp, N, HP, Np, m_rt, ikf, lnkf, cd1, cd2, gs, acc);
      const size_t o = (size_t)row * HPn + lp;
#pragma unroll
      for (int s = 0; s < NS; s++)
#pragma unroll
        for (int a = 0; a < 3; a++) out[(3 * s + a) * nl + o] = make_float2(acc[s][2 * a], acc[s][2 * a + 1]);
    }
  }
  for (unsigned q = blockIdx.x * kFoldNT + threadIdx.x; q < 2 * rows; q += gridDim.x * kFoldNT) {
    const unsigned row = q >> 1;
    const int lp = (q & 1) ? H : 0;
    const int jp = (int)(row % (unsigned)Np), ip = (int)(row / (unsigned)Np);
    float acc[NS][6];
    fold_mode<MF, NS, GShared<NS>, true>(ip, jp, lp, N, HP, Np, m_rt, ikf, lnkf, cd1, cd2, gs, acc);
    const size_t o = (size_t)row * HPn + lp;
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
      for (int a = 0; a < 3; a++) out[(3 * s + a) * nl + o] = make_float2(acc[s][2 * a], acc[s][2 * a + 1]);
  }
}

// The fold of scale i n_a/n^2 X, a = 0..2, with the multipliers and the sums in FP64:
// component a's spectrum at out + a nl.  One thread per output mode, first the kz
// between the planes, row by row, then the kz = 0 and Nsample/2 modes of all rows, so
// that a wave takes one path.  Bound by the read of the mesh's spectrum, row segments
// of the m^2 aliases up and down (384 to 192: 105 us, 2.9 TB/s).
template <int MF, bool PLANES>
__device__ __forceinline__ void disp_fold(int ip, int jp, int lp, const float2 *__restrict__ X, int N, int HP, int Np,
                                          int m_rt, double acc[6]) {
  const int m = MF > 0 ? MF : m_rt;
#pragma unroll
  for (int q = 0; q < 6; q++) acc[q] = 0.0;
  if (ip == 0 && jp == 0 && lp == 0) return;
  // (re, im) += (wr, wi) (i n_a/n^2 X(i, j, l)), component by component
  auto add = [&](int i, int j, int l, double wr, double wi) {
    const float2 d = X[((size_t)i * N + j) * HP + l];
    const int n[3] = {kint(i, N), kint(j, N), kint(l, N)}, n2 = n[0] * n[0] + n[1] * n[1] + n[2] * n[2];
    const double w = n2 > 0 ? recip(n2) : 0.0, x = wr * w * d.y, y = wi * w * d.x;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      acc[2 * a] -= (double)n[a] * x;
      acc[2 * a + 1] += (double)n[a] * y;
    }
  };
#pragma unroll
  for (int a = 0; a < m; a++) {
    const int i = ip + a * Np, mi = i == 0 ? 0 : N - i;
#pragma unroll
    for (int b = 0; b < m; b++) {
      const int j = jp + b * Np, mj = j == 0 ? 0 : N - j;
#pragma unroll
      for (int c = 0; c < m; c++) {
        const int l = lp + c * Np;
        if (l > 0 && l < N / 2) {
          add(i, j, l, 1.0, 1.0);
        } else if (l > N / 2) {
          add(mi, mj, N - l, 1.0, -1.0);
        } else if (PLANES) {  // kz = 0 or N/2 plane: (X(k) + conj X(-k)) / 2
          add(i, j, l, 0.5, 0.5);
          add(mi, mj, l, 0.5, -0.5);
        }
      }
    }
  }
}
template <int MF>
__global__ __launch_bounds__(kBlock) void k_disp_fold(const float2 *__restrict__ X, int N, int HP, int Np, int HPn,
                                                      int m_rt, double scale, float2 *__restrict__ out, size_t nl,
                                                      size_t zs) {
  X = zbuf(X, zs);
  out = zbuf(out, zs);
  const size_t rows = (size_t)Np * Np, H = Np / 2, inner = rows * (H - 1);
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  double acc[6];
  size_t row;
  int lp;
  if (e < inner) {
    row = e / (H - 1);
    lp = 1 + (int)(e % (H - 1));
    disp_fold<MF, false>((int)(row / Np), (int)(row % Np), lp, X, N, HP, Np, m_rt, acc);
  } else {
    if (e >= inner + 2 * rows) return;
    row = (e - inner) >> 1;
    lp = (e - inner) & 1 ? (int)H : 0;
    disp_fold<MF, true>((int)(row / Np), (int)(row % Np), lp, X, N, HP, Np, m_rt, acc);
  }
#pragma unroll
  for (int a = 0; a < 3; a++)
    out[a * nl + row * HPn + lp] = make_float2((float)(scale * acc[2 * a]), (float)(scale * acc[2 * a + 1]));
}

__global__ __launch_bounds__(kBlock) void k_d2f(size_t n, const double *__restrict__ a, float *__restrict__ b) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (float)a[i];
}

// g_o(|n|^2) = norm_o num_o(ln k) / den_o(ln k) from cubic Hermite slices on a
// uniform ln k grid; t = [num, dnum, den, dden] (4*ny doubles)
struct KSl {
  double y0, dy, norm;
  int ny;
};
__device__ __forceinline__ double herm(const double *__restrict__ v, const double *__restrict__ dv, const KSl &s,
                                       double y) {
  const double ymax = s.y0 + s.dy * (s.ny - 1);
  if (y < s.y0) y = s.y0;
  if (y > ymax) y = ymax;
  int j = (int)floor((y - s.y0) / s.dy);
  if (j > s.ny - 2) j = s.ny - 2;
  if (j < 0) j = 0;
  const double h = s.dy, t = (y - (s.y0 + j * s.dy)) / h, t2 = t * t, t3 = t2 * t;
  return (2 * t3 - 3 * t2 + 1) * v[j] + (t3 - 2 * t2 + t) * h * dv[j] + (-2 * t3 + 3 * t2) * v[j + 1] +
         (t3 - t2) * h * dv[j + 1];
}
__global__ __launch_bounds__(kBlock) void k_growth_n2(size_t n2len, double kf, KSl s1, const double *__restrict__ t1,
                                                      KSl s2, const double *__restrict__ t2, double *__restrict__ g1,
                                                      double *__restrict__ g2, float *__restrict__ g1f,
                                                      float *__restrict__ g2f) {
  const size_t n2 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n2 >= n2len) return;
  double a = 0.0, b = 0.0;
  if (n2 > 0) {
    const double lk = log(kf * sqrt((double)n2));
    a = s1.norm * (herm(t1, t1 + s1.ny, s1, lk) / herm(t1 + 2 * s1.ny, t1 + 3 * s1.ny, s1, lk));
    b = s2.norm * (herm(t2, t2 + s2.ny, s2, lk) / herm(t2 + 2 * s2.ny, t2 + 3 * s2.ny, s2, lk));
  }
  g1[n2] = a;
  g2[n2] = b;
  g1f[n2] = (float)a;
  g2f[n2] = (float)b;
}

// ---------------------------------------------------------------- massive neutrinos
// The factor of PtoMesh's neutrino term per |n|^2 from a ln k slice:
// fac = norm num/den at ln(kf |n|) (OmegaNu/Omega N^3 T_nu(k, a)/T_cb(k, 1)).
__global__ __launch_bounds__(kBlock) void k_nu_fac(size_t n2len, double kf, KSl s, const double *__restrict__ t,
                                                   double *__restrict__ fac) {
  const size_t n2 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n2 >= n2len) return;
  double v = 0.0;
  if (n2 > 0) {
    const double lk = log(kf * sqrt((double)n2));
    v = s.norm * (herm(t, t + s.ny, s, lk) / herm(t + 2 * s.ny, t + 3 * s.ny, s, lk));
  }
  fac[n2] = v;
}

// PtoMesh's neutrino term (src/auxPM.c:383-420) on every stored mode but k = 0:
// delta = cdmfac delta + fac(|n|^2) cdelta_IC, in FP64 as the reference.  Grid
// (N*N rows, kz blocks).
__global__ __launch_bounds__(kBlock) void k_nu_add(float2 *__restrict__ dk, const float2 *__restrict__ cd, int N,
                                                   int HP, const double *__restrict__ fac, double cdmfac) {
  const int k = blockIdx.y * blockDim.x + threadIdx.x;
  if (k > N / 2) return;
  const unsigned row = blockIdx.x;
  const int j = (int)(row % (unsigned)N), i = (int)(row / (unsigned)N);
  if (i == 0 && j == 0 && k == 0) return;
  const int d0 = i > N / 2 ? N - i : i, d1 = j > N / 2 ? N - j : j;
  const double f = fac[d0 * d0 + d1 * d1 + k * k];
  const size_t e = (size_t)row * HP + k;
  const float2 v = dk[e], c = cd[e];
  dk[e] = make_float2((float)(cdmfac * (double)v.x + f * (double)c.x), (float)(cdmfac * (double)v.y + f * (double)c.y));
}

// Waits for the stream on every way out of the block: the host memory that it copies
// from stays until the copies are done, also where a later call fails.
struct StreamWait {
  mgpu_ctx *ctx;
  ~StreamWait() {
    if (ctx) (void)hipStreamSynchronize(ctx->stream);
  }
};

// The seed tables of count realizations (ctx's, at the batch stride) into table (on the
// device): the states the chunks of each stream start from go to slot 1, which the
// initial conditions overwrite afterwards.  A chunk is 16 advances of 12 values, or
// what makes 2048 chunks; in small tables, which the chunks' own length would hold up, as
// many as balance the host's jumps (0.35 us each) with a thread's advances (3.4 us each):
// scale-dependent initial conditions 236 -> 145 us at 16, 262 -> 180 us at 32 (202 and 231
// us with the table made by the host).
// inverted (or nullptr): the realizations' inversion flags, one behind each table.
int seed_tables(mgpu_ctx *ctx, int count, const unsigned long *seeds, const int *inverted, unsigned *table,
                std::vector<double> &st) {
  const int N = ctx->N;
  const unsigned advances = cdiv((size_t)N * N, 12);
  const unsigned adv = std::max({1u, std::min(16u, (unsigned)std::lround(std::sqrt(advances / 9.7))), cdiv(advances, 2048)});
  const unsigned n = cdiv(advances, adv);
  const size_t len = 13 * (size_t)n + 1;
  if (len * sizeof(double) > ctx->slot_elems * sizeof(float2))
    return mgpu_fail(ctx, MGPU_E_INVALID, "seed states do not fit a mesh slot");
  const rlx::Num jump = rlx::step_power(202ull * adv);
  st.resize(len * count);
  for (int r = 0; r < count; r++) {
    double *o = st.data() + len * r;
    Ranlxd1 g;
    g.seed(seeds[r]);
    rlx::Num X = rlx::from_state(g);
    for (unsigned t = 0; t < n; t++) {
      for (int q = 0; q < 12; q++) o[(size_t)q * n + t] = g.y[q];
      o[(size_t)12 * n + t] = g.carry;
      if (t + 1 < n) rlx::to_state(X = rlx::mul(X, jump), g);
    }
    o[len - 1] = inverted && inverted[r] ? 1.0 : 0.0;
    MGPU_HIP(ctx, hipMemcpyAsync((char *)ctx->slot[1] + ctx->zs * r, o, len * sizeof(double), hipMemcpyHostToDevice,
                                 ctx->stream));
  }
  hipLaunchKernelGGL(k_seed_table, dim3(cdiv(n, 64), 1, count), dim3(64), 0, ctx->stream, (const double *)ctx->slot[1],
                     n, adv, N, inverted != nullptr, table, ctx->zs);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

int spectrum(mgpu_ctx *ctx, int mode, const float2 *cd, const float2 *cd2, float2 *out, int a,
             const double *g1 = nullptr, const double *g2 = nullptr) {
  const double kf = 2 * MGPU_PI / ctx->p.box;
  const double modes = (double)ctx->N * ctx->N * (ctx->N / 2 + 1);
  {
    KScope ks(ctx, MGPU_K_LPT, 8.0 * modes * (cd2 ? 3 : 2));
    hipLaunchKernelGGL(k_lpt_spectrum, dim3(cdiv(ctx->slot_elems, kBlock), 1, ctx->bz), dim3(kBlock), 0, ctx->stream,
                       mode, cd, cd2, out, ctx->N, ctx->HP, kf, a, g1, g2, ctx->zs);
  }
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

// lattice read-out of a real mesh into dst ([np] floats) with mean removal
int readout(mgpu_ctx *ctx, const float2 *mesh, double scale, float *dst) {
  const size_t np = ctx->np;
  const unsigned nb = cdiv(np, kBlock);
  {
    // compulsory: one mesh sample read and one float written per lattice point
    KScope ks(ctx, MGPU_K_READOUT, 8.0 * np);
    hipLaunchKernelGGL(k_lattice_read, dim3(nb, 1, ctx->bz), dim3(kBlock), 0, ctx->stream, (const float *)mesh, ctx->N,
                       ctx->Np, 2 * ctx->HP, scale, dst, ctx->partial, ctx->zs);
  }
  MGPU_HIP(ctx, hipGetLastError());
  hipLaunchKernelGGL(k_reduce1, dim3(1, 1, ctx->bz), dim3(1024), 0, ctx->stream, ctx->partial, (int)nb, ctx->dsum,
                     ctx->zs);
  MGPU_HIP(ctx, hipGetLastError());
  hipLaunchKernelGGL(k_sub_mean, dim3(nb, 1, ctx->bz), dim3(kBlock), 0, ctx->stream, dst, np, ctx->dsum,
                     1.0 / (double)np, ctx->zs);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

int upload_n2(mgpu_ctx *ctx, int which, const double *h) {
  MGPU_HIP(ctx, hipMemcpyAsync(ctx->n2tab[which], h, ctx->n2len * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_d2f, dim3(cdiv(ctx->n2len, kBlock)), dim3(kBlock), 0, ctx->stream, ctx->n2len,
                     (const double *)ctx->n2tab[which], ctx->n2tabf[which]);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

}  // namespace

// The device address of this GPU's seed-table scratch, looked up once per
// device (with that device current) and kept for the process.
int ic_scratch_init(mgpu_ctx *ctx) {
  if (ctx->device < 0 || ctx->device >= kMaxDevices)
    return mgpu_fail(ctx, MGPU_E_INVALID, "device index beyond the seed-table scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[ctx->device]) {
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      (void)hipGetLastError();
      return mgpu_fail(ctx, MGPU_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    }
    g_scratch_ptr[ctx->device] = (unsigned *)p;
  }
  ctx->ic_scratch = g_scratch_ptr[ctx->device];
  return MGPU_OK;
}

// displacement_fields.  The seed table goes to seed_dev (the per-device scratch) or,
// with nullptr, to slot 2 (work space of the initial conditions); nothing is
// allocated on the device either way.
int ic_displacement_fields(mgpu_ctx *ctx, unsigned long seed, int sphere_mode, int amp_fixed, int inverted,
                           const double *pk_n2, unsigned *seed_dev) {
  PhaseTimer pt(ctx, &ctx->t.ic);
  const int N = ctx->N;
  int rc;
  std::vector<double> st;
  StreamWait wait{ctx};
  unsigned *dseed = seed_dev ? seed_dev : (unsigned *)ctx->slot[2];
  if ((rc = seed_tables(ctx, 1, &seed, nullptr, dseed, st))) return rc;
  if ((rc = upload_n2(ctx, 0, pk_n2))) return rc;
  float2 *cd = ctx->p.scale_dependent ? ctx->cdelta[0] : ctx->slot[0];
  MGPU_HIP(ctx, hipMemsetAsync(cd, 0, ctx->slot_elems * sizeof(float2), ctx->stream));
  hipLaunchKernelGGL(k_ic_delta, dim3(cdiv((size_t)N * N, kBlock)), dim3(kBlock), 0, ctx->stream, dseed, N, ctx->Np,
                     ctx->HP, ctx->p.box, sphere_mode, amp_fixed, inverted, ctx->n2tab[0], cd, (size_t)0,
                     (const int *)nullptr);
  MGPU_HIP(ctx, hipGetLastError());
  if ((rc = ic_lpt_from_delta(ctx, cd))) return rc;
  wait.ctx = nullptr;
  MGPU_HIP(ctx, hipStreamSynchronize(ctx->stream));  // the uploads' host memory goes out of scope
  return MGPU_OK;
}

// The lattice displacements i k_a/k^2 X scale of spectrum X in slot in (0 or 1), mean
// removed, into LPT slot o; slots 2 and 3 are work space.  Where the mesh is a multiple
// of the lattice the read-out has weight 1 on one node, and the spectra are folded onto
// the lattice's own (192 of 384: three
// fields in 205 us with their transforms, where each took 500 us on the mesh); else, and at Nmesh =
// Nsample where there is nothing to fold, the mesh's transform is read out.
static int ic_read_displacements(mgpu_ctx *ctx, const float2 *X, double scale, int o) {
  int rc;
  if (ctx->fft_read.n > 0) {
    const FFTPlan *plan = &ctx->fft_read;
    const int Np = ctx->Np, m = ctx->N / Np;
    const size_t nl = (size_t)Np * Np * plan->hp;  // 3 nl <= N^2 HP: m >= 2
    float2 *buf = ctx->slot[2];
    {
      KScope ks(ctx, MGPU_K_LPT, ctx->bz * 8.0 * ((double)ctx->N * ctx->N * (ctx->N / 2 + 1) + 3.0 * Np * Np * (Np / 2 + 1)));
      auto kern = m == 2 ? k_disp_fold<2> : m == 3 ? k_disp_fold<3> : k_disp_fold<0>;
      hipLaunchKernelGGL(kern, dim3(cdiv((size_t)Np * Np * (Np / 2 + 1), kBlock), 1, ctx->bz), dim3(kBlock), 0,
                         ctx->stream, X, ctx->N, ctx->HP, Np, plan->hp, m, scale * ctx->p.box / (2 * MGPU_PI), buf, nl,
                         ctx->zs);
    }
    MGPU_HIP(ctx, hipGetLastError());
    if (ctx->bz == 1) {
      float *out[2] = {ctx->lpt[o], nullptr};
      return fft_c2r_fields(ctx, plan, buf, nl, 1, out, ctx->np);
    }
    for (int a = 0; a < 3; a++)
      if ((rc = fft_c2r_3d(ctx, plan, buf + a * nl, ctx->lpt[o] + a * ctx->np))) return rc;
    return MGPU_OK;
  }
  for (int a = 0; a < 3; a++) {
    if ((rc = lpt_x_pass(ctx, X, ctx->slot[3], nullptr, nullptr, LptFields{1, {a}, {-1}}))) return rc;
    if ((rc = fft_pass_col(ctx, &ctx->fft, ctx->slot[3], 1, 0))) return rc;
    if ((rc = fft_pass_z(ctx, &ctx->fft, ctx->slot[3], 0))) return rc;
    if ((rc = readout(ctx, ctx->slot[3], scale, ctx->lpt[o] + (size_t)a * ctx->np))) return rc;
  }
  return MGPU_OK;
}

// From delta(k) in cd on: the 2LPT source and the ZA and 2LPT lattice
// displacements (or, scale-dependent, the stored -source).  Every launch covers
// ctx->bz realizations (a batch's member 0 with bz = count).
int ic_lpt_from_delta(mgpu_ctx *ctx, float2 *cd) {
  int rc;
  const FFTPlan *plan = &ctx->fft;
  float2 *s = ctx->slot[1], *d1 = ctx->slot[2], *d2 = ctx->slot[3];
  // displacement gradients -> 2LPT source, built in slot 1 with two more slots of work
  // space: the diagonal ones, two off the diagonal, the last one and the r2c
  if ((rc = lpt_x_pass(ctx, cd, s, d1, d2, LptFields{3, {0, 1, 2}, {0, 1, 2}}))) return rc;
  for (float2 *d : {s, d1, d2})
    if ((rc = fft_pass_col(ctx, plan, d, 1, 0))) return rc;
  if ((rc = lpt_source_pass(ctx, LPT_DIAG, s, d1, d2))) return rc;
  if ((rc = lpt_x_pass(ctx, cd, d1, d2, nullptr, LptFields{2, {0, 0}, {1, 2}}))) return rc;
  for (float2 *d : {d1, d2})
    if ((rc = fft_pass_col(ctx, plan, d, 1, 0))) return rc;
  if ((rc = lpt_source_pass(ctx, LPT_OFF2, s, d1, d2))) return rc;
  if ((rc = lpt_x_pass(ctx, cd, d1, nullptr, nullptr, LptFields{1, {1}, {2}}))) return rc;
  if ((rc = fft_pass_col(ctx, plan, d1, 1, 0))) return rc;
  if ((rc = lpt_source_pass(ctx, LPT_OFF1, s, d1, nullptr))) return rc;
  if ((rc = fft_pass_col(ctx, plan, s, 1, 1))) return rc;
  if ((rc = fft_pass_col(ctx, plan, s, 0, 1))) return rc;

  if (ctx->p.scale_dependent) return spectrum(ctx, SPEC_NEG, s, nullptr, ctx->cdelta[1], 0);
  // ZA and 2LPT displacements at the lattice, mean removed (cdisp, src/2LPT.c:417-490;
  // cdisp2 = -i k_a/k^2 src, src/2LPT.c:1359-1370, read out with -3/7 N^-3)
  const double inv_n3 = 1.0 / ((double)ctx->N * ctx->N * ctx->N);
  if ((rc = ic_read_displacements(ctx, cd, 1.0, 0))) return rc;
  if ((rc = ic_read_displacements(ctx, s, 3. / 7. * inv_n3, 1))) return rc;
  MGPU_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return MGPU_OK;
}

int ic_displacement_fields_batch(mgpu_ctx *const *m, int count, const unsigned long *seeds, int sphere_mode,
                                 int amp_fixed, const int *inverted, const double *pk_n2) {
  mgpu_ctx *ctx = m[0];
  PhaseTimer pt(ctx, &ctx->t.ic);
  if (ctx->p.scale_dependent)
    return mgpu_fail(ctx, MGPU_E_STATE, "batched initial conditions: not for scale-dependent runs");
  const int N = ctx->N;
  const size_t nn = (size_t)N * N;
  int rc;
  std::vector<double> st;
  StreamWait wait{ctx};
  // the seed tables, and behind them the inversion flags, in the members' slot 2
  if ((rc = seed_tables(ctx, count, seeds, inverted, (unsigned *)ctx->slot[2], st))) return rc;
  for (int r = 0; r < count; r++) {
    // every member holds the table (later calls on a member alone read its own)
    if ((rc = upload_n2(m[r], 0, pk_n2))) return rc;
    MGPU_HIP(ctx, hipMemsetAsync(m[r]->slot[0], 0, ctx->slot_elems * sizeof(float2), ctx->stream));
  }
  struct Restore {
    mgpu_ctx *c;
    ~Restore() { c->bz = 1; }
  } restore{ctx};
  ctx->bz = (unsigned)count;
  float2 *cd = ctx->slot[0];
  hipLaunchKernelGGL(k_ic_delta, dim3(cdiv(nn, kBlock), 1, count), dim3(kBlock), 0, ctx->stream,
                     (const unsigned *)ctx->slot[2], N, ctx->Np, ctx->HP, ctx->p.box, sphere_mode, amp_fixed, 0,
                     ctx->n2tab[0], cd, ctx->zs, (const int *)ctx->slot[2] + nn);
  MGPU_HIP(ctx, hipGetLastError());
  if ((rc = ic_lpt_from_delta(ctx, cd))) return rc;
  wait.ctx = nullptr;
  MGPU_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return MGPU_OK;
}

int ic_init_particles(mgpu_ctx *ctx, double Di, double Di2) {
  PhaseTimer pt(ctx, &ctx->t.ic);
  if (ctx->np == 0) return MGPU_OK;
  hipLaunchKernelGGL(k_init_particles, dim3(cdiv(ctx->np, kBlock)), dim3(kBlock), 0, ctx->stream, ctx->pos, ctx->vel,
                     ctx->lpt[0], ctx->lpt[1], ctx->Np, ctx->p.box, ctx->p.scale_dependent, Di, Di2,
                     ctx->p.use_cola, 0.0, 0.0);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

// shared-grid slices as the fold kernel takes them (node float4s in ctx->slice_buf)
struct SliceFold {
  float y0, dy, idy, ymax, norm1, norm2;
  int ny;
};

template <int MF, int NS>
int launch_fold_gs(mgpu_ctx *ctx, const SliceFold &f, float lnkf, float ikf, float2 *out, size_t nl) {
  GShared<NS> gs{};
  gs.sl = nullptr;
  gs.y0 = f.y0;
  gs.dy = f.dy;
  gs.idy = f.idy;
  gs.ymax = f.ymax;
  gs.norm1 = f.norm1;
  gs.norm2 = f.norm2;
  gs.ny = f.ny;
  const int Np = ctx->Np;
  const size_t lds = sizeof(float4) * (size_t)f.ny * (1 + NS);
  int lpw = 16;
  while (lpw < Np / 2 && lpw < kFoldNT) lpw *= 2;
  // as many blocks as the LDS and the registers keep resident, each copying the slices once
  // (both slots at 512 / 768 with 256 particles a side: 912 / 1412 us; twice as many blocks
  // 1004 / 1648 us, four times 929 / 1431; up to 256 the three are equal)
  const unsigned per_cu = (unsigned)std::max<size_t>(1, std::min<size_t>(2, ctx->lds_max / std::max<size_t>(lds, 1)));
  const unsigned nb = (unsigned)std::min<size_t>(cdiv((size_t)Np * Np, kFoldNT / lpw), (size_t)ctx->cus * per_cu);
  hipLaunchKernelGGL((k_lpt_fold_gs<MF, NS>), dim3(nb), dim3(kFoldNT), lds, ctx->stream, ctx->cdelta[0],
                     ctx->cdelta[1], (const float4 *)ctx->slice_buf, gs, lnkf, ctx->N, ctx->HP, Np,
                     ctx->fft_lattice.hp, ctx->N / Np, ikf, lpw, out, nl);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}

// LPT fields of ns slots (slots[s]).  With sl (shared-grid growth slices of
// every slot, already in ctx->slice_buf) the lattice fold evaluates the growth
// in LDS; otherwise (ns = 1) from the n2 tables.
static int lattice_fields(mgpu_ctx *ctx, int ns, const int *slots, const SliceFold *sl) {
  int rc;
  if (ctx->lattice_slot) {
    // exact lattice fold: N = m * Nsample; spectrum (s, a) at lattice_slot + (3 s + a) nl
    const int Np = ctx->Np, HPn = ctx->fft_lattice.hp, m = ctx->N / Np;
    const size_t nl = (size_t)Np * Np * HPn;
    const float ikf = (float)(ctx->p.box / (2 * MGPU_PI)), lnkf = (float)std::log(2 * MGPU_PI / ctx->p.box);
    {
      // compulsory: both stored spectra read once (the 1LPT one inside the IC cube only), 3 ns folded outputs written
      const double modes = (double)ctx->N * ctx->N * (ctx->N / 2 + 1);
      KScope ks(ctx, MGPU_K_FOLD, 8.0 * modes * (1.0 + 1.0 / (double)(m * m * m)) + 3.0 * ns * 8.0 * nl);
      if (sl && ns == 2) {
        rc = m == 1 ? launch_fold_gs<1, 2>(ctx, *sl, lnkf, ikf, ctx->lattice_slot, nl)
             : m == 2 ? launch_fold_gs<2, 2>(ctx, *sl, lnkf, ikf, ctx->lattice_slot, nl)
             : m == 3 ? launch_fold_gs<3, 2>(ctx, *sl, lnkf, ikf, ctx->lattice_slot, nl)
                      : launch_fold_gs<0, 2>(ctx, *sl, lnkf, ikf, ctx->lattice_slot, nl);
      } else if (sl) {
        rc = m == 1 ? launch_fold_gs<1, 1>(ctx, *sl, lnkf, ikf, ctx->lattice_slot, nl)
             : m == 2 ? launch_fold_gs<2, 1>(ctx, *sl, lnkf, ikf, ctx->lattice_slot, nl)
             : m == 3 ? launch_fold_gs<3, 1>(ctx, *sl, lnkf, ikf, ctx->lattice_slot, nl)
                      : launch_fold_gs<0, 1>(ctx, *sl, lnkf, ikf, ctx->lattice_slot, nl);
      } else {
        auto kern = m == 1 ? k_lpt_fold<1> : m == 2 ? k_lpt_fold<2> : m == 3 ? k_lpt_fold<3> : k_lpt_fold<0>;
        hipLaunchKernelGGL(kern, dim3((unsigned)((size_t)Np * Np), cdiv(Np / 2 + 1, kBlock)), dim3(kBlock), 0,
                           ctx->stream, ctx->cdelta[0], ctx->cdelta[1], GTab{ctx->n2tabf[0], ctx->n2tabf[1]}, ctx->N,
                           ctx->HP, Np, HPn, m, ikf, ctx->lattice_slot, nl);
        rc = MGPU_OK;
      }
      if (rc) return rc;
    }
    MGPU_HIP(ctx, hipGetLastError());
    // the 3 ns fields' transforms, one launch per pass (the z pass one per slot)
    float *out[2] = {ctx->lpt[slots[0]], ns > 1 ? ctx->lpt[slots[1]] : nullptr};
    return fft_c2r_fields(ctx, &ctx->fft_lattice, ctx->lattice_slot, nl, ns, out, ctx->np);
  }
  if (ns != 1) return mgpu_fail(ctx, MGPU_E_INVALID, "several LPT slots at once need the lattice fold");
  for (int a = 0; a < 3; a++) {
    if ((rc = spectrum(ctx, SPEC_FIELD, ctx->cdelta[0], ctx->cdelta[1], ctx->slot[3], a, ctx->n2tab[0],
                       ctx->n2tab[1])))
      return rc;
    if ((rc = fft_c2r_3d(ctx, &ctx->fft, ctx->slot[3]))) return rc;
    if ((rc = readout(ctx, ctx->slot[3], 1.0, ctx->lpt[slots[0]] + (size_t)a * ctx->np))) return rc;
  }
  return MGPU_OK;
}

// pinned host staging of n bytes; the previous upload from it must be complete before it is refilled
static int slice_staging(mgpu_ctx *ctx, size_t bytes, void **host) {
  if (ctx->slice_ev) MGPU_HIP(ctx, hipEventSynchronize(ctx->slice_ev));
  else MGPU_HIP(ctx, hipEventCreateWithFlags(&ctx->slice_ev, hipEventDisableTiming));
  const size_t nd = (bytes + sizeof(double) - 1) / sizeof(double);
  if (ctx->slice_host_len < nd) {
    if (ctx->slice_host) MGPU_HIP(ctx, hipHostFree(ctx->slice_host));
    ctx->slice_host = nullptr;
    MGPU_HIP(ctx, hipHostMalloc((void **)&ctx->slice_host, nd * sizeof(double), hipHostMallocDefault));
    ctx->slice_host_len = nd;
  }
  if (!ctx->slice_buf || ctx->slice_len < nd) {
    if (ctx->slice_buf) {
      MGPU_HIP(ctx, hipStreamSynchronize(ctx->stream));
      MGPU_HIP(ctx, hipFree(ctx->slice_buf));
    }
    ctx->slice_buf = nullptr;
    MGPU_HIP(ctx, hipMalloc(&ctx->slice_buf, nd * sizeof(double)));
    ctx->slice_len = nd;
  }
  *host = ctx->slice_host;
  return MGPU_OK;
}
static int slice_upload(mgpu_ctx *ctx, size_t bytes) {
  MGPU_HIP(ctx, hipMemcpyAsync(ctx->slice_buf, ctx->slice_host, bytes, hipMemcpyHostToDevice, ctx->stream));
  MGPU_HIP(ctx, hipEventRecord(ctx->slice_ev, ctx->stream));
  return MGPU_OK;
}

// ns slots, slices q[2 s + o] for (slot s, order o + 1)
int ic_lpt_fields_slices_n(mgpu_ctx *ctx, int ns, const int *slots, const mgpu_kslice *const *q) {
  PhaseTimer pt(ctx, &ctx->t.lpt_fields);
  if (!ctx->p.scale_dependent) return mgpu_fail(ctx, MGPU_E_STATE, "LPT fields need a scale-dependent context");
  for (int e = 0; e < 2 * ns; e++)
    if (!q[e] || q[e]->nk < 2 || q[e]->nk > 8192 || q[e]->dlnk <= 0)
      return mgpu_fail(ctx, MGPU_E_INVALID, "bad growth slice");
  const int ny = q[0]->nk;
  // the shared-grid fold needs one ln k grid for every slice, and (two slots) the
  // same denominators and norms in both slots
  bool shared = ctx->lattice_slot != nullptr && 16 * (size_t)ny * (1 + ns) <= 65536;
  for (int e = 1; e < 2 * ns && shared; e++)
    shared = q[e]->nk == ny && q[e]->lnk0 == q[0]->lnk0 && q[e]->dlnk == q[0]->dlnk;
  for (int o = 0; o < 2 && shared && ns == 2; o++)
    shared = q[2 + o]->norm == q[o]->norm && std::equal(q[o]->den, q[o]->den + ny, q[2 + o]->den) &&
             std::equal(q[o]->dden, q[o]->dden + ny, q[2 + o]->dden);
  if (!shared && ns == 2) {
    int rc = ic_lpt_fields_slices_n(ctx, 1, slots, q);
    return rc ? rc : ic_lpt_fields_slices_n(ctx, 1, slots + 1, q + 2);
  }
  int rc;
  if (shared) {
    const size_t bytes = sizeof(float) * 4 * (size_t)ny * (1 + ns);
    void *h;
    if ((rc = slice_staging(ctx, bytes, &h))) return rc;
    float *f = (float *)h;
    for (int j = 0; j < ny; j++) {
      *f++ = (float)q[0]->den[j];
      *f++ = (float)q[0]->dden[j];
      *f++ = (float)q[1]->den[j];
      *f++ = (float)q[1]->dden[j];
      for (int s = 0; s < ns; s++) {
        *f++ = (float)q[2 * s]->num[j];
        *f++ = (float)q[2 * s]->dnum[j];
        *f++ = (float)q[2 * s + 1]->num[j];
        *f++ = (float)q[2 * s + 1]->dnum[j];
      }
    }
    if ((rc = slice_upload(ctx, bytes))) return rc;
    SliceFold sf;
    sf.y0 = (float)q[0]->lnk0;
    sf.dy = (float)q[0]->dlnk;
    sf.idy = (float)(1.0 / q[0]->dlnk);
    sf.ymax = (float)(q[0]->lnk0 + q[0]->dlnk * (ny - 1));
    sf.norm1 = (float)q[0]->norm;
    sf.norm2 = (float)q[1]->norm;
    sf.ny = ny;
    return lattice_fields(ctx, ns, slots, &sf);
  }
  // general slices: the per-|n|^2 growth tables first (FP64 Hermite), then the table path
  const size_t total = 4 * (size_t)(q[0]->nk + q[1]->nk);
  void *h;
  if ((rc = slice_staging(ctx, total * sizeof(double), &h))) return rc;
  double *p = (double *)h;
  for (int e = 0; e < 2; e++)
    for (const double *src : {q[e]->num, q[e]->dnum, q[e]->den, q[e]->dden}) {
      std::copy(src, src + q[e]->nk, p);
      p += q[e]->nk;
    }
  if ((rc = slice_upload(ctx, total * sizeof(double)))) return rc;
  const KSl k0{q[0]->lnk0, q[0]->dlnk, q[0]->norm, q[0]->nk}, k1{q[1]->lnk0, q[1]->dlnk, q[1]->norm, q[1]->nk};
  hipLaunchKernelGGL(k_growth_n2, dim3(cdiv(ctx->n2len, kBlock)), dim3(kBlock), 0, ctx->stream, ctx->n2len,
                     2 * MGPU_PI / ctx->p.box, k0, (const double *)ctx->slice_buf, k1,
                     (const double *)ctx->slice_buf + 4 * q[0]->nk, ctx->n2tab[0], ctx->n2tab[1], ctx->n2tabf[0],
                     ctx->n2tabf[1]);
  MGPU_HIP(ctx, hipGetLastError());
  return lattice_fields(ctx, 1, slots, nullptr);
}

int ic_lpt_fields_slices(mgpu_ctx *ctx, int slot, const mgpu_kslice *o1, const mgpu_kslice *o2) {
  const mgpu_kslice *q[2] = {o1, o2};
  return ic_lpt_fields_slices_n(ctx, 1, &slot, q);
}

int ic_lpt_fields(mgpu_ctx *ctx, int slot, const double *g1_n2, const double *g2_n2) {
  PhaseTimer pt(ctx, &ctx->t.lpt_fields);
  if (!ctx->p.scale_dependent) return mgpu_fail(ctx, MGPU_E_STATE, "LPT fields need a scale-dependent context");
  int rc;
  if ((rc = upload_n2(ctx, 0, g1_n2))) return rc;
  if ((rc = upload_n2(ctx, 1, g2_n2))) return rc;
  if ((rc = lattice_fields(ctx, 1, &slot, nullptr))) return rc;
  MGPU_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return MGPU_OK;
}


// the neutrino term's factors for the next PtoMesh (f == NULL: off)
int ic_nu_set(mgpu_ctx *ctx, double cdmfac, const mgpu_kslice *f) {
  if (!f) {
    ctx->nu_on = false;
    return MGPU_OK;
  }
  if (!f->num || !f->dnum || !f->den || !f->dden || f->nk < 2 || f->nk > 8192 || f->dlnk <= 0)
    return mgpu_fail(ctx, MGPU_E_INVALID, "bad neutrino slice");
  if (!ctx->cdelta[0]) return mgpu_fail(ctx, MGPU_E_STATE, "the neutrino term needs the stored IC spectrum (scale-dependent context)");
  const size_t n = 4 * (size_t)f->nk;
  std::vector<double> h(n);
  std::copy(f->num, f->num + f->nk, h.begin());
  std::copy(f->dnum, f->dnum + f->nk, h.begin() + f->nk);
  std::copy(f->den, f->den + f->nk, h.begin() + 2 * f->nk);
  std::copy(f->dden, f->dden + f->nk, h.begin() + 3 * f->nk);
  if (ctx->nu_slice_len < n) {
    MGPU_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (ctx->nu_slice) MGPU_HIP(ctx, hipFree(ctx->nu_slice));
    ctx->nu_slice = nullptr;
    MGPU_HIP(ctx, hipMalloc((void **)&ctx->nu_slice, n * sizeof(double)));
    ctx->nu_slice_len = n;
  }
  if (!ctx->nu_fac) MGPU_HIP(ctx, hipMalloc((void **)&ctx->nu_fac, ctx->n2len * sizeof(double)));
  MGPU_HIP(ctx, hipMemcpyAsync(ctx->nu_slice, h.data(), n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
  const KSl ks{f->lnk0, f->dlnk, f->norm, f->nk};
  hipLaunchKernelGGL(k_nu_fac, dim3(cdiv(ctx->n2len, kBlock)), dim3(kBlock), 0, ctx->stream, ctx->n2len,
                     2 * MGPU_PI / ctx->p.box, ks, (const double *)ctx->nu_slice, ctx->nu_fac);
  MGPU_HIP(ctx, hipGetLastError());
  MGPU_HIP(ctx, hipStreamSynchronize(ctx->stream));  // h goes out of scope
  ctx->nu_cdmfac = cdmfac;
  ctx->nu_on = true;
  return MGPU_OK;
}

// the neutrino term on delta(k) in slot 0
int ic_nu_apply(mgpu_ctx *ctx) {
  if (!ctx->nu_on) return mgpu_fail(ctx, MGPU_E_STATE, "no neutrino factors: call mgpu_set_neutrinos first");
  const int N = ctx->N;
  KScope ks(ctx, MGPU_K_SPECTRAL, 24.0 * (double)N * N * (N / 2 + 1));
  hipLaunchKernelGGL(k_nu_add, dim3((unsigned)((size_t)N * N), cdiv((size_t)(N / 2 + 1), kBlock)), dim3(kBlock), 0,
                     ctx->stream, ctx->slot[0], ctx->cdelta[0], N, ctx->HP, (const double *)ctx->nu_fac,
                     ctx->nu_cdmfac);
  MGPU_HIP(ctx, hipGetLastError());
  return MGPU_OK;
}
