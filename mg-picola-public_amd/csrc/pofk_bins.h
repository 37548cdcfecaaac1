// P(k) bin of a mode from its |n|^2, shared by the passes that bin P(k).
//
// The bin is compute_power_spectrum's FP64 formula (src/compute_pofk.c:112-126),
// which rises with |n|^2, so the host evaluates it once and keeps each bin's first
// |n|^2 (edge[b], b = 0..nbins; edge[nbins] ends the last bin).  A lane estimates the
// bin in FP32 and corrects it against the edges, so every mode falls in exactly the
// formula's bin.  The edges are a few KB, read from LDS; a table of the bin of every
// |n|^2 (1.5 MB at 1024) costs a gather whose 64 lanes touch up to 64 cache lines:
// the density x pass that bins P(k) at 1024 took 4.79 ms with it against 3.78 ms
// without binning.  Bins too many for their edges to share the LDS, or that do not rise
// with |n|^2 (a last bin below the first), are taken from the table.
#pragma once
#include <hip/hip_runtime.h>

struct PkBinFn {
  const int *edge = nullptr;       // nbins + 1 first |n|^2 of the bins (device memory)
  const int16_t *table = nullptr;  // bin of every |n|^2, -1 outside (device memory)
  int nbins = 0, logbins = 0;
  float a = 0.f, b = 0.f;  // estimate: a |n| + b, or a log2 |n|^2 + b
};

// e: the edges (LDS or global), e0 = e[0], e1 = e[nbins]; -1 outside the bins
static __device__ __forceinline__ int pk_bin_of(int n2, const PkBinFn &f, const int *e, int e0, int e1) {
  if (n2 < e0 || n2 >= e1) return -1;
  const float x = f.logbins ? __log2f((float)n2) * f.a + f.b : sqrtf((float)n2) * f.a + f.b;
  int nk = min(max((int)x, 0), f.nbins - 1);
  // e0 <= n2 < e1 and the edges rise, so both walks end inside the bins
  while (n2 < e[nk]) --nk;
  while (n2 >= e[nk + 1]) ++nk;
  return nk;
}
