// stencil27.h -- what the multigrid kernels' translation units share: the
// batched-launch argument container, indexing and the 27-point stencil.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>

#include "pmg_device.h"

namespace pmg {
namespace {

constexpr int kBlock = 256;

// Kernel-argument container of a batched launch: one argument set per
// calculation (at most kMaxBatch).
template <class P>
struct Batch {
  P v[kMaxBatch];
};

__host__ __device__ inline size_t IX(int i, int j, int k, int nx, int ny) {
  return ((size_t)k * ny + j) * nx + i;
}

inline dim3 grid_interior(int nx, int ny, int nz) {
  long cnt = (long)(nx - 2) * (ny - 2);
  return dim3((unsigned)((cnt + kBlock - 1) / kBlock), (unsigned)(nz - 2), 1);
}

// Vectors of 16 or 8 bytes at any element alignment, and windows of N + 2
// elements.
template <class T, int N>
__device__ __forceinline__ void vld16(T (&v)[N], const T* p) {
  static_assert(sizeof(T) * N == 16 || sizeof(T) * N == 8, "8- or 16-byte vectors");
  typedef T vT __attribute__((ext_vector_type(N)));
  vT a;
  __builtin_memcpy(&a, p, sizeof(T) * N);
#pragma unroll
  for (int i = 0; i < N; i++) v[i] = a[i];
}

template <class T, int N>
__device__ __forceinline__ void vst16(T* p, const T (&v)[N]) {
  static_assert(sizeof(T) * N == 16 || sizeof(T) * N == 8, "8- or 16-byte vectors");
  typedef T vT __attribute__((ext_vector_type(N)));
  vT a;
#pragma unroll
  for (int i = 0; i < N; i++) a[i] = v[i];
  __builtin_memcpy(p, &a, sizeof(T) * N);
}

template <class T, int N>
__device__ __forceinline__ void vldw(T (&w)[N + 2], const T* p) {
  static_assert(sizeof(T) * N == 16 || sizeof(T) * N == 8, "8- or 16-byte vectors");
  typedef T vT __attribute__((ext_vector_type(N)));
  typedef T v2 __attribute__((ext_vector_type(2)));
  vT a;
  v2 b;
  __builtin_memcpy(&a, p, sizeof(T) * N);
  __builtin_memcpy(&b, p + N, 2 * sizeof(T));
#pragma unroll
  for (int i = 0; i < N; i++) w[i] = a[i];
  w[N] = b[0];
  w[N + 1] = b[1];
}

// ----------------------------------------------------------------- 27-point
template <class T>
struct P27 {
  T o, u, d;
};

template <class T>
__device__ inline P27<T> part27(const T* const* a, const T* __restrict__ x, size_t p, int nx,
                                size_t nxy) {
  const T *oE = a[1], *oN = a[2], *uC = a[3], *oNE = a[4], *oNW = a[5], *uE = a[6], *uW = a[7],
          *uN = a[8], *uS = a[9], *uNE = a[10], *uNW = a[11], *uSE = a[12], *uSW = a[13];
  P27<T> r;
  T o = oN[p] * x[p + nx];
  o += oN[p - nx] * x[p - nx];
  o += oE[p] * x[p + 1];
  o += oE[p - 1] * x[p - 1];
  o += oNE[p] * x[p + nx + 1];
  o += oNW[p] * x[p + nx - 1];
  o += oNW[p - nx + 1] * x[p - nx + 1];
  o += oNE[p - nx - 1] * x[p - nx - 1];
  const size_t q = p + nxy;
  T u = uC[p] * x[q];
  u += uN[p] * x[q + nx];
  u += uS[p] * x[q - nx];
  u += uE[p] * x[q + 1];
  u += uW[p] * x[q - 1];
  u += uNE[p] * x[q + nx + 1];
  u += uNW[p] * x[q + nx - 1];
  u += uSE[p] * x[q - nx + 1];
  u += uSW[p] * x[q - nx - 1];
  const size_t m = p - nxy;
  T d = uC[m] * x[m];
  d += uS[m + nx] * x[m + nx];
  d += uN[m - nx] * x[m - nx];
  d += uW[m + 1] * x[m + 1];
  d += uE[m - 1] * x[m - 1];
  d += uSW[m + nx + 1] * x[m + nx + 1];
  d += uSE[m + nx - 1] * x[m + nx - 1];
  d += uNW[m - nx + 1] * x[m - nx + 1];
  d += uNE[m - nx - 1] * x[m - nx - 1];
  r.o = o;
  r.u = u;
  r.d = d;
  return r;
}

template <class T>
struct Ops27 {
  const T* a[14];
};

// One calculation of a 27-point smoothing, residual or damping launch.
template <class T>
struct Args27 {
  Ops27<T> A;
  const T* D;
  const T* f;
  T* x;
  T* y;  // plane form: the neighbour planes' values; residual: the output
  T* z;  // plane form: the output
};

template <class T>
Ops27<T> to27(const Ops<T>& A) {
  Ops27<T> o;
  for (int s = 0; s < 14; s++) o.a[s] = A.a[s];
  return o;
}

// A batched launch takes at most kMaxBatch calculations.
inline void check_batch(int nb) {
  if (nb < 1 || nb > kMaxBatch) {
    fprintf(stderr, "pmg: a batched launch takes 1 to %d calculations, not %d\n", kMaxBatch, nb);
    abort();
  }
}

}  // namespace
}  // namespace pmg
