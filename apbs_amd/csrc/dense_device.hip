// dense_device.hip -- the coarsest level's dense operator: assembly, inverse
// and product.
#include "stencil27.h"

#include <cfloat>

namespace pmg {
namespace {

// forward offsets of the 14 stored coefficients
__constant__ int c_fwd[14][3] = {{0, 0, 0},  {1, 0, 0},  {0, 1, 0},  {0, 0, 1}, {1, 1, 0},
                                 {-1, 1, 0}, {1, 0, 1},  {-1, 0, 1}, {0, 1, 1}, {0, -1, 1},
                                 {1, 1, 1},  {-1, 1, 1}, {1, -1, 1}, {-1, -1, 1}};

// kAsmRows rows per workgroup, 16 lanes per row: the rows are cleared with
// consecutive stores, then each lane writes up to two of the row's 26
// couplings (forward ones from this point's coefficients, backward ones from
// the neighbour's) and lane 0 the diagonal.
constexpr int kAsmRows = kBlock / 16;

__global__ void __launch_bounds__(kBlock)
    k_dense_assemble(int nx, int ny, int nz, Batch<InvertArgs> B, int N) {
  const Ops<double>& A = B.v[blockIdx.y].A;
  const double* D = B.v[blockIdx.y].D;
  double* M = B.v[blockIdx.y].M;
  const int r0 = blockIdx.x * kAsmRows, rows = min(kAsmRows, N - r0);
  double* Mb = M + (size_t)r0 * N;
  for (int t = threadIdx.x; t < rows * N; t += kBlock) Mb[t] = 0.0;
  __syncthreads();
  const int r = r0 + threadIdx.x / 16, lane = threadIdx.x % 16;
  if (r >= N) return;
  const int ni = nx - 2, nj = ny - 2;
  const int i = r % ni + 1, j = (r / ni) % nj + 1, k = r / (ni * nj) + 1;
  if (lane == 0) M[(size_t)r * N + r] = D[IX(i, j, k, nx, ny)];
  for (int e = lane; e < 26; e += 16) {
    const int s = 1 + e / 2, dir = (e & 1) ? 1 : -1;
    const int i2 = i + dir * c_fwd[s][0], j2 = j + dir * c_fwd[s][1], k2 = k + dir * c_fwd[s][2];
    if (i2 < 1 || i2 > nx - 2 || j2 < 1 || j2 > ny - 2 || k2 < 1 || k2 > nz - 2) continue;
    const int c = (i2 - 1) + ni * ((j2 - 1) + nj * (k2 - 1));
    const double v = dir > 0 ? -A.a[s][IX(i, j, k, nx, ny)] : -A.a[s][IX(i2, j2, k2, nx, ny)];
    M[(size_t)r * N + c] = v;
  }
}

// A pivot that is not positive and finite means the operator is not positive
// definite (Vdpbfa's leading-minor test, mlinpckd.c:194-233): the 1-based
// index of the first one goes to *flag (host-mapped memory) with a
// system-scope store; a flag that an earlier block raised is kept.
__device__ inline void flag_pivot(int k, double* flag) {
  if (flag && __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == 0.0)
    __hip_atomic_store(flag, (double)(k + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The Gauss-Jordan inverse in one workgroup with the matrix held in LDS
// (N*N + 2N doubles, N <= 89).  Per pivot: stage column k and the scaled
// pivot row (v / piv), then update every element; each thread's (i, j) pairs
// are decoded once.
constexpr int kInvPer = 8;  // elements per thread: 89 * 89 <= 8 * 1024

__global__ void __launch_bounds__(1024) k_dense_invert_lds(Batch<InvertArgs> B, int N) {
  double* Mg = B.v[blockIdx.x].M;
  double* flag = B.v[blockIdx.x].flag;
  extern __shared__ double sm[];
  double* M = sm;
  double* col = sm + (size_t)N * N;
  double* prow = col + N;
  const int tid = threadIdx.x;
  int ei[kInvPer], ej[kInvPer];
  int ne = 0;
  for (int e = tid; e < N * N && ne < kInvPer; e += 1024, ne++) {
    ei[ne] = e / N;
    ej[ne] = e - ei[ne] * N;
  }
  for (int e = tid; e < N * N; e += 1024) M[e] = Mg[e];
  __syncthreads();
  int bad = -1;
  for (int k = 0; k < N; k++) {
    if (tid == 0 && bad < 0 && !(M[k * N + k] > 0.0 && M[k * N + k] <= DBL_MAX)) bad = k;
    if (tid < N) {
      col[tid] = M[tid * N + k];
      const double v = (tid == k) ? 1.0 : M[k * N + tid];
      prow[tid] = v / M[k * N + k];
    }
    __syncthreads();
    for (int q = 0; q < ne; q++) {
      const int i = ei[q], j = ej[q];
      if (i == k) {
        M[i * N + j] = prow[j];
      } else {
        const double base = (j == k) ? 0.0 : M[i * N + j];
        M[i * N + j] = base - col[i] * prow[j];
      }
    }
    __syncthreads();
  }
  for (int e = tid; e < N * N; e += 1024) Mg[e] = M[e];
  if (tid == 0 && bad >= 0) flag_pivot(bad, flag);
}

// The same Gauss-Jordan inverse for N <= 64 with the matrix in registers: 1,024
// threads, thread t holds entries 4 (t % 16) .. + 3 of row t / 16.  Each pivot
// step publishes the pivot row and column through double-buffered LDS (one
// barrier per pivot) and scales the pivot row by the pivot's reciprocal, so a
// step is an LDS round trip, a division and four updates.  With 16 entries on
// each of 256 threads the updates and their selects were the longest part of
// the step: 71 us at N = 64 beside the cycle's kernels, 47 us so.
// Reads N rows of src (leading dimension lds), writes dst (ldd; rows and
// columns up to nout, zero past N); pivot p is reported as base + p.
constexpr int kRegT = 1024;

__device__ __forceinline__ void invert_reg_body(const double* src, size_t lds, double* dst,
                                                size_t ldd, int N, int nout, int base,
                                                double* flag) {
  __shared__ double colb[2][64], rowb[2][64];
  const int t = threadIdx.x, r = t >> 4, cb = t & 15, c0 = cb * 4;
  double m[4];
#pragma unroll
  for (int q = 0; q < 4; q++)
    m[q] = (r < N && c0 + q < N) ? src[(size_t)r * lds + c0 + q] : 0.0;
  int bad = -1;
  for (int k = 0; k < N; k++) {
    const int b = k & 1;
    if ((k >> 2) == cb) {
      double v = m[0];
#pragma unroll
      for (int q = 1; q < 4; q++)
        if (q == (k & 3)) v = m[q];
      colb[b][r] = v;
    }
    if (r == k) {
#pragma unroll
      for (int q = 0; q < 4; q++) rowb[b][c0 + q] = m[q];
    }
    __syncthreads();
    const double piv = rowb[b][k];
    if (t == 0 && bad < 0 && !(piv > 0.0 && piv <= DBL_MAX)) bad = k;
    const double inv = 1.0 / piv;
    const double ci = colb[b][r];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int j = c0 + q;
      const double pj = ((j == k) ? 1.0 : rowb[b][j]) * inv;
      m[q] = (r == k) ? pj : ((j == k) ? 0.0 : m[q]) - ci * pj;
    }
  }
#pragma unroll
  for (int q = 0; q < 4; q++)
    if (r < nout && c0 + q < nout)
      dst[(size_t)r * ldd + c0 + q] = (r < N && c0 + q < N) ? m[q] : 0.0;
  if (t == 0 && bad >= 0) flag_pivot(base + bad, flag);
}

__global__ void __launch_bounds__(kRegT) k_dense_invert_reg(Batch<InvertArgs> B, int N) {
  double* Mg = B.v[blockIdx.x].M;
  invert_reg_body(Mg, N, Mg, N, N, N, 0, B.v[blockIdx.x].flag);
}

// Larger N (a coarsest level that cannot halve again, as 12^3 under 353^3:
// N = 1000): Gauss-Jordan by blocks of kGJ = 64 pivots.  Per block k, with P
// the inverse of the diagonal block, C the block's column panel and
// R = P A[k, :] its row panel: A[i, j] -= C_i R_j, A[k, :] = R,
// A[:, k] = -C P, A[k, k] = P.  Three launches a block: the diagonal block
// (registers, one workgroup), the panels, and the rank-64 update in 64 x 64
// tiles on the FP64 matrix cores.  One pivot at a time over the whole matrix
// takes three launches a pivot and 16 N^2 bytes of traffic each: 9.4 ms and
// 3,000 launches at N = 1000, the largest part of a 353^3 solve.
constexpr int kGJ = 64;
constexpr int kGjLda = 36, kGjLdb = 72;  // LDS strides: every bank twice per access

typedef double gj_d4 __attribute__((ext_vector_type(4)));

// acc[ti][tj] += the 16 x 16 tiles of A B over K = 64 owned by this wavefront
// (rows 32 (w / 2) + 16 ti, columns 32 (w % 2) + 16 tj): A is am x ak (lda),
// B ak x bn (ldb), taken as zero outside.
__device__ __forceinline__ void gj_mm(const double* __restrict__ A, size_t lda, int am, int ak,
                                      const double* __restrict__ B, size_t ldb, int bn,
                                      gj_d4 (&acc)[2][2]) {
  __shared__ double sA[kGJ * kGjLda], sB[32 * kGjLdb];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int r0 = 32 * (w >> 1), c0 = 32 * (w & 1), li = lane & 15, lk = lane >> 4;
  for (int h = 0; h < 2; h++) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int x = t + 256 * e;
      const int ar = x >> 5, ac = x & 31;
      sA[ar * kGjLda + ac] = (ar < am && 32 * h + ac < ak) ? A[ar * lda + 32 * h + ac] : 0.0;
      const int br = x >> 6, bc = x & 63;
      sB[br * kGjLdb + bc] = (32 * h + br < ak && bc < bn) ? B[(32 * h + br) * ldb + bc] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 32; kk += 4) {
      double a[2], b[2];
#pragma unroll
      for (int q = 0; q < 2; q++) {
        a[q] = sA[(r0 + 16 * q + li) * kGjLda + kk + lk];
        b[q] = sB[(kk + lk) * kGjLdb + c0 + 16 * q + li];
      }
#pragma unroll
      for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
          acc[ti][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ti], b[tj], acc[ti][tj], 0, 0, 0);
    }
    __syncthreads();
  }
}

// Calls f(row, column, value) for the tile elements this lane holds.
template <class F>
__device__ __forceinline__ void gj_each(const gj_d4 (&acc)[2][2], F f) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int ti = 0; ti < 2; ti++)
#pragma unroll
    for (int tj = 0; tj < 2; tj++)
#pragma unroll
      for (int v = 0; v < 4; v++)
        f(32 * (w >> 1) + 16 * ti + 4 * v + (lane >> 4), 32 * (w & 1) + 16 * tj + (lane & 15),
          acc[ti][tj][v]);
}

// work: P (64 x 64), R (64 x N), C (N x 64)
struct GjWork {
  double *P, *R, *C;
  __device__ explicit GjWork(double* w, int N)
      : P(w), R(w + kGJ * kGJ), C(w + kGJ * kGJ + (size_t)kGJ * N) {}
};

__global__ void __launch_bounds__(kRegT) k_gj_diag(Batch<InvertArgs> B, int N, int kb) {
  const InvertArgs& a = B.v[blockIdx.x];
  const GjWork W(a.work, N);
  const int p0 = kb * kGJ;
  invert_reg_body(a.M + (size_t)p0 * N + p0, N, W.P, kGJ, min(kGJ, N - p0), kGJ, p0, a.flag);
}

// blockIdx.y 0: R of column tile blockIdx.x; 1: C of row tile blockIdx.x.
__global__ void __launch_bounds__(256) k_gj_panels(Batch<InvertArgs> B, int N, int kb) {
  const InvertArgs& a = B.v[blockIdx.z];
  const GjWork W(a.work, N);
  const int q0 = blockIdx.x * kGJ, p0 = kb * kGJ, bk = min(kGJ, N - p0), bq = min(kGJ, N - q0);
  if ((int)blockIdx.x == kb) return;
  if (blockIdx.y == 0) {
    gj_d4 acc[2][2] = {};
    gj_mm(W.P, kGJ, bk, bk, a.M + (size_t)p0 * N + q0, N, bq, acc);
    gj_each(acc, [&](int r, int c, double v) {
      if (r < bk && c < bq) W.R[(size_t)r * N + q0 + c] = v;
    });
  } else {
    for (int x = threadIdx.x; x < kGJ * kGJ; x += 256) {
      const int r = x >> 6, c = x & 63;
      if (r < bq && c < bk) W.C[(size_t)(q0 + r) * kGJ + c] = a.M[(size_t)(q0 + r) * N + p0 + c];
    }
  }
}

__global__ void __launch_bounds__(256) k_gj_update(Batch<InvertArgs> B, int N, int kb) {
  const InvertArgs& a = B.v[blockIdx.z];
  const GjWork W(a.work, N);
  const int j0 = blockIdx.x * kGJ, i0 = blockIdx.y * kGJ, p0 = kb * kGJ;
  const int bi = min(kGJ, N - i0), bj = min(kGJ, N - j0), bk = min(kGJ, N - p0);
  const bool prow = (int)blockIdx.y == kb, pcol = (int)blockIdx.x == kb;
  double* T = a.M + (size_t)i0 * N + j0;
  if (prow) {
    for (int x = threadIdx.x; x < kGJ * kGJ; x += 256) {
      const int r = x >> 6, c = x & 63;
      if (r < bi && c < bj) T[(size_t)r * N + c] = pcol ? W.P[x] : W.R[(size_t)r * N + j0 + c];
    }
    return;
  }
  gj_d4 acc[2][2] = {};
  if (pcol)
    gj_mm(W.C + (size_t)i0 * kGJ, kGJ, bi, bk, W.P, kGJ, bj, acc);
  else
    gj_mm(W.C + (size_t)i0 * kGJ, kGJ, bi, bk, W.R + j0, N, bj, acc);
  gj_each(acc, [&](int r, int c, double v) {
    if (r < bi && c < bj) T[(size_t)r * N + c] = (pcol ? 0.0 : T[(size_t)r * N + c]) - v;
  });
}

// x_r = sum_c Minv[r][c] f_c over the interior unknowns, N <= kDenseSmall:
// one workgroup gathers f into LDS, then each row sums in column order.
constexpr int kDenseSmall = 96;

template <class T>
__global__ void __launch_bounds__(128) k_dense_solve(int nx, int ny, int nz, Batch<DenseArgs<T>> B,
                                                     int N) {
  __shared__ double fv[kDenseSmall];
  const double* Minv = B.v[blockIdx.x].Minv;
  const T* f = B.v[blockIdx.x].f;
  T* x = B.v[blockIdx.x].x;
  const int ni = nx - 2, nj = ny - 2;
  for (int c = threadIdx.x; c < N; c += blockDim.x) {
    const int i = c % ni + 1, j = (c / ni) % nj + 1, k = c / (ni * nj) + 1;
    fv[c] = (double)f[IX(i, j, k, nx, ny)];
  }
  __syncthreads();
  const int r = threadIdx.x;
  if (r >= N) return;
  const double* row = Minv + (size_t)r * N;
  double s = 0.0;
#pragma unroll 8
  for (int c = 0; c < N; c++) s += row[c] * fv[c];
  const int i = r % ni + 1, j = (r / ni) % nj + 1, k = r / (ni * nj) + 1;
  x[IX(i, j, k, nx, ny)] = (T)s;
}

// The same product for larger N: one wavefront per row (its lanes stride over
// the columns, so a row is read in whole lines), f gathered into LDS in chunks.
// One thread per row took 413 us at N = 1000 (four workgroups, a chain of
// 1,000 additions).
constexpr int kDenseChunk = 2048;

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_dense_solve_rows(int nx, int ny, int nz, Batch<DenseArgs<T>> B, int N) {
  __shared__ double fv[kDenseChunk];
  const double* Minv = B.v[blockIdx.y].Minv;
  const T* f = B.v[blockIdx.y].f;
  T* x = B.v[blockIdx.y].x;
  const int ni = nx - 2, nj = ny - 2;
  const int lane = threadIdx.x & 63, r = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  double s = 0.0;
  for (int c0 = 0; c0 < N; c0 += kDenseChunk) {
    const int m = min(kDenseChunk, N - c0);
    __syncthreads();
    for (int t = threadIdx.x; t < m; t += kBlock) {
      const int c = c0 + t, i = c % ni + 1, j = (c / ni) % nj + 1, k = c / (ni * nj) + 1;
      fv[t] = (double)f[IX(i, j, k, nx, ny)];
    }
    __syncthreads();
    if (r < N) {
      const double* row = Minv + (size_t)r * N + c0;
#pragma unroll 4
      for (int t = lane; t < m; t += 64) s += row[t] * fv[t];
    }
  }
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if (r >= N || lane != 0) return;
  const int i = r % ni + 1, j = (r / ni) % nj + 1, k = r / (ni * nj) + 1;
  x[IX(i, j, k, nx, ny)] = (T)s;
}

}  // namespace

size_t dense_work(int N) {
  return N <= kGJ ? (size_t)N : (size_t)kGJ * kGJ + 2 * (size_t)kGJ * N;
}

static void dense_invert_batch(hipStream_t s, const Batch<InvertArgs>& B, int N, int nb,
                               int form) {
  if (N <= 64 && form != 1) {
    k_dense_invert_reg<<<nb, kRegT, 0, s>>>(B, N);
    return;
  }
  const size_t lds = ((size_t)N * N + 2 * N) * sizeof(double);
  if (lds <= 64 * 1024 && (size_t)N * N <= (size_t)kInvPer * 1024) {
    k_dense_invert_lds<<<nb, 1024, lds, s>>>(B, N);
    return;
  }
  const unsigned nt = (unsigned)((N + kGJ - 1) / kGJ);
  for (unsigned kb = 0; kb < nt; kb++) {
    k_gj_diag<<<nb, kRegT, 0, s>>>(B, N, (int)kb);
    k_gj_panels<<<dim3(nt, 2, nb), 256, 0, s>>>(B, N, (int)kb);
    k_gj_update<<<dim3(nt, nt, nb), 256, 0, s>>>(B, N, (int)kb);
  }
}

void dense_assemble_invert_batch(hipStream_t s, int nx, int ny, int nz, int N,
                                 const InvertArgs* c, int nb, int form) {
  check_batch(nb);
  Batch<InvertArgs> B;
  for (int b = 0; b < nb; b++) B.v[b] = c[b];
  k_dense_assemble<<<dim3((N + kAsmRows - 1) / kAsmRows, nb), kBlock, 0, s>>>(nx, ny, nz, B, N);
  dense_invert_batch(s, B, N, nb, form);
}

void dense_invert_batch(hipStream_t s, int N, const InvertArgs* c, int nb, int form) {
  check_batch(nb);
  Batch<InvertArgs> B;
  for (int b = 0; b < nb; b++) B.v[b] = c[b];
  dense_invert_batch(s, B, N, nb, form);
}

void dense_assemble(hipStream_t s, int nx, int ny, int nz, const Ops<double>& A, const double* D,
                    double* M, int N) {
  Batch<InvertArgs> B;
  B.v[0] = InvertArgs{A, D, M, nullptr, nullptr};
  k_dense_assemble<<<dim3((N + kAsmRows - 1) / kAsmRows, 1), kBlock, 0, s>>>(nx, ny, nz, B, N);
}

void dense_invert(hipStream_t s, double* M, double* work, int N, int form, double* flag) {
  const InvertArgs c{Ops<double>{}, nullptr, M, work, flag};
  dense_invert_batch(s, N, &c, 1, form);
}

template <class T>
void dense_solve_batch(hipStream_t s, int nx, int ny, int nz, int N, const DenseArgs<T>* c,
                       int nb) {
  check_batch(nb);
  Batch<DenseArgs<T>> B;
  for (int b = 0; b < nb; b++) B.v[b] = c[b];
  if (((size_t)N * N + N) * sizeof(double) <= 64 * 1024 && N <= kDenseSmall)
    k_dense_solve<T><<<nb, 128, 0, s>>>(nx, ny, nz, B, N);
  else
    k_dense_solve_rows<T><<<dim3((N + kBlock / 64 - 1) / (kBlock / 64), nb), kBlock, 0, s>>>(
        nx, ny, nz, B, N);
}

template <class T>
void dense_solve(hipStream_t s, int nx, int ny, int nz, const double* Minv, int N, const T* f,
                 T* x) {
  const DenseArgs<T> c{Minv, f, x};
  dense_solve_batch<T>(s, nx, ny, nz, N, &c, 1);
}

#define INST(T)                                                                                \
  template void dense_solve<T>(hipStream_t, int, int, int, const double*, int, const T*, T*);   \
  template void dense_solve_batch<T>(hipStream_t, int, int, int, int, const DenseArgs<T>*, int);
INST(double)
INST(float)
#undef INST

}  // namespace pmg
