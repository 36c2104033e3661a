// pmg_device.hip -- PMG multigrid kernels for CDNA4 (gfx950).
//
// The fine 7-point kernels evaluate exactly the reference's expressions in the
// reference's order (src/pmgc/gsd.c:95-165, matvecd.c:461-496) and are built
// without FMA contraction, so one sweep is bitwise identical to the reference
// arithmetic.  Coarse 27-point levels are smoothed with an 8-colour
// Gauss-Seidel ordering (parity of i, j, k) instead of the reference's
// in-place lexicographic sweep (gsd.c:230-327), whose dependencies are serial.
#include "pmg_device.h"

#include "stencil27.h"

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

namespace pmg {

namespace {

// ------------------------------------------------------------------ 7-point
// fc + north + south + east + west + down + up, left to right.
template <class T>
__device__ inline T acc7(T init, const T* __restrict__ oE, const T* __restrict__ oN,
                         const T* __restrict__ uC, const T* __restrict__ x, size_t p, int nx,
                         size_t nxy) {
  T s = init;
  s += oN[p] * x[p + nx];
  s += oN[p - nx] * x[p - nx];
  s += oE[p] * x[p + 1];
  s += oE[p - 1] * x[p - 1];
  s += uC[p - nxy] * x[p - nxy];
  s += uC[p] * x[p + nxy];
  return s;
}

// One colour of the red-black sweep: points with (i+j+k)&1 == par (0-based).
// The reference's "red" points (1-based i+j+k even) have par == 1.
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_gsrb7(int nx, int ny, int nz, const T* __restrict__ oE, const T* __restrict__ oN,
            const T* __restrict__ uC, const T* __restrict__ D, const T* __restrict__ fc, T* x,
            int par) {
  const int npair = (nx - 1) / 2;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int ip = t % npair;
  const int j = 1 + t / npair;
  if (j > ny - 2) return;
  const int i = 1 + (((1 + j + k) ^ par) & 1) + 2 * ip;
  if (i > nx - 2) return;
  const size_t nxy = (size_t)nx * ny;
  const size_t p = IX(i, j, k, nx, ny);
  x[p] = acc7(fc[p], oE, oN, uC, x, p, nx, nxy) / D[p];
}

// One colour of the 8-colour sweep: 0-based parities (c&1, (c>>1)&1, (c>>2)&1).
// Latency-bound on the small coarse levels: up to 128 VGPRs, so that all 54
// operands of a point are in flight at once.
template <class T>
__device__ __forceinline__ void gsrb27_body(int nx, int ny, int nz, const Ops27<T>& A,
                                            const T* __restrict__ D, const T* __restrict__ fc,
                                            T* x, int c) {
  const int ci = c & 1, cj = (c >> 1) & 1, ck = (c >> 2) & 1;
  const int i0 = ci ? 1 : 2, j0 = cj ? 1 : 2, k0 = ck ? 1 : 2;
  const int ni = (nx - 2 - i0) / 2 + 1, nj = (ny - 2 - j0) / 2 + 1;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = k0 + 2 * (int)blockIdx.y;
  if (k > nz - 2 || ni <= 0 || nj <= 0) return;
  const int ti = t % ni, tj = t / ni;
  if (tj >= nj) return;
  const int i = i0 + 2 * ti, j = j0 + 2 * tj;
  if (i > nx - 2 || j > ny - 2) return;
  const size_t nxy = (size_t)nx * ny;
  const size_t p = IX(i, j, k, nx, ny);
  P27<T> s = part27<T>(A.a, x, p, nx, nxy);
  x[p] = (fc[p] + (s.o + s.u + s.d)) / D[p];
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_gsrb27(int nx, int ny, int nz, Batch<Args27<T>> B, int c) {
  const Args27<T>& a = B.v[blockIdx.z];
  gsrb27_body<T>(nx, ny, nz, a.A, a.D, a.f, a.x, c);
}

// Two colours of that sweep in one launch: A = c and B = c ^ 1, which differ
// only in the parity of i and follow each other in both sweep orders.  An
// A point and a B point are neighbours only along i within one row, and the
// rows of one (j, k) parity do not touch each other, so a wavefront owns a
// row: lane t updates the A point iA0 + 2t, writes it, and takes the new A
// values beside its B point iB0 + 2t from the neighbouring lanes.  Rows of up
// to 128 interior points.  The arithmetic is part27's, term for term.
template <class T>
__device__ inline T lane_value(T v, int src) {
  return __shfl(v, src < 0 ? 0 : (src > 63 ? 63 : src), 64);
}

template <class T>
__device__ __forceinline__ void pair_body(int nx, int ny, int nz, const Ops27<T>& A,
                                          const T* __restrict__ D, const T* __restrict__ fc, T* x,
                                          int pa, int cj, int ck) {
  const T *oE = A.a[1], *oN = A.a[2], *uC = A.a[3], *oNE = A.a[4], *oNW = A.a[5], *uE = A.a[6],
          *uW = A.a[7], *uN = A.a[8], *uS = A.a[9], *uNE = A.a[10], *uNW = A.a[11],
          *uSE = A.a[12], *uSW = A.a[13];
  const int j0 = cj ? 1 : 2, k0 = ck ? 1 : 2;
  const int nj = (ny - 2 - j0) / 2 + 1;
  const int row = (int)((blockIdx.x * (unsigned)kBlock + threadIdx.x) / 64);
  const int lane = (int)(threadIdx.x % 64);
  const int nk = (nz - 2 - k0) / 2 + 1;
  if (row >= nj * nk) return;  // uniform per wavefront
  const int j = j0 + 2 * (row % nj), k = k0 + 2 * (row / nj);
  const size_t nxy = (size_t)nx * ny;
  const size_t rowp = (size_t)k * nxy + (size_t)j * nx;
  const int iA = (pa ? 1 : 2) + 2 * lane, iB = (pa ? 2 : 1) + 2 * lane;
  T a = 0;
  if (iA <= nx - 2) {
    const size_t p = rowp + iA;
    P27<T> r = part27<T>(A.a, x, p, nx, nxy);
    a = (fc[p] + (r.o + r.u + r.d)) / D[p];
    x[p] = a;
  }
  // new A values at iB - 1 and iB + 1: lanes t - 1 and t when A is even,
  // t and t + 1 when A is odd
  const T am = lane_value(a, pa ? lane : lane - 1);
  const T ap = lane_value(a, pa ? lane + 1 : lane);
  if (iB > nx - 2) return;
  const size_t p = rowp + iB;
  const T xm = (iB - 1 >= 1) ? am : x[p - 1];
  const T xp = (iB + 1 <= nx - 2) ? ap : x[p + 1];
  T o = oN[p] * x[p + nx];
  o += oN[p - nx] * x[p - nx];
  o += oE[p] * xp;
  o += oE[p - 1] * xm;
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
  x[p] = (fc[p] + (o + u + d)) / D[p];
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_gsrb27_pair(int nx, int ny, int nz, Batch<Args27<T>> B, int pa, int cj, int ck) {
  const Args27<T>& a = B.v[blockIdx.z];
  pair_body<T>(nx, ny, nz, a.A, a.D, a.f, a.x, pa, cj, ck);
}

// The vector form of the colour-pair launch.  In the form above a lane loads
// one word per operand, with the lanes two words apart, so its 54 loads per
// point keep the texture addresser (four lanes per clock) busy for most of
// the launch.  Here a lane owns a run of kV consecutive points of a row (8 or
// 16 bytes, both colours): each of the 26 coefficient terms, f and D is one
// load, and each of the 9 neighbouring rows of
// x one window of kV + 2 values.  The A points of the run are updated first
// (their row neighbours are B points, still old) and written to a row buffer
// in LDS; after a barrier the B points take their new A neighbours from it.
// The last run of a row is moved inwards so that every load stays inside its
// row; overlapping runs compute and write the same values.  part27's terms in
// its order, so the results are the scalar form's bit for bit.
// R runs per row, RB rows per workgroup; LDS holds RB rows of new A values.
template <class T, int kV>
__global__ void __launch_bounds__(kBlock)
    k_gsrb27_vpair(int nx, int ny, int nz, Batch<Args27<T>> B, int pa, int cj, int ck, int R,
                   int RB) {
  constexpr int kH = kV / 2;
  extern __shared__ unsigned char vpair_smem[];
  T* na = reinterpret_cast<T*>(vpair_smem);
  const Args27<T>& ar = B.v[blockIdx.z];
  const T *oE = ar.A.a[1], *oN = ar.A.a[2], *uC = ar.A.a[3], *oNE = ar.A.a[4],
          *oNW = ar.A.a[5], *uE = ar.A.a[6], *uW = ar.A.a[7], *uN = ar.A.a[8], *uS = ar.A.a[9],
          *uNE = ar.A.a[10], *uNW = ar.A.a[11], *uSE = ar.A.a[12], *uSW = ar.A.a[13];
  const T *D = ar.D, *fc = ar.f;
  T* x = ar.x;
  const int j0 = cj ? 1 : 2, k0 = ck ? 1 : 2;
  const int nj = (ny - 2 - j0) / 2 + 1, nk = (nz - 2 - k0) / 2 + 1;
  const int lr = (int)threadIdx.x / R, run = (int)threadIdx.x % R;
  const int row = (int)blockIdx.x * RB + lr;
  const bool act = lr < RB && row < nj * nk;
  const int rr = act ? row : 0;  // idle lanes load row 0 of the class (unused)
  const int j = j0 + 2 * (rr % nj), k = k0 + 2 * (rr / nj);
  const int ib = min(1 + kV * run, nx - 1 - kV);
  const size_t nxy = (size_t)nx * ny;
  const size_t p = (size_t)k * nxy + (size_t)j * nx + ib;
  const size_t q = p + nxy, m = p - nxy;
  T* nrow = na + (size_t)(act ? lr : 0) * nx;

  // coefficient vectors (columns ib .. ib+kV-1 of each term)
  T c[28][kV];
  vld16(c[0], oN + p);
  vld16(c[1], oN + p - nx);
  vld16(c[2], oE + p);
  vld16(c[3], oE + p - 1);
  vld16(c[4], oNE + p);
  vld16(c[5], oNW + p);
  vld16(c[6], oNW + p - nx + 1);
  vld16(c[7], oNE + p - nx - 1);
  vld16(c[8], uC + p);
  vld16(c[9], uN + p);
  vld16(c[10], uS + p);
  vld16(c[11], uE + p);
  vld16(c[12], uW + p);
  vld16(c[13], uNE + p);
  vld16(c[14], uNW + p);
  vld16(c[15], uSE + p);
  vld16(c[16], uSW + p);
  vld16(c[17], uC + m);
  vld16(c[18], uS + m + nx);
  vld16(c[19], uN + m - nx);
  vld16(c[20], uW + m + 1);
  vld16(c[21], uE + m - 1);
  vld16(c[22], uSW + m + nx + 1);
  vld16(c[23], uSE + m + nx - 1);
  vld16(c[24], uNW + m - nx + 1);
  vld16(c[25], uNE + m - nx - 1);
  vld16(c[26], fc + p);
  vld16(c[27], D + p);
  // x windows (columns ib-1 .. ib+kV) of the 9 rows: 0 (j,k), 1 (j+1,k),
  // 2 (j-1,k), 3 (j,k+1), 4 (j+1,k+1), 5 (j-1,k+1), 6 (j,k-1), 7 (j+1,k-1),
  // 8 (j-1,k-1)
  T w[9][kV + 2];
  vldw<T, kV>(w[0], x + p - 1);
  vldw<T, kV>(w[1], x + p + nx - 1);
  vldw<T, kV>(w[2], x + p - nx - 1);
  vldw<T, kV>(w[3], x + q - 1);
  vldw<T, kV>(w[4], x + q + nx - 1);
  vldw<T, kV>(w[5], x + q - nx - 1);
  vldw<T, kV>(w[6], x + m - 1);
  vldw<T, kV>(w[7], x + m + nx - 1);
  vldw<T, kV>(w[8], x + m - nx - 1);

  // the value of element e0 + 2*mm (e0 = 0 or 1): selects between values
  auto point = [&](int e0, int mm, T xm, T xp) {
    auto pc = [&](int t) {
      const T lo = c[t][2 * mm], hi = c[t][2 * mm + 1];
      return e0 ? hi : lo;
    };
    auto pw = [&](int r, int d) {
      const T lo = w[r][2 * mm + d], hi = w[r][2 * mm + 1 + d];
      return e0 ? hi : lo;
    };
    T o = pc(0) * pw(1, 1);
    o += pc(1) * pw(2, 1);
    o += pc(2) * xp;
    o += pc(3) * xm;
    o += pc(4) * pw(1, 2);
    o += pc(5) * pw(1, 0);
    o += pc(6) * pw(2, 2);
    o += pc(7) * pw(2, 0);
    T u = pc(8) * pw(3, 1);
    u += pc(9) * pw(4, 1);
    u += pc(10) * pw(5, 1);
    u += pc(11) * pw(3, 2);
    u += pc(12) * pw(3, 0);
    u += pc(13) * pw(4, 2);
    u += pc(14) * pw(4, 0);
    u += pc(15) * pw(5, 2);
    u += pc(16) * pw(5, 0);
    T d = pc(17) * pw(6, 1);
    d += pc(18) * pw(7, 1);
    d += pc(19) * pw(8, 1);
    d += pc(20) * pw(6, 2);
    d += pc(21) * pw(6, 0);
    d += pc(22) * pw(7, 2);
    d += pc(23) * pw(7, 0);
    d += pc(24) * pw(8, 2);
    d += pc(25) * pw(8, 0);
    return (pc(26) + (o + u + d)) / pc(27);
  };

  // A points (column parity pa): row neighbours are old B values.  The
  // element pairs are handled with constant indices (the calls below, not a
  // loop), so every selected value is a register, never an address.
  const int eA = (pa - ib) & 1, eB = eA ^ 1;
  T av[kH];
  auto stageA = [&](auto mmc) {
    constexpr int mm = decltype(mmc)::value;
    const T xm = eA ? w[0][2 * mm + 1] : w[0][2 * mm];
    const T xp = eA ? w[0][2 * mm + 3] : w[0][2 * mm + 2];
    av[mm] = point(eA, mm, xm, xp);
    if (act) nrow[ib + eA + 2 * mm] = av[mm];
  };
  stageA(std::integral_constant<int, 0>{});
  if constexpr (kH > 1) stageA(std::integral_constant<int, 1>{});
  __syncthreads();
  // B points: new A neighbours from the row buffer, boundary columns old
  T out[kV];
  auto stageB = [&](auto mmc) {
    constexpr int mm = decltype(mmc)::value;
    const int col = ib + eB + 2 * mm;
    const T om = eB ? w[0][2 * mm + 1] : w[0][2 * mm];
    const T op = eB ? w[0][2 * mm + 3] : w[0][2 * mm + 2];
    const T xm = col - 1 >= 1 ? nrow[col - 1] : om;
    const T xp = col + 1 <= nx - 2 ? nrow[col + 1] : op;
    const T bv = point(eB, mm, xm, xp);
    out[2 * mm] = eA ? bv : av[mm];
    out[2 * mm + 1] = eA ? av[mm] : bv;
  };
  stageB(std::integral_constant<int, 0>{});
  if constexpr (kH > 1) stageB(std::integral_constant<int, 1>{});
  if (act) vst16(x + p, out);
}

template <class T>
__device__ __forceinline__ void resid7_body(int nx, int ny, int nz, const T* __restrict__ oE,
                                            const T* __restrict__ oN, const T* __restrict__ uC,
                                            const T* __restrict__ D, const T* __restrict__ fc,
                                            const T* __restrict__ x, T* __restrict__ r) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int i = 1 + t % (nx - 2), j = 1 + t / (nx - 2);
  if (j > ny - 2) return;
  const size_t nxy = (size_t)nx * ny;
  const size_t p = IX(i, j, k, nx, ny);
  r[p] = acc7(fc[p], oE, oN, uC, x, p, nx, nxy) - D[p] * x[p];
}

template <class T>
__global__ void __launch_bounds__(kBlock) k_resid7(int nx, int ny, int nz, Batch<Args27<T>> B) {
  const Args27<T>& a = B.v[blockIdx.z];
  resid7_body<T>(nx, ny, nz, a.A.a[1], a.A.a[2], a.A.a[3], a.D, a.f, a.x, a.y);
}

// The 7-point residual with one lane per 16-byte run of a row (4 floats or
// 2 doubles): every operand is one 16-byte load, x of the row a window of
// kV + 2 values, r one 16-byte store.  The last run of a row is moved inwards
// so that every load stays inside its row (overlapping runs write the same
// values).  acc7's terms and order, so the values are k_resid7's bit for bit.
template <class T>
__global__ void __launch_bounds__(kBlock) k_resid7v(int nx, int ny, int nz, Batch<Args27<T>> B) {
  constexpr int kV = 16 / (int)sizeof(T);
  const Args27<T>& a = B.v[blockIdx.z];
  const T *oE = a.A.a[1], *oN = a.A.a[2], *uC = a.A.a[3], *D = a.D, *fc = a.f, *x = a.x;
  T* r = a.y;
  const int R = (nx - 2 + kV - 1) / kV;
  const int t = (int)(blockIdx.x * kBlock + threadIdx.x);
  const int run = t % R, row = t / R;
  if (row >= (ny - 2) * (nz - 2)) return;
  const int j = 1 + row % (ny - 2), k = 1 + row / (ny - 2);
  const int ib = min(1 + kV * run, nx - 1 - kV);
  const size_t nxy = (size_t)nx * ny;
  const size_t p = (size_t)k * nxy + (size_t)j * nx + ib;
  T vf[kV], vN[kV], vNm[kV], vE[kV], vEm[kV], vUm[kV], vU[kV], vD[kV];
  T xn[kV], xs[kV], xu[kV], xd[kV], xw[kV + 2];
  vld16(vf, fc + p);
  vld16(vN, oN + p);
  vld16(vNm, oN + p - nx);
  vld16(vE, oE + p);
  vld16(vEm, oE + p - 1);
  vld16(vUm, uC + p - nxy);
  vld16(vU, uC + p);
  vld16(vD, D + p);
  vld16(xn, x + p + nx);
  vld16(xs, x + p - nx);
  vld16(xu, x + p + nxy);
  vld16(xd, x + p - nxy);
  vldw<T, kV>(xw, x + p - 1);
  T out[kV];
#pragma unroll
  for (int e = 0; e < kV; e++) {
    T sv = vf[e];
    sv += vN[e] * xn[e];
    sv += vNm[e] * xs[e];
    sv += vE[e] * xw[e + 2];
    sv += vEm[e] * xw[e];
    sv += vUm[e] * xd[e];
    sv += vU[e] * xu[e];
    out[e] = sv - vD[e] * xw[e + 1];
  }
  vst16(r + p, out);
}

template <class T>
__device__ __forceinline__ void resid27_body(int nx, int ny, int nz, const Ops27<T>& A,
                                             const T* __restrict__ D, const T* __restrict__ fc,
                                             const T* __restrict__ x, T* __restrict__ r) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int i = 1 + t % (nx - 2), j = 1 + t / (nx - 2);
  if (j > ny - 2) return;
  const size_t nxy = (size_t)nx * ny;
  const size_t p = IX(i, j, k, nx, ny);
  P27<T> s = part27<T>(A.a, x, p, nx, nxy);
  r[p] = fc[p] + s.o + s.u + s.d - D[p] * x[p];
}

template <class T>
__global__ void __launch_bounds__(kBlock) k_resid27(int nx, int ny, int nz, Batch<Args27<T>> B) {
  const Args27<T>& a = B.v[blockIdx.z];
  resid27_body<T>(nx, ny, nz, a.A, a.D, a.f, a.x, a.y);
}

// --------------------------------------------------------------- reductions
__device__ inline double block_sum(double v, double* sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  double r = sh[0];
  __syncthreads();
  return r;
}

// How the fine-grid reductions walk the interior: tiles of 256 consecutive
// (i, j) columns, a column a thread, cut along k into runs of kc planes so that
// there are at most kParts runs (one a block) where there are that few tiles.
// XCD x (blocks x, x + 8, ...) owns a contiguous eighth of the runs.  A thread
// keeps its column's operands of planes k - 1 and k in registers; with points
// dealt in contiguous chunks every block read them again, and most came from
// beyond the L2 (130 bytes a point for the 80 of k_jres_trial at 353^3).
// Microseconds so, and before: k_jres_trial 82 (94) at 161^3 in FP64, 1078
// (1217) at 353^3 with an FP32 correction; k_nresid7_xpay 76 (83), 434 (530).
struct PartRuns {
  int ntile, kc, items;
};

inline PartRuns part_runs(int nx, int ny, int nz) {
  const int nk = std::max(1, nz - 2);
  const int ntile = std::max(1, ((nx - 2) * (ny - 2) + kBlock - 1) / kBlock);
  const int want = std::max(1, std::min(nk, kParts / ntile));
  const int kc = (nk + want - 1) / want;
  return {ntile, kc, ntile * ((nk + kc - 1) / kc)};
}

// f(first point, planes) for each run of this block
template <class F>
__device__ __forceinline__ void part_columns(int nx, int ny, int nz, PartRuns R, F f) {
  const int ni = nx - 2, nij = ni * (ny - 2);
  const int per = (R.items + 7) / 8, x = blockIdx.x % 8;
  for (int e = blockIdx.x / 8; e < per; e += kParts / 8) {
    const int item = x * per + e;
    if (item >= R.items) break;
    const int ch = item / R.ntile, t = (item - ch * R.ntile) * kBlock + threadIdx.x;
    if (t >= nij) continue;
    const int j = 1 + t / ni, i = 1 + t - (j - 1) * ni, k0 = 1 + ch * R.kc;
    f(IX(i, j, k0, nx, ny), min(R.kc, nz - 1 - k0));
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_nrm1_part(int nx, int ny, int nz, PartRuns R, const T* __restrict__ x, double* part) {
  __shared__ double sh[kBlock];
  const size_t nxy = (size_t)nx * ny;
  double acc = 0.0;
  part_columns(nx, ny, nz, R, [&](size_t p, int planes) {
#pragma unroll 4
    for (int m = 0; m < planes; m++, p += nxy) acc += fabs((double)x[p]);
  });
  double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// The 7-point residual and the partial sums of its L1 norm in one pass: the
// points are visited in k_nrm1_part's order (part_columns), so the norm is
// bitwise that of storing r and calling k_nrm1_part.  r is stored when
// non-null.
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_resid7_nrm(int nx, int ny, int nz, PartRuns R, const T* __restrict__ oE,
                 const T* __restrict__ oN, const T* __restrict__ uC, const T* __restrict__ D,
                 const T* __restrict__ fc, const T* __restrict__ x, T* __restrict__ r,
                 float* __restrict__ r32, double* part) {
  __shared__ double sh[kBlock];
  const size_t nxy = (size_t)nx * ny;
  double acc = 0.0;
  part_columns(nx, ny, nz, R, [&](size_t p, int planes) {
    T xkm = x[p - nxy], x0 = x[p], vUm = uC[p - nxy];
    for (int m = 0; m < planes; m++, p += nxy) {
      // every operand first; acc7's terms and order
      const T xjp = x[p + nx], xjm = x[p - nx], xip = x[p + 1], xim = x[p - 1];
      const T xkp = x[p + nxy];
      const T vN = oN[p], vNm = oN[p - nx], vE = oE[p], vEm = oE[p - 1];
      const T vU = uC[p], vD = D[p];
      T sv = fc[p];
      sv += vN * xjp;
      sv += vNm * xjm;
      sv += vE * xip;
      sv += vEm * xim;
      sv += vUm * xkm;
      sv += vU * xkp;
      const T v = sv - vD * x0;
      if (r) r[p] = v;
      if (r32) r32[p] = (float)v;
      acc += fabs((double)v);
      xkm = x0;
      x0 = xkp;
      vUm = vU;
    }
  });
  double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// The L1 norm partials of x (k_nrm1_part's order) and y = (float) x on the
// interior, in one pass.
__global__ void __launch_bounds__(kBlock)
    k_nrm1_to32(int nx, int ny, int nz, PartRuns R, const double* __restrict__ x, float* __restrict__ y,
                double* part) {
  __shared__ double sh[kBlock];
  const size_t nxy = (size_t)nx * ny;
  double acc = 0.0;
  part_columns(nx, ny, nz, R, [&](size_t p, int planes) {
#pragma unroll 4
    for (int m = 0; m < planes; m++, p += nxy) {
      const double v = x[p];
      y[p] = (float)v;
      acc += fabs(v);
    }
  });
  double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// One calculation of a reduction's finishing launch.
struct FinishArgs {
  const double* part;
  double* out;
  double* hout;
};

struct FinishBatch {
  FinishArgs v[2 * kMaxBatch];
};

// out[0] = sum(part[0..kParts-1]); ratio: out[0] = sum(a)/sum(b)
// (and hout[0] = out[0] when hout is given); calculation blockIdx.x.  Only
// the first nparts partial sums are read: the others are taken as +0.0, which
// leaves the sum's bits as they are (no partial sum is -0.0).
__global__ void __launch_bounds__(kBlock) k_finish(FinishBatch B, int ratio, int nparts) {
  __shared__ double sh[kBlock];
  const double* part = B.v[blockIdx.x].part;
  double* out = B.v[blockIdx.x].out;
  double* hout = B.v[blockIdx.x].hout;
  double a = 0.0, b = 0.0;
  for (int t = threadIdx.x; t < nparts; t += kBlock) {
    a += part[t];
    if (ratio) b += part[kParts + t];
  }
  double sa = block_sum(a, sh);
  double sb = ratio ? block_sum(b, sh) : 0.0;
  if (threadIdx.x == 0) {
    if (ratio) {
      out[0] = sa / sb;
      out[1] = sa;
      out[2] = sb;
    } else {
      out[0] = sa;
    }
    // a system-scope store: the value reaches host memory past the GPU caches
    if (hout) __hip_atomic_store(hout, ratio ? sa / sb : sa, __ATOMIC_RELEASE,
                                 __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// One calculation of a damping launch: the level's operator, the coarse
// correction x and right-hand side w0, and its partial sums.
template <class T>
struct DampPart {
  Ops27<T> A;
  const T* D;
  const T* x;
  const T* w0;
  double* part;
};

template <class T>
__device__ __forceinline__ void damp_body(int nx, int ny, int nz, const Ops27<T>& A,
                                          const T* __restrict__ D, const T* __restrict__ x,
                                          const T* __restrict__ w0, double* part) {
  __shared__ double sh[kBlock];
  const long ni = nx - 2, nij = ni * (ny - 2), n = nij * (nz - 2);
  const size_t nxy = (size_t)nx * ny;
  double num = 0.0, den = 0.0;
  for (long t = (long)blockIdx.x * kBlock + threadIdx.x; t < n; t += (long)kParts * kBlock) {
    const int i = 1 + (int)(t % ni), j = 1 + (int)((t / ni) % (ny - 2)), k = 1 + (int)(t / nij);
    const size_t p = IX(i, j, k, nx, ny);
    P27<T> s = part27<T>(A.a, x, p, nx, nxy);
    const T ax = (-s.o) + (-s.u) + (-s.d) + D[p] * x[p];
    num += (double)x[p] * (double)w0[p];
    den += (double)x[p] * (double)ax;
  }
  double sn = block_sum(num, sh);
  double sd = block_sum(den, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = sn;
    part[kParts + blockIdx.x] = sd;
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock) k_damp_part(int nx, int ny, int nz, Batch<DampPart<T>> B) {
  const DampPart<T>& a = B.v[blockIdx.z];
  damp_body<T>(nx, ny, nz, a.A, a.D, a.x, a.w0, a.part);
}

// ---------------------------------------------------------------- transfers
// Restriction P^T (matvecd.c:801-913) with weights 1, 1/2, 1/4, 1/8.
template <class T>
__device__ __forceinline__ T restrict_at(int nxf, int nyf, int I, int J, int K,
                                         const T* __restrict__ in) {
  const T W1 = T(1.0), W2 = T(0.5), W4 = T(0.25), W8 = T(0.125);
  const int ii = 2 * I, jj = 2 * J, kk = 2 * K;
  const size_t sx = 1, sy = nxf, sz = (size_t)nxf * nyf;
  const size_t c = IX(ii, jj, kk, nxf, nyf);
  T o = W1 * in[c];
  o += W2 * in[c + sy];
  o += W2 * in[c - sy];
  o += W2 * in[c + sx];
  o += W2 * in[c - sx];
  o += W4 * in[c + sx + sy];
  o += W4 * in[c - sx + sy];
  o += W4 * in[c + sx - sy];
  o += W4 * in[c - sx - sy];
  const size_t u0 = c + sz;
  T u = W2 * in[u0];
  u += W4 * in[u0 + sy];
  u += W4 * in[u0 - sy];
  u += W4 * in[u0 + sx];
  u += W4 * in[u0 - sx];
  u += W8 * in[u0 + sx + sy];
  u += W8 * in[u0 - sx + sy];
  u += W8 * in[u0 + sx - sy];
  u += W8 * in[u0 - sx - sy];
  const size_t d0 = c - sz;
  T d = W2 * in[d0];
  d += W4 * in[d0 + sy];
  d += W4 * in[d0 - sy];
  d += W4 * in[d0 + sx];
  d += W4 * in[d0 - sx];
  d += W8 * in[d0 + sx + sy];
  d += W8 * in[d0 - sx + sy];
  d += W8 * in[d0 + sx - sy];
  d += W8 * in[d0 - sx - sy];
  return o + u + d;
}

template <class T>
__device__ __forceinline__ void restrict_body(int nxf, int nyf, int nxc, int nyc,
                                              const T* __restrict__ in, T* __restrict__ out,
                                              T* __restrict__ zero) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int K = blockIdx.y + 1;
  const int I = 1 + t % (nxc - 2), J = 1 + t / (nxc - 2);
  if (J > nyc - 2) return;
  out[IX(I, J, K, nxc, nyc)] = restrict_at<T>(nxf, nyf, I, J, K, in);
  if (zero) zero[IX(I, J, K, nxc, nyc)] = T(0);
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_restrict(int nxf, int nyf, int nzf, int nxc, int nyc, int nzc, Batch<TransferArgs<T>> B) {
  const TransferArgs<T>& a = B.v[blockIdx.z];
  restrict_body<T>(nxf, nyf, nxc, nyc, a.in, a.out, a.zero);
}

// restrict3 and the level's Jacobian diagonal, every point a thread: the
// boundary layer of c keeps its values.  Launched apart for each calculation
// and level with one pass over all diagonals behind them, a Newton step of
// eight calculations at 65^3 took 48 launches here, 4 so.
__device__ __forceinline__ void restrict_diag_body(int nxf, int nyf, int nxc, int nyc, int nzc,
                                                   const double* __restrict__ in,
                                                   double* __restrict__ out,
                                                   const double* __restrict__ oC,
                                                   double* __restrict__ D,
                                                   float* __restrict__ Df) {
  const unsigned t = blockIdx.x * kBlock + threadIdx.x, nx = nxc, ny = nyc;
  const int I = (int)(t % nx), J = (int)(t / nx % ny), K = (int)(t / nx / ny);
  if (K >= nzc) return;
  const size_t p = IX(I, J, K, nxc, nyc);
  double c;
  if (I >= 1 && I <= nxc - 2 && J >= 1 && J <= nyc - 2 && K >= 1 && K <= nzc - 2)
    out[p] = c = restrict_at<double>(nxf, nyf, I, J, K, in);
  else
    c = out[p];
  const double v = oC[p] + c;
  D[p] = v;
  if (Df) Df[p] = (float)v;
}

__global__ void __launch_bounds__(kBlock)
    k_restrict_diag(int nxf, int nyf, int nxc, int nyc, int nzc, Batch<DiagArgs> B) {
  const DiagArgs& a = B.v[blockIdx.z];
  restrict_diag_body(nxf, nyf, nxc, nyc, nzc, a.in, a.out, a.oC, a.D, a.Df);
}

// Trilinear prolongation and correction x_f += damp * P x_c (matvecd.c:935-1076
// followed by Vxaxpy, mgcsd.c:485-487).  The reference gives coarse boundary
// points weight 0; the coarse solution's boundary layer is zero (never
// written), so here they are read and add +0: the same terms in the same
// order, W * x_c with W = 1/2^(number of odd fine indices), without the
// per-term boundary tests.
// A lane updates the 16 bytes of a row from fine index kN m on (kN = 4 floats
// or 2 doubles: one load and one store of x_f, kN / 2 + 1 coarse values of
// each row the point's parities call for).  A point a lane, its parities
// diverging along the row, was bound by the addresser: 21.4 us onto 161^3 in
// FP32 (11.7 so; 8 bytes a point at the copy rate take 6), 29 in FP64 (17.9),
// 235 onto 353^3 in FP32 (94); onto 65^3 and below no difference.
template <class T>
__device__ __forceinline__ void prolong_body(int nxc, int nyc, int nxf, int nyf,
                                             const T* __restrict__ xc, T* __restrict__ xf,
                                             const double* __restrict__ damp) {
  constexpr int kN = 16 / (int)sizeof(T);
  const int nv = (nxf - 1 + kN - 1) / kN;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int m = t % nv, j = 1 + t / nv;
  if (j > nyf - 2) return;
  const int by = j & 1, bz = k & 1, i0 = kN * m, I0 = i0 / 2;
  const T W = (by ? T(0.5) : T(1.0)) * (bz ? T(0.5) : T(1.0));
  const size_t sy = nxc, sz = (size_t)nxc * nyc;
  const size_t row = IX(0, j >> 1, k >> 1, nxc, nyc);
  const size_t p = IX(i0, j, k, nxf, nyf);
  // (i0 + kN <= nxf - 1: the whole run is inside the row)
  const bool whole = m > 0 && i0 + kN <= nxf - 1;
  T x[kN], v[kN];
  if (whole) vld16(x, xf + p);
#pragma unroll
  for (int e = 0; e < kN; e++) v[e] = T(0);
  // terms in the order (0,0,0), (1,0,0), (0,1,0), (1,1,0), then the same at kk + 1
  auto add = [&](size_t r, bool first) {
    T c[kN / 2 + 1];
#pragma unroll
    for (int q = 0; q <= kN / 2; q++) c[q] = xc[r + min(I0 + q, nxc - 1)];
#pragma unroll
    for (int e = 0; e < kN; e++) {
      const T w = (e & 1) ? W * T(0.5) : W;
      v[e] = first ? w * c[e / 2] : v[e] + w * c[e / 2];
      if (e & 1) v[e] += w * c[e / 2 + 1];
    }
  };
  add(row, true);
  if (by) add(row + sy, false);
  if (bz) {
    add(row + sz, false);
    if (by) add(row + sz + sy, false);
  }
  const T dm = T(damp[0]);
  if (whole) {
#pragma unroll
    for (int e = 0; e < kN; e++) x[e] = x[e] + dm * v[e];
    vst16(xf + p, x);
  } else {
#pragma unroll
    for (int e = 0; e < kN; e++)
      if (i0 + e >= 1 && i0 + e <= nxf - 2) xf[p + e] = xf[p + e] + dm * v[e];
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_prolong_add(int nxc, int nyc, int nxf, int nyf, Batch<TransferArgs<T>> B) {
  const TransferArgs<T>& a = B.v[blockIdx.z];
  prolong_body<T>(nxc, nyc, nxf, nyf, a.in, a.out, a.damp);
}

// ------------------------------------------------------------- vector kit
template <class T>
__global__ void k_fill(T* x, size_t n, T v) {
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (size_t)gridDim.x * kBlock)
    x[t] = v;
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_axpy_int(int nx, int ny, int nz, double a, const T* __restrict__ x, T* __restrict__ y) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int i = 1 + t % (nx - 2), j = 1 + t / (nx - 2);
  if (j > ny - 2) return;
  const size_t p = IX(i, j, k, nx, ny);
  y[p] += T(a) * x[p];
}

__global__ void __launch_bounds__(kBlock)
    k_xpay_int(int nx, int ny, int nz, const double* __restrict__ x, double a,
               const double* __restrict__ z, double* __restrict__ y) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int i = 1 + t % (nx - 2), j = 1 + t / (nx - 2);
  if (j > ny - 2) return;
  const size_t p = IX(i, j, k, nx, ny);
  double v = x[p];
  v += a * z[p];
  y[p] = v;
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_copy_int(int nx, int ny, int nz, const T* __restrict__ x, T* __restrict__ y) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int i = 1 + t % (nx - 2), j = 1 + t / (nx - 2);
  if (j > ny - 2) return;
  const size_t p = IX(i, j, k, nx, ny);
  y[p] = x[p];
}

template <class T>
__global__ void k_add_diag(size_t n, const T* __restrict__ oC, const T* __restrict__ cc,
                           T* __restrict__ D, float* __restrict__ Df) {
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (size_t)gridDim.x * kBlock) {
    const T v = oC[t] + cc[t];
    D[t] = v;
    if (Df) Df[t] = (float)v;
  }
}

// Zero up to kZeroMax arrays in one launch.  Each array owns a contiguous
// range of blocks (found once per block).  A whole array is cleared in 16-byte
// stores, kZeroChunk words per block; a shell array one outer-layer element
// per thread: the planes k = 0 and nz-1, then per inner plane the rows j = 0
// and ny-1 and the ends i = 0 and nx-1 of the other rows.
constexpr unsigned kZeroChunk = 4 * 4 * kBlock;

__device__ inline size_t shell_index(int nx, int ny, int nz, size_t e) {
  const size_t plane = (size_t)nx * ny;
  if (e < plane) return e;
  if (e < 2 * plane) return (size_t)(nz - 1) * plane + (e - plane);
  const size_t r0 = e - 2 * plane;
  const size_t per = 2 * (size_t)nx + 2 * (size_t)(ny - 2);
  const size_t k = 1 + r0 / per;
  const size_t r = r0 % per;
  size_t i, j;
  if (r < (size_t)nx) {
    i = r;
    j = 0;
  } else if (r < 2 * (size_t)nx) {
    i = r - nx;
    j = ny - 1;
  } else {
    const size_t q = r - 2 * (size_t)nx;
    j = 1 + q / 2;
    i = (q & 1) ? nx - 1 : 0;
  }
  return (k * ny + j) * nx + i;
}

__global__ void __launch_bounds__(kBlock) k_zero_many(ZeroArgs Z) {
  const unsigned b = blockIdx.x;
  int a = 0;
  while (a + 1 < Z.n && b >= Z.blk[a + 1]) a++;
  const unsigned lb = b - Z.blk[a];
  unsigned* base = Z.p[a];
  if (Z.nx[a] == 0) {
    const size_t w0 = (size_t)lb * kZeroChunk;
    const size_t w1 = min(w0 + kZeroChunk, Z.words[a]);
    const size_t v1 = w0 + ((w1 - w0) & ~(size_t)3);
    uint4* v = reinterpret_cast<uint4*>(base + w0);
    for (size_t t = threadIdx.x; w0 + 4 * t < v1; t += kBlock) v[t] = make_uint4(0u, 0u, 0u, 0u);
    for (size_t w = v1 + threadIdx.x; w < w1; w += kBlock) base[w] = 0u;
  } else {
    const size_t e = (size_t)lb * kBlock + threadIdx.x;
    if (e >= Z.words[a]) return;
    const size_t p = shell_index(Z.nx[a], Z.ny[a], Z.nz[a], e) * Z.wpe[a];
    for (int w = 0; w < Z.wpe[a]; w++) base[p + w] = 0u;
  }
}

// D_l = oC_l + c_l on every level in one launch (and Df_l = (float) D_l
// where Df_l is given): the same values as one add_diag per level.
__global__ void __launch_bounds__(kBlock) k_add_diag_levels(DiagLevels L) {
  const size_t tot = L.off[L.nl];
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < tot;
       t += (size_t)gridDim.x * kBlock) {
    int l = 0;
    while (t >= L.off[l + 1]) l++;
    const size_t i = t - L.off[l];
    const double v = L.oC[l][i] + L.c[l][i];
    L.D[l][i] = v;
    if (L.Df[l]) L.Df[l][i] = (float)v;
  }
}

// y += a * (double) x on the interior: an FP32 correction added to an FP64
// solution, the same bits as converting x first and calling axpy_interior
__global__ void __launch_bounds__(kBlock)
    k_axpy_int_f32(int nx, int ny, int nz, double a, const float* __restrict__ x,
                   double* __restrict__ y, int assign) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int i = 1 + t % (nx - 2), j = 1 + t / (nx - 2);
  if (j > ny - 2) return;
  const size_t p = IX(i, j, k, nx, ny);
  // assign: y starts at zero, and 0.0 + v rounds like the update of a zero y
  double v = assign ? 0.0 : y[p];
  v += a * (double)x[p];
  y[p] = v;
}

__global__ void k_scale(size_t n, double a, const double* __restrict__ x, double* __restrict__ y) {
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (size_t)gridDim.x * kBlock)
    y[t] = a * x[t];
}

template <class Tin, class Tout>
__global__ void k_convert(size_t n, const Tin* __restrict__ in, Tout* __restrict__ out) {
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (size_t)gridDim.x * kBlock)
    out[t] = (Tout)in[t];
}

// array blockIdx.y of the list
__global__ void __launch_bounds__(kBlock) k_convert_many(ConvArgs C) {
  const double* __restrict__ in = C.in[blockIdx.y];
  float* __restrict__ out = C.out[blockIdx.y];
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < C.n;
       t += (size_t)gridDim.x * kBlock)
    out[t] = (float)in[t];
}

// VfboundPMG (mikpckd.c:209-256): x faces, then y faces, then z faces, so
// edge points take the value of the last face written.
__global__ void k_faces(int nx, int ny, int nz, double* u, const double* gx, const double* gy,
                        const double* gz, int pass) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (pass == 0) {
    if (t >= ny * nz) return;
    const int j = t % ny, k = t / ny;
    u[IX(0, j, k, nx, ny)] = gx[j + ny * k];
    u[IX(nx - 1, j, k, nx, ny)] = gx[j + ny * k + (size_t)ny * nz];
  } else if (pass == 1) {
    if (t >= nx * nz) return;
    const int i = t % nx, k = t / nx;
    u[IX(i, 0, k, nx, ny)] = gy[i + nx * k];
    u[IX(i, ny - 1, k, nx, ny)] = gy[i + nx * k + (size_t)nx * nz];
  } else {
    if (t >= nx * ny) return;
    const int i = t % nx, j = t / nx;
    u[IX(i, j, 0, nx, ny)] = gz[i + nx * j];
    u[IX(i, j, nz - 1, nx, ny)] = gz[i + nx * j + (size_t)nx * ny];
  }
}

// ---------------------------------------------------------------- nonlinear
// sum over species of (-c_s q_s) cc exp(clamp(-q_s u)) (mypdec.c:145-223)
__device__ inline double ncvec(double coef, double u, const Ions& I) {
  double out = 0;
  for (int s = 0; s < I.nion; s++) {
    const double zcf2 = -1.0 * I.sconc[s] * I.q[s];
    const double zu2 = -1.0 * I.q[s];
    double az = fabs(zcf2 * coef);
    const double am_zero = (1.0e-20 <= az ? 1.0e-20 : az) * 1.0e20;
    double a = zu2 * u;
    double mn = (a <= 0.0) ? a : 0.0;
    const double am_neg = (mn >= -85.0) ? mn : -85.0;
    double mx = (a >= 0.0) ? a : 0.0;
    const double am_pos = (mx <= 85.0) ? mx : 85.0;
    const double arg = am_zero * (am_neg + am_pos);
    out = out + zcf2 * coef * exp(arg);
  }
  return out;
}

__global__ void __launch_bounds__(kBlock)
    k_nresid7(int nx, int ny, int nz, const double* __restrict__ oC, const double* __restrict__ oE,
              const double* __restrict__ oN, const double* __restrict__ uC,
              const double* __restrict__ cc, const double* __restrict__ fc,
              const double* __restrict__ x, double* __restrict__ r, Ions ions) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int i = 1 + t % (nx - 2), j = 1 + t / (nx - 2);
  if (j > ny - 2) return;
  const size_t nxy = (size_t)nx * ny;
  const size_t p = IX(i, j, k, nx, ny);
  const double w = ncvec(cc[p], x[p], ions);
  r[p] = acc7(fc[p], oE, oN, uC, x, p, nx, nxy) - oC[p] * x[p] - w;
}

// k_nresid7 with the L1-norm partials of the residual (order of k_nrm1_part).
__global__ void __launch_bounds__(kBlock)
    k_nresid7_nrm(int nx, int ny, int nz, PartRuns R, const double* __restrict__ oC,
                  const double* __restrict__ oE, const double* __restrict__ oN,
                  const double* __restrict__ uC, const double* __restrict__ cc,
                  const double* __restrict__ fc, const double* __restrict__ x,
                  double* __restrict__ r, Ions ions, double* part) {
  __shared__ double sh[kBlock];
  const size_t nxy = (size_t)nx * ny;
  double acc = 0.0;
  part_columns(nx, ny, nz, R, [&](size_t p, int planes) {
    double xkm = x[p - nxy], x0 = x[p], vUm = uC[p - nxy];
    for (int m = 0; m < planes; m++, p += nxy) {
      // every operand first; acc7's terms and order
      const double xjp = x[p + nx], xjm = x[p - nx], xip = x[p + 1], xim = x[p - 1];
      const double xkp = x[p + nxy];
      const double vN = oN[p], vNm = oN[p - nx], vE = oE[p], vEm = oE[p - 1];
      const double vU = uC[p], vC = oC[p], vcc = cc[p], vfc = fc[p];
      const double w = ncvec(vcc, x0, ions);
      double s7 = vfc;
      s7 += vN * xjp;
      s7 += vNm * xjm;
      s7 += vE * xip;
      s7 += vEm * xim;
      s7 += vUm * xkm;
      s7 += vU * xkp;
      const double v = s7 - vC * x0 - w;
      r[p] = v;
      acc += fabs(v);
      xkm = x0;
      x0 = xkp;
      vUm = vU;
    }
  });
  double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// k_nresid7_nrm at the trial point y = x + a z (k_xpay_int's arithmetic,
// evaluated for every stencil point it reads), storing y and the residual:
// the same bits as k_xpay_int then k_nresid7_nrm.  The boundary layers of x
// and z are zero, as y's is.
__global__ void __launch_bounds__(kBlock)
    k_nresid7_xpay(int nx, int ny, int nz, PartRuns R, const double* __restrict__ oC,
                   const double* __restrict__ oE, const double* __restrict__ oN,
                   const double* __restrict__ uC, const double* __restrict__ cc,
                   const double* __restrict__ fc, const double* __restrict__ x, double a,
                   const double* __restrict__ z, double* __restrict__ y,
                   double* __restrict__ r, Ions ions, double* part) {
  __shared__ double sh[kBlock];
  const size_t nxy = (size_t)nx * ny;
  double acc = 0.0;
  auto trial = [&](size_t q) {
    double v = x[q];
    v += a * z[q];
    return v;
  };
  part_columns(nx, ny, nz, R, [&](size_t p, int planes) {
    double ykm = trial(p - nxy), y0 = trial(p), vUm = uC[p - nxy];
    for (int m = 0; m < planes; m++, p += nxy) {
      // every operand first: the neighbours +j, -j, +i, -i and +k
      const size_t q[5] = {p + nx, p - nx, p + 1, p - 1, p + nxy};
      double xc[5], zc[5];
#pragma unroll
      for (int u = 0; u < 5; u++) {
        xc[u] = x[q[u]];
        zc[u] = z[q[u]];
      }
      const double vN = oN[p], vNm = oN[p - nx], vE = oE[p], vEm = oE[p - 1];
      const double vU = uC[p], vC = oC[p], vcc = cc[p], vfc = fc[p];
      double yc[5];
#pragma unroll
      for (int u = 0; u < 5; u++) {
        double v = xc[u];
        v += a * zc[u];
        yc[u] = v;
      }
      const double w = ncvec(vcc, y0, ions);
      double s7 = vfc;
      s7 += vN * yc[0];
      s7 += vNm * yc[1];
      s7 += vE * yc[2];
      s7 += vEm * yc[3];
      s7 += vUm * ykm;
      s7 += vU * yc[4];
      const double v = s7 - vC * y0 - w;
      acc += fabs(v);
      y[p] = y0;
      r[p] = v;
      ykm = y0;
      y0 = yc[4];
      vUm = vU;
    }
  });
  double s = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// The end of a Newton step's inner cycle and the step's first trial point in
// one pass.  With z the correction the cycle produced (its boundary layer
// zero; read as (double) zf when zf is given, the values an FP32 correction
// assigned to z would have): the inner residual fz + J z of the Jacobian
// system (J's diagonal D), its FP32 image in r32 and its L1 partials in
// part[0, kParts) (k_resid7_nrm<double>'s values and order); and y = x + a z
// with the nonlinear residual at y in rn (its FP32 image in rn32 when given),
// its L1 partials in part[kParts, 2 kParts) (k_nresid7_xpay's values and
// order).  The two stencils share their operator loads.
// Every operand of a point is loaded before the arithmetic (the two stencils
// read z and x at the same seven points); kZF selects z from zf.
template <bool kZF>
__device__ __forceinline__ void jres_body(
    int nx, int ny, int nz, const PartRuns& R, const double* __restrict__ oC,
    const double* __restrict__ oE, const double* __restrict__ oN, const double* __restrict__ uC,
    const double* __restrict__ D, const double* __restrict__ cc, const double* __restrict__ fc,
    const double* __restrict__ fz, const double* __restrict__ x, double a,
    const double* __restrict__ z, const float* __restrict__ zf, double* __restrict__ y,
    double* __restrict__ rn, float* __restrict__ r32, float* __restrict__ rn32, const Ions& ions,
    double* part) {
  __shared__ double sh[kBlock];
  const size_t nxy = (size_t)nx * ny;
  double acc_j = 0.0, acc_n = 0.0;
  auto zval = [&](size_t q) { return kZF ? (double)zf[q] : z[q]; };
  part_columns(nx, ny, nz, R, [&](size_t p, int planes) {
    // z and the trial value y = x + a z (k_xpay_int's arithmetic) of planes
    // k - 1 and k
    double zkm = zval(p - nxy), z0 = zval(p), ykm = x[p - nxy], y0 = x[p], vUm = uC[p - nxy];
    ykm += a * zkm;
    y0 += a * z0;
    for (int m = 0; m < planes; m++, p += nxy) {
      // the neighbours +j, -j, +i, -i and +k
      const size_t q[5] = {p + nx, p - nx, p + 1, p - 1, p + nxy};
      double zc[5], xc[5];
#pragma unroll
      for (int u = 0; u < 5; u++) {
        zc[u] = zval(q[u]);
        xc[u] = x[q[u]];
      }
      const double vfz = fz[p], vN = oN[p], vNm = oN[p - nx], vE = oE[p], vEm = oE[p - 1];
      const double vU = uC[p], vD = D[p], vC = oC[p], vcc = cc[p], vfc = fc[p];
      // acc7's terms and order at z
      double sj = vfz;
      sj += vN * zc[0];
      sj += vNm * zc[1];
      sj += vE * zc[2];
      sj += vEm * zc[3];
      sj += vUm * zkm;
      sj += vU * zc[4];
      const double vj = sj - vD * z0;
      acc_j += fabs(vj);
      double yc[5];
#pragma unroll
      for (int u = 0; u < 5; u++) {
        double v = xc[u];
        v += a * zc[u];
        yc[u] = v;
      }
      const double w = ncvec(vcc, y0, ions);
      double s7 = vfc;
      s7 += vN * yc[0];
      s7 += vNm * yc[1];
      s7 += vE * yc[2];
      s7 += vEm * yc[3];
      s7 += vUm * ykm;
      s7 += vU * yc[4];
      const double v = s7 - vC * y0 - w;
      acc_n += fabs(v);
      if (r32) r32[p] = (float)vj;
      y[p] = y0;
      rn[p] = v;
      if (rn32) rn32[p] = (float)v;
      zkm = z0;
      z0 = zc[4];
      ykm = y0;
      y0 = yc[4];
      vUm = vU;
    }
  });
  const double bj = block_sum(acc_j, sh);
  const double bn = block_sum(acc_n, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = bj;
    part[kParts + blockIdx.x] = bn;
  }
}

template <bool kZF>
__global__ void __launch_bounds__(kBlock)
    k_jres_trial(int nx, int ny, int nz, PartRuns R, double a, Batch<JresArgs> B) {
  const JresArgs& c = B.v[blockIdx.y];
  jres_body<kZF>(nx, ny, nz, R, c.A.a[0], c.A.a[1], c.A.a[2], c.A.a[3], c.D, c.cc, c.fc, c.fz, c.x,
                 a, c.z, c.zf, c.y, c.rn, c.r32, c.rn32, c.ions, c.part);
}

// Vdc_vecpmg (mypdec.c:366-433) at every point; with oC given also the
// diagonal D = oC + N'(x) and, with Df, its FP32 image (k_add_diag_levels'
// values for this level) in the same pass.
__device__ __forceinline__ void dcvec_body(size_t n, const double* __restrict__ cc,
                                           const double* __restrict__ x, double* __restrict__ out,
                                           const Ions& I, const double* __restrict__ oC,
                                           double* __restrict__ D, float* __restrict__ Df) {
  for (size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x; t < n; t += (size_t)gridDim.x * kBlock) {
    double o = 0.0;
    const double coef = cc[t], u = x[t];
    for (int s = 0; s < I.nion; s++) {
      const double zcf2 = I.sconc[s] * I.q[s] * I.q[s];
      const double zu2 = -1.0 * I.q[s];
      double az = fabs(zcf2 * coef);
      const double am_zero = (1.0e-20 <= az ? 1.0e-20 : az) * 1.0e20;
      double a = zu2 * u;
      double mn = (a <= 0.0) ? a : 0.0;
      const double am_neg = (mn >= -85.0) ? mn : -85.0;
      double mx = (a >= 0.0) ? a : 0.0;
      const double am_pos = (mx <= 85.0) ? mx : 85.0;
      const double arg = am_zero * (am_neg + am_pos);
      o += zcf2 * coef * exp(arg);
    }
    out[t] = o;
    if (oC) {
      const double v = oC[t] + o;
      D[t] = v;
      if (Df) Df[t] = (float)v;
    }
  }
}

__global__ void __launch_bounds__(kBlock) k_dcvec(size_t n, Batch<DcArgs> B) {
  const DcArgs& a = B.v[blockIdx.y];
  dcvec_body(n, a.cc, a.x, a.out, a.ions, a.oC, a.D, a.Df);
}

// ---------------------------------------------------------------- operators
// VbuildA_fv (buildAd.c:105-281), face terms folded into fc in the order
// east, north, up, west, south, down.
__global__ void __launch_bounds__(kBlock)
    k_buildA(int nx, int ny, int nz, const double* xf, const double* yf, const double* zf,
             const double* gx, const double* gy, const double* gz, const double* a1,
             const double* a2, const double* a3, const double* ccf, const double* fcf,
             double* oC, double* cc, double* fc, double* oE, double* oN, double* uC) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const int k = blockIdx.y + 1;
  const int i = 1 + t % (nx - 2), j = 1 + t / (nx - 2);
  if (j > ny - 2) return;
  const double diag = 1.0;
  const double hzm1 = zf[k] - zf[k - 1], hz = zf[k + 1] - zf[k];
  const double hym1 = yf[j] - yf[j - 1], hy = yf[j + 1] - yf[j];
  const double hxm1 = xf[i] - xf[i - 1], hx = xf[i + 1] - xf[i];
  const double c_oE = diag * (hym1 + hy) * (hzm1 + hz) / (4.0 * hx);
  const double c_oEm1 = diag * (hym1 + hy) * (hzm1 + hz) / (4.0 * hxm1);
  const double c_oN = diag * (hxm1 + hx) * (hzm1 + hz) / (4.0 * hy);
  const double c_oNm1 = diag * (hxm1 + hx) * (hzm1 + hz) / (4.0 * hym1);
  const double c_uC = diag * (hxm1 + hx) * (hym1 + hy) / (4.0 * hz);
  const double c_uCm1 = diag * (hxm1 + hx) * (hym1 + hy) / (4.0 * hzm1);
  const double c_fc = diag * (hxm1 + hx) * (hym1 + hy) * (hzm1 + hz) / 8.0;
  const size_t nxy = (size_t)nx * ny;
  const size_t p = IX(i, j, k, nx, ny);
  double f = c_fc * fcf[p];
  cc[p] = c_fc * ccf[p];
  double d = c_oE * a1[p];
  d += c_oEm1 * a1[p - 1];
  d += c_oN * a2[p];
  d += c_oNm1 * a2[p - nx];
  d += c_uC * a3[p];
  d += c_uCm1 * a3[p - nxy];
  oC[p] = d;
  if (i != nx - 2) {
    oE[p] = c_oE * a1[p];
  } else {
    oE[p] = 0.0;
    f += c_oE * a1[p] * gx[j + ny * k + (size_t)ny * nz];
  }
  if (j != ny - 2) {
    oN[p] = c_oN * a2[p];
  } else {
    oN[p] = 0.0;
    f += c_oN * a2[p] * gy[i + nx * k + (size_t)nx * nz];
  }
  if (k != nz - 2) {
    uC[p] = c_uC * a3[p];
  } else {
    uC[p] = 0.0;
    f += c_uC * a3[p] * gz[i + nx * j + (size_t)nx * ny];
  }
  if (i == 1) f += c_oEm1 * a1[p - 1] * gx[j + ny * k];
  if (j == 1) f += c_oNm1 * a2[p - nx] * gy[i + nx * k];
  if (k == 1) f += c_uCm1 * a3[p - nxy] * gz[i + nx * j];
  fc[p] = f;
}

inline unsigned nblocks(size_t n) {
  size_t b = (n + kBlock - 1) / kBlock;
  if (b > 65535) b = 65535;
  if (b == 0) b = 1;
  return (unsigned)b;
}

}  // namespace

// =================================================================== wrappers

template <class T>
void gsrb7(hipStream_t s, int nx, int ny, int nz, const Ops<T>& A, const T* D, const T* fc, T* x,
           int nu, int iadjoint) {
  const int npair = (nx - 1) / 2;
  const long cnt = (long)npair * (ny - 2);
  dim3 g((unsigned)((cnt + kBlock - 1) / kBlock), (unsigned)(nz - 2));
  for (int it = 0; it < nu; it++) {
    // red (par 1) then black (par 0); swapped for the adjoint sweep
    const int first = iadjoint ? 0 : 1;
    k_gsrb7<T><<<g, kBlock, 0, s>>>(nx, ny, nz, A.a[1], A.a[2], A.a[3], D, fc, x, first);
    k_gsrb7<T><<<g, kBlock, 0, s>>>(nx, ny, nz, A.a[1], A.a[2], A.a[3], D, fc, x, 1 - first);
  }
}

int gsrb7_launches(int nu) { return 2 * nu; }

template <class T>
static Batch<Args27<T>> args27(const LevelArgs<T>* c, int nb) {
  Batch<Args27<T>> B;
  for (int b = 0; b < nb; b++)
    B.v[b] = Args27<T>{to27(c[b].A), c[b].D, c[b].f, c[b].x, c[b].r, nullptr};
  return B;
}

template <class T>
void gsrb27_batch(hipStream_t s, int nx, int ny, int nz, const LevelArgs<T>* c, int nb, int nu,
                  int iadjoint) {
  check_batch(nb);
  const Batch<Args27<T>> B = args27(c, nb);
  for (int it = 0; it < nu; it++)
    for (int cc = 0; cc < 8; cc++) {
      const int col = iadjoint ? 7 - cc : cc;
      const int i0 = (col & 1) ? 1 : 2, j0 = ((col >> 1) & 1) ? 1 : 2, k0 = ((col >> 2) & 1) ? 1 : 2;
      const int ni = (nx - 2 - i0) / 2 + 1, nj = (ny - 2 - j0) / 2 + 1, nk = (nz - 2 - k0) / 2 + 1;
      if (ni <= 0 || nj <= 0 || nk <= 0) continue;
      dim3 g((unsigned)(((long)ni * nj + kBlock - 1) / kBlock), (unsigned)nk, (unsigned)nb);
      k_gsrb27<T><<<g, kBlock, 0, s>>>(nx, ny, nz, B, col);
    }
}

template <class T>
void gsrb27(hipStream_t s, int nx, int ny, int nz, const Ops<T>& A, const T* D, const T* fc, T* x,
            int nu, int iadjoint) {
  const LevelArgs<T> c{A, D, fc, x, nullptr, nullptr};
  gsrb27_batch<T>(s, nx, ny, nz, &c, 1, nu, iadjoint);
}

// The colour-pair sweeps with the vector kernel.
constexpr int kPairRun = 2;  // points of a run

template <class T>
static void vpair_launch(hipStream_t s, int nx, int ny, int nz, const Batch<Args27<T>>& B,
                         int nb, int nu, int iadjoint) {
  const int R = (nx - 2 + kPairRun - 1) / kPairRun;
  // workgroup size: whole rows, fewest idle lanes
  int NT = kBlock, idle = 1 << 30;
  for (int t = 64; t <= kBlock; t += 64) {
    if (t < R) continue;
    const int id = t - (t / R) * R;
    if (id * kBlock < idle * t) {  // compare idle fractions
      idle = id;
      NT = t;
    }
  }
  const int RB = NT / R;
  for (int it = 0; it < nu; it++)
    for (int h = 0; h < 4; h++) {
      // forward: (0,1) (2,3) (4,5) (6,7); adjoint: (7,6) (5,4) (3,2) (1,0)
      const int col = iadjoint ? 7 - 2 * h : 2 * h;
      const int pa = col & 1, cj = (col >> 1) & 1, ck = (col >> 2) & 1;
      const int j0 = cj ? 1 : 2, k0 = ck ? 1 : 2;
      if (j0 > ny - 2 || k0 > nz - 2) continue;
      const long rows = (long)((ny - 2 - j0) / 2 + 1) * ((nz - 2 - k0) / 2 + 1);
      const dim3 g((unsigned)((rows + RB - 1) / RB), 1, (unsigned)nb);
      k_gsrb27_vpair<T, kPairRun><<<g, NT, (size_t)RB * nx * sizeof(T), s>>>(nx, ny, nz, B, pa,
                                                                             cj, ck, R, RB);
    }
}

// The colour-pair form, for the levels that gsrb27_use_planes leaves: rows of
// fewer than 40 points on planes of more than 49 rows, and in FP64 rows of 115 to
// 130.  Form 0 (the default): the vector kernel with runs of two points where a
// row holds one run plus its boundary points and fits one workgroup, else the
// one-point-per-lane kernel; form 1 that kernel.  Per sweep (4 launches), us, runs
// and one point per lane: 129^3 FP64 93.9 and 161.7; 33x65x65 18.5 and 20.9 (FP32
// 14.7 and 15.0).
template <class T>
void gsrb27_pairs_form(hipStream_t s, int nx, int ny, int nz, const LevelArgs<T>* c, int nb,
                       int nu, int iadjoint, int form) {
  check_batch(nb);
  const Batch<Args27<T>> B = args27(c, nb);
  if (form == 0 && nx >= kPairRun + 2 && (nx - 2 + kPairRun - 1) / kPairRun <= kBlock) {
    vpair_launch<T>(s, nx, ny, nz, B, nb, nu, iadjoint);
    return;
  }
  for (int it = 0; it < nu; it++)
    for (int h = 0; h < 4; h++) {
      const int col = iadjoint ? 7 - 2 * h : 2 * h;
      const int pa = col & 1, cj = (col >> 1) & 1, ck = (col >> 2) & 1;
      const int j0 = cj ? 1 : 2, k0 = ck ? 1 : 2;
      if (j0 > ny - 2 || k0 > nz - 2) continue;
      const long rows = (long)((ny - 2 - j0) / 2 + 1) * ((nz - 2 - k0) / 2 + 1);
      const dim3 g((unsigned)((rows * 64 + kBlock - 1) / kBlock), 1, (unsigned)nb);
      k_gsrb27_pair<T><<<g, kBlock, 0, s>>>(nx, ny, nz, B, pa, cj, ck);
    }
}

template <class T>
void gsrb27_pairs_batch(hipStream_t s, int nx, int ny, int nz, const LevelArgs<T>* c, int nb,
                        int nu, int iadjoint) {
  gsrb27_pairs_form<T>(s, nx, ny, nz, c, nb, nu, iadjoint, 0);
}

template <class T>
void gsrb27_pairs(hipStream_t s, int nx, int ny, int nz, const Ops<T>& A, const T* D,
                  const T* fc, T* x, int nu, int iadjoint) {
  const LevelArgs<T> c{A, D, fc, x, nullptr, nullptr};
  gsrb27_pairs_batch<T>(s, nx, ny, nz, &c, 1, nu, iadjoint);
}

bool gsrb27_use_pairs(int nx) { return nx >= 3 && nx <= 130; }

template <class T>
void resid_batch(hipStream_t s, int st, int nx, int ny, int nz, const LevelArgs<T>* c, int nb) {
  check_batch(nb);
  dim3 g = grid_interior(nx, ny, nz);
  g.z = (unsigned)nb;
  const Batch<Args27<T>> B = args27(c, nb);
  constexpr int kV = 16 / (int)sizeof(T);
  if (st == 7 && nx >= kV + 2) {
    const long lanes = (long)((nx - 2 + kV - 1) / kV) * (ny - 2) * (nz - 2);
    const dim3 gv((unsigned)((lanes + kBlock - 1) / kBlock), 1, (unsigned)nb);
    k_resid7v<T><<<gv, kBlock, 0, s>>>(nx, ny, nz, B);
  } else if (st == 7)
    k_resid7<T><<<g, kBlock, 0, s>>>(nx, ny, nz, B);
  else
    k_resid27<T><<<g, kBlock, 0, s>>>(nx, ny, nz, B);
}

template <class T>
void resid(hipStream_t s, int st, int nx, int ny, int nz, const Ops<T>& A, const T* D, const T* fc,
           const T* x, T* r) {
  const LevelArgs<T> c{A, D, fc, const_cast<T*>(x), nullptr, r};
  resid_batch<T>(s, st, nx, ny, nz, &c, 1);
}

void nresid7(hipStream_t s, int nx, int ny, int nz, const Ops<double>& A, const double* cc,
             const double* fc, const double* x, double* r, const Ions& ions) {
  k_nresid7<<<grid_interior(nx, ny, nz), kBlock, 0, s>>>(nx, ny, nz, A.a[0], A.a[1], A.a[2],
                                                         A.a[3], cc, fc, x, r, ions);
}

void dcvec_batch(hipStream_t s, size_t n, const DcArgs* c, int nb) {
  check_batch(nb);
  Batch<DcArgs> B;
  for (int b = 0; b < nb; b++) B.v[b] = c[b];
  k_dcvec<<<dim3(nblocks(n), nb), kBlock, 0, s>>>(n, B);
}

void dcvec(hipStream_t s, size_t n, const double* cc, const double* x, double* out,
           const Ions& ions, const double* oC, double* D, float* Df) {
  const DcArgs c{cc, x, out, oC, D, Df, ions};
  dcvec_batch(s, n, &c, 1);
}

void restrict_diag_batch(hipStream_t s, int nxf, int nyf, int nzf, int nxc, int nyc, int nzc,
                         const DiagArgs* c, int nb) {
  check_batch(nb);
  Batch<DiagArgs> B;
  for (int b = 0; b < nb; b++) B.v[b] = c[b];
  const size_t n = (size_t)nxc * nyc * nzc;
  k_restrict_diag<<<dim3((unsigned)((n + kBlock - 1) / kBlock), 1, nb), kBlock, 0, s>>>(
      nxf, nyf, nxc, nyc, nzc, B);
}

template <class T>
void restrict3_batch(hipStream_t s, int nxf, int nyf, int nzf, int nxc, int nyc, int nzc,
                     const TransferArgs<T>* c, int nb) {
  check_batch(nb);
  Batch<TransferArgs<T>> B;
  for (int b = 0; b < nb; b++) B.v[b] = c[b];
  dim3 g = grid_interior(nxc, nyc, nzc);
  g.z = (unsigned)nb;
  k_restrict<T><<<g, kBlock, 0, s>>>(nxf, nyf, nzf, nxc, nyc, nzc, B);
}

template <class T>
void restrict3(hipStream_t s, int nxf, int nyf, int nzf, int nxc, int nyc, int nzc, const T* in,
               T* out, T* zero) {
  const TransferArgs<T> c{in, out, zero, nullptr};
  restrict3_batch<T>(s, nxf, nyf, nzf, nxc, nyc, nzc, &c, 1);
}

template <class T>
void prolong_add_batch(hipStream_t s, int nxc, int nyc, int nzc, int nxf, int nyf, int nzf,
                       const TransferArgs<T>* c, int nb) {
  check_batch(nb);
  Batch<TransferArgs<T>> B;
  for (int b = 0; b < nb; b++) B.v[b] = c[b];
  constexpr int kN = 16 / (int)sizeof(T);
  const long cnt = (long)((nxf - 1 + kN - 1) / kN) * (nyf - 2);
  const dim3 g((unsigned)((cnt + kBlock - 1) / kBlock), (unsigned)(nzf - 2), (unsigned)nb);
  k_prolong_add<T><<<g, kBlock, 0, s>>>(nxc, nyc, nxf, nyf, B);
}

template <class T>
void prolong_add(hipStream_t s, int nxc, int nyc, int nzc, int nxf, int nyf, int nzf, const T* xc,
                 T* xf, const double* damp) {
  const TransferArgs<T> c{xc, xf, nullptr, damp};
  prolong_add_batch<T>(s, nxc, nyc, nzc, nxf, nyf, nzf, &c, 1);
}

template <class T>
void nrm1(hipStream_t s, int nx, int ny, int nz, const T* x, double* part, double* out,
          double* hout) {
  const PartRuns R = part_runs(nx, ny, nz);
  k_nrm1_part<T><<<kParts, kBlock, 0, s>>>(nx, ny, nz, R, x, part);
  {
    FinishBatch F;
    F.v[0] = FinishArgs{part, out, hout};
    k_finish<<<1, kBlock, 0, s>>>(F, 0, kParts);
  }
}

template <class T>
void resid7_nrm1(hipStream_t s, int nx, int ny, int nz, const Ops<T>& A, const T* D, const T* fc,
                 const T* x, T* r, double* part, double* out, double* hout, float* r32) {
  const PartRuns R = part_runs(nx, ny, nz);
  k_resid7_nrm<T><<<kParts, kBlock, 0, s>>>(nx, ny, nz, R, A.a[1], A.a[2], A.a[3], D, fc, x, r,
                                            r32, part);
  {
    FinishBatch F;
    F.v[0] = FinishArgs{part, out, hout};
    k_finish<<<1, kBlock, 0, s>>>(F, 0, kParts);
  }
}

void nrm1_to32(hipStream_t s, int nx, int ny, int nz, const double* x, float* y, double* part,
               double* out, double* hout) {
  const PartRuns R = part_runs(nx, ny, nz);
  k_nrm1_to32<<<kParts, kBlock, 0, s>>>(nx, ny, nz, R, x, y, part);
  FinishBatch F;
  F.v[0] = FinishArgs{part, out, hout};
  k_finish<<<1, kBlock, 0, s>>>(F, 0, kParts);
}

void nresid7_xpay_nrm1(hipStream_t s, int nx, int ny, int nz, const Ops<double>& A,
                       const double* cc, const double* fc, const double* x, double a,
                       const double* z, double* y, double* r, const Ions& ions, double* part,
                       double* out, double* hout) {
  const PartRuns R = part_runs(nx, ny, nz);
  k_nresid7_xpay<<<kParts, kBlock, 0, s>>>(nx, ny, nz, R, A.a[0], A.a[1], A.a[2], A.a[3], cc, fc,
                                           x, a, z, y, r, ions, part);
  FinishBatch F;
  F.v[0] = FinishArgs{part, out, hout};
  k_finish<<<1, kBlock, 0, s>>>(F, 0, kParts);
}

void jres_trial_nrm1_batch(hipStream_t s, int nx, int ny, int nz, double a, const JresArgs* c,
                           int nb) {
  check_batch(nb);
  const PartRuns R = part_runs(nx, ny, nz);
  Batch<JresArgs> B;
  FinishBatch F;
  for (int b = 0; b < nb; b++) {
    B.v[b] = c[b];
    F.v[2 * b] = FinishArgs{c[b].part, c[b].out, c[b].hout};
    F.v[2 * b + 1] = FinishArgs{c[b].part + kParts, c[b].out2, c[b].hout2};
  }
  if (c[0].zf)
    k_jres_trial<true><<<dim3(kParts, nb), kBlock, 0, s>>>(nx, ny, nz, R, a, B);
  else
    k_jres_trial<false><<<dim3(kParts, nb), kBlock, 0, s>>>(nx, ny, nz, R, a, B);
  k_finish<<<2 * nb, kBlock, 0, s>>>(F, 0, kParts);
}

void jres_trial_nrm1(hipStream_t s, int nx, int ny, int nz, const Ops<double>& A,
                     const double* D, const double* cc, const double* fc, const double* fz,
                     const double* x, double a, const double* z, const float* zf, double* y,
                     double* rn, float* r32, float* rn32, const Ions& ions, double* part,
                     double* out, double* hout, double* out2, double* hout2) {
  const JresArgs c{A,  D,   cc,   fc,   fz,  x,    z,    zf,    y,
                   rn, r32, rn32, part, out, hout, out2, hout2, ions};
  jres_trial_nrm1_batch(s, nx, ny, nz, a, &c, 1);
}

void nresid7_nrm1(hipStream_t s, int nx, int ny, int nz, const Ops<double>& A, const double* cc,
                  const double* fc, const double* x, double* r, const Ions& ions, double* part,
                  double* out, double* hout) {
  const PartRuns R = part_runs(nx, ny, nz);
  k_nresid7_nrm<<<kParts, kBlock, 0, s>>>(nx, ny, nz, R, A.a[0], A.a[1], A.a[2], A.a[3], cc, fc, x,
                                          r, ions, part);
  {
    FinishBatch F;
    F.v[0] = FinishArgs{part, out, hout};
    k_finish<<<1, kBlock, 0, s>>>(F, 0, kParts);
  }
}

template <class T>
void damp_factor_batch(hipStream_t s, int nx, int ny, int nz, const DampArgs<T>* c, int nb) {
  check_batch(nb);
  Batch<DampPart<T>> B;
  FinishBatch F;
  for (int b = 0; b < nb; b++) {
    B.v[b] = DampPart<T>{to27(c[b].A), c[b].D, c[b].x, c[b].w0, c[b].part};
    F.v[b] = FinishArgs{c[b].part, c[b].out, nullptr};
  }
  // a level of fewer than kParts * kBlock interior points leaves the blocks
  // past its last point empty (partial sums +0.0): they are not launched
  const long n = (long)(nx - 2) * (ny - 2) * (nz - 2);
  const int np = (int)std::min<long>(kParts, std::max<long>(1, (n + kBlock - 1) / kBlock));
  k_damp_part<T><<<dim3(np, 1, nb), kBlock, 0, s>>>(nx, ny, nz, B);
  k_finish<<<nb, kBlock, 0, s>>>(F, 1, np);
}

template <class T>
void damp_factor(hipStream_t s, int nx, int ny, int nz, const Ops<T>& A, const T* D, const T* x,
                 const T* w0, double* part, double* out) {
  const DampArgs<T> c{A, D, x, w0, part, out};
  damp_factor_batch<T>(s, nx, ny, nz, &c, 1);
}

template <class T>
void fill(hipStream_t s, T* x, size_t n, T v) {
  k_fill<T><<<nblocks(n), kBlock, 0, s>>>(x, n, v);
}

template <class T>
void axpy_interior(hipStream_t s, int nx, int ny, int nz, double a, const T* x, T* y) {
  k_axpy_int<T><<<grid_interior(nx, ny, nz), kBlock, 0, s>>>(nx, ny, nz, a, x, y);
}

void xpay_interior(hipStream_t s, int nx, int ny, int nz, const double* x, double a,
                   const double* z, double* y) {
  k_xpay_int<<<grid_interior(nx, ny, nz), kBlock, 0, s>>>(nx, ny, nz, x, a, z, y);
}

template <class T>
void copy_interior(hipStream_t s, int nx, int ny, int nz, const T* x, T* y) {
  k_copy_int<T><<<grid_interior(nx, ny, nz), kBlock, 0, s>>>(nx, ny, nz, x, y);
}

template <class T>
void add_diag(hipStream_t s, size_t n, const T* oC, const T* cc, T* D, float* Df) {
  k_add_diag<T><<<nblocks(n), kBlock, 0, s>>>(n, oC, cc, D, Df);
}

void ZeroList::add(void* ptr, size_t bytes) {
  if (!ptr || bytes < 4) return;
  if (z.n == kZeroMax) flush();
  z.p[z.n] = (unsigned*)ptr;
  z.words[z.n] = bytes / 4;
  z.nx[z.n] = z.ny[z.n] = z.nz[z.n] = 0;
  z.wpe[z.n] = 0;
  z.blk[z.n + 1] = z.blk[z.n] + (unsigned)((bytes / 4 + kZeroChunk - 1) / kZeroChunk);
  z.n++;
}

void ZeroList::add_shell(void* ptr, int nx, int ny, int nz, size_t elem_bytes) {
  if (!ptr || nx < 1 || ny < 1 || nz < 1) return;
  if (nx < 3 || ny < 3 || nz < 3) {  // every point is on the boundary
    add(ptr, (size_t)nx * ny * nz * elem_bytes);
    return;
  }
  if (z.n == kZeroMax) flush();
  const size_t pts = 2 * (size_t)nx * ny + (size_t)(nz - 2) * (2 * (size_t)nx + 2 * (size_t)(ny - 2));
  z.p[z.n] = (unsigned*)ptr;
  z.words[z.n] = pts;
  z.nx[z.n] = nx;
  z.ny[z.n] = ny;
  z.nz[z.n] = nz;
  z.wpe[z.n] = (int)(elem_bytes / 4);
  z.blk[z.n + 1] = z.blk[z.n] + (unsigned)((pts + kBlock - 1) / kBlock);
  z.n++;
}

void ZeroList::flush() {
  if (z.n > 0 && z.blk[z.n] > 0) k_zero_many<<<z.blk[z.n], kBlock, 0, s>>>(z);
  z.n = 0;
  z.blk[0] = 0;
}

void add_diag_levels(hipStream_t s, const DiagLevels& L) {
  k_add_diag_levels<<<nblocks(L.off[L.nl]), kBlock, 0, s>>>(L);
}

void axpy_interior_f32(hipStream_t s, int nx, int ny, int nz, double a, const float* x,
                       double* y, bool assign) {
  k_axpy_int_f32<<<grid_interior(nx, ny, nz), kBlock, 0, s>>>(nx, ny, nz, a, x, y,
                                                               assign ? 1 : 0);
}

void scale(hipStream_t s, size_t n, double a, const double* x, double* y) {
  k_scale<<<nblocks(n), kBlock, 0, s>>>(n, a, x, y);
}

void convert_many(hipStream_t s, const ConvArgs& c) {
  if (c.m <= 0 || c.n == 0) return;
  if (c.m > kConvMax) {
    fprintf(stderr, "convert_many: %d arrays, at most %d\n", c.m, kConvMax);
    abort();
  }
  k_convert_many<<<dim3(nblocks(c.n), (unsigned)c.m), kBlock, 0, s>>>(c);
}

template <class Tin, class Tout>
void convert(hipStream_t s, size_t n, const Tin* in, Tout* out) {
  k_convert<Tin, Tout><<<nblocks(n), kBlock, 0, s>>>(n, in, out);
}

void set_faces(hipStream_t s, int nx, int ny, int nz, double* u, const double* gx,
               const double* gy, const double* gz) {
  k_faces<<<nblocks((size_t)ny * nz), kBlock, 0, s>>>(nx, ny, nz, u, gx, gy, gz, 0);
  k_faces<<<nblocks((size_t)nx * nz), kBlock, 0, s>>>(nx, ny, nz, u, gx, gy, gz, 1);
  k_faces<<<nblocks((size_t)nx * ny), kBlock, 0, s>>>(nx, ny, nz, u, gx, gy, gz, 2);
}

void buildA_fv(hipStream_t s, int nx, int ny, int nz, const double* xf, const double* yf,
               const double* zf, const double* gx, const double* gy, const double* gz,
               const double* a1, const double* a2, const double* a3, const double* ccf,
               const double* fcf, double* oC, double* cc, double* fc, double* oE, double* oN,
               double* uC) {
  k_buildA<<<grid_interior(nx, ny, nz), kBlock, 0, s>>>(nx, ny, nz, xf, yf, zf, gx, gy, gz, a1,
                                                        a2, a3, ccf, fcf, oC, cc, fc, oE, oN, uC);
}

// ------------------------------------------------------ explicit instances
#define INST(T)                                                                                 \
  template void gsrb7<T>(hipStream_t, int, int, int, const Ops<T>&, const T*, const T*, T*, int, \
                         int);                                                                  \
  template void gsrb27<T>(hipStream_t, int, int, int, const Ops<T>&, const T*, const T*, T*, int, \
                          int);                                                                 \
  template void gsrb27_pairs<T>(hipStream_t, int, int, int, const Ops<T>&, const T*, const T*,   \
                                T*, int, int);                                                  \
  template void resid<T>(hipStream_t, int, int, int, int, const Ops<T>&, const T*, const T*,     \
                         const T*, T*);                                                         \
  template void restrict3<T>(hipStream_t, int, int, int, int, int, int, const T*, T*, T*);      \
  template void prolong_add<T>(hipStream_t, int, int, int, int, int, int, const T*, T*,         \
                               const double*);                                                  \
  template void nrm1<T>(hipStream_t, int, int, int, const T*, double*, double*, double*);       \
  template void resid7_nrm1<T>(hipStream_t, int, int, int, const Ops<T>&, const T*, const T*,   \
                               const T*, T*, double*, double*, double*, float*);                \
  template void damp_factor<T>(hipStream_t, int, int, int, const Ops<T>&, const T*, const T*,   \
                               const T*, double*, double*);                                     \
  template void fill<T>(hipStream_t, T*, size_t, T);                                            \
  template void axpy_interior<T>(hipStream_t, int, int, int, double, const T*, T*);             \
  template void copy_interior<T>(hipStream_t, int, int, int, const T*, T*);                     \
  template void add_diag<T>(hipStream_t, size_t, const T*, const T*, T*, float*);               \
  template void gsrb27_batch<T>(hipStream_t, int, int, int, const LevelArgs<T>*, int, int, int); \
  template void gsrb27_pairs_batch<T>(hipStream_t, int, int, int, const LevelArgs<T>*, int, int, \
                                      int);                                                     \
  template void gsrb27_pairs_form<T>(hipStream_t, int, int, int, const LevelArgs<T>*, int, int,  \
                                     int, int);                                                 \
  template void resid_batch<T>(hipStream_t, int, int, int, int, const LevelArgs<T>*, int);       \
  template void restrict3_batch<T>(hipStream_t, int, int, int, int, int, int,                     \
                                   const TransferArgs<T>*, int);                                \
  template void prolong_add_batch<T>(hipStream_t, int, int, int, int, int, int,                   \
                                     const TransferArgs<T>*, int);                              \
  template void damp_factor_batch<T>(hipStream_t, int, int, int, const DampArgs<T>*, int);
INST(double)
INST(float)
#undef INST
template void convert<double, float>(hipStream_t, size_t, const double*, float*);
template void convert<float, double>(hipStream_t, size_t, const float*, double*);

}  // namespace pmg
