// coarse_device.hip -- smoothing of the small 27-point levels, where a launch
// is bound by latency and not by bandwidth.
#include "stencil27.h"

namespace pmg {
namespace {

// The four colours of one plane parity of the 8-colour sweep in one launch:
// colours 4ck .. 4ck+3 (4ck+3 .. 4ck for the adjoint sweep).  Planes of one
// parity do not touch each other, so a workgroup owns a TX x TY tile of one
// plane.  It loads the plane's values over the tile and a 4-point margin into
// LDS and runs the four colours there in order: colour s over the tile grown
// by 3 - s points, so the margin holds every value the tile's later colours
// read.  Margin points are computed by several workgroups, identically, and
// only the tile is written.  In-plane values come from src, the neighbouring
// planes from nbr, and the result goes to dst, so no workgroup reads what
// another writes.  The arithmetic is part27's, term for term.
//
// Each colour has W wavefronts of its own, one point per lane.  All of them
// load their points' coefficients, right-hand sides and neighbour planes at
// once and form the two neighbour-plane sums before the first colour runs, so
// a launch waits for memory once and a colour step is eight LDS reads, a
// chain of additions and a division.  With all wavefronts walking the colours
// together, each colour waited for its own loads: four round trips.
// us per sweep of two launches (together, then so): 41^3 FP64 22.1, 12.7,
// FP32 13.3, 10.7; 21^3 15.7, 9.4 and 10.4, 8.2; 11^3 14.6, 8.9 and 10.3, 7.6.
template <class T, int TX, int TY, int W>
__global__ void __launch_bounds__(256 * W)
    k_gs27_plane(int nx, int ny, int nz, Batch<Args27<T>> B, int ck, int adj) {
  constexpr int M = 4, LX = TX + 2 * M, LY = TY + 2 * M, NTH = 256 * W;
  static_assert(((TX + 6 + 1) / 2) * ((TY + 6 + 1) / 2) <= 64 * W, "one lane per point");
  __shared__ T sx[LX * LY];
  const Args27<T>& ar = B.v[blockIdx.z];
  const T* const* a = ar.A.a;
  const T *src = ar.x, *nbr = ar.y;
  T* dst = ar.z;
  const int tilesx = (nx - 2 + TX - 1) / TX;
  const int tx0 = 1 + (int)(blockIdx.x % tilesx) * TX;
  const int ty0 = 1 + (int)(blockIdx.x / tilesx) * TY;
  const int k = (ck ? 1 : 2) + 2 * (int)blockIdx.y;
  const size_t nxy = (size_t)nx * ny;
  const size_t kp = (size_t)k * nxy;
  const int bx = tx0 - M, by = ty0 - M;  // grid coordinates of sx[0]
  // this wavefront's colour (i parity pi, j parity pj; parity 0 is the even
  // indices, first interior point 2) and this lane's point of it
  const int s = (int)threadIdx.x / (64 * W), t = (int)threadIdx.x % (64 * W);
  const int q = adj ? 3 - s : s, pi = q & 1, pj = q >> 1, g = 3 - s;
  int ilo = max(1, tx0 - g), jlo = max(1, ty0 - g);
  const int ihi = min(nx - 2, tx0 + TX - 1 + g), jhi = min(ny - 2, ty0 + TY - 1 + g);
  ilo += (ilo & 1) != pi;
  jlo += (jlo & 1) != pj;
  const int ni = ilo <= ihi ? (ihi - ilo) / 2 + 1 : 0;
  const int nj = jlo <= jhi ? (jhi - jlo) / 2 + 1 : 0;
  const bool act = t < ni * nj;
  const int i = act ? ilo + 2 * (t % ni) : 1, j = act ? jlo + 2 * (t / ni) : 1;
  const int e = (j - by) * LX + (i - bx);
  T co[8], f = T(0), D = T(1), u = T(0), d = T(0);
  if (act) {
    const T *oE = a[1], *oN = a[2], *uC = a[3], *oNE = a[4], *oNW = a[5], *uE = a[6], *uW = a[7],
            *uN = a[8], *uS = a[9], *uNE = a[10], *uNW = a[11], *uSE = a[12], *uSW = a[13];
    const size_t p = kp + (size_t)j * nx + i;
    co[0] = oN[p];
    co[1] = oN[p - nx];
    co[2] = oE[p];
    co[3] = oE[p - 1];
    co[4] = oNE[p];
    co[5] = oNW[p];
    co[6] = oNW[p - nx + 1];
    co[7] = oNE[p - nx - 1];
    f = ar.f[p];
    D = ar.D[p];
    const size_t qa = p + nxy, m = p - nxy;
    u = uC[p] * nbr[qa];
    u += uN[p] * nbr[qa + nx];
    u += uS[p] * nbr[qa - nx];
    u += uE[p] * nbr[qa + 1];
    u += uW[p] * nbr[qa - 1];
    u += uNE[p] * nbr[qa + nx + 1];
    u += uNW[p] * nbr[qa + nx - 1];
    u += uSE[p] * nbr[qa - nx + 1];
    u += uSW[p] * nbr[qa - nx - 1];
    d = uC[m] * nbr[m];
    d += uS[m + nx] * nbr[m + nx];
    d += uN[m - nx] * nbr[m - nx];
    d += uW[m + 1] * nbr[m + 1];
    d += uE[m - 1] * nbr[m - 1];
    d += uSW[m + nx + 1] * nbr[m + nx + 1];
    d += uSE[m + nx - 1] * nbr[m + nx - 1];
    d += uNW[m - nx + 1] * nbr[m - nx + 1];
    d += uNE[m - nx - 1] * nbr[m - nx - 1];
  }
  for (int r = threadIdx.x; r < LX * LY; r += NTH) {
    const int ii = bx + r % LX, jj = by + r / LX;
    sx[r] = (ii >= 0 && ii < nx && jj >= 0 && jj < ny) ? src[kp + (size_t)jj * nx + ii] : T(0);
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 4; c++) {
    if (s == c && act) {
      T o = co[0] * sx[e + LX];
      o += co[1] * sx[e - LX];
      o += co[2] * sx[e + 1];
      o += co[3] * sx[e - 1];
      o += co[4] * sx[e + LX + 1];
      o += co[5] * sx[e + LX - 1];
      o += co[6] * sx[e - LX + 1];
      o += co[7] * sx[e - LX - 1];
      sx[e] = (f + (o + u + d)) / D;
    }
    __syncthreads();
  }
  for (int r = threadIdx.x; r < TX * TY; r += NTH) {
    const int ii = tx0 + r % TX, jj = ty0 + r / TX;
    if (ii <= nx - 2 && jj <= ny - 2)
      dst[kp + (size_t)jj * nx + ii] = sx[(jj - by) * LX + (ii - bx)];
  }
}


// The plane-parity sweep over whole rows: a workgroup owns 2m consecutive rows
// of a plane and a lane a run of kV consecutive points of a row (both colours).
// With whole rows only the rows one above and one below the tile are computed
// twice (the square tiles above recompute 3 columns and rows a side), and a
// lane's 26 coefficient terms, f and D are one 8- or 16-byte load each, where
// the form above loads single words two apart, four of its 46 loads a point
// going through the addresser at a time.  Lanes: the m + 1 rows of the first
// row parity (colours 0 and 1 of the plane), then the m rows of the second.
// The neighbour planes' sums are formed before the first colour; a colour step
// reads the plane's values from LDS.  part27's terms in its order.
// us per sweep of two launches (the best other form, then this one): 49^3 FP64
// 14.3, 11.4, FP32 11.1, 10.7; 65^3 20.3, 15.4 and 15.3, 11.7; 81^3 35.4, 26.9
// and 22.8, 18.4; 97^3 45.7, 41.8 and 29.2, 24.4; 177^3 506, 266 and 262, 122
// (one launch per colour: its rows are too long for the pair form).
template <class T, int kV>
__global__ void __launch_bounds__(512)
    k_gs27_rows(int nx, int ny, int nz, Batch<Args27<T>> B, int ck, int adj, int R, int m) {
  extern __shared__ unsigned char rows_smem[];
  T* sx = reinterpret_cast<T*>(rows_smem);
  const Args27<T>& ar = B.v[blockIdx.z];
  const T* const* a = ar.A.a;
  const T *src = ar.x, *nbr = ar.y;
  const int j0 = 1 + (int)blockIdx.x * 2 * m;  // the tile's first row
  const int k = (ck ? 1 : 2) + 2 * (int)blockIdx.y;
  const size_t nxy = (size_t)nx * ny;
  const size_t kp = (size_t)k * nxy;
  // row parity of the first two colours; the lane's row and run
  const int first = adj ? 1 : 0;
  const int lr = (int)threadIdx.x / R, run = (int)threadIdx.x % R;
  const int g = lr <= m ? 0 : 1;  // row group
  int j = g == 0 ? j0 - 1 + 2 * lr + (((j0 - 1) & 1) != first)
                 : j0 + 2 * (lr - m - 1) + ((j0 & 1) == first);
  const bool act = lr < 2 * m + 1 && j >= 1 && j <= ny - 2;
  if (!act) j = 1;
  const int ib = min(1 + kV * run, nx - 1 - kV);
  const size_t p = kp + (size_t)j * nx + ib;
  const int e = (j - (j0 - 2)) * nx + ib;  // LDS index of the run
  T co[8][kV], f[kV], D[kV], u[kV], d[kV];
  if (act) {
    const T *oE = a[1], *oN = a[2], *uC = a[3], *oNE = a[4], *oNW = a[5], *uE = a[6], *uW = a[7],
            *uN = a[8], *uS = a[9], *uNE = a[10], *uNW = a[11], *uSE = a[12], *uSW = a[13];
    vld16(co[0], oN + p);
    vld16(co[1], oN + p - nx);
    vld16(co[2], oE + p);
    vld16(co[3], oE + p - 1);
    vld16(co[4], oNE + p);
    vld16(co[5], oNW + p);
    vld16(co[6], oNW + p - nx + 1);
    vld16(co[7], oNE + p - nx - 1);
    vld16(f, ar.f + p);
    vld16(D, ar.D + p);
    const size_t q = p + nxy, mm = p - nxy;
    T c[9][kV], w0[kV + 2], w1[kV + 2], w2[kV + 2];
    vld16(c[0], uC + p);
    vld16(c[1], uN + p);
    vld16(c[2], uS + p);
    vld16(c[3], uE + p);
    vld16(c[4], uW + p);
    vld16(c[5], uNE + p);
    vld16(c[6], uNW + p);
    vld16(c[7], uSE + p);
    vld16(c[8], uSW + p);
    vldw<T, kV>(w0, nbr + q - 1);
    vldw<T, kV>(w1, nbr + q + nx - 1);
    vldw<T, kV>(w2, nbr + q - nx - 1);
#pragma unroll
    for (int v = 0; v < kV; v++) {
      T s = c[0][v] * w0[v + 1];
      s += c[1][v] * w1[v + 1];
      s += c[2][v] * w2[v + 1];
      s += c[3][v] * w0[v + 2];
      s += c[4][v] * w0[v];
      s += c[5][v] * w1[v + 2];
      s += c[6][v] * w1[v];
      s += c[7][v] * w2[v + 2];
      s += c[8][v] * w2[v];
      u[v] = s;
    }
    vld16(c[0], uC + mm);
    vld16(c[1], uS + mm + nx);
    vld16(c[2], uN + mm - nx);
    vld16(c[3], uW + mm + 1);
    vld16(c[4], uE + mm - 1);
    vld16(c[5], uSW + mm + nx + 1);
    vld16(c[6], uSE + mm + nx - 1);
    vld16(c[7], uNW + mm - nx + 1);
    vld16(c[8], uNE + mm - nx - 1);
    vldw<T, kV>(w0, nbr + mm - 1);
    vldw<T, kV>(w1, nbr + mm + nx - 1);
    vldw<T, kV>(w2, nbr + mm - nx - 1);
#pragma unroll
    for (int v = 0; v < kV; v++) {
      T s = c[0][v] * w0[v + 1];
      s += c[1][v] * w1[v + 1];
      s += c[2][v] * w2[v + 1];
      s += c[3][v] * w0[v + 2];
      s += c[4][v] * w0[v];
      s += c[5][v] * w1[v + 2];
      s += c[6][v] * w1[v];
      s += c[7][v] * w2[v + 2];
      s += c[8][v] * w2[v];
      d[v] = s;
    }
  }
  // the plane's values: rows j0 - 2 .. j0 + 2m + 1 (rows outside the grid are
  // not read by any point)
  for (int r = threadIdx.x; r < (2 * m + 4) * nx; r += blockDim.x) {
    const int jj = j0 - 2 + r / nx;
    sx[r] = jj >= 0 && jj < ny ? src[kp + (size_t)(j0 - 2) * nx + r] : T(0);
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 4; s++) {
    if (act && g == s / 2) {
      // colours in order: column parity 0 then 1 (adjoint: 1 then 0)
      const int pi = (s & 1) ^ first;
      const int e0 = (pi - ib) & 1;
#pragma unroll
      for (int h = 0; h < kV / 2; h++) {
        auto pk = [&](const T(&v)[kV]) {
          const T lo = v[2 * h], hi = v[2 * h + 1];
          return e0 ? hi : lo;
        };
        const T* x = sx + e + e0 + 2 * h;
        T o = pk(co[0]) * x[nx];
        o += pk(co[1]) * x[-nx];
        o += pk(co[2]) * x[1];
        o += pk(co[3]) * x[-1];
        o += pk(co[4]) * x[nx + 1];
        o += pk(co[5]) * x[nx - 1];
        o += pk(co[6]) * x[-nx + 1];
        o += pk(co[7]) * x[-nx - 1];
        sx[e + e0 + 2 * h] = (pk(f) + (o + pk(u) + pk(d))) / pk(D);
      }
    }
    __syncthreads();
  }
  if (act && j >= j0 && j < j0 + 2 * m) {
    T out[kV];
#pragma unroll
    for (int v = 0; v < kV; v++) out[v] = sx[e + v];
    vst16(ar.z + p, out);
  }
}

// ------------------------------------------------------------ bottom of the cycle
// The last smoothed level and the coarsest one in one workgroup: restriction of
// the residual above, the pre-smoothing sweeps from zero, the residual and its
// restriction, the product with the dense inverse, the damping factor, the
// prolongation, the adjoint sweeps, and the damping factor of the level itself.
// Launched one by one these are 17 launches of 3 to 9 us on data that fits one
// CU.  Here a thread owns a point: its 26 coefficients, diagonal and right-hand
// side stay in registers and the level's values in LDS.  Points are dealt to
// threads colour by colour, so a colour step is a few whole wavefronts; the
// sums over the neighbour planes are formed once per plane parity by all its
// points together, so a step is eight LDS reads, one sum and a division between
// two barriers.  us per launch, points in grid order with all 26 reads a step,
// then so: 11^3 FP64 45, 29, FP32 28, 24.5; 9^3 FP64 34, 19.5.  Every
// value is formed by the separate kernels' expressions in their order (the
// reductions in the trees of k_damp_part and k_finish), so the cycle keeps its
// bits.
constexpr int kBotPts = 1728;     // points of the level with its boundary, by parity class
constexpr int kBotInner = 1024;   // interior points, one per thread
constexpr int kBotCoarse = 512;   // points of the coarsest level with its boundary
constexpr int kBotN = 64;         // unknowns of the coarsest level

template <class T>
struct BottomPart {
  Ops27<T> A, Ac;
  const T *D, *Dc;
  const T* r;
  T* x;
  const double* Minv;
  double* damp;
};

// A point of the level in LDS.  The eight parity classes of (i, j, k) are eight
// contiguous blocks of S points, so the points of a colour and every one of
// their neighbours' classes lie next to each other and a colour step reads LDS
// without bank conflicts (with points in grid order a colour's lanes are two or
// more words apart).  xm .. zp lead to the neighbours, whose classes differ.
struct BotPoint {
  int e, xm, xp, ym, yp, zm, zp;
  __device__ BotPoint(int i, int j, int k, int nx, int ny, int nz) {
    const int mx = (nx + 1) / 2, my = (ny + 1) / 2, S = mx * my * ((nz + 1) / 2);
    const int bi = i & 1, bj = j & 1, bk = k & 1;
    e = (4 * bk + 2 * bj + bi) * S + ((k >> 1) * my + (j >> 1)) * mx + (i >> 1);
    xp = bi ? 1 - S : S;
    xm = bi ? -S : S - 1;
    yp = bj ? mx - 2 * S : 2 * S;
    ym = bj ? -2 * S : 2 * S - mx;
    zp = bk ? mx * my - 4 * S : 4 * S;
    zm = bk ? -4 * S : 4 * S - mx * my;
  }
};

// part27's three sums at a point, with the 26 coefficients in its order.
template <class T>
__device__ __forceinline__ T sum_o(const T (&c)[26], const T* x, const BotPoint& p) {
  const T *r = x + p.e, *rp = r + p.yp, *rm = r + p.ym;
  T o = c[0] * rp[0];
  o += c[1] * rm[0];
  o += c[2] * r[p.xp];
  o += c[3] * r[p.xm];
  o += c[4] * rp[p.xp];
  o += c[5] * rp[p.xm];
  o += c[6] * rm[p.xp];
  o += c[7] * rm[p.xm];
  return o;
}

template <class T>
__device__ __forceinline__ T sum_u(const T (&c)[26], const T* x, const BotPoint& p) {
  const T *r = x + p.e + p.zp, *rp = r + p.yp, *rm = r + p.ym;
  T u = c[8] * r[0];
  u += c[9] * rp[0];
  u += c[10] * rm[0];
  u += c[11] * r[p.xp];
  u += c[12] * r[p.xm];
  u += c[13] * rp[p.xp];
  u += c[14] * rp[p.xm];
  u += c[15] * rm[p.xp];
  u += c[16] * rm[p.xm];
  return u;
}

template <class T>
__device__ __forceinline__ T sum_d(const T (&c)[26], const T* x, const BotPoint& p) {
  const T *r = x + p.e + p.zm, *rp = r + p.yp, *rm = r + p.ym;
  T d = c[17] * r[0];
  d += c[18] * rp[0];
  d += c[19] * rm[0];
  d += c[20] * r[p.xp];
  d += c[21] * r[p.xm];
  d += c[22] * rp[p.xp];
  d += c[23] * rp[p.xm];
  d += c[24] * rm[p.xp];
  d += c[25] * rm[p.xm];
  return d;
}

template <class T>
__device__ __forceinline__ void coef27(T (&c)[26], const Ops27<T>& A, size_t p, int nx,
                                       size_t nxy) {
  const T *oE = A.a[1], *oN = A.a[2], *uC = A.a[3], *oNE = A.a[4], *oNW = A.a[5], *uE = A.a[6],
          *uW = A.a[7], *uN = A.a[8], *uS = A.a[9], *uNE = A.a[10], *uNW = A.a[11],
          *uSE = A.a[12], *uSW = A.a[13];
  const size_t m = p - nxy;
  c[0] = oN[p];
  c[1] = oN[p - nx];
  c[2] = oE[p];
  c[3] = oE[p - 1];
  c[4] = oNE[p];
  c[5] = oNW[p];
  c[6] = oNW[p - nx + 1];
  c[7] = oNE[p - nx - 1];
  c[8] = uC[p];
  c[9] = uN[p];
  c[10] = uS[p];
  c[11] = uE[p];
  c[12] = uW[p];
  c[13] = uNE[p];
  c[14] = uNW[p];
  c[15] = uSE[p];
  c[16] = uSW[p];
  c[17] = uC[m];
  c[18] = uS[m + nx];
  c[19] = uN[m - nx];
  c[20] = uW[m + 1];
  c[21] = uE[m - 1];
  c[22] = uSW[m + nx + 1];
  c[23] = uSE[m + nx - 1];
  c[24] = uNW[m - nx + 1];
  c[25] = uNE[m - nx - 1];
}

// restrict_body's sum at index c of in (strides 1, sy, sz).
template <class T, class I>
__device__ __forceinline__ T restrict27(const T* in, I c, I sy, I sz) {
  const T W1 = T(1.0), W2 = T(0.5), W4 = T(0.25), W8 = T(0.125);
  T o = W1 * in[c];
  o += W2 * in[c + sy];
  o += W2 * in[c - sy];
  o += W2 * in[c + 1];
  o += W2 * in[c - 1];
  o += W4 * in[c + 1 + sy];
  o += W4 * in[c - 1 + sy];
  o += W4 * in[c + 1 - sy];
  o += W4 * in[c - 1 - sy];
  const I u0 = c + sz, d0 = c - sz;
  T u = W2 * in[u0];
  u += W4 * in[u0 + sy];
  u += W4 * in[u0 - sy];
  u += W4 * in[u0 + 1];
  u += W4 * in[u0 - 1];
  u += W8 * in[u0 + 1 + sy];
  u += W8 * in[u0 - 1 + sy];
  u += W8 * in[u0 + 1 - sy];
  u += W8 * in[u0 - 1 - sy];
  T d = W2 * in[d0];
  d += W4 * in[d0 + sy];
  d += W4 * in[d0 - sy];
  d += W4 * in[d0 + 1];
  d += W4 * in[d0 - 1];
  d += W8 * in[d0 + 1 + sy];
  d += W8 * in[d0 - 1 + sy];
  d += W8 * in[d0 + 1 - sy];
  d += W8 * in[d0 - 1 - sy];
  return o + u + d;
}

// The halving sum of a 64-entry block over a wavefront; valid in lane 0.
__device__ __forceinline__ double wave_tree(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// kNT: the most threads of the launch (its register budget); kQ: Minv's entries
// per thread.
template <class T, int kNT, int kQ>
__global__ void __launch_bounds__(kNT)
    k_bottom(int nxf, int nyf, int nx, int ny, int nz, int nxc, int nyc, int nzc,
             Batch<BottomPart<T>> B, int nu) {
  __shared__ T sx[kBotPts];
  __shared__ double pool[kBotN * (kBotN + 1)];  // residual, then Minv, then the level's products
  __shared__ T sxc[kBotCoarse];
  __shared__ double sfc[kBotN], spart[8], sdamp;
  const BottomPart<T>& a = B.v[blockIdx.x];
  const int tid = threadIdx.x, NT = blockDim.x;
  const int ni = nx - 2, nj = ny - 2, nk = nz - 2, n = ni * nj * nk, nxy = nx * ny;
  const int cni = nxc - 2, cnj = nyc - 2, N = cni * cnj * (nzc - 2), cxy = nxc * nyc;
  T* sr = reinterpret_cast<T*>(pool);
  // the thread's point: colour by colour, x fastest within a colour
  int col = -1, i = 1, j = 1, k = 1;
  if (tid < n) {
    int t = tid;
    for (int c = 0; c < 8; c++) {
      const int i0 = (c & 1) ? 1 : 2, j0 = (c & 2) ? 1 : 2, k0 = (c & 4) ? 1 : 2;
      const int ci = max(0, (nx - 2 - i0) / 2 + 1), cj = max(0, (ny - 2 - j0) / 2 + 1),
                ck = max(0, (nz - 2 - k0) / 2 + 1);
      const int m = nx - 2 < i0 || ny - 2 < j0 || nz - 2 < k0 ? 0 : ci * cj * ck;
      if (t < m) {
        col = c;
        i = i0 + 2 * (t % ci);
        j = j0 + 2 * ((t / ci) % cj);
        k = k0 + 2 * (t / (ci * cj));
        break;
      }
      t -= m;
    }
  }
  const bool act = col >= 0;
  const int e = k * nxy + j * nx + i;
  const BotPoint pt(i, j, k, nx, ny, nz);
  T c[26], D = T(1), f = T(0);
  if (act) {
    coef27<T>(c, a.A, (size_t)e, nx, (size_t)nxy);
    D = a.D[e];
    f = restrict27<T, size_t>(a.r, IX(2 * i, 2 * j, 2 * k, nxf, nyf), (size_t)nxf,
                              (size_t)nxf * nyf);
  } else {
#pragma unroll
    for (int q = 0; q < 26; q++) c[q] = T(0);
  }
  // Minv's entries, in flight through the first sweeps
  double mv[kQ];
#pragma unroll
  for (int q = 0; q < kQ; q++) {
    const int t = tid + q * NT;
    mv[q] = t < N * N ? a.Minv[t] : 0.0;
  }
  for (int t = tid; t < kBotPts; t += NT) sx[t] = T(0);
  for (int t = tid; t < cxy * nzc; t += NT) sxc[t] = T(0);
  __syncthreads();
  auto smooth = [&](bool adj) {
    for (int it = 0; it < nu; it++)
      for (int h = 0; h < 2; h++) {
        const int ck = adj ? 1 - h : h;
        T u = T(0), d = T(0);
        if (act && (k & 1) == ck) {
          u = sum_u<T>(c, sx, pt);
          d = sum_d<T>(c, sx, pt);
        }
        for (int cc = 0; cc < 4; cc++) {
          if (act && col == 4 * ck + (adj ? 3 - cc : cc))
            sx[pt.e] = (f + (sum_o<T>(c, sx, pt) + u + d)) / D;
          __syncthreads();
        }
      }
  };
  smooth(false);
  if (act) {
    const T o = sum_o<T>(c, sx, pt), u = sum_u<T>(c, sx, pt), d = sum_d<T>(c, sx, pt);
    sr[e] = f + o + u + d - D * sx[pt.e];
  }
  __syncthreads();
  const int ci = tid % cni + 1, cj = (tid / cni) % cnj + 1, ck = tid / (cni * cnj) + 1;
  if (tid < N)
    sfc[tid] = (double)restrict27<T, int>(sr, (2 * ck * ny + 2 * cj) * nx + 2 * ci, nx, nxy);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kQ; q++) {
    const int t = tid + q * NT;
    if (t < N * N) pool[(t / N) * (kBotN + 1) + t % N] = mv[q];
  }
  __syncthreads();
  if (tid < N) {
    const double* row = pool + tid * (kBotN + 1);
    double s = 0.0;
#pragma unroll 8
    for (int q = 0; q < N; q++) s += row[q] * sfc[q];
    sxc[(ck * nyc + cj) * nxc + ci] = (T)s;
  }
  __syncthreads();
  if (tid < 64) {  // the coarsest level's damping factor (one block of k_damp_part)
    double num = 0.0, den = 0.0;
    if (tid < N) {
      const int p = (ck * nyc + cj) * nxc + ci;
      const P27<T> s = part27<T>(a.Ac.a, sxc, (size_t)p, nxc, (size_t)cxy);
      const T xv = sxc[p];
      const T ax = (-s.o) + (-s.u) + (-s.d) + a.Dc[p] * xv;
      num += (double)xv * sfc[tid];
      den += (double)xv * (double)ax;
    }
    num = wave_tree(num);
    den = wave_tree(den);
    if (tid == 0) sdamp = num / den;
  }
  __syncthreads();
  if (act) {  // prolong_body
    const int bx = i & 1, by = j & 1, bz = k & 1;
    const T W = (bx ? T(0.5) : T(1.0)) * (by ? T(0.5) : T(1.0)) * (bz ? T(0.5) : T(1.0));
    const int c0 = ((k >> 1) * nyc + (j >> 1)) * nxc + (i >> 1);
    T v = W * sxc[c0];
    if (bx) v += W * sxc[c0 + 1];
    if (by) {
      v += W * sxc[c0 + nxc];
      if (bx) v += W * sxc[c0 + nxc + 1];
    }
    if (bz) {
      v += W * sxc[c0 + cxy];
      if (bx) v += W * sxc[c0 + cxy + 1];
      if (by) {
        v += W * sxc[c0 + cxy + nxc];
        if (bx) v += W * sxc[c0 + cxy + nxc + 1];
      }
    }
    sx[pt.e] = sx[pt.e] + T(sdamp) * v;
  }
  __syncthreads();
  smooth(true);
  // the level's damping factor: products in interior order (x fastest), one
  // block of 256 per wavefront as k_damp_part sums them, then k_finish's sum
  double* num = pool;
  double* den = pool + kBotInner;
  for (int t = tid; t < 2 * kBotInner; t += NT) pool[t] = 0.0;
  __syncthreads();
  if (act) {
    const T o = sum_o<T>(c, sx, pt), u = sum_u<T>(c, sx, pt), d = sum_d<T>(c, sx, pt);
    const T xv = sx[pt.e];
    const T ax = (-o) + (-u) + (-d) + D * xv;
    const int q = (i - 1) + ni * ((j - 1) + nj * (k - 1));
    double nv = 0.0, dv = 0.0;
    nv += (double)xv * (double)f;
    dv += (double)xv * (double)ax;
    num[q] = nv;
    den[q] = dv;
    a.x[e] = xv;
  }
  __syncthreads();
  const int w = tid >> 6, lane = tid & 63;
  if (w < 4) {
    auto block = [&](const double* v) {
      const double* b = v + 256 * w;
      const double b0 = b[lane] + b[lane + 128], b1 = b[lane + 64] + b[lane + 192];
      return wave_tree(b0 + b1);
    };
    const double sn = block(num), sd = block(den);
    if (lane == 0) {
      spart[w] = sn;
      spart[4 + w] = sd;
    }
  }
  __syncthreads();
  if (tid == 0) {
    const double sa = (spart[0] + spart[2]) + (spart[1] + spart[3]);
    const double sb = (spart[4] + spart[6]) + (spart[5] + spart[7]);
    a.damp[0] = sa / sb;
    a.damp[1] = sa;
    a.damp[2] = sb;
  }
}

}  // namespace

bool bottom_fits(int nx, int ny, int nz, int nxc, int nyc, int nzc) {
  if (nx < 3 || ny < 3 || nz < 3 || nxc < 3 || nyc < 3 || nzc < 3) return false;
  return (long)(nx - 2) * (ny - 2) * (nz - 2) <= kBotInner &&
         8L * ((nx + 1) / 2) * ((ny + 1) / 2) * ((nz + 1) / 2) <= kBotPts &&
         (long)(nxc - 2) * (nyc - 2) * (nzc - 2) <= kBotN && (long)nxc * nyc * nzc <= kBotCoarse;
}

template <class T>
void bottom_batch(hipStream_t s, const int above[3], const int level[3], const int coarsest[3],
                  const BottomArgs<T>* c, int nb, int nu) {
  check_batch(nb);
  Batch<BottomPart<T>> B;
  for (int b = 0; b < nb; b++)
    B.v[b] = BottomPart<T>{to27(c[b].A), to27(c[b].Ac), c[b].D,    c[b].Dc,
                           c[b].r,       c[b].x,        c[b].Minv, c[b].damp};
  const int n = (level[0] - 2) * (level[1] - 2) * (level[2] - 2);
  // whole wavefronts, 256 threads or more: four of them sum the level's products
  const int nt = n <= 256 ? 256 : (n + 63) / 64 * 64;
  auto launch = [&](auto kernel) {
    kernel<<<nb, nt, 0, s>>>(above[0], above[1], level[0], level[1], level[2], coarsest[0],
                             coarsest[1], coarsest[2], B, nu);
  };
  static_assert(kBotN * kBotN <= 16 * 256 && kBotN * kBotN <= 8 * 576, "Minv fits the threads");
  if (nt <= 512)
    launch(k_bottom<T, 512, 16>);
  else if (nt <= 768)
    launch(k_bottom<T, 768, 8>);
  else
    launch(k_bottom<T, 1024, 8>);
}

// Whether a rows code (100 kV + m) fits a level: a run and its boundary points
// in a row, the tile's runs in one workgroup.
static bool rows_fit(int nx, int word, int code) {
  const int kV = code / 100, m = code % 100;
  if ((kV != 2 && !(kV == 4 && word == 4)) || m < 1 || nx < kV + 2) return false;
  const int R = (nx - 2 + kV - 1) / kV;
  return (2 * m + 1) * R <= 512 && (long)(2 * m + 4) * nx * word <= 64 * 1024;
}

// Points of a run in the rows form of rows of nx points, or 0 for another form.
// Below rows of 40 points the square tiles are faster (33^3: FP64 9.5 us a sweep
// against 10.9, FP32 9.0 against 9.7), from 115 to 130 in FP64 the colour pairs
// are the faster or close (117^3 77.3 against 74.5, 121^3 79.8 and 79.7, 125^3
// 85.2 and 88.8, 129^3 92.8 and 95.3).  FP32 takes 8-byte runs up to rows of 104 points (89^3
// 20.8 us against 21.3 with 16 bytes, 97^3 24.4 and 24.4), 16-byte runs above
// (113^3 34.8 against 37.5, 129^3 47.9 and 50.5).
static int rows_run(int nx, int word) {
  if (nx < 40 || (word == 8 && nx > 114 && nx <= 130)) return 0;
  const int kV = word == 4 && nx > 104 ? 4 : 2;
  return rows_fit(nx, word, 100 * kV + 1) ? kV : 0;
}

// The rows form of nb levels swept together, or 0.  The row pairs m of a
// workgroup, 1 to 6: a launch takes as long as the CU with the most work, which
// runs ceil(workgroups / 256) workgroups of so many wavefronts each (and their
// barriers, about half a wavefront's time), so m is the one that makes this
// least, the largest on a tie, where fewer rows are computed twice.  us a sweep
// (m: time): 49^3 FP64 2: 14.7, 3: 11.2, 4: 13.2; 65^3 3: 18.2, 4: 15.6, 5: 17.2;
// 73^3 4: 23.5, 5: 24.0, 6: 20.4; 97^3 2: 45.3, 3: 42.0, 4: 45.5; eight levels
// of 45^3 3: 37.8, 6: 32.9; FP32 81^3 4: 18.4, 5: 17.1.  Over 148 shapes (40 to
// 177 points a row, ragged ones and batches of eight among them) the rule's m
// is 1.2 % slower than the fastest on average; at worst 9 % (eight levels of
// 105^3 in FP32) and 8 % (77^3, m = 2 for 3).
static int rows_code(int nx, int ny, int nz, int word, int nb) {
  const int kV = rows_run(nx, word);
  if (kV == 0) return 0;
  const int R = (nx - 2 + kV - 1) / kV;
  int best = 0;
  long least = 0;
  for (int m = 1; m <= 6; m++) {
    if (!rows_fit(nx, word, 100 * kV + m)) continue;
    const long groups = (long)((ny - 2 + 2 * m - 1) / (2 * m)) * ((nz - 1) / 2) * nb;
    const long cost = (groups + 255) / 256 * (2 * (((2 * m + 1) * R + 63) / 64) + 1);
    if (best == 0 || cost <= least) {
      best = 100 * kV + m;
      least = cost;
    }
  }
  return best;
}

// The square tiles are for levels of at most 49^2 points a plane: larger planes
// with short rows take the colour pairs.
bool gsrb27_use_planes(int nx, int ny, int nz, int word) {
  return nz >= 3 && (rows_run(nx, word) != 0 || (nx <= 49 && ny <= 49));
}

bool gsrb27_planes_fits(int nx, int word, int tile) {
  return tile == 8 || tile == 16 || rows_fit(nx, word, tile);
}

int gsrb27_planes_tile(int nx, int ny, int nz, int word, int nb) {
  if (const int code = rows_code(nx, ny, nz, word, nb)) return code;
  const long groups = (long)((nx - 2 + 15) / 16) * ((ny - 2 + 15) / 16) * ((nz - 2) / 2);
  return groups >= 64 ? 16 : 8;
}

template <class T>
void gsrb27_planes_batch(hipStream_t s, int nx, int ny, int nz, const LevelArgs<T>* c, int nb,
                         int nu, int iadjoint, int tile) {
  check_batch(nb);
  if (nx < 3 || ny < 3 || nz < 3) return;
  constexpr int word = (int)sizeof(T);
  if (!gsrb27_planes_fits(nx, word, tile)) tile = gsrb27_planes_tile(nx, ny, nz, word, nb);
  const bool rows = tile >= 100;
  for (int it = 0; it < nu; it++) {
    // sweep it reads x (even it) or xs and writes the other one
    const int first = iadjoint ? 1 : 0;
    for (int h = 0; h < 2; h++) {
      const int ck = h == 0 ? first : 1 - first;
      const int k0 = ck ? 1 : 2;
      if (k0 > nz - 2) continue;
      const int nk = (nz - 2 - k0) / 2 + 1;
      Batch<Args27<T>> B;
      for (int b = 0; b < nb; b++) {
        T* in = (it & 1) ? c[b].xs : c[b].x;
        T* out = (it & 1) ? c[b].x : c[b].xs;
        B.v[b] = Args27<T>{to27(c[b].A), c[b].D, c[b].f, in, h == 0 ? in : out, out};
      }
      if (rows) {
        const int kV = tile / 100, m = tile % 100, R = (nx - 2 + kV - 1) / kV;
        const int nt = ((2 * m + 1) * R + 63) / 64 * 64;
        const dim3 gr((unsigned)((ny - 2 + 2 * m - 1) / (2 * m)), (unsigned)nk, (unsigned)nb);
        const size_t lds = (size_t)(2 * m + 4) * nx * sizeof(T);
        if (kV == 4) {
          if constexpr (sizeof(T) == 4)
            k_gs27_rows<T, 4><<<gr, nt, lds, s>>>(nx, ny, nz, B, ck, iadjoint, R, m);
        } else {
          k_gs27_rows<T, 2><<<gr, nt, lds, s>>>(nx, ny, nz, B, ck, iadjoint, R, m);
        }
        continue;
      }
      const unsigned tiles = (unsigned)(((nx - 2 + tile - 1) / tile) * ((ny - 2 + tile - 1) / tile));
      const dim3 g(tiles, (unsigned)nk, (unsigned)nb);
      if (tile == 16)
        k_gs27_plane<T, 16, 16, 2><<<g, 512, 0, s>>>(nx, ny, nz, B, ck, iadjoint);
      else
        k_gs27_plane<T, 8, 8, 1><<<g, 256, 0, s>>>(nx, ny, nz, B, ck, iadjoint);
    }
  }
  if (nu & 1)
    for (int b = 0; b < nb; b++) copy_interior<T>(s, nx, ny, nz, c[b].xs, c[b].x);
}

template <class T>
void gsrb27_planes(hipStream_t s, int nx, int ny, int nz, const Ops<T>& A, const T* D,
                   const T* fc, T* x, T* xs, int nu, int iadjoint, int tile) {
  const LevelArgs<T> c{A, D, fc, x, xs, nullptr};
  gsrb27_planes_batch<T>(s, nx, ny, nz, &c, 1, nu, iadjoint, tile);
}

#define INST(T)                                                                                \
  template void gsrb27_planes<T>(hipStream_t, int, int, int, const Ops<T>&, const T*, const T*, \
                                 T*, T*, int, int, int);                                       \
  template void gsrb27_planes_batch<T>(hipStream_t, int, int, int, const LevelArgs<T>*, int,    \
                                       int, int, int);                                         \
  template void bottom_batch<T>(hipStream_t, const int[3], const int[3], const int[3],          \
                                const BottomArgs<T>*, int, int);
INST(double)
INST(float)
#undef INST

}  // namespace pmg
