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


}  // namespace

int gsrb27_planes_tile(int nx, int ny, int nz) {
  const long groups = (long)((nx - 2 + 15) / 16) * ((ny - 2 + 15) / 16) * ((nz - 2) / 2);
  return groups >= 64 ? 16 : 8;
}

template <class T>
void gsrb27_planes_batch(hipStream_t s, int nx, int ny, int nz, const LevelArgs<T>* c, int nb,
                         int nu, int iadjoint, int tile) {
  check_batch(nb);
  if (nx < 3 || ny < 3 || nz < 3) return;
  if (tile != 8 && tile != 16 && tile != 32) tile = gsrb27_planes_tile(nx, ny, nz);
  if (tile == 32) tile = 16;
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
                                       int, int, int);
INST(double)
INST(float)
#undef INST

}  // namespace pmg
