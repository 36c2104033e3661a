// galerkin_device.hip -- Galerkin coarse operators A_c = P^T A P for CDNA4
// (gfx950): the 14 stored coefficients of the 27-point coarse stencil from a
// 7- or 27-point fine one (VbuildG_7 / VbuildG_27, src/pmgc/buildGd.c:450-3115).
#include "pmg_device.h"

#include "stencil27.h"

namespace pmg {
namespace {

// forward offsets of the 14 stored coefficients
__constant__ int c_fwd[14][3] = {{0, 0, 0},  {1, 0, 0},  {0, 1, 0},  {0, 0, 1}, {1, 1, 0},
                                 {-1, 1, 0}, {1, 0, 1},  {-1, 0, 1}, {0, 1, 1}, {0, -1, 1},
                                 {1, 1, 1},  {-1, 1, 1}, {1, -1, 1}, {-1, -1, 1}};

// stored direction of each offset (sx,sy,sz) at (sz+1)*9+(sy+1)*3+(sx+1): +s forward, -s backward
__constant__ int c_ent[27] = {-10, -8, -11, -6, -3, -7, -12, -9, -13, -4, -2, -5, -1, 0, 1, 5, 2, 4, 13, 9, 12, 7, 3, 6, 11, 8, 10};

__device__ inline double pweight(int dx, int dy, int dz) {
  if (dx < -1 || dx > 1 || dy < -1 || dy > 1 || dz < -1 || dz > 1) return 0.0;
  const int m = abs(dx) + abs(dy) + abs(dz);
  return m == 0 ? 1.0 : (m == 1 ? 0.5 : (m == 2 ? 0.25 : 0.125));
}

// A(f, f+s) of the fine operator without cc (same search order as the
// oracle's restatement: first matching stored coefficient, forward then back).
__device__ inline double fine_entry(int st, const Ops27<double>& A, int nxf, int nyf, int fi,
                                    int fj, int fk, int sx, int sy, int sz) {
  if (sx == 0 && sy == 0 && sz == 0) return A.a[0][IX(fi, fj, fk, nxf, nyf)];
  // each offset is exactly one stored direction, forward (+) or backward (-)
  const int e = c_ent[(sz + 1) * 9 + (sy + 1) * 3 + (sx + 1)];
  const int s = e > 0 ? e : -e;
  if (s >= (st == 7 ? 4 : 14)) return 0.0;
  if (e > 0) return -A.a[s][IX(fi, fj, fk, nxf, nyf)];
  return -A.a[s][IX(fi + sx, fj + sy, fk + sz, nxf, nyf)];
}

struct OutPtrs {
  double* a[14];
};

// Inner sum of the Galerkin product for coarse point (I, J, K), stored
// direction to (I2, J2, K2) and fine neighbour d = 9(dz+1) + 3(dy+1) + (dx+1)
// of the fine point 2(I, J, K) (the reference's loop order).  The loops visit
// only the terms with a non-zero second weight pweight(f + s - g0), i.e.
// |f + s - g0| <= 1 per axis, in the full scan's order, so the sum is the
// full scan's.
__device__ __forceinline__ double galerkin_tt(int st, const Ops27<double>& Af, int nxf, int nyf,
                                              int I, int J, int K, int I2, int J2, int K2,
                                              int d) {
  const int dz = d / 9 - 1, dy = (d / 3) % 3 - 1, dx = d % 3 - 1;
  const int fx = 2 * I + dx, fy = 2 * J + dy, fz = 2 * K + dz;
  const int g0x = 2 * I2, g0y = 2 * J2, g0z = 2 * K2;
  const int sx0 = max(-1, g0x - 1 - fx), sx1 = min(1, g0x + 1 - fx);
  const int sy0 = max(-1, g0y - 1 - fy), sy1 = min(1, g0y + 1 - fy);
  const int sz0 = max(-1, g0z - 1 - fz), sz1 = min(1, g0z + 1 - fz);
  double tt = 0.0;
  for (int sz = sz0; sz <= sz1; sz++)
    for (int sy = sy0; sy <= sy1; sy++)
      for (int sx = sx0; sx <= sx1; sx++) {
        if (st == 7 && abs(sx) + abs(sy) + abs(sz) > 1) continue;
        const double p2 = pweight(fx + sx - g0x, fy + sy - g0y, fz + sz - g0z);
        tt += fine_entry(st, Af, nxf, nyf, fx, fy, fz, sx, sy, sz) * p2;
      }
  return tt;
}

// The general sum by one thread per (coarse interior point, stored coefficient),
// 64 consecutive coarse points per wavefront and one direction s per
// wavefront, so the pruned loop bounds (which depend on s only) never
// diverge within a wavefront.
__global__ void __launch_bounds__(kBlock)
    k_galerkin_point(int st, int nxf, int nyf, int nzf, Ops27<double> Af, int nxc, int nyc,
                     int nzc, OutPtrs out) {
  const long ni = nxc - 2, nj = nyc - 2, nk = nzc - 2;
  const long nq = ni * nj * nk;
  const long t = (long)blockIdx.x * kBlock + threadIdx.x;
  const long w = t / 64;
  const int s = (int)(w % 14);
  const long q = (w / 14) * 64 + (t % 64);
  if (q >= nq) return;
  const int I = 1 + (int)(q % ni), J = 1 + (int)((q / ni) % nj), K = 1 + (int)(q / (ni * nj));
  const int I2 = I + c_fwd[s][0], J2 = J + c_fwd[s][1], K2 = K + c_fwd[s][2];
  const size_t pc = IX(I, J, K, nxc, nyc);
  if (I2 < 1 || I2 > nxc - 2 || J2 < 1 || J2 > nyc - 2 || K2 < 1 || K2 > nzc - 2) {
    out.a[s][pc] = 0.0;
    return;
  }
  double sum = 0.0;
  for (int d = 0; d < 27; d++)
    sum += pweight(d % 3 - 1, (d / 3) % 3 - 1, d / 9 - 1) *
           galerkin_tt(st, Af, nxf, nyf, I, J, K, I2, J2, K2, d);
  out.a[s][pc] = (s == 0) ? sum : -sum;
}

// The same sum with every loop unrolled at compile time for one stencil
// width ST and one stored direction S: the pruned loop bounds, both
// prolongation weights and the stored array of each fine offset become
// constants, so a term is one load and one multiply-add.  Terms whose fine
// entry is a structural zero (the diagonal offsets of a 7-point operator) add
// +0.0 to a partial sum that starts at +0.0 and so cannot be -0.0; they are
// left out without changing a bit.
namespace gal {
constexpr int kFwd[14][3] = {{0, 0, 0},  {1, 0, 0},  {0, 1, 0},  {0, 0, 1}, {1, 1, 0},
                             {-1, 1, 0}, {1, 0, 1},  {-1, 0, 1}, {0, 1, 1}, {0, -1, 1},
                             {1, 1, 1},  {-1, 1, 1}, {1, -1, 1}, {-1, -1, 1}};
__host__ __device__ constexpr int iabs(int v) { return v < 0 ? -v : v; }
__host__ __device__ constexpr int imax(int a, int b) { return a > b ? a : b; }
__host__ __device__ constexpr int imin(int a, int b) { return a < b ? a : b; }
// stored direction of offset (sx, sy, sz): +s forward, -s backward
__host__ __device__ constexpr int ent(int sx, int sy, int sz) {
  for (int s = 0; s < 14; s++) {
    if (kFwd[s][0] == sx && kFwd[s][1] == sy && kFwd[s][2] == sz) return s;
    if (kFwd[s][0] == -sx && kFwd[s][1] == -sy && kFwd[s][2] == -sz) return -s;
  }
  return 99;
}
__host__ __device__ constexpr double pw(int dx, int dy, int dz) {
  return (dx < -1 || dx > 1 || dy < -1 || dy > 1 || dz < -1 || dz > 1)
             ? 0.0
             : (iabs(dx) + iabs(dy) + iabs(dz) == 0
                    ? 1.0
                    : (iabs(dx) + iabs(dy) + iabs(dz) == 1
                           ? 0.5
                           : (iabs(dx) + iabs(dy) + iabs(dz) == 2 ? 0.25 : 0.125)));
}

// tt_d for stored direction S (0 where every second weight is zero)
template <int ST, int S>
__device__ __forceinline__ double inner(const Ops27<double>& A, size_t pf, int nx, size_t nxy,
                                        int d) {
  constexpr int FX = kFwd[S][0], FY = kFwd[S][1], FZ = kFwd[S][2];
  const int dz = d / 9 - 1, dy = (d / 3) % 3 - 1, dx = d % 3 - 1;
  const int ox = 2 * FX - dx, oy = 2 * FY - dy, oz = 2 * FZ - dz;
  const long f = (long)dx + (long)dy * nx + (long)dz * (long)nxy;
  double tt = 0.0;
#pragma unroll
  for (int sz = -1; sz <= 1; sz++)
#pragma unroll
    for (int sy = -1; sy <= 1; sy++)
#pragma unroll
      for (int sx = -1; sx <= 1; sx++) {
        if (sx < imax(-1, ox - 1) || sx > imin(1, ox + 1) || sy < imax(-1, oy - 1) ||
            sy > imin(1, oy + 1) || sz < imax(-1, oz - 1) || sz > imin(1, oz + 1))
          continue;
        if (ST == 7 && iabs(sx) + iabs(sy) + iabs(sz) > 1) continue;
        const double p2 = pw(sx - ox, sy - oy, sz - oz);
        const int e = ent(sx, sy, sz);
        double v;
        if (e == 0)
          v = A.a[0][pf + f];
        else if (e > 0)
          v = -A.a[e][pf + f];
        else
          v = -A.a[-e][pf + f + (long)sx + (long)sy * nx + (long)sz * (long)nxy];
        tt += v * p2;
      }
  return tt;
}

// The sums of several directions at a coarse point, which share their loads.
// (Their terms stay inside the fine grid also where the direction leaves the
// coarse interior and the coefficient is zero.)
template <int ST, int... S>
__device__ __forceinline__ void coefs(const Ops27<double>& A, size_t pf, int nx, size_t nxy,
                                      int I, int J, int K, int nxc, int nyc, int nzc,
                                      double* const* out) {
  constexpr int n = sizeof...(S), dir[n] = {S...};
  double sum[n] = {};
#pragma unroll
  for (int d = 0; d < 27; d++) {
    const double w = pw(d % 3 - 1, (d / 3) % 3 - 1, d / 9 - 1);
    int m = 0;
    ((sum[m++] += w * inner<ST, S>(A, pf, nx, nxy, d)), ...);
  }
  const size_t pc = IX(I, J, K, nxc, nyc);
#pragma unroll
  for (int m = 0; m < n; m++) {
    const int s = dir[m];
    const int I2 = I + kFwd[s][0], J2 = J + kFwd[s][1], K2 = K + kFwd[s][2];
    const bool in = I2 >= 1 && I2 <= nxc - 2 && J2 >= 1 && J2 <= nyc - 2 && K2 <= nzc - 2;
    out[s][pc] = in ? (s == 0 ? sum[m] : -sum[m]) : 0.0;
  }
}

}  // namespace gal

// A wavefront forms the sums of 64 consecutive coarse points, all fourteen of
// them (kGroups = 1) or one group of four.  What bounded one sum per
// wavefront was operand traffic: the fourteen sums of a point use 570 distinct
// values of a 27-point operator (150 of a 7-point one) but read 1270 (430),
// and neighbouring workgroups, dealt to different XCDs, each read them from
// memory again.  So the sums share their loads, and each XCD takes one
// contiguous range of points.  A 27-point operator takes four groups:
// directions that read the same coefficients, few enough values to stay in
// 256 registers (242, and 180 for the 7-point one; none spilled), and a
// quarter of the 45 KB of straight-line code for a wavefront of a small level
// to fetch.  Microseconds a call, before -> now: 7-point fine levels of 65^3
// 11.1 -> 6.0, 161^3 118 -> 37, 353^3 1481 -> 525; 27-point 21^3 17.1 -> 8.4,
// 41^3 20.8 -> 9.1, 81^3 126 -> 29, 177^3 1327 -> 354.  The 7-point operator
// in four groups: 161^3 55, 353^3 900; the 27-point one in one group: 21^3
// 28, 81^3 53, 177^3 595; in two, 81^3 58.
template <int ST, int kGroups>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))
    k_galerkin(int nxf, int nyf, Ops27<double> Af, int nxc, int nyc, int nzc, OutPtrs out) {
  static_assert(kGroups == 1 || kGroups == 4, "the groups below");
  const long ni = nxc - 2, nj = nyc - 2, nk = nzc - 2;
  const long nq = ni * nj * nk;
  const int per = gridDim.x / 8;
  const long t = ((long)(blockIdx.x % 8) * per + blockIdx.x / 8) * kBlock + threadIdx.x;
  const int part = __builtin_amdgcn_readfirstlane((int)(t / 64 % kGroups));
  const long q = t / 64 / kGroups * 64 + t % 64;
  if (q >= nq) return;
  const int I = 1 + (int)(q % ni), J = 1 + (int)((q / ni) % nj), K = 1 + (int)(q / (ni * nj));
  const size_t nxy = (size_t)nxf * nyf;
  const size_t pf = IX(2 * I, 2 * J, 2 * K, nxf, nyf);
  if (kGroups == 1)
    gal::coefs<ST, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13>(Af, pf, nxf, nxy, I, J, K, nxc,
                                                                 nyc, nzc, out.a);
  else if (part == 0)
    gal::coefs<ST, 0, 1>(Af, pf, nxf, nxy, I, J, K, nxc, nyc, nzc, out.a);
  else if (part == 1)
    gal::coefs<ST, 2, 4, 5>(Af, pf, nxf, nxy, I, J, K, nxc, nyc, nzc, out.a);
  else if (part == 2)
    gal::coefs<ST, 3, 6, 7>(Af, pf, nxf, nxy, I, J, K, nxc, nyc, nzc, out.a);
  else
    gal::coefs<ST, 8, 9, 10, 11, 12, 13>(Af, pf, nxf, nxy, I, J, K, nxc, nyc, nzc, out.a);
}

// The general sum by one 32-lane group per (coarse interior point, stored coefficient); lane d < 27
// computes tt_d, lane 0 then adds p1_d * tt_d for d = 0..26 in order, the
// same sum as k_galerkin_point's.
constexpr int kGalGroups = kBlock / 32;

__global__ void __launch_bounds__(kBlock)
    k_galerkin_group(int st, int nxf, int nyf, int nzf, Ops27<double> Af, int nxc, int nyc,
                     int nzc, OutPtrs out) {
  __shared__ double tt_sh[kGalGroups][27];
  const long ni = nxc - 2, nj = nyc - 2, nk = nzc - 2;
  const long nq = ni * nj * nk;
  const int grp = threadIdx.x / 32, d = threadIdx.x % 32;
  const long g = (long)blockIdx.x * kGalGroups + grp;
  const int s = (int)(g % 14);
  const long q = g / 14;
  const bool live = q < nq;
  int I = 0, J = 0, K = 0, I2 = 0, J2 = 0, K2 = 0;
  if (live) {
    I = 1 + (int)(q % ni);
    J = 1 + (int)((q / ni) % nj);
    K = 1 + (int)(q / (ni * nj));
    I2 = I + c_fwd[s][0];
    J2 = J + c_fwd[s][1];
    K2 = K + c_fwd[s][2];
  }
  const bool inside = live && !(I2 < 1 || I2 > nxc - 2 || J2 < 1 || J2 > nyc - 2 || K2 < 1 ||
                                K2 > nzc - 2);
  if (inside && d < 27) tt_sh[grp][d] = galerkin_tt(st, Af, nxf, nyf, I, J, K, I2, J2, K2, d);
  __syncthreads();
  if (!live || d != 0) return;
  const size_t pc = IX(I, J, K, nxc, nyc);
  if (!inside) {
    out.a[s][pc] = 0.0;
    return;
  }
  double sum = 0.0;
  for (int e = 0; e < 27; e++) sum += pweight(e % 3 - 1, (e / 3) % 3 - 1, e / 9 - 1) * tt_sh[grp][e];
  out.a[s][pc] = (s == 0) ? sum : -sum;
}

}  // namespace

void galerkin(hipStream_t s, int st, int nxf, int nyf, int nzf, const Ops<double>& Af, int nxc,
              int nyc, int nzc, double* const ac[14], int form) {
  OutPtrs o;
  for (int k = 0; k < 14; k++) o.a[k] = ac[k];
  const long nq = (long)(nxc - 2) * (nyc - 2) * (nzc - 2);
  if (form != 1 && form != 2) {
    const int groups = st == 7 ? 1 : 4;
    const long nb = ((nq + 63) / 64 * groups * 64 + kBlock - 1) / kBlock;
    const unsigned g = (unsigned)((nb + 7) / 8 * 8);  // whole rounds of the 8 XCDs
    if (st == 7)
      k_galerkin<7, 1><<<g, kBlock, 0, s>>>(nxf, nyf, to27(Af), nxc, nyc, nzc, o);
    else
      k_galerkin<27, 4><<<g, kBlock, 0, s>>>(nxf, nyf, to27(Af), nxc, nyc, nzc, o);
  } else if (form == 2) {
    const long groups = nq * 14;
    k_galerkin_group<<<(unsigned)((groups + kGalGroups - 1) / kGalGroups), kBlock, 0, s>>>(
        st, nxf, nyf, nzf, to27(Af), nxc, nyc, nzc, o);
  } else {
    const long tot = ((nq + 63) / 64) * 64 * 14;
    k_galerkin_point<<<(unsigned)((tot + kBlock - 1) / kBlock), kBlock, 0, s>>>(
        st, nxf, nyf, nzf, to27(Af), nxc, nyc, nzc, o);
  }
}

}  // namespace pmg
