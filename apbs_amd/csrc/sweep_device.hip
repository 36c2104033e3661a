// sweep_device.hip -- the fused red-black sweep of the fine 7-point level.
//
// The kernels evaluate the reference's expressions in the reference's order
// (src/pmgc/gsd.c:95-165) without FMA contraction.
#include "stencil27.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace pmg {

namespace {

// One complete red-black sweep, out of place: xo = sweep(xi).  In the 7-point
// stencil every neighbour of a point has the other colour, so the first colour
// F reads only old values of the second colour S, and S reads only new F
// values.  A workgroup owns a TX x TY tile of (i, j) and marches over a chunk
// of k planes: the new F values of plane k+1 (tile plus a one-point halo) go
// to a three-plane LDS ring, then the S points of plane k are updated from the
// ring and the whole tile row of plane k is written.  Each value is the
// in-place sweep's value bit for bit (same terms, same order, no FMA).
// Points outside the interior are not written.
constexpr int kFT = 256, kXCD = 8;

// kTX columns (even), kTY rows and kKC planes per workgroup of kNT threads.
// The arrays of one calculation in a fused-sweep launch.
template <class T>
struct SweepArgs {
  const T *oE, *oN, *uC, *D, *fc, *xi;
  T* xo;
};

// kZeroX: xi is zero everywhere (a solve of the correction equation from a
// zero start); its values are not read, and the sweep's values are those of
// reading the zeros.
template <class T, int kTY, int kKC, int kTX, int kNT, bool kZeroX>
__device__ __forceinline__ void fused_body(int nx, int ny, int nz, int tile,
                                           const T* __restrict__ oE, const T* __restrict__ oN,
                                           const T* __restrict__ uC, const T* __restrict__ D,
                                           const T* __restrict__ fc, const T* __restrict__ xi,
                                           T* __restrict__ xo, int first) {
  constexpr int RX = kTX + 2, RY = kTY + 2, RN = RX * RY;
  constexpr int FPR = RX / 2, FN = FPR * RY;  // F points per region row / per plane
  __shared__ T ring[3][RN];
  const int tid = threadIdx.x;
  const int nbx = (nx - 2 + kTX - 1) / kTX, nby = (ny - 2 + kTY - 1) / kTY;
  const int i0 = 1 + (tile % nbx) * kTX, j0 = 1 + ((tile / nbx) % nby) * kTY;
  const int k0 = 1 + (tile / (nbx * nby)) * kKC;
  const int k1 = min(k0 + kKC, nz - 1);  // planes k0 .. k1-1
  const size_t nxy = (size_t)nx * ny;
  const int F = first;                   // parity of the first colour

  // New F values of plane kk over the tile and its halo, one thread per F
  // point in kFR rounds.  loadF issues every round's loads at once into
  // registers; storeF computes the values (acc7's terms and order) into the
  // plane's LDS slot.
  constexpr int kFR = (FN + kNT - 1) / kNT;
  struct FRegs {
    T v[kFR][14];
    int slot[kFR];  // LDS index in the ring plane
    int kind[kFR];  // 0 nothing, 1 boundary copy, 2 interior update
  };
  auto loadF = [&](int kk, FRegs& R) {
#pragma unroll
    for (int u = 0; u < kFR; u++) {
      R.kind[u] = 0;
      const int f = tid + u * kNT;
      if (f >= FN) continue;
      const int row = f / FPR, c = f % FPR;
      const int j = j0 - 1 + row;
      const int ib = i0 - 1;
      const int i = ib + ((F - ib - j - kk) & 1) + 2 * c;
      if (i > nx - 1 || j > ny - 1) continue;
      const size_t p = ((size_t)kk * ny + j) * nx + i;
      R.slot[u] = row * RX + (i - ib);
      if (i >= 1 && i <= nx - 2 && j >= 1 && j <= ny - 2 && kk >= 1 && kk <= nz - 2) {
        R.kind[u] = 2;
        R.v[u][0] = fc[p];
        R.v[u][1] = oN[p];
        R.v[u][2] = kZeroX ? T(0) : xi[p + nx];
        R.v[u][3] = oN[p - nx];
        R.v[u][4] = kZeroX ? T(0) : xi[p - nx];
        R.v[u][5] = oE[p];
        R.v[u][6] = kZeroX ? T(0) : xi[p + 1];
        R.v[u][7] = oE[p - 1];
        R.v[u][8] = kZeroX ? T(0) : xi[p - 1];
        R.v[u][9] = uC[p - nxy];
        R.v[u][10] = kZeroX ? T(0) : xi[p - nxy];
        R.v[u][11] = uC[p];
        R.v[u][12] = kZeroX ? T(0) : xi[p + nxy];
        R.v[u][13] = D[p];
      } else {
        R.kind[u] = 1;
        R.v[u][0] = kZeroX ? T(0) : xi[p];
      }
    }
  };
  auto storeF = [&](int kk, const FRegs& R) {
    T* r = ring[kk % 3];
#pragma unroll
    for (int u = 0; u < kFR; u++) {
      if (R.kind[u] == 2) {
        T acc = R.v[u][0];
        acc += R.v[u][1] * R.v[u][2];
        acc += R.v[u][3] * R.v[u][4];
        acc += R.v[u][5] * R.v[u][6];
        acc += R.v[u][7] * R.v[u][8];
        acc += R.v[u][9] * R.v[u][10];
        acc += R.v[u][11] * R.v[u][12];
        r[R.slot[u]] = acc / R.v[u][13];
      } else if (R.kind[u] == 1) {
        r[R.slot[u]] = R.v[u][0];
      }
    }
  };

  // The S step: thread u owns the (i, i+1) pair u % 32 of tile row u / 32 (one
  // F and one S point).  The eight operands of the S point of plane kk are
  // loaded one plane ahead, together with stageF(kk), so each coefficient
  // line is fetched once for both colours while it is still cached.
  constexpr int kSP = (kTX / 2 * kTY + kNT - 1) / kNT;
  T cur[kSP][8], nxt[kSP][8];
  auto loadS = [&](int kk, T (&r)[kSP][8]) {
#pragma unroll
    for (int u = 0; u < kSP; u++) {
      const int sidx = tid + u * kNT;
      if (sidx >= kTX / 2 * kTY) continue;
      const int j = j0 + sidx / (kTX / 2);
      const int is = i0 + 2 * (sidx % (kTX / 2)) + ((1 - F - i0 - j - kk) & 1);
      if (is > nx - 2 || j > ny - 2) continue;
      const size_t p = ((size_t)kk * ny + j) * nx + is;
      r[u][0] = fc[p];
      r[u][1] = oN[p];
      r[u][2] = oN[p - nx];
      r[u][3] = oE[p];
      r[u][4] = oE[p - 1];
      r[u][5] = uC[p - nxy];
      r[u][6] = uC[p];
      r[u][7] = D[p];
    }
  };

  FRegs fr;
  loadS(k0, cur);
  loadF(k0 - 1, fr);
  storeF(k0 - 1, fr);
  loadF(k0, fr);
  storeF(k0, fr);
  loadF(k0 + 1, fr);
  for (int k = k0; k < k1; k++) {
    // F(k+1) from registers loaded one step earlier; the loads of F(k+2) and
    // of S(k+1)'s operands are in flight while S(k) is computed
    if (k + 1 < k1) loadS(k + 1, nxt);
    storeF(k + 1, fr);
    __syncthreads();
    if (k + 1 < k1) loadF(k + 2, fr);
    const T* rm = ring[(k - 1) % 3];
    const T* r0 = ring[k % 3];
    const T* rp = ring[(k + 1) % 3];
#pragma unroll
    for (int u = 0; u < kSP; u++) {
      const int sidx = tid + u * kNT;
      if (sidx >= kTX / 2 * kTY) continue;
      const int jj = sidx / (kTX / 2);
      const int j = j0 + jj;
      if (j > ny - 2) continue;
      const int ia = i0 + 2 * (sidx % (kTX / 2));
      const int is = ia + ((1 - F - i0 - j - k) & 1);
      const int iF = ia + ((F - i0 - j - k) & 1);
      const size_t row = ((size_t)k * ny + j) * nx;
      if (iF <= nx - 2) xo[row + iF] = r0[(jj + 1) * RX + (iF - i0 + 1)];
      if (is <= nx - 2) {
        const int e = (jj + 1) * RX + (is - i0 + 1);
        T acc = cur[u][0];
        acc += cur[u][1] * r0[e + RX];
        acc += cur[u][2] * r0[e - RX];
        acc += cur[u][3] * r0[e + 1];
        acc += cur[u][4] * r0[e - 1];
        acc += cur[u][5] * rm[e];
        acc += cur[u][6] * rp[e];
        xo[row + is] = acc / cur[u][7];
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kSP; u++)
#pragma unroll
      for (int w = 0; w < 8; w++) cur[u][w] = nxt[u][w];
  }
}

// Workgroups are dealt round-robin to the 8 XCDs: XCD x gets the (calculation,
// tile) items [x*per, (x+1)*per) in calculation-major, z-major order, so tiles
// that share halo rows and planes share an L2.
template <class T, int kTY, int kKC, int kTX, int kNT, bool kZeroX = false>
__global__ void __launch_bounds__(kNT)
    k_gsrb7_fused(int nx, int ny, int nz, Batch<SweepArgs<T>> B, int nreq, int first) {
  const int nbx = (nx - 2 + kTX - 1) / kTX, nby = (ny - 2 + kTY - 1) / kTY;
  const int nb = nbx * nby * ((nz - 2 + kKC - 1) / kKC);
  const int total = nb * nreq;
  const int per = (total + kXCD - 1) / kXCD;
  const int item = (blockIdx.x % kXCD) * per + blockIdx.x / kXCD;
  if (item >= total) return;
  const SweepArgs<T>& a = B.v[item / nb];
  fused_body<T, kTY, kKC, kTX, kNT, kZeroX>(nx, ny, nz, item % nb, a.oE, a.oN, a.uC, a.D, a.fc,
                                            a.xi, a.xo, first);
}

// The vector form of the fused sweep.  The scalar form above loads one
// 4- or 8-byte word per lane and operand with the lanes two words apart, so
// the texture addresser (four lanes per clock) and the L1 limit it long
// before memory does.  Here a lane owns a run of kV consecutive elements of
// one row (16 bytes: 4 floats or 2 doubles, both colours) and loads every
// operand as a 16-byte vector; the coefficient vectors that the F step of
// plane k loads are the S step's operands of plane k one step later, so the
// S step loads nothing from memory.  Values and their order are the scalar
// form's (acc7's terms, no FMA).
//
// Lanes: region row r (0 .. kTY+1, row j = j0-1+r) and run c of that row
// (columns i0-1+kV*c ..); a run is moved inwards to [1, nx-1-kV] when it would
// cross the first or last interior column, so every load stays inside the
// row and runs near the grid edge may overlap (they then write the same
// values).  The boundary columns 0 and nx-1 come from the x(p-1) / x(p+1)
// vectors of the runs beside them.
template <class T, int kTY, int kKC, int kTX, int kNT, bool kZeroX>
__device__ __forceinline__ void vfused_body(int nx, int ny, int nz, int tile,
                                            const T* __restrict__ oE, const T* __restrict__ oN,
                                            const T* __restrict__ uC, const T* __restrict__ D,
                                            const T* __restrict__ fc, const T* __restrict__ xi,
                                            T* __restrict__ xo, int first) {
  constexpr int kV = 16 / (int)sizeof(T), kH = kV / 2;
  constexpr int RX = kTX + 2, RY = kTY + 2, RN = RX * RY;
  constexpr int NSEG = (RX + kV - 1) / kV;
  static_assert(RY * NSEG <= kNT, "one lane per run");
  __shared__ T ring[3][RN];
  const int tid = threadIdx.x;
  const int nbx = (nx - 2 + kTX - 1) / kTX, nby = (ny - 2 + kTY - 1) / kTY;
  const int i0 = 1 + (tile % nbx) * kTX, j0 = 1 + ((tile / nbx) % nby) * kTY;
  const int k0 = 1 + (tile / (nbx * nby)) * kKC;
  const int k1 = min(k0 + kKC, nz - 1);  // planes k0 .. k1-1
  const size_t nxy = (size_t)nx * ny;
  const int F = first;

  const bool lane = tid < RY * NSEG;
  const int r = lane ? tid / NSEG : 0, c = lane ? tid % NSEG : 0;
  const int j = j0 - 1 + r;
  const bool rowin = lane && j <= ny - 1;
  const bool rowint = j >= 1 && j <= ny - 2;
  const bool srow = lane && r >= 1 && r <= kTY && j <= ny - 2;
  const int jr = min(j, ny - 1), jc = min(max(j, 1), ny - 2);
  const int is = i0 - 1 + kV * c;
  const int ib = min(max(is, 1), nx - 1 - kV);
  const int chi = min(i0 + kTX - 1, nx - 2);  // last column this tile writes
  // a lane holds, per plane: fc, oN, oN(-nx), oE, oE(-1), uC(-nxy), uC, D and
  // x(+nx), x(-nx), x(+1), x(-1), x(+nxy), x(-nxy), each at columns ib ..
  struct Set {
    T a[8][kV];
    T x[6][kV];
  };
  auto load = [&](int kk, Set& S) {
    const int kc = min(max(kk, 1), nz - 2);
    const size_t q = ((size_t)kc * ny + jc) * nx + ib;   // interior row / plane
    const size_t pr = ((size_t)kk * ny + jr) * nx + ib;  // the lane's own row and plane
    vld16(S.a[0], fc + q);
    vld16(S.a[1], oN + q);
    vld16(S.a[2], oN + q - nx);
    vld16(S.a[3], oE + q);
    vld16(S.a[4], oE + q - 1);
    vld16(S.a[5], uC + q - nxy);
    vld16(S.a[6], uC + q);
    vld16(S.a[7], D + q);
    if (!kZeroX) {
      vld16(S.x[0], xi + q + nx);
      vld16(S.x[1], xi + q - nx);
      vld16(S.x[2], xi + pr + 1);
      vld16(S.x[3], xi + pr - 1);
      vld16(S.x[4], xi + q + nxy);
      vld16(S.x[5], xi + q - nxy);
    } else {
#pragma unroll
      for (int v = 0; v < 6; v++)
#pragma unroll
        for (int e = 0; e < kV; e++) S.x[v][e] = T(0);
    }
  };
  // New F values of plane kk into the ring (and fv: the lane's F elements
  // e0, e0+2, ..., with e0 the first element of F colour)
  auto stageF = [&](int kk, const Set& S, T (&fv)[kH]) {
    if (!rowin) return;
    T* rg = ring[kk % 3] + r * RX - (i0 - 1);
    const bool inner = rowint && kk >= 1 && kk <= nz - 2;
    const int e0 = (F - ib - j - kk) & 1;
#pragma unroll
    for (int m = 0; m < kH; m++) {
      // (selects between values, not addresses, so the vectors stay in registers)
      auto pk = [&](const T(&v)[kV]) {
        const T lo = v[2 * m], hi = v[2 * m + 1];
        return e0 ? hi : lo;
      };
      T val;
      if (inner) {
        T acc = pk(S.a[0]);
        acc += pk(S.a[1]) * pk(S.x[0]);
        acc += pk(S.a[2]) * pk(S.x[1]);
        acc += pk(S.a[3]) * pk(S.x[2]);
        acc += pk(S.a[4]) * pk(S.x[3]);
        acc += pk(S.a[5]) * pk(S.x[5]);
        acc += pk(S.a[6]) * pk(S.x[4]);
        val = acc / pk(S.a[7]);
      } else {
        // a boundary row or plane keeps its values: x at element e is
        // x(p-1)[e+1], or x(p+1)[e-1] for the last element
        const T xe = 2 * m + 2 < kV ? S.x[3][(2 * m + 2) % kV] : S.x[2][2 * m];
        const T xo1 = S.x[3][2 * m + 1];
        val = e0 ? xe : xo1;
      }
      fv[m] = val;
      const int col = ib + e0 + 2 * m;
      if (col >= i0 - 1 && col <= i0 + kTX) rg[col] = val;
    }
    // boundary columns 0 and nx-1 when they are in the region and of F colour
    if (is <= 0 && ((j + kk) & 1) == F) rg[0] = S.x[3][0];
    if (ib == nx - 1 - kV && nx - 1 <= i0 + kTX && ((nx - 1 + j + kk) & 1) == F)
      rg[nx - 1] = S.x[2][kV - 1];
  };
  // S values of plane k from the coefficient vectors of plane k and the ring;
  // both colours of the lane's tile columns are written
  auto stageS = [&](int k, const Set& S, const T(&fv)[kH]) {
    if (!srow) return;
    const int off = r * RX - (i0 - 1);
    const T* rm = ring[(k - 1) % 3] + off;
    const T* r0 = ring[k % 3] + off;
    const T* rp = ring[(k + 1) % 3] + off;
    const int e0 = (F - ib - j - k) & 1;
    T* row = xo + ((size_t)k * ny + j) * nx;
    // a run wholly inside the tile's columns is written with one 16-byte
    // store; the runs at the tile's edges element by element
    const bool full = ib >= i0 && ib + kV - 1 <= chi;
    T out[kV];
#pragma unroll
    for (int m = 0; m < kH; m++) {
      const int cf = ib + e0 + 2 * m;
      const int cs = ib + (1 - e0) + 2 * m;
      T sv = T(0);
      if (full || (cs >= i0 && cs <= chi)) {
        auto pk = [&](const T(&v)[kV]) {
          const T lo = v[2 * m], hi = v[2 * m + 1];
          return e0 ? lo : hi;
        };
        T acc = pk(S.a[0]);
        acc += pk(S.a[1]) * r0[cs + RX];
        acc += pk(S.a[2]) * r0[cs - RX];
        acc += pk(S.a[3]) * r0[cs + 1];
        acc += pk(S.a[4]) * r0[cs - 1];
        acc += pk(S.a[5]) * rm[cs];
        acc += pk(S.a[6]) * rp[cs];
        sv = acc / pk(S.a[7]);
      }
      const T f = fv[m];
      out[2 * m] = e0 ? sv : f;
      out[2 * m + 1] = e0 ? f : sv;
      if (!full) {
        if (cf >= i0 && cf <= chi) row[cf] = f;
        if (cs >= i0 && cs <= chi) row[cs] = sv;
      }
    }
    if (full) vst16(row + ib, out);
  };
  // one plane step: F(k+1) from n (loaded one step earlier), then S(k) from
  // c, whose registers then take the loads of plane k+2
  auto step = [&](int k, Set& cur, T(&fc_)[kH], const Set& nxt, T(&fn)[kH]) {
    stageF(k + 1, nxt, fn);
    __syncthreads();
    stageS(k, cur, fc_);
    if (k + 2 <= k1) load(k + 2, cur);
    __syncthreads();
  };

  Set A, B;
  T fa[kH], fb[kH];
  load(k0 - 1, A);
  stageF(k0 - 1, A, fa);
  load(k0, A);
  stageF(k0, A, fa);
  load(k0 + 1, B);
  int k = k0;
  for (; k + 1 < k1; k += 2) {
    step(k, A, fa, B, fb);
    step(k + 1, B, fb, A, fa);
  }
  if (k < k1) step(k, A, fa, B, fb);
}

template <class T, int kTY, int kKC, int kTX, int kNT, bool kZeroX = false>
__global__ void __launch_bounds__(kNT)
    k_gsrb7_vfused(int nx, int ny, int nz, Batch<SweepArgs<T>> B, int nreq, int first) {
  const int nbx = (nx - 2 + kTX - 1) / kTX, nby = (ny - 2 + kTY - 1) / kTY;
  const int nb = nbx * nby * ((nz - 2 + kKC - 1) / kKC);
  const int total = nb * nreq;
  const int per = (total + kXCD - 1) / kXCD;
  const int item = (blockIdx.x % kXCD) * per + blockIdx.x / kXCD;
  if (item >= total) return;
  const SweepArgs<T>& a = B.v[item / nb];
  vfused_body<T, kTY, kKC, kTX, kNT, kZeroX>(nx, ny, nz, item % nb, a.oE, a.oN, a.uC, a.D, a.fc,
                                             a.xi, a.xo, first);
}

}  // namespace

template <class T, int TY, int KC, int TX, int NT = kFT, bool ZX = false>
void fused_sweep(hipStream_t s, int nx, int ny, int nz, const Batch<SweepArgs<T>>& B, int nb,
                 int first) {
  const int tiles = ((nx - 2 + TX - 1) / TX) * ((ny - 2 + TY - 1) / TY) * ((nz - 2 + KC - 1) / KC);
  const long total = (long)tiles * nb;
  const unsigned g = (unsigned)(((total + kXCD - 1) / kXCD) * kXCD);
  k_gsrb7_fused<T, TY, KC, TX, NT, ZX><<<g, NT, 0, s>>>(nx, ny, nz, B, nb, first);
}

// The vector form: one lane per 16-byte run of a region row, the workgroup
// rounded up to whole wavefronts.
template <class T, int TY, int KC, int TX, bool ZX = false>
void vfused_sweep(hipStream_t s, int nx, int ny, int nz, const Batch<SweepArgs<T>>& B, int nb,
                  int first) {
  constexpr int kV = 16 / (int)sizeof(T);
  constexpr int NT = (((TY + 2) * ((TX + 2 + kV - 1) / kV) + 63) / 64) * 64;
  const int tiles = ((nx - 2 + TX - 1) / TX) * ((ny - 2 + TY - 1) / TY) * ((nz - 2 + KC - 1) / KC);
  const long total = (long)tiles * nb;
  const unsigned g = (unsigned)(((total + kXCD - 1) / kXCD) * kXCD);
  k_gsrb7_vfused<T, TY, KC, TX, NT, ZX><<<g, NT, 0, s>>>(nx, ny, nz, B, nb, first);
}

// The vector-form shapes (70TP or 7TPP: TY rows x P planes) need rows of at
// least 16 bytes plus the two boundary points.
static bool vector_shape(int rp) {
  switch (rp) {
    case 7048: case 7088: case 7410: case 7412: case 7416: case 7816:
      return true;
    default:
      return false;
  }
}

// Launches the vector form of shape rp (vector_shape(rp) holds).
template <class T, int TX, bool ZX>
void vfused_dispatch(hipStream_t s, int rp, int nx, int ny, int nz, const Batch<SweepArgs<T>>& B,
                     int nb, int first) {
  switch (rp) {
    case 7048: vfused_sweep<T, 4, 8, TX, ZX>(s, nx, ny, nz, B, nb, first); break;
    case 7088: vfused_sweep<T, 8, 8, TX, ZX>(s, nx, ny, nz, B, nb, first); break;
    case 7410: vfused_sweep<T, 4, 10, TX, ZX>(s, nx, ny, nz, B, nb, first); break;
    case 7412: vfused_sweep<T, 4, 12, TX, ZX>(s, nx, ny, nz, B, nb, first); break;
    case 7416: vfused_sweep<T, 4, 16, TX, ZX>(s, nx, ny, nz, B, nb, first); break;
    default: vfused_sweep<T, 8, 16, TX, ZX>(s, nx, ny, nz, B, nb, first); break;
  }
}

// The scalar shapes 4 rows x 8 planes and 8 rows x 8 planes with 512
// threads and every vector shape also come in the zero-start form; other
// shapes start from a cleared x.
static bool zero_start_shape(int rp) { return rp == 48 || rp == 5088 || vector_shape(rp); }

static bool valid_tile(int v) {
  const int w = v / 10000, rp = v % 10000;
  const bool shape = rp == 416 || rp == 48 || rp == 816 || rp == 88 || rp == 84 || rp == 1616 ||
                     rp == 832 || rp == 44 || rp == 68 || rp == 5088 || rp == 5084 ||
                     rp == 5816 || vector_shape(rp);
  return shape && (w == 0 || w == 64 || w == 80 || w == 96);
}

// tile shape of the fused sweep: rows x planes per workgroup
// An APBS_PMG_FUSED_TILE shape, or 0.
static int fused_tile_env() {
  static int t = [] {
    const char* e = getenv("APBS_PMG_FUSED_TILE");
    if (!e) return 0;
    const int v = atoi(e);
    return valid_tile(v) ? v : 0;
  }();
  return t;
}

// The march's default shape for a grid and word size (the grids block_tile
// leaves to it): the vector form, with the rows x
// planes per workgroup that were fastest in standalone sweeps (us per sweep;
// the best shape moves with how the workgroups fill the chip).  The shapes for
// fewer points serve long rows and batches; a single 65^3 or 97^3 grid, and
// 129^3 in FP32, take a block:
//   FP32: up to 2.5M points 4 x 8 (65^3 12.2, 97^3 15.0, 129^3 20.3); up to
//         5.5M 4 x 10 (161^3 29.7 against 36.5 for 4 x 8 and 50.2 for the
//         scalar form); up to 20M 8 x 16 (193^3 49.3 against 70.8 for the
//         scalar 8 x 8 with 512 threads); above 8 x 16 in 96-column tiles
//         (353^3 403, against 421 in 64-column tiles and 573 scalar).
//   FP64: up to 0.5M points 4 x 8 (65^3 12.9); up to 1M 4 x 10 (97^3 18.7);
//         up to 3M 4 x 12 (129^3 31.8); up to 5.5M 4 x 10 (161^3 48.9 against
//         65.4 scalar); up to 20M 4 x 12 (193^3 125.4 against 137.9); above
//         4 x 12 in 80-column tiles (353^3 786, against 822 for 4 x 16 in
//         64-column tiles and 931 scalar).
// The column width otherwise follows fused_width; at 353^3 the widths above
// leave fewer idle lanes (a run is 16 bytes, the workgroup whole wavefronts).
int fused_tile(int nx, int ny, int nz, int word) {
  if (const int t = fused_tile_env()) return t;
  const long n = (long)nx * ny * nz;
  if (word == 4) {
    if (n <= 2500000L) return 7048;
    if (n <= 5500000L) return 7410;
    return n <= 20000000L ? 7816 : 967816;
  }
  if (n <= 500000L) return 7048;
  if (n <= 1000000L) return 7410;
  if (n <= 3000000L) return 7412;
  if (n <= 5500000L) return 7410;
  return n <= 20000000L ? 7412 : 807412;
}

// Block shape (block_sweep_device.hip) of nb grids swept together, or 0 where
// the march is taken: above 1.5M points in all in FP64 (113^3 block 26.2 us a
// sweep, march 29.1; 129^3 31.2 and 30.8) and 3.1M in FP32 (145^3 22.4 and 27.5,
// 161^3 31.9 and 30.0; long rows meet earlier, 225x97x97 20.9 and 20.2).  The
// shape is the one of 256 or more workgroups (one a CU; all shapes of a grid too
// small for that) that loads the fewest runs per run written, the larger
// workgroup on a tie.  Rows of more than 130 points in FP64 (258 in FP32) leave
// shapes that load three runs and more for one written; from 100,000 points such
// a grid keeps the march, which is right for the larger (161x97x97 FP64 28.1 and
// 24.5) and not for the smaller ones (161x65x65 13.5 and 18.1).  At 129 points the
// shape of 2 rows and 3 planes, 2.7 runs for one, is the faster: 129x129x65 18.2
// and 23.5, 129x97x97 17.9 and 23.5, 129x65x65 10.3 and 16.8.
static int block_tile(int nx, int ny, int nz, int word, int nb) {
  const double pts = (double)nx * ny * nz * nb;
  if (pts > (word == 8 ? 1.5e6 : 3.1e6)) return 0;
  const int kV = 16 / word, R = (nx - 2 + kV - 1) / kV;
  auto groups = [&](int TY, int KC) {
    return (long)((ny - 2 + TY - 1) / TY) * ((nz - 2 + KC - 1) / KC) * nb;
  };
  const long want = std::min(256L, groups(1, 1));
  int best = 0, lanes = 0;
  double eff = 0.0;
  for (int TY = 1; TY <= 8; TY++)
    for (int KC = 1; KC <= 8; KC++) {
      const int code = 100 * TY + KC, runs = (TY + 2) * KC + 2 * TY;
      if (!block_sweep_fits(nx, word, code) || groups(TY, KC) < want) continue;
      const double e = (double)TY * KC / runs;
      if (e > eff + 1e-9 || (e > eff - 1e-9 && R * runs > lanes)) {
        best = code;
        eff = e;
        lanes = R * runs;
      }
    }
  return eff >= 0.37 || pts < 1.0e5 ? best : 0;
}

// Whether the default fused sweep of a grid runs in the vector form.
bool fused_vector(int nx, int ny, int nz, int word) {
  return nx >= 16 / word + 2 && (vector_shape(fused_tile(nx, ny, nz, word) % 10000) ||
                                 block_tile(nx, ny, nz, word, 1) != 0);
}

// Tile width for an x extent: the one of 64 / 80 / 96 columns that leaves
// the fewest idle columns in the last tile (64 on a tie).
int fused_width(int nx) {
  int best = 64, waste = 1 << 30;
  for (int w : {64, 80, 96}) {
    const int m = ((nx - 2 + w - 1) / w) * w - (nx - 2);
    if (m < waste) {
      waste = m;
      best = w;
    }
  }
  return best;
}

template <class T, int TX>
static void fused_sweep_w(hipStream_t s, int rp, int nx, int ny, int nz,
                          const Batch<SweepArgs<T>>& B, int nb, int first, bool zero_x) {
  if (zero_x) {
    if (rp == 48)
      fused_sweep<T, 4, 8, TX, kFT, true>(s, nx, ny, nz, B, nb, first);
    else if (vector_shape(rp))
      vfused_dispatch<T, TX, true>(s, rp, nx, ny, nz, B, nb, first);
    else
      fused_sweep<T, 8, 8, TX, 512, true>(s, nx, ny, nz, B, nb, first);
    return;
  }
  if (vector_shape(rp)) {
    vfused_dispatch<T, TX, false>(s, rp, nx, ny, nz, B, nb, first);
    return;
  }
  switch (rp) {
    case 416: fused_sweep<T, 4, 16, TX>(s, nx, ny, nz, B, nb, first); break;
    case 48: fused_sweep<T, 4, 8, TX>(s, nx, ny, nz, B, nb, first); break;
    case 44: fused_sweep<T, 4, 4, TX>(s, nx, ny, nz, B, nb, first); break;
    // 512-thread workgroups: 8 or 12 rows with one F round and one S round
    case 5088: fused_sweep<T, 8, 8, TX, 512>(s, nx, ny, nz, B, nb, first); break;
    case 5084: fused_sweep<T, 8, 4, TX, 512>(s, nx, ny, nz, B, nb, first); break;
    case 5816: fused_sweep<T, 8, 16, TX, 512>(s, nx, ny, nz, B, nb, first); break;
    case 68: fused_sweep<T, 6, 8, TX>(s, nx, ny, nz, B, nb, first); break;
    case 88: fused_sweep<T, 8, 8, TX>(s, nx, ny, nz, B, nb, first); break;
    case 84: fused_sweep<T, 8, 4, TX>(s, nx, ny, nz, B, nb, first); break;
    case 1616: fused_sweep<T, 16, 16, TX>(s, nx, ny, nz, B, nb, first); break;
    case 832: fused_sweep<T, 8, 32, TX>(s, nx, ny, nz, B, nb, first); break;
    default: fused_sweep<T, 8, 16, TX>(s, nx, ny, nz, B, nb, first); break;
  }
}

template <class T>
void gsrb7_fused_batch(hipStream_t s, int nx, int ny, int nz, const LevelArgs<T>* c, int nb,
                       int nu, int iadjoint, int tile_shape, bool zero_x) {
  check_batch(nb);
  const int first = iadjoint ? 0 : 1;
  int block = tile_shape >= kBlockTile ? tile_shape - kBlockTile : 0;
  if (tile_shape == 0 && !fused_tile_env()) block = block_tile(nx, ny, nz, (int)sizeof(T), nb);
  if (block && block_sweep_fits(nx, (int)sizeof(T), block)) {
    for (int it = 0; it < nu; it++)
      gsrb7_block_sweep<T>(s, nx, ny, nz, c, nb, first, (it & 1) != 0, zero_x && it == 0, block);
    if (nu & 1)
      for (int b = 0; b < nb; b++) copy_interior<T>(s, nx, ny, nz, c[b].xs, c[b].x);
    return;
  }
  const int tile =
      tile_shape > 0 && valid_tile(tile_shape) ? tile_shape
                                               : fused_tile(nx, ny, nz, (int)sizeof(T));
  int rp = tile % 10000;
  const int w = tile / 10000 ? tile / 10000 : fused_width(nx);
  if (vector_shape(rp) && nx < 16 / (int)sizeof(T) + 2) rp = 48;
  if (zero_x && !zero_start_shape(rp)) {
    for (int b = 0; b < nb; b++) fill<T>(s, c[b].x, (size_t)nx * ny * nz, T(0));
    zero_x = false;
  }
  for (int it = 0; it < nu; it++) {
    // sweep it reads x (even it) or xs and writes the other one
    Batch<SweepArgs<T>> B;
    for (int b = 0; b < nb; b++) {
      const LevelArgs<T>& a = c[b];
      B.v[b] = SweepArgs<T>{a.A.a[1], a.A.a[2], a.A.a[3], a.D, a.f,
                            (it & 1) ? a.xs : a.x, (it & 1) ? a.x : a.xs};
    }
    const bool zx = zero_x && it == 0;
    if (w == 80)
      fused_sweep_w<T, 80>(s, rp, nx, ny, nz, B, nb, first, zx);
    else if (w == 96)
      fused_sweep_w<T, 96>(s, rp, nx, ny, nz, B, nb, first, zx);
    else
      fused_sweep_w<T, 64>(s, rp, nx, ny, nz, B, nb, first, zx);
  }
  if (nu & 1)
    for (int b = 0; b < nb; b++) copy_interior<T>(s, nx, ny, nz, c[b].xs, c[b].x);
}

template <class T>
void gsrb7_fused(hipStream_t s, int nx, int ny, int nz, const Ops<T>& A, const T* D, const T* fc,
                 T* x, T* tmp, int nu, int iadjoint, int tile_shape) {
  const LevelArgs<T> c{A, D, fc, x, tmp, nullptr};
  gsrb7_fused_batch<T>(s, nx, ny, nz, &c, 1, nu, iadjoint, tile_shape);
}

int gsrb7_fused_launches(int nu) { return nu + (nu & 1); }

#define INST(T)                                                                                 \
  template void gsrb7_fused<T>(hipStream_t, int, int, int, const Ops<T>&, const T*, const T*, T*, \
                               T*, int, int, int);                                              \
  template void gsrb7_fused_batch<T>(hipStream_t, int, int, int, const LevelArgs<T>*, int, int,  \
                                     int, int, bool);
INST(double)
INST(float)
#undef INST

}  // namespace pmg
