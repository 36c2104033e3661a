// block_sweep_device.hip -- the fused red-black sweep for fine grids that the
// marching form leaves short of work.
#include "stencil27.h"

namespace pmg {
namespace {

// One complete red-black sweep of the 7-point level, out of place, like
// k_gsrb7_vfused and bit for bit its values, without the march: a workgroup
// owns TY whole rows of KC planes, and every run of kV points (16 bytes, both
// colours) of those planes, of the rows one above and below and of the planes
// one above and below has a lane of its own.  All lanes load their operands at
// once, the first colour's values go to LDS, and after one barrier the second
// colour is updated from them.  So a launch is one wait for memory and one
// barrier, where a marching workgroup waits and meets twice for each plane; the
// price is that ((TY + 2) KC + 2 TY) / (TY KC) runs are loaded per run written.
// On grids whose march does not fill the chip (65^3: 128 workgroups of 8 dependent
// planes) the wait is what the sweep costs.  us per sweep, marching, then so:
// 33^3 FP64 13.1, 3.4, FP32 13.1, 3.4; 65^3 13.1, 5.1 and 12.5, 4.3; 97^3 18.4,
// 13.8 and 15.1, 7.2; 129^3 FP32 20.3, 14.8.
template <class T>
struct BlockArgs {
  const T *oE, *oN, *uC, *D, *fc, *xi;
  T* xo;
};

constexpr int kXcd = 8;

template <class T, bool kZeroX>
__global__ void __launch_bounds__(1024)
    k_gsrb7_block(int nx, int ny, int nz, Batch<BlockArgs<T>> B, int nreq, int F, int R, int TY,
                  int KC) {
  constexpr int kV = 16 / (int)sizeof(T), kH = kV / 2;
  extern __shared__ unsigned char block_smem[];
  T* buf = reinterpret_cast<T*>(block_smem);  // [KC + 2][TY + 2][nx]
  // workgroups are dealt round-robin to the XCDs: contiguous tiles share an L2
  const int nby = (ny - 2 + TY - 1) / TY, nb = nby * ((nz - 2 + KC - 1) / KC);
  const int total = nb * nreq, per = (total + kXcd - 1) / kXcd;
  const int item = (int)(blockIdx.x % kXcd) * per + (int)(blockIdx.x / kXcd);
  if (item >= total) return;
  const BlockArgs<T>& a = B.v[item / nb];
  const int tile = item % nb;
  const int j0 = 1 + (tile % nby) * TY, k0 = 1 + (tile / nby) * KC;
  // lanes: TY + 2 rows of each of the KC planes, then TY rows of the planes
  // below and above
  const int row = (int)threadIdx.x / R, run = (int)threadIdx.x % R;
  const int inner_rows = (TY + 2) * KC;
  int pl, r;  // plane (0 .. KC + 1) and row (0 .. TY + 1) of the block
  if (row < inner_rows) {
    pl = 1 + row / (TY + 2);
    r = row % (TY + 2);
  } else {
    const int q = row - inner_rows;
    pl = q < TY ? 0 : KC + 1;
    r = 1 + (q < TY ? q : q - TY);
  }
  const int j = j0 - 1 + r, k = k0 - 1 + pl;
  const bool act = row < inner_rows + 2 * TY && j <= ny - 1 && k <= nz - 1;
  const bool interior = act && j >= 1 && j <= ny - 2 && k >= 1 && k <= nz - 2;
  const int ib = min(1 + kV * run, nx - 1 - kV);
  const size_t nxy = (size_t)nx * ny;
  const size_t p = ((size_t)(act ? k : 0) * ny + (act ? j : 0)) * nx + ib;
  T* line = buf + (size_t)(pl * (TY + 2) + r) * nx;
  const int e0 = (F - ib - j - k) & 1;  // first element of the first colour
  T c[8][kV], fv[kH];
  if (interior) {
    T x[6][kV];
    vld16(c[0], a.fc + p);
    vld16(c[1], a.oN + p);
    vld16(c[2], a.oN + p - nx);
    vld16(c[3], a.oE + p);
    vld16(c[4], a.oE + p - 1);
    vld16(c[5], a.uC + p - nxy);
    vld16(c[6], a.uC + p);
    vld16(c[7], a.D + p);
    if (!kZeroX) {
      vld16(x[0], a.xi + p + nx);
      vld16(x[1], a.xi + p - nx);
      vld16(x[2], a.xi + p + 1);
      vld16(x[3], a.xi + p - 1);
      vld16(x[4], a.xi + p + nxy);
      vld16(x[5], a.xi + p - nxy);
    } else {
#pragma unroll
      for (int v = 0; v < 6; v++)
#pragma unroll
        for (int q = 0; q < kV; q++) x[v][q] = T(0);
    }
#pragma unroll
    for (int m = 0; m < kH; m++) {
      auto pk = [&](const T(&v)[kV]) {
        const T lo = v[2 * m], hi = v[2 * m + 1];
        return e0 ? hi : lo;
      };
      T acc = pk(c[0]);
      acc += pk(c[1]) * pk(x[0]);
      acc += pk(c[2]) * pk(x[1]);
      acc += pk(c[3]) * pk(x[2]);
      acc += pk(c[4]) * pk(x[3]);
      acc += pk(c[5]) * pk(x[5]);
      acc += pk(c[6]) * pk(x[4]);
      fv[m] = acc / pk(c[7]);
      line[ib + e0 + 2 * m] = fv[m];
    }
    // the boundary columns keep their values
    if (run == 0) line[0] = x[3][0];
    if (run == R - 1) line[nx - 1] = x[2][kV - 1];
  } else if (act) {
    // a boundary row or plane keeps its values
    T x[kV];
    if (!kZeroX) {
      vld16(x, a.xi + p);
    } else {
#pragma unroll
      for (int q = 0; q < kV; q++) x[q] = T(0);
    }
#pragma unroll
    for (int q = 0; q < kV; q++) line[ib + q] = x[q];
  }
  __syncthreads();
  if (!interior || pl < 1 || pl > KC || r < 1 || r > TY) return;
  const T *up = line + nx, *dn = line - nx;
  const T *ab = line + (size_t)(TY + 2) * nx, *be = line - (size_t)(TY + 2) * nx;
  T out[kV];
#pragma unroll
  for (int m = 0; m < kH; m++) {
    const int s = ib + (1 - e0) + 2 * m;
    auto pk = [&](const T(&v)[kV]) {
      const T lo = v[2 * m], hi = v[2 * m + 1];
      return e0 ? lo : hi;
    };
    T acc = pk(c[0]);
    acc += pk(c[1]) * up[s];
    acc += pk(c[2]) * dn[s];
    acc += pk(c[3]) * line[s + 1];
    acc += pk(c[4]) * line[s - 1];
    acc += pk(c[5]) * be[s];
    acc += pk(c[6]) * ab[s];
    const T sv = acc / pk(c[7]);
    out[2 * m] = e0 ? sv : fv[m];
    out[2 * m + 1] = e0 ? fv[m] : sv;
  }
  vst16(a.xo + p, out);
}

}  // namespace

// Block shape code 100 TY + KC; whether it fits a grid: a run and its boundary
// points in a row, the block's runs in one workgroup, its rows in LDS.
bool block_sweep_fits(int nx, int word, int code) {
  const int TY = code / 100, KC = code % 100, kV = 16 / word;
  if (TY < 1 || KC < 1 || nx < kV + 2) return false;
  const int R = (nx - 2 + kV - 1) / kV;
  return R * ((TY + 2) * KC + 2 * TY) <= 1024 &&
         (long)(KC + 2) * (TY + 2) * nx * word <= 64 * 1024;
}

template <class T>
void gsrb7_block_sweep(hipStream_t s, int nx, int ny, int nz, const LevelArgs<T>* c, int nb,
                       int first, bool flip, bool zero_x, int code) {
  check_batch(nb);
  constexpr int kV = 16 / (int)sizeof(T);
  const int TY = code / 100, KC = code % 100, R = (nx - 2 + kV - 1) / kV;
  Batch<BlockArgs<T>> B;
  for (int b = 0; b < nb; b++)
    B.v[b] = BlockArgs<T>{c[b].A.a[1], c[b].A.a[2],           c[b].A.a[3],          c[b].D,
                          c[b].f,      flip ? c[b].xs : c[b].x, flip ? c[b].x : c[b].xs};
  const long total = (long)((ny - 2 + TY - 1) / TY) * ((nz - 2 + KC - 1) / KC) * nb;
  const unsigned g = (unsigned)((total + kXcd - 1) / kXcd * kXcd);
  const int nt = (R * ((TY + 2) * KC + 2 * TY) + 63) / 64 * 64;
  const size_t lds = (size_t)(KC + 2) * (TY + 2) * nx * sizeof(T);
  if (zero_x)
    k_gsrb7_block<T, true><<<g, nt, lds, s>>>(nx, ny, nz, B, nb, first, R, TY, KC);
  else
    k_gsrb7_block<T, false><<<g, nt, lds, s>>>(nx, ny, nz, B, nb, first, R, TY, KC);
}

#define INST(T)                                                                              \
  template void gsrb7_block_sweep<T>(hipStream_t, int, int, int, const LevelArgs<T>*, int, int, \
                                     bool, bool, int);
INST(double)
INST(float)
#undef INST

}  // namespace pmg
