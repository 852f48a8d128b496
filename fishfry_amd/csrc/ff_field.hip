// Driver kernels of the benchmark: the right-hand side f (FishFry.hpp:14-45)
// and the error sums against the exact potential (FishFry.hpp:57-101).
//
// Both are extended with a phase shift, an amplitude and a list of extra
// Fourier modes (used by the batched and mixed-precision workloads); with
// shift 0, scale 1 and no modes they evaluate exactly the reference's
// expressions in the reference's operation order.  The error sums use a
// fixed-shape two-stage reduction instead of the reference's double atomics,
// so they are bit-reproducible run to run.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/fishfry.h"
#include "ff_internal.hpp"

namespace ff {

struct FieldArgs {
  int ni, nj, nk;
  double xlo, ylo, zlo, dx, dy, dz;
  double sx, sy, sz;  // shift
  double scale;
  int nmodes;
  int mk[FF_MAX_MODES][3];
  double ma[FF_MAX_MODES], mb[FF_MAX_MODES];
  double minv[FF_MAX_MODES];  // -1/lambda_k of each mode (exact potential)
};

// Every term of f and of the exact potential is a product of one factor per
// axis, so a tile evaluates the factors of its coordinates once into LDS
// and forms the points from them: the analytic part in FishFry.hpp's order, and
// each mode as Re((a - ib) e^{i kx x} e^{i ky y} e^{i kz z}).  For one plane
// i that sum is a matrix product (rows j, columns k, two inner terms per mode),
// which runs on the FP64 matrix instruction with the analytic part as its
// addend.
//
// A workgroup of four waves owns 16 rows (j) by 64 columns (k) of up to
// kMaxPlanes planes (i), its waves taking the planes in turn.  One sincos per
// (coordinate, mode) of the tile then serves 16 * 64 * planes points; taken at
// every point they bounded the kernel (512^3 with 16 modes: 5.50 ms, now
// 0.24 ms, of which the 1.07 GB written take 0.19 ms; 32^3: 9.0 and 8.4 us).
// Rounding: the angle of one axis is smaller than that of all three, so its
// factor carries less error than the cosine of the sum did (relative to 64-bit
// reference values at 484^3: 1.3e-15, now 1.2e-15).
constexpr int kRows = 16, kCols = 64, kMaxPlanes = 64;
constexpr int kFieldThreads = 256;
constexpr int kFieldGroups = 1024;  // workgroups that fill the chip (four per CU)

typedef double f64x4 __attribute__((ext_vector_type(4)));

struct FieldTiles {
  int planes;           // planes per tile
  int tj, tk;           // tiles along j and k
  long long tiles;      // all tiles
  int modes4;           // modes held (0, 16 or 32; the ones past nmodes have amplitude zero)
  __host__ __device__ size_t doubles() const {
    return 2 * (size_t)(planes + kRows + kCols) * (size_t)(modes4 + 1);
  }
};

struct cplx {
  double x, y;
};

// The tile's factors in LDS: modes, then the analytic part, each axis of the
// tile's planes, rows and columns in turn.
struct FieldLds {
  cplx *mx, *my, *mz;  // [mode][plane], [mode][row], [mode][column]; mx holds (a - ib) e^{i kx x}
  cplx *ax, *ay, *az;  // f: (px, dpx), (py, dpy), (pz, dpz); potential: (px, 0), (py, 0), (pz, 0)
};

__device__ __forceinline__ FieldLds field_lds(double* lds, const FieldTiles& t) {
  FieldLds l;
  cplx* c = reinterpret_cast<cplx*>(lds);
  l.mx = c;
  l.my = l.mx + (size_t)t.modes4 * t.planes;
  l.mz = l.my + (size_t)t.modes4 * kRows;
  l.ax = l.mz + (size_t)t.modes4 * kCols;
  l.ay = l.ax + t.planes;
  l.az = l.ay + kRows;
  return l;
}

// Coordinates past the grid's edge have no factors: a row or column of the
// product depends on its own coordinate only, and theirs are not stored.
// (One axis per wave for the analytic part, and one sincos for all three axes
// of the modes: on the smallest grids this chain is the kernel's time.)
template <bool POTENTIAL>
__device__ __forceinline__ void field_factors(const FieldArgs& a, const FieldTiles& t, const FieldLds& l, int i0,
                                              int j0, int k0) {
  const int np = min(t.planes, a.ni - i0), nr = min(kRows, a.nj - j0), nc = min(kCols, a.nk - k0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // FishFry.hpp:22-44 and :71-86, same expressions and order
  if (wave == 0 && lane < np) {
    const double x = a.xlo + (i0 + lane) * a.dx + a.sx;
    const double cx = cos(x);
    const double sx = sin(x);
    const double ex = exp(sx);
    l.ax[lane] = cplx{cx * ex, POTENTIAL ? 0.0 : -ex * sx * cx * (sx + 3.0)};
  } else if (wave == 1 && lane < nr) {
    const double y = a.ylo + (j0 + lane) * a.dy + a.sy;
    const double cy = cos(y);
    const double sy = sin(y);
    const double ey = exp(cy);
    l.ay[lane] = cplx{sy * ey, POTENTIAL ? 0.0 : sy * ey * (sy * sy - 3.0 * cy - 1.0)};
  } else if (wave == 2 && lane < nc) {
    const double z = a.zlo + (k0 + lane) * a.dz + a.sz;
    const double cz = cos(z);
    const double sz = sin(z);
    const double ez = exp(cz);
    l.az[lane] = cplx{cz * ez, POTENTIAL ? 0.0 : ez * (3.0 * sz * sz - cz * cz * cz - 1.0)};
  }
  const int coords = np + nr + nc;
  for (int e = kFieldThreads - 1 - threadIdx.x; e < coords * t.modes4; e += kFieldThreads) {
    const int m = e / coords, q = e - m * coords;
    const int axis = q < np ? 0 : (q < np + nr ? 1 : 2);
    const int r = q - (axis == 0 ? 0 : (axis == 1 ? np : np + nr));
    const bool on = m < a.nmodes;  // padding modes have amplitude zero
    const int mm = on ? m : 0;
    const double w = axis == 0 ? a.xlo + (i0 + r) * a.dx + a.sx
                               : (axis == 1 ? a.ylo + (j0 + r) * a.dy + a.sy : a.zlo + (k0 + r) * a.dz + a.sz);
    double s, c;
    sincos(a.mk[mm][axis] * w, &s, &c);
    if (axis == 0) {
      const double iv = POTENTIAL ? a.minv[mm] : 1.0;
      const double ma = iv * a.ma[mm], mb = iv * a.mb[mm];
      l.mx[m * t.planes + r] = on ? cplx{ma * c + mb * s, ma * s - mb * c} : cplx{0.0, 0.0};
    } else if (axis == 1) {
      l.my[m * kRows + r] = cplx{c, s};
    } else {
      l.mz[m * kCols + r] = cplx{c, s};
    }
  }
}

// The points of plane i0 + ii of the tile, in the accumulator layout of the
// 16 x 16 x 4 FP64 product: element v of point block b is row 4 v + lane / 16,
// column 16 b + lane % 16.  M4: modes / 4 held in registers.
template <bool POTENTIAL, int M4>
__device__ __forceinline__ void field_points(const FieldArgs& a, const FieldTiles& t, const FieldLds& l, int ii,
                                             const cplx (&zf)[M4 ? M4 : 1][4], const cplx (&yf)[M4 ? M4 : 1],
                                             f64x4 (&acc)[4]) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const cplx px = l.ax[ii];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const cplx py = l.ay[4 * v + g];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const cplx pz = l.az[16 * b + c];
      if constexpr (POTENTIAL) acc[b][v] = a.scale * (px.x * py.x * pz.x);
      else acc[b][v] = a.scale * (px.x * py.x * pz.y + px.x * py.y * pz.x + px.y * py.x * pz.x);
    }
  }
#pragma unroll
  for (int s = 0; s < M4; ++s) {
    const cplx ex = l.mx[(4 * s + g) * t.planes + ii];
    const double re = ex.x * yf[s].x - ex.y * yf[s].y;
    const double im = ex.x * yf[s].y + ex.y * yf[s].x;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(re, zf[s][b].x, acc[b], 0, 0, 0);
      acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(-im, zf[s][b].y, acc[b], 0, 0, 0);
    }
  }
}

// Runs the workgroup's tiles: point(offset, value) for each point of the grid
// that a lane holds.
template <bool POTENTIAL, int M4, typename Point>
__device__ __forceinline__ void field_tiles(const FieldArgs& a, const FieldTiles& t, const Point& point) {
  extern __shared__ __align__(16) double field_smem[];
  const FieldLds l = field_lds(field_smem, t);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  for (long long tile = xcd_remap(blockIdx.x, gridDim.x); tile < t.tiles; tile += gridDim.x) {
    const long long ji = tile / t.tk;
    const int k0 = (int)(tile - ji * t.tk) * kCols;
    const int i0 = (int)(ji / t.tj) * t.planes;
    const int j0 = (int)(ji % t.tj) * kRows;
    __syncthreads();  // the last tile's factors have been read
    field_factors<POTENTIAL>(a, t, l, i0, j0, k0);
    __syncthreads();
    cplx zf[M4 ? M4 : 1][4], yf[M4 ? M4 : 1];
#pragma unroll
    for (int s = 0; s < M4; ++s) {
      yf[s] = l.my[(4 * s + g) * kRows + c];
#pragma unroll
      for (int b = 0; b < 4; ++b) zf[s][b] = l.mz[(4 * s + g) * kCols + 16 * b + c];
    }
    for (int ii = wave; ii < t.planes && i0 + ii < a.ni; ii += kFieldThreads / 64) {
      f64x4 acc[4];
      field_points<POTENTIAL, M4>(a, t, l, ii, zf, yf, acc);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int j = j0 + 4 * v + g;
        if (j >= a.nj) continue;
        const long long row = ((long long)(i0 + ii) * a.nj + j) * a.nk;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int k = k0 + 16 * b + c;
          if (k < a.nk) point(row + k, acc[b][v]);
        }
      }
    }
  }
}

template <int M4>
__global__ __launch_bounds__(kFieldThreads) void k_field_init(const FieldArgs a, const FieldTiles t,
                                                              double* __restrict__ f) {
  field_tiles<false, M4>(a, t, [&](long long off, double v) { f[off] = v; });
}

constexpr int DIFF_THREADS = kFieldThreads;
constexpr int DIFF_BLOCKS = 1024;

// Stage 1: workgroup b accumulates tiles b, b+G, ... (a lane its own points, in
// order; 512^3 with 16 modes: 5.9 ms, now 0.70 ms), then a fixed tree in LDS.  partial[3*b + {0,1,2}] = (sum|e|, sum e^2,
// max|e|).
template <int M4>
__global__ __launch_bounds__(DIFF_THREADS) void k_field_diff(const FieldArgs a, const FieldTiles t,
                                                             const double* __restrict__ phi,
                                                             double* __restrict__ partial) {
  __shared__ double s1[DIFF_THREADS], s2[DIFF_THREADS], sm[DIFF_THREADS];
  double t1 = 0.0, t2 = 0.0, tm = 0.0;
  field_tiles<true, M4>(a, t, [&](long long off, double v) {
    const double d = fabs(v - (phi ? phi[off] : 0.0));
    t1 += d;
    t2 += d * d;
    tm = d > tm ? d : tm;
  });
  s1[threadIdx.x] = t1;
  s2[threadIdx.x] = t2;
  sm[threadIdx.x] = tm;
  __syncthreads();
  for (int w = DIFF_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      s1[threadIdx.x] += s1[threadIdx.x + w];
      s2[threadIdx.x] += s2[threadIdx.x + w];
      sm[threadIdx.x] = sm[threadIdx.x] > sm[threadIdx.x + w] ? sm[threadIdx.x] : sm[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partial[3 * blockIdx.x + 0] = s1[0];
    partial[3 * blockIdx.x + 1] = s2[0];
    partial[3 * blockIdx.x + 2] = sm[0];
  }
}

// Stage 2: one block folds the partials in a fixed order.
__global__ __launch_bounds__(DIFF_THREADS) void k_field_diff_final(const double* __restrict__ partial, int nb,
                                                                   double* __restrict__ out) {
  __shared__ double s1[DIFF_THREADS], s2[DIFF_THREADS], sm[DIFF_THREADS];
  double t1 = 0.0, t2 = 0.0, tm = 0.0;
  for (int b = threadIdx.x; b < nb; b += DIFF_THREADS) {
    t1 += partial[3 * b + 0];
    t2 += partial[3 * b + 1];
    tm = partial[3 * b + 2] > tm ? partial[3 * b + 2] : tm;
  }
  s1[threadIdx.x] = t1;
  s2[threadIdx.x] = t2;
  sm[threadIdx.x] = tm;
  __syncthreads();
  for (int w = DIFF_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      s1[threadIdx.x] += s1[threadIdx.x + w];
      s2[threadIdx.x] += s2[threadIdx.x + w];
      sm[threadIdx.x] = sm[threadIdx.x] > sm[threadIdx.x + w] ? sm[threadIdx.x] : sm[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = s1[0];
    out[1] = s2[0];
    out[2] = sm[0];
  }
}

static void field_args(const ff_field& f, FieldArgs& a) {
  a.ni = f.n[0];
  a.nj = f.n[1];
  a.nk = f.n[2];
  a.xlo = f.lo[0];
  a.ylo = f.lo[1];
  a.zlo = f.lo[2];
  a.dx = f.d[0];
  a.dy = f.d[1];
  a.dz = f.d[2];
  a.sx = f.shift[0];
  a.sy = f.shift[1];
  a.sz = f.shift[2];
  a.scale = f.scale;
  a.nmodes = f.nmodes;
  for (int m = 0; m < f.nmodes; ++m) {
    for (int c = 0; c < 3; ++c) a.mk[m][c] = f.mode_k[m][c];
    a.ma[m] = f.mode_a[m];
    a.mb[m] = f.mode_b[m];
    double lam = 0.0;
    for (int c = 0; c < 3; ++c) {
      const int n = f.n[c];
      int kk = f.mode_k[m][c] % n;
      if (kk < 0) kk += n;
      const int km = kk < n - kk ? kk : n - kk;
      const double t = double(km) * f.dd[c];
      lam += t * t;
    }
    a.minv[m] = lam > 0.0 ? -1.0 / lam : 0.0;
  }
}

// Register tiles of the mode loop: none, 16 modes or 32 (FF_MAX_MODES).
static int field_m4(const FieldArgs& a) { return a.nmodes == 0 ? 0 : (a.nmodes <= 16 ? 4 : 8); }

// Planes per tile: as many as leave kFieldGroups tiles, so that the factors
// of a tile serve many points on a large grid and a small one still fills the
// chip; at least 4, one per wave.
static FieldTiles field_tiling(const FieldArgs& a) {
  FieldTiles t;
  // (extents up to 2^31 - 1: no sum with a tile's width)
  t.tj = 1 + (a.nj - 1) / kRows;
  t.tk = 1 + (a.nk - 1) / kCols;
  const long long across = (long long)t.tj * t.tk;
  t.planes = (int)std::max<long long>(4, std::min<long long>(kMaxPlanes, a.ni * across / kFieldGroups));
  t.tiles = across * (1 + (a.ni - 1) / t.planes);
  t.modes4 = 4 * field_m4(a);
  return t;
}

// A kernel over the tiles with the dynamic LDS of their factors: 76 KB at 64
// planes and 32 modes.  Above 64 KB a kernel has to be given it first.
static hipError_t field_launch(const void* fn, unsigned grid, const FieldTiles& t, void** argv, hipStream_t s) {
  const size_t lds = t.doubles() * sizeof(double);
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  return hipLaunchKernel(fn, dim3(grid), dim3(kFieldThreads), argv, lds, s);
}

ff_status field_check(const ff_field* f) {
  if (!f) return set_error(FF_ERR_INVALID, "ff_field: null descriptor");
  for (int c = 0; c < 3; ++c)
    if (f->n[c] < 1) return set_error(FF_ERR_INVALID, "ff_field: extents must be >= 1");
  if (f->nmodes < 0 || f->nmodes > FF_MAX_MODES) return set_error(FF_ERR_INVALID, "ff_field: nmodes out of range");
  if ((long long)f->n[0] * f->n[1] >= (1LL << 31)) return set_error(FF_ERR_INVALID, "ff_field: grid too large");
  return FF_OK;
}

ff_status field_init(const ff_field* f, double* out, hipStream_t s) {
  ff_status st = field_check(f);
  if (st != FF_OK) return st;
  if (!out) return set_error(FF_ERR_INVALID, "ff_field_init: null output");
  FieldArgs a;
  field_args(*f, a);
  const FieldTiles t = field_tiling(a);
  const unsigned grid = (unsigned)std::min<long long>(t.tiles, 1 << 20);
  const void* const fns[3] = {(const void*)&k_field_init<0>, (const void*)&k_field_init<4>,
                              (const void*)&k_field_init<8>};
  void* argv[] = {&a, const_cast<FieldTiles*>(&t), &out};
  return hip_check(field_launch(fns[field_m4(a) / 4], grid, t, argv, s), "k_field_init launch");
}

static_assert(kDiffDoubles == 3 * DIFF_BLOCKS + 3 && kDiffResult == 3 * DIFF_BLOCKS, "diff work area");

ff_status field_diff(const ff_field* f, const double* phi, double out[3], hipStream_t s) {
  if (!out) return set_error(FF_ERR_INVALID, "ff_field_diff: null output");
  double* partial = nullptr;
  ff_status st = device_scratch(3 * DIFF_BLOCKS + 3, &partial);
  if (st != FF_OK) return st;
  st = field_diff_enqueue(f, phi, partial, s);
  if (st != FF_OK) return st;
  st = hip_check(hipMemcpyAsync(out, partial + 3 * DIFF_BLOCKS, 3 * sizeof(double), hipMemcpyDeviceToHost, s),
                 "diff copy");
  if (st != FF_OK) return st;
  return hip_check(hipStreamSynchronize(s), "diff sync");
}

ff_status field_diff_enqueue(const ff_field* f, const double* phi, double* partial, hipStream_t s) {
  ff_status st = field_check(f);
  if (st != FF_OK) return st;
  FieldArgs a;
  field_args(*f, a);
  const FieldTiles t = field_tiling(a);
  const int nb = (int)std::min<long long>(t.tiles, DIFF_BLOCKS);
  const void* const fns[3] = {(const void*)&k_field_diff<0>, (const void*)&k_field_diff<4>,
                              (const void*)&k_field_diff<8>};
  void* argv[] = {&a, const_cast<FieldTiles*>(&t), &phi, &partial};
  st = hip_check(field_launch(fns[field_m4(a) / 4], (unsigned)nb, t, argv, s), "k_field_diff launch");
  if (st != FF_OK) return st;
  hipLaunchKernelGGL(k_field_diff_final, dim3(1), dim3(DIFF_THREADS), 0, s, partial, nb, partial + 3 * DIFF_BLOCKS);
  return hip_check(hipGetLastError(), "k_field_diff_final launch");
}

}  // namespace ff
