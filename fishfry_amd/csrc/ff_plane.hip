// Plane kernels (see ff_plane.hpp).  FF_PLANE selects the row length nz of one
// build unit (0: the launchers).
//
// What bounds them: the passes of a small grid are bound by launches and ramps
// (64^3: five kernels of 4 us each, of which half is the launch) and those of a
// batch by their reads and writes.  A plane of up to 10000 complex values
// fits one CU: its rows live in registers (E values per thread, as in the row
// kernels), go through LDS between their passes, then once across to the
// columns' threads, whose passes exchange through the same LDS.  The spectrum
// between the z and y transforms never leaves the CU.
#include "ff_plane.hpp"

#ifndef FF_PLANE
#error "FF_PLANE must be defined"
#endif

namespace ff {

// The row transform of nz (E values per thread at positions r0 + i*L of row
// `line`) and the column transform of ny (column c).  Threads beyond the rows
// or columns repeat the last one's work: they write the values its owner writes
// and store nothing.
// The thread's number behind an opaque copy: each phase derives its LDS addresses
// and twiddle positions anew.  Left visible, the compiler keeps those of one
// phase live into the next and spills.
__device__ __forceinline__ int phase_thread() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

template <int NZ, int NY>
struct PlaneRow {
  static constexpr int M = NZ / 2, NH = M + 1, E = kPlaneLens[plane_index(NZ)].ez, L = M / E;
  int line, r0;
  bool own;
  RowIdx idx;
  __device__ __forceinline__ PlaneRow() {
    const int t = phase_thread(), q = t / L;
    own = q < NY;
    line = own ? q : NY - 1;
    r0 = t - q * L;
    idx = RowIdx{line * plane_row_pitch(NZ), 4};
  }
};

template <int NZ, int NY>
struct PlaneCol {
  static constexpr int E = kPlaneLens[plane_index(NY)].ey, L = NY / E, NH = NZ / 2 + 1;
  int c, r0;
  bool own;
  ColIdx idx;
  __device__ __forceinline__ PlaneCol() {
    const int t = phase_thread(), q = t / NH;
    own = q < L;
    r0 = own ? q : L - 1;
    c = t - q * NH;
    idx = ColIdx{NH, c, kColPadShift};
  }
};

// The plane in LDS as the columns see it: entry (row j, kh) at [j][kh].
template <int NZ>
__device__ __forceinline__ int plane_at(int j, int kh) {
  return j * (NZ / 2 + 1) + kh + (j >> kColPadShift);
}

// Column half of the forward kernel: takes the row spectra x (and, from the
// thread of kh = 0, the Nyquist entry) and writes the plane.
template <int NZ, int NY, typename F, int EZ>
__device__ __forceinline__ void plane_cols_fwd(const RowArgs& a, cx<F>* lds, cx<F> (&x)[EZ], F nyq, FF_GLB cx<F>* dst) {
  using R = PlaneRow<NZ, NY>;
  using C = PlaneCol<NZ, NY>;
  const R row;
  const C col;
  cx<F> u[C::E];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < EZ; ++i) lds[plane_at<NZ>(row.line, row.r0 + i * R::L)] = x[i];
  if (row.r0 == 0) lds[plane_at<NZ>(row.line, R::M)] = cx<F>{nyq, F(0)};
  __syncthreads();
#pragma unroll
  for (int i = 0; i < C::E; ++i) u[i] = lds[col.idx(col.r0 + i * C::L)];
  const cx<F>* __restrict__ tw = reinterpret_cast<const cx<F>*>(a.tw2);
  const C at;
  fft_line_static<NY, C::E, -1, F, ColIdx, false>(u, tw, lds, at.idx, at.r0);
  const C to;
  if (to.own) {
#pragma unroll
    for (int i = 0; i < C::E; ++i) dst[(to.r0 + i * C::L) * R::NH + to.c] = u[i];
  }
}

template <int NZ, int NY, typename F, typename IN>
__global__ __launch_bounds__(plane_threads(NZ, NY)) void k_plane_r2c(const RowArgs a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cx<F>* lds = reinterpret_cast<cx<F>*>(smem_raw);
  using R = PlaneRow<NZ, NY>;
  const PassInst io = inst_of(a);
  const long long plane = xcd_remap(blockIdx.x, a.nblocks);
  cx<F> v[R::E];
  {
    const R row;
    const FF_GLB cx<IN>* src = (const FF_GLB cx<IN>*)(glb<const IN>(io.src) + (plane * NY + row.line) * NZ);
#pragma unroll
    for (int i = 0; i < R::E; ++i) {
      const cx<IN> p = src[row.r0 + i * R::L];
      v[i] = cx<F>{F(p.x), F(p.y)};
    }
    const cx<F>* __restrict__ tw = reinterpret_cast<const cx<F>*>(a.tw);
    fft_line_static<R::M, R::E, -1, F, RowIdx, false>(v, tw, lds, row.idx, row.r0);
  }
  // the half spectrum of the row, as r2c_tile forms it; Z[M - k] through LDS
  const F nyq = v[0].x - v[0].y;  // (of the thread that holds k = 0)
  auto spectrum = [&](cx<F> zk, cx<F> z, cx<F> w) {
    const cx<F> zm = conj(z);
    const cx<F> ev = {F(0.5) * (zk.x + zm.x), F(0.5) * (zk.y + zm.y)};
    const cx<F> od = {F(0.5) * (zk.y - zm.y), F(-0.5) * (zk.x - zm.x)};
    return ev + twmul<-1>(od, w);
  };
  __syncthreads();
  {
    const R row;
#pragma unroll
    for (int i = 0; i < R::E; ++i) lds[row.idx(row.r0 + i * R::L)] = v[i];
    __syncthreads();
  }
  const R row;
  const FF_GLB cx<F>* twp = glb<const cx<F>>(a.twpost) + row.r0;
#pragma unroll
  for (int i = 0; i < R::E; ++i) {
    const int k = row.r0 + i * R::L;
    v[i] = spectrum(v[i], lds[row.idx(k ? R::M - k : 0)], cx<F>(twp[i * R::L]));
  }
  FF_GLB cx<F>* dst = glb<cx<F>>(io.dst) + plane * NY * R::NH;
  plane_cols_fwd<NZ, NY, F>(a, lds, v, nyq, dst);
}

// Column half of the inverse kernel: the plane's columns transformed and handed
// to the rows' threads as the packed values z[k] merged from X[k] and X[M - k]
// (c2r_tile).
template <int NZ, int NY, typename F, int EZ>
__device__ __forceinline__ void plane_cols_inv(const RowArgs& a, cx<F>* lds, const FF_GLB cx<F>* src, cx<F> (&v)[EZ]) {
  using R = PlaneRow<NZ, NY>;
  using C = PlaneCol<NZ, NY>;
  cx<F> u[C::E];
  {
    const C from;
#pragma unroll
    for (int i = 0; i < C::E; ++i) u[i] = src[(from.r0 + i * C::L) * R::NH + from.c];
    const C at;
    const cx<F>* __restrict__ tw = reinterpret_cast<const cx<F>*>(a.tw2);
    fft_line_static<NY, C::E, +1, F, ColIdx, false>(u, tw, lds, at.idx, at.r0);
  }
  const R row;
  const C col;
  const cx<F>* __restrict__ twp = reinterpret_cast<const cx<F>*>(a.twpost);
  auto merge = [&](int k, cx<F> xk, cx<F> xm) {
    if (k == 0) {
      xk.y = F(0);
      xm.y = F(0);
    }
    const cx<F> cm = conj(xm);
    const cx<F> A = xk + cm;
    const cx<F> B = twmul<+1>(xk - cm, twp[k]);
    return cx<F>{A.x - B.y, A.y + B.x};
  };
  __syncthreads();
#pragma unroll
  for (int i = 0; i < C::E; ++i) lds[col.idx(col.r0 + i * C::L)] = u[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < EZ; ++i) {
    const int k = row.r0 + i * R::L;
    v[i] = merge(k, lds[plane_at<NZ>(row.line, k)], lds[plane_at<NZ>(row.line, R::M - k)]);
  }
}

template <int NZ, int NY, typename F, typename OUT, int EPI>
__global__ __launch_bounds__(plane_threads(NZ, NY)) void k_plane_c2r(const RowArgs a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cx<F>* lds = reinterpret_cast<cx<F>*>(smem_raw);
  using R = PlaneRow<NZ, NY>;
  const PassInst io = inst_of(a);
  const long long plane = xcd_remap(blockIdx.x, a.nblocks);
  const FF_GLB cx<F>* src = glb<const cx<F>>(io.src) + plane * NY * R::NH;
  cx<F> v[R::E];
  plane_cols_inv<NZ, NY, F>(a, lds, src, v);
  {
    const R at;
    const cx<F>* __restrict__ tw = reinterpret_cast<const cx<F>*>(a.tw);
    fft_line_static<R::M, R::E, +1, F, RowIdx, false>(v, tw, lds, at.idx, at.r0);
  }
  const R row;
  if (row.own) {
    const double shift = io.shiftp ? a.shift * *glb<const double>(io.shiftp) : a.shift;
    const long long off = (plane * NY + row.line) * NZ;
    FF_GLB OUT* out = glb<OUT>(io.dst) + off;
    const FF_GLB double* f = glb<const double>(io.aux) + (EPI == EPI_RESIDUAL ? off : 0);
#pragma unroll
    for (int i = 0; i < R::E; ++i)
      c2r_out2<EPI, OUT>(out, f, row.r0 + i * R::L, to_d(v[i].x), to_d(v[i].y), a.scale, shift);
  }
}

template <int NZ>
const void* plane_r2c_fn(int ny, int f32, int in_f32);
template <int NZ>
const void* plane_c2r_fn(int ny, int f32, int out_kind, int epi);

#if FF_PLANE > 0
template <int NY>
static const void* r2c_of(int f32, int in_f32) {
  if constexpr (plane_threads(FF_PLANE, NY) == 0) return nullptr;
  else if (!f32) return in_f32 ? nullptr : (const void*)&k_plane_r2c<FF_PLANE, NY, double, double>;
  else return in_f32 ? (const void*)&k_plane_r2c<FF_PLANE, NY, float, float> : (const void*)&k_plane_r2c<FF_PLANE, NY, float, double>;
}
template <int NY>
static const void* c2r_of(int f32, int out_kind, int epi) {
  if constexpr (plane_threads(FF_PLANE, NY) > 0) {
    if (!f32) {
      if (epi == EPI_STORE && out_kind == 0) return (const void*)&k_plane_c2r<FF_PLANE, NY, double, double, EPI_STORE>;
      if (epi == EPI_RESIDUAL && out_kind == 1) return (const void*)&k_plane_c2r<FF_PLANE, NY, double, float, EPI_RESIDUAL>;
    } else {
      if (epi == EPI_STORE && out_kind == 0) return (const void*)&k_plane_c2r<FF_PLANE, NY, float, double, EPI_STORE>;
      if (epi == EPI_ACCUM && out_kind == 0) return (const void*)&k_plane_c2r<FF_PLANE, NY, float, double, EPI_ACCUM>;
    }
  }
  return nullptr;
}
#define FF_PLANE_NY(CALL)        \
  switch (ny) {                  \
    case 32: return CALL(32);      \
    case 36: return CALL(36);      \
    case 40: return CALL(40);      \
    case 48: return CALL(48);      \
    case 50: return CALL(50);      \
    case 64: return CALL(64);      \
    case 72: return CALL(72);      \
    case 80: return CALL(80);      \
    case 96: return CALL(96);      \
    case 100: return CALL(100);    \
    case 108: return CALL(108);    \
    case 128: return CALL(128);    \
    case 160: return CALL(160);    \
    default: return nullptr;     \
  }
template <>
const void* plane_r2c_fn<FF_PLANE>(int ny, int f32, int in_f32) {
#define FF_FN(NY) r2c_of<NY>(f32, in_f32)
  FF_PLANE_NY(FF_FN)
#undef FF_FN
}
template <>
const void* plane_c2r_fn<FF_PLANE>(int ny, int f32, int out_kind, int epi) {
#define FF_FN(NY) c2r_of<NY>(f32, out_kind, epi)
  FF_PLANE_NY(FF_FN)
#undef FF_FN
}
#undef FF_PLANE_NY
#else
#define FF_PLANE_DECL(NZ)                                    \
  template <>                                                \
  const void* plane_r2c_fn<NZ>(int ny, int f32, int in_f32); \
  template <>                                                \
  const void* plane_c2r_fn<NZ>(int ny, int f32, int out_kind, int epi);
FF_PLANE_DECL(32)
FF_PLANE_DECL(36)
FF_PLANE_DECL(40)
FF_PLANE_DECL(48)
FF_PLANE_DECL(50)
FF_PLANE_DECL(64)
FF_PLANE_DECL(72)
FF_PLANE_DECL(80)
FF_PLANE_DECL(96)
FF_PLANE_DECL(100)
FF_PLANE_DECL(108)
FF_PLANE_DECL(128)
#undef FF_PLANE_DECL

static hipError_t plane_launch(const void* fn, const Launch& l, const RowArgs& a) {
  if (!fn) return hipErrorInvalidValue;
  if (l.lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l.lds);
    if (e != hipSuccess) return e;
  }
  void* argv[] = {const_cast<RowArgs*>(&a)};
  return hipLaunchKernel(fn, l.grid, l.block, argv, l.lds, l.stream);
}
#define FF_PLANE_NZ(CALL)                           \
  switch (a.nz) {                                   \
    case 32: return plane_launch(CALL(32), l, a);   \
    case 36: return plane_launch(CALL(36), l, a);   \
    case 40: return plane_launch(CALL(40), l, a);   \
    case 48: return plane_launch(CALL(48), l, a);   \
    case 50: return plane_launch(CALL(50), l, a);   \
    case 64: return plane_launch(CALL(64), l, a);   \
    case 72: return plane_launch(CALL(72), l, a);   \
    case 80: return plane_launch(CALL(80), l, a);   \
    case 96: return plane_launch(CALL(96), l, a);   \
    case 100: return plane_launch(CALL(100), l, a); \
    case 108: return plane_launch(CALL(108), l, a); \
    case 128: return plane_launch(CALL(128), l, a); \
    default: return hipErrorInvalidValue;           \
  }
hipError_t plane_r2c(int f32, int in_f32, const Launch& l, const RowArgs& a) {
#define FF_FN(NZ) plane_r2c_fn<NZ>(a.ny, f32, in_f32)
  FF_PLANE_NZ(FF_FN)
#undef FF_FN
}
hipError_t plane_c2r(int f32, int out_kind, int epi, const Launch& l, const RowArgs& a) {
#define FF_FN(NZ) plane_c2r_fn<NZ>(a.ny, f32, out_kind, epi)
  FF_PLANE_NZ(FF_FN)
#undef FF_FN
}
#undef FF_PLANE_NZ
#endif

}  // namespace ff
