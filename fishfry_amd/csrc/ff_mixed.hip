// Mixed-radix pass kernels (see ff_mixed.hpp): the y and x passes over
// columns and the z passes over rows, for the lengths the register engine has
// no direct plan for.  FF_MIX_PART selects the kernels of one build unit.
//
// What bounds them (MI355X, FP64, 385x301x338, one pass reading and writing 630
// MB: 0.11 ms at the rate of the row kernels): Bluestein's lines were bound by
// their four transforms of at least twice the length and by the registers of
// the kernels that hold them (x 1.27 ms, y 0.32, z forward 0.50, z inverse 0.61);
// here x takes 0.31 ms, y 0.22, z 0.18 and 0.20, bound by the LDS exchanges and
// index arithmetic of the stages.  A tile is about 2048 FP64 (4096 FP32) values
// in two buffers (49 KB of LDS at 385), more where row segments of 64 bytes and the
// eight lines of a dense stage ask for it (67 KB at 127, 132 KB at 1017 in FP64), so that two
// to four workgroups of 256 threads share a CU, one at the longest lines, and one's memory
// phase covers another's stages.  Two buffers in turn cost one barrier per
// stage instead of two, and let a stage's butterflies be spread over all
// threads whatever its radix.
#include <type_traits>

#include "ff_mixed.hpp"

#ifndef FF_MIX_PART
#error "FF_MIX_PART must be defined"
#endif

namespace ff {

// ---------------------------------------------------------------------------
// Butterflies of the radices only these kernels use.

// Odd prime R: with s[m] = a[m] + a[R-m], d[m] = a[m] - a[R-m],
//   X[k], X[R-k] = (a0 + sum cos(2 pi k m / R) s[m]) -+ i (sum sin(2 pi k m / R) d[m])   (forward).
template <int R, int K, int M, typename F>
__device__ __forceinline__ void odd_terms(const cx<F>* s, const cx<F>* d, cx<F>& p, cx<F>& q) {
  if constexpr (M <= (R - 1) / 2) {
    constexpr F c = F(kcos(R, K * M)), sn = F(ksin(R, K * M));
    p = {fmadd(c, s[M - 1].x, p.x), fmadd(c, s[M - 1].y, p.y)};
    if constexpr (M == 1) q = {sn * d[0].x, sn * d[0].y};
    else q = {fmadd(sn, d[M - 1].x, q.x), fmadd(sn, d[M - 1].y, q.y)};
    odd_terms<R, K, M + 1, F>(s, d, p, q);
  }
}

template <int R, int K, int DIR, typename F>
__device__ __forceinline__ void odd_outputs(cx<F>* a, cx<F> a0, const cx<F>* s, const cx<F>* d) {
  if constexpr (K <= (R - 1) / 2) {
    cx<F> p = a0, q{};
    odd_terms<R, K, 1, F>(s, d, p, q);
    const cx<F> t = mul_mi<DIR>(q);
    a[K] = p + t;
    a[R - K] = p - t;
    odd_outputs<R, K + 1, DIR, F>(a, a0, s, d);
  }
}

template <int R, int DIR, typename F>
__device__ __forceinline__ void dft_odd(cx<F>* a) {
  constexpr int H = (R - 1) / 2;
  cx<F> s[H], d[H];
  const cx<F> a0 = a[0];
  cx<F> sum = a0;
#pragma unroll
  for (int m = 1; m <= H; ++m) {
    s[m - 1] = a[m] + a[R - m];
    d[m - 1] = a[m] - a[R - m];
    sum = sum + s[m - 1];
  }
  a[0] = sum;
  odd_outputs<R, 1, DIR, F>(a, a0, s, d);
}

template <int R, int DIR, typename F>
__device__ __forceinline__ void mix_dft(cx<F>* a) {
  if constexpr (R == 7 || R == 11 || R == 13) dft_odd<R, DIR, F>(a);
  else if constexpr (R == 9) dft_ct<3, 3, DIR, F>(a);
  else Dft<R, DIR, F>::run(a);
}

// ---------------------------------------------------------------------------
// Stages.

// The tile's lines in LDS: columns [position][line], rows [line][pitch].
template <typename F, bool ROW>
struct MixTile {
  cx<F>* buf;        // this buffer
  int T, lgT, pitch;
  const cx<F>* tab;  // the dense stages' (cos, sin) tables
  __device__ __forceinline__ int at(int line, int pos) const {
    return ROW ? line * pitch + pos : (pos << lgT) + line;
  }
};

__device__ __forceinline__ int div_by(int v, int by, uint32_t inv) {
  return by > 1 ? (int)__umulhi((uint32_t)v, inv) : v;
}

// The plan in device memory, read through the scalar path: plans are never
// written while a kernel that reads them runs.
#if defined(__HIP_DEVICE_COMPILE__)
#define FF_CST __attribute__((address_space(4)))
#else
#define FF_CST
#endif
typedef const FF_CST MixPlan* MixPlanPtr;
__device__ __forceinline__ MixStage mix_stage(MixPlanPtr mp, int p) {
  MixStage s;
  s.R = mp->st[p].R;
  s.dense = mp->st[p].dense;
  s.ns = mp->st[p].ns;
  s.cnt = mp->st[p].cnt;
  s.nsinv = mp->st[p].nsinv;
  s.cntinv = mp->st[p].cntinv;
  s.twstep = mp->st[p].twstep;
  s.twnext = mp->st[p].twnext;
  s.rinv = mp->st[p].rinv;
  s.ktiles = mp->st[p].ktiles;
  s.ltab = mp->st[p].ltab;
  return s;
}

// The twiddles of the dense stage after this one (on 0: none).
struct NextTw {
  int on, ns, cnt, twstep;
  uint32_t nsinv, cntinv;
};
__device__ __forceinline__ NextTw next_tw(MixPlanPtr mp, int p, int twnext) {
  if (!twnext) return NextTw{0, 1, 1, 0, 0, 0};
  return NextTw{1, mp->st[p].ns, mp->st[p].cnt, mp->st[p].twstep, mp->st[p].nsinv, mp->st[p].cntinv};
}

// Twiddle exponent of a dense stage at natural position pos: m' * k' * twstep
// with pos = j' + m' * cnt, k' = j' mod ns.
__device__ __forceinline__ int dense_twiddle(const NextTw& s, int pos) {
  const int m = div_by(pos, s.cnt, s.cntinv);
  const int j = pos - m * s.cnt;
  const int k = s.ns > 1 ? fast_mod(j, s.ns, s.nsinv) : 0;
  return m * k * s.twstep;
}

// One stage of radix R.  A source gives src.at(line)(position), a sink takes
// snk.at(line)(position, value).
// Lanes run along the lines of a column tile and along the butterflies of a
// row tile, so both global sides are contiguous.
template <int R, int DIR, typename F, bool ROW, typename Src, typename Snk>
__device__ __forceinline__ void small_stage(const MixStage& s, const MixTile<F, ROW>& t, const FF_GLB cx<F>* tw,
                                            const Src& src, const Snk& snk) {
  const int items = s.cnt * t.T;
  for (int it = threadIdx.x; it < items; it += kMixThreads) {
    int line, j;
    if constexpr (ROW) {
      line = div_by(it, s.cnt, s.cntinv);
      j = it - line * s.cnt;
    } else {
      line = it & (t.T - 1);
      j = it >> t.lgT;
    }
    const auto from = src.at(line);
    const auto to = snk.at(line);
    cx<F> a[R];
#pragma unroll
    for (int m = 0; m < R; ++m) a[m] = from(j + m * s.cnt);
    int k = 0;
    if (s.ns > 1) {
      k = fast_mod(j, s.ns, s.nsinv);
      const int e = k * s.twstep;
#pragma unroll
      for (int m = 1; m < R; ++m) a[m] = twmul<DIR>(a[m], cx<F>(tw[m * e]));
    }
    mix_dft<R, DIR, F>(a);
    const int base = (j - k) * R + k;
#pragma unroll
    for (int m = 0; m < R; ++m) to(base + m * s.ns, a[m]);
  }
}

template <int DIR, typename F, bool ROW, typename Src, typename Snk>
__device__ __forceinline__ void any_small_stage(const MixStage& s, const MixTile<F, ROW>& t, const FF_GLB cx<F>* tw,
                                                const Src& src, const Snk& snk) {
  switch (s.R) {
    case 2: small_stage<2, DIR>(s, t, tw, src, snk); break;
    case 3: small_stage<3, DIR>(s, t, tw, src, snk); break;
    case 4: small_stage<4, DIR>(s, t, tw, src, snk); break;
    case 5: small_stage<5, DIR>(s, t, tw, src, snk); break;
    case 6: small_stage<6, DIR>(s, t, tw, src, snk); break;
    case 7: small_stage<7, DIR>(s, t, tw, src, snk); break;
    case 8: small_stage<8, DIR>(s, t, tw, src, snk); break;
    case 9: small_stage<9, DIR>(s, t, tw, src, snk); break;
    case 10: small_stage<10, DIR>(s, t, tw, src, snk); break;
    case 11: small_stage<11, DIR>(s, t, tw, src, snk); break;
    case 13: small_stage<13, DIR>(s, t, tw, src, snk); break;
    default: break;
  }
}

// The matrix product of four inner terms: 16 x 16 x 4, one k row by column
// lane; element v of the result is row acc_row(v, lane / 16), column lane % 16.
template <typename F>
struct MixAcc;
template <>
struct MixAcc<double> {
  typedef double V __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ V mfma(double a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int v, int g) { return 4 * v + g; }
};
template <>
struct MixAcc<float> {
  typedef float V __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ V mfma(float a, float b, V c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int v, int g) { return 4 * g + v; }
};

// The dense stage of prime radix D: for each butterfly the outputs k and D - k
// are P[k] -+ i Q[k] with P = x0 + C s, Q = S d, C and S the ((D+1)/2 x
// (D-1)/2) cosine and sine matrices and s, d the sums and differences of the
// inputs m and D - m: half the operations of the full matrix.  The product's
// columns are the real and imaginary parts of 8 (line, butterfly) pairs; the
// sine product's columns are fed the other part with the sign of -i, so P +- Q
// needs no exchange between lanes.  A wave takes KB tiles of 16 k for one block
// of 8 pairs, so the inputs are read once for all of them.  The matrix entries
// come from (cos, sin)(2 pi t / D), t = k m mod D, in LDS: a matrix in memory
// (D = 131: 87 KB for a tile of 17 KB) kept the kernel on its reads through L2.
// The sums are taken in chunks of 4 * kDenseChunk terms: one chain of N terms
// rounds N^2 / 2 times a term's square, chunks of c terms N c / 2 + N^2 / 2c (at
// 199 and above the plain chain was up to twice as far from the exact result as
// Bluestein's transforms).
// The sink takes snk.at(line)(position, part, value); the lanes of the two parts
// are neighbours.
constexpr int kDenseChunk = 4;

// Entry t of a table sits at tab_at(t): the 16 k of a product step by m entries,
// and a step that is a multiple of 2, 4, 8 or 16 would put them on few banks.
__device__ __forceinline__ int tab_at(int t) { return t ^ ((t >> 4) & 15); }

template <int KB, int DIR, typename F, bool ROW, typename Snk>
__device__ __forceinline__ void dense_tiles(const MixStage& s, const MixTile<F, ROW>& t, const cx<F>* tab,
                                            const Snk& snk) {
  using A = MixAcc<F>;
  const int D = s.R, H = (D - 1) / 2;
  const int lane = threadIdx.x & 63, g = lane >> 4, part = lane & 1;
  const int Q = s.cnt * t.T;
  const int blocks = (Q + 7) >> 3, groups = (s.ktiles + KB - 1) / KB;
  const int step = ROW ? s.cnt : s.cnt << t.lgT;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  for (int u = wave; u < blocks * groups; u += kMixThreads / 64) {
    const int cb = u / groups, kt = (u - cb * groups) * KB;
    const int q = cb * 8 + ((lane & 15) >> 1);
    const int qc = q < Q ? q : Q - 1;
    int line, j;
    if constexpr (ROW) {
      line = div_by(qc, s.cnt, s.cntinv);
      j = qc - line * s.cnt;
    } else {
      line = qc & (t.T - 1);
      j = qc >> t.lgT;
    }
    const cx<F>* x = t.buf + t.at(line, j);
    const F x0 = part ? x[0].y : x[0].x;
    typename A::V P[KB], S[KB];
    int e[KB], de[KB];  // k m mod D and its step over four m
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      P[b] = typename A::V{x0, x0, x0, x0};
      S[b] = typename A::V{F(0), F(0), F(0), F(0)};
      const int k = 16 * (kt + b) + (lane & 15);  // (rows past H are not stored)
      e[b] = fast_mod(k * (g + 1), D, s.rinv);
      de[b] = fast_mod(4 * k, D, s.rinv);
    }
    // m = 4 i + g + 1 in step i; the terms past H (at most seven, and the loads
    // one step ahead) stay within the line, D being 17 or more, and count as zero
    const cx<F>* lo = x + (g + 1) * step;
    const cx<F>* hi = x + (D - 1 - g) * step;
    cx<F> a = *lo, c = *hi, w[KB];
#pragma unroll
    for (int b = 0; b < KB; ++b) w[b] = tab[tab_at(e[b])];
    int left = H - 1 - g;
    for (int i = (H + 3) >> 2; i > 0; i -= kDenseChunk) {
      typename A::V p[KB], q[KB];
#pragma unroll
      for (int b = 0; b < KB; ++b) p[b] = q[b] = typename A::V{F(0), F(0), F(0), F(0)};
      for (int r = min(i, kDenseChunk); r > 0; --r, left -= 4) {
        F sum = part ? a.y + c.y : a.x + c.x, dif = part ? c.x - a.x : a.y - c.y;
        if (left < 0) sum = dif = F(0);
        cx<F> wn[KB];
        lo += 4 * step;
        hi -= 4 * step;
        a = *lo;
        c = *hi;
#pragma unroll
        for (int b = 0; b < KB; ++b) {
          e[b] += de[b];
          e[b] -= e[b] >= D ? D : 0;
          wn[b] = tab[tab_at(e[b])];
        }
#pragma unroll
        for (int b = 0; b < KB; ++b) {
          p[b] = A::mfma(w[b].x, sum, p[b]);
          q[b] = A::mfma(w[b].y, dif, q[b]);
          w[b] = wn[b];
        }
      }
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        P[b] += p[b];
        S[b] += q[b];
      }
    }
    const int kk = s.ns > 1 ? fast_mod(j, s.ns, s.nsinv) : 0;
    const int base = (j - kk) * D + kk;
    const auto to = snk.at(line);
#pragma unroll
    for (int b = 0; b < KB; ++b) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int k = 16 * (kt + b) + A::row(v, g);
        if (k <= H && q < Q) {
          const F plus = P[b][v] + S[b][v], minus = P[b][v] - S[b][v];
          to(base + k * s.ns, part, DIR < 0 ? plus : minus);
          if (k) to(base + (D - k) * s.ns, part, DIR < 0 ? minus : plus);
        }
      }
    }
  }
}

// One to three k tiles per wave: the split whose busiest wave has the fewest.
template <int DIR, typename F, bool ROW, typename Snk>
__device__ __forceinline__ void dense_stage(const MixStage& s, const MixTile<F, ROW>& t, const Snk& snk) {
  const cx<F>* tab = t.tab + s.ltab;
  constexpr int W = kMixThreads / 64;
  const int blocks = (s.cnt * t.T + 7) >> 3;
  const int t1 = (blocks * s.ktiles + W - 1) / W;
  const int t2 = (blocks * ((s.ktiles + 1) >> 1) + W - 1) / W * 2;
  const int t3 = (blocks * ((s.ktiles + 2) / 3) + W - 1) / W * 3;
  if (t3 <= t2 && t3 <= t1) dense_tiles<3, DIR, F, ROW>(s, t, tab, snk);
  else if (t2 <= t1) dense_tiles<2, DIR, F, ROW>(s, t, tab, snk);
  else dense_tiles<1, DIR, F, ROW>(s, t, tab, snk);
}

// The other part of a complex value held by two neighbouring lanes.
__device__ __forceinline__ float other_part(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));  // quad_perm 1,0,3,2
}
__device__ __forceinline__ double other_part(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0xB1, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Sources and sinks in LDS.
template <typename F, bool ROW>
struct LdsSrc {
  MixTile<F, ROW> t;
  struct Line {
    const cx<F>* p;
    int lg;
    __device__ __forceinline__ cx<F> operator()(int pos) const { return p[ROW ? pos : pos << lg]; }
  };
  __device__ __forceinline__ Line at(int line) const { return Line{t.buf + t.at(line, 0), t.lgT}; }
};

// next: the stage after this one where it is dense (its twiddles are applied
// here: a dense stage reads every input once per pair of k tiles).
template <int DIR, typename F, bool ROW>
struct LdsSnk {
  MixTile<F, ROW> t;
  NextTw next;
  const FF_GLB cx<F>* tw;
  struct Line {
    cx<F>* p;
    int lg;
    NextTw next;
    const FF_GLB cx<F>* tw;
    __device__ __forceinline__ void operator()(int pos, cx<F> v) const {
      if (next.on) v = twmul<DIR>(v, cx<F>(tw[dense_twiddle(next, pos)]));
      p[ROW ? pos : pos << lg] = v;
    }
    __device__ __forceinline__ void operator()(int pos, int part, F v) const {
      if (next.on) {
        const cx<F> w = tw[dense_twiddle(next, pos)];
        const F o = other_part(v);
        // forward: x wx - y wy, y wx + x wy; inverse: x wx + y wy, y wx - x wy
        const bool minus = (part == 0) == (DIR < 0);
        v = minus ? fmadd(v, w.x, -(o * w.y)) : fmadd(v, w.x, o * w.y);
      }
      reinterpret_cast<F*>(p + (ROW ? pos : pos << lg))[part] = v;
    }
  };
  __device__ __forceinline__ Line at(int line) const {
    return Line{t.buf + t.at(line, 0), t.lgT, next, tw};
  }
};

// The tile of buffer b.
template <typename F, bool ROW>
__device__ __forceinline__ MixTile<F, ROW> mix_tile(cx<F>* lds, int b, int stride, int T, int lgT, int pitch,
                                                    const cx<F>* tab) {
  return MixTile<F, ROW>{lds + b * stride, T, lgT, pitch, tab};
}

// Runs stages [p0, np) of the transform of the lines in buffer b, the last one
// into snk.  Barriers: one per stage (two buffers in turn).
template <int DIR, typename F, bool ROW, typename Snk>
__device__ __forceinline__ void mix_stages(MixPlanPtr mp, int p0, cx<F>* lds, int& b, int stride, int T, int lgT,
                                           int pitch, const FF_GLB cx<F>* tw, const cx<F>* tab, const Snk& snk) {
  for (int p = p0; p < mp->np; ++p) {
    const MixStage s = mix_stage(mp, p);
    const MixTile<F, ROW> t = mix_tile<F, ROW>(lds, b, stride, T, lgT, pitch, tab);
    const LdsSrc<F, ROW> src{t};
    if (p + 1 == mp->np) {
      if (s.dense) dense_stage<DIR, F, ROW>(s, t, snk);
      else any_small_stage<DIR, F, ROW>(s, t, tw, src, snk);
    } else {
      const LdsSnk<DIR, F, ROW> to{mix_tile<F, ROW>(lds, b ^ 1, stride, T, lgT, pitch, tab),
                                   next_tw(mp, p + 1, s.twnext), tw};
      if (s.dense) dense_stage<DIR, F, ROW>(s, t, to);
      else any_small_stage<DIR, F, ROW>(s, t, tw, src, to);
      b ^= 1;
      __syncthreads();
    }
  }
}

// Calls fn(line, position) for n positions of T lines (ninv: ceil(2^32 / n)),
// neighbouring lanes on neighbouring positions.
template <typename Fn>
__device__ __forceinline__ void each_line(int T, int n, uint32_t ninv, const Fn& fn) {
  for (int it = threadIdx.x; it < n * T; it += kMixThreads) {
    const int line = div_by(it, n, ninv);
    fn(line, it - line * n);
  }
}

// load(item) -> store(item, value) over the items, four loads ahead of their
// stores: an item at a time waits for memory once per item.
template <typename Load, typename Store>
__device__ __forceinline__ void copy_items(int items, const Load& load, const Store& store) {
  for (int it = threadIdx.x; it < items; it += 4 * kMixThreads) {
    decltype(load(0)) v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = load(min(it + q * kMixThreads, items - 1));
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (it + q * kMixThreads < items) store(it + q * kMixThreads, v[q]);
  }
}

// The dense stages' tables to LDS (complete after the next barrier).
template <typename F>
__device__ __forceinline__ void load_tables(MixPlanPtr mp, const void* plan, cx<F>* tab) {
  const FF_GLB cx<F>* src = glb<const cx<F>>(static_cast<const unsigned char*>(plan) + mp->tables);
  const int n = mp->ntab;
  for (int e = threadIdx.x; e < n; e += kMixThreads) tab[e] = src[e];  // (stored in tab_at order)
}

// The first stage, from src into buffer b, or, where that stage is dense or
// the only one, a copy of the line; returns the stages done.
template <int DIR, typename F, bool ROW, typename Src>
__device__ __forceinline__ int mix_first(MixPlanPtr mp, cx<F>* lds, int b, int stride, int T, int lgT, int pitch,
                                         const FF_GLB cx<F>* tw, const cx<F>* tab, const Src& src) {
  const MixTile<F, ROW> t = mix_tile<F, ROW>(lds, b, stride, T, lgT, pitch, tab);
  const MixStage s = mix_stage(mp, 0);
  if (mp->np == 1 || s.dense) {
    if constexpr (ROW) {
      const uint32_t ninv = mp->ninv;
      const int n = mp->n;
      auto where = [n, ninv](int it, int& line) {
        line = div_by(it, n, ninv);
        return it - line * n;
      };
      copy_items(
          n * T,
          [&](int it) {
            int line;
            const int pos = where(it, line);
            return src.at(line)(pos);
          },
          [&](int it, cx<F> v) {
            int line;
            const int pos = where(it, line);
            t.buf[t.at(line, pos)] = v;
          });
    } else {
      copy_items(
          mp->n * T, [&](int it) { return src.at(it & (T - 1))(it >> lgT); },
          [&](int it, cx<F> v) { t.buf[it] = v; });  // [position][line]
    }
    __syncthreads();
    return 0;
  }
  const LdsSnk<DIR, F, ROW> to{t, next_tw(mp, 1, s.twnext), tw};
  any_small_stage<DIR, F, ROW>(s, t, tw, src, to);
  __syncthreads();
  return 1;
}

// ---------------------------------------------------------------------------
// Column passes.

template <typename F>
struct ColSrc {
  const FF_GLB cx<F>* src;
  SpecSide in;
  int outer, col0, ncols;
  __device__ __forceinline__ auto at(int line) const {
    const int col = col0 + line;
    long long base, step;
    // columns past the plane load its last one (never stored)
    side_addr(in, outer, col < ncols ? col : ncols - 1, 0, 1, base, step);
    const FF_GLB cx<F>* p = src + base;
    return [p, step](int pos) { return cx<F>(p[pos * step]); };
  }
};

template <typename F>
struct ColSnk {
  FF_GLB cx<F>* dst;
  SpecSide out;
  int outer, col0, ncols;
  struct Line {
    FF_GLB cx<F>* p;
    long long step;
    bool ok;
    __device__ __forceinline__ void operator()(int pos, cx<F> v) const {
      if (ok) p[pos * step] = v;
    }
    __device__ __forceinline__ void operator()(int pos, int part, F v) const {
      if (ok) ((FF_GLB F*)(p + pos * step))[part] = v;
    }
  };
  __device__ __forceinline__ Line at(int line) const {
    const int col = col0 + line;
    long long base, step;
    side_addr(out, outer, col < ncols ? col : ncols - 1, 0, 1, base, step);
    return Line{dst + base, step, col < ncols};
  }
};

// The spectral filter of ParisPencil.cpp:269-284 (or its symbol, or the
// finite-difference one) between the transforms of the x pass, in the same
// operations as the register engine's (col_line in ff_kernels.hpp).
template <typename F, int MODE>
struct FilterSnk {
  MixTile<F, false> t;
  int outer, col0, ncols, cols_j, nx, ny;
  double ddi, ddj, ddk;
  const FF_GLB double *symx, *symy, *symz;
  FF_GLB double* dc;
  int dc_add;
  struct Line {
    cx<F>* p;
    int lg, jk, nx;       // jk: j | kh
    double dj, dk, ddi;   // spectral: (j dd)^2 and kh dd; finite differences: the j and kh terms' factors
    double ddk;
    const FF_GLB double* symx;
    FF_GLB double* dc;
    int dc_add;
    __device__ __forceinline__ F factor(int ii) const {
      if constexpr (MODE == COL_FILTER_FD) {
        const double s2 = fmadd(dk, ddk, fmadd(symx[ii], ddi, dj));
        return F((ii | jk) ? -1.0 / s2 : 0.0);
      } else {
        const double di = double(ii < nx - ii ? ii : nx - ii) * ddi;
        const double s2 = fmadd(dk, dk, fmadd(di, di, dj));
        if constexpr (MODE == COL_FILTER) return F((ii | jk) ? -1.0 / s2 : 0.0);
        else return F(-s2);
      }
    }
    // the (0,0,0) term before the multiply is the sum of the input field
    __device__ __forceinline__ void put_dc(F v) const { *dc = std::is_same<F, float>::value && dc_add ? *dc + double(v) : double(v); }
    __device__ __forceinline__ void operator()(int pos, cx<F> v) const {
      const F d = factor(pos);
      if (dc && !(pos | jk)) put_dc(v.x);
      p[pos << lg] = cx<F>{d * v.x, d * v.y};
    }
    __device__ __forceinline__ void operator()(int pos, int part, F v) const {
      const F d = factor(pos);
      if (dc && !(pos | jk | part)) put_dc(v);
      reinterpret_cast<F*>(p + (pos << lg))[part] = d * v;
    }
  };
  __device__ __forceinline__ Line at(int line) const {
    // (columns past the plane take its last one's symbol)
    const int col = col0 + line < ncols ? col0 + line : ncols - 1;
    const int jj = cols_j ? col : outer, kk = cols_j ? outer : col;
    Line l;
    l.p = t.buf + t.at(line, 0);
    l.lg = t.lgT;
    l.jk = jj | kk;
    l.nx = nx;
    l.ddi = ddi;
    l.ddk = ddk;
    l.dc = dc;
    l.dc_add = dc_add;
    l.symx = symx;
    if constexpr (MODE == COL_FILTER_FD) {
      l.dj = symy[jj] * ddj;
      l.dk = symz[kk];
    } else {
      l.dj = sqr(double(jj < ny - jj ? jj : ny - jj) * ddj);
      l.dk = double(kk) * ddk;
    }
    return l;
  }
};

// A workgroup owns T neighbouring columns of one plane.  An in-place pass is
// safe: a tile's columns are in LDS before the first of them is stored.
template <typename F, int MODE>
__global__ __launch_bounds__(kMixThreads) void k_mix_col(const ColArgs a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cx<F>* lds = reinterpret_cast<cx<F>*>(smem_raw);
  const MixPlanPtr mp = (MixPlanPtr)(a.mix);
  const PassInst io = inst_of(a);
  const int blk = xcd_remap(blockIdx.x, a.nblocks);
  const int outer = blk / a.tiles, col0 = (blk - outer * a.tiles) * a.T;
  const FF_GLB cx<F>* tw = glb<const cx<F>>(a.tw);
  const int stride = mp->n * a.T;
  cx<F>* tab = lds + a.nbuf * stride;
  load_tables(mp, a.mix, tab);
  const ColSrc<F> src{glb<const cx<F>>(io.src), a.in, outer, col0, a.ncols};
  const ColSnk<F> snk{glb<cx<F>>(io.dst), a.out, outer, col0, a.ncols};
  int b = 0;
  if constexpr (MODE == COL_INV) {
    const int p = mix_first<+1, F, false>(mp, lds, b, stride, a.T, a.lgT, 0, tw, tab, src);
    mix_stages<+1, F, false>(mp, p, lds, b, stride, a.T, a.lgT, 0, tw, tab, snk);
  } else {
    const int p = mix_first<-1, F, false>(mp, lds, b, stride, a.T, a.lgT, 0, tw, tab, src);
    if constexpr (MODE == COL_FWD) {
      mix_stages<-1, F, false>(mp, p, lds, b, stride, a.T, a.lgT, 0, tw, tab, snk);
    } else {
      // the filtered spectrum lands in the buffer the last stage does not read
      const int last = (mp->np - 1 - p) & 1 ? b ^ 1 : b;
      const FilterSnk<F, MODE> filter{mix_tile<F, false>(lds, last ^ 1, stride, a.T, a.lgT, 0, tab),
                                      outer, col0, a.ncols, a.cols_j, a.nx, a.ny, io.ddi, io.ddj, io.ddk,
                                      glb<const double>(a.symx), glb<const double>(a.symy),
                                      glb<const double>(a.symz), glb<double>(io.dc_out), a.dc_add};
      mix_stages<-1, F, false>(mp, p, lds, b, stride, a.T, a.lgT, 0, tw, tab, filter);
      __syncthreads();
      b = last ^ 1;
      mix_stages<+1, F, false>(mp, 0, lds, b, stride, a.T, a.lgT, 0, tw, tab, snk);
    }
  }
}

// ---------------------------------------------------------------------------
// Row passes.  Even nz: a line is a row packed as nz/2 complex values.  Odd nz:
// a line is two neighbouring rows of one plane, x1 + i x2, whose spectra are
// X1[k], X2[k] = (Z[k] + conj Z[n-k]) / 2, (Z[k] - conj Z[n-k]) / 2i: half the
// lines of transforming each row on its own.  With ny odd a plane's last row
// is paired with zeros.

// The lines of a workgroup and their rows.  Lines past the end take the last one
// (in bounds, never stored).  Odd nz: line l is pair l % hy of plane l / hy (hy
// pairs to a plane); the tile's first line is split once, the others by 32-bit
// steps from it.
template <bool ODD>
struct RowLines {
  long long line0, nlines, row0;  // row0: first row of the plane of line0 (odd nz)
  int pair0, ny, hy;
  uint32_t hyinv;
  __device__ __forceinline__ RowLines(const RowArgs& a, long long first) : line0(first), nlines(a.nlines), ny(a.ny) {
    if constexpr (ODD) {
      hy = (ny + 1) >> 1;
      hyinv = a.hyinv;
      const long long i = line0 / hy;
      pair0 = (int)(line0 - i * hy);
      row0 = i * ny;
    }
  }
  __device__ __forceinline__ bool have(int line) const { return line0 + line < nlines; }
  // first row of a line; two: a second one follows
  __device__ __forceinline__ long long row(int line, bool& two) const {
    const int last = (int)min(nlines - 1 - line0, (long long)65535);
    line = line < last ? line : last;
    if constexpr (!ODD) {
      two = false;
      return line0 + line;
    } else {
      const int q = pair0 + line;
      const int up = div_by(q, hy, hyinv);
      const int jp = 2 * (q - up * hy);
      two = jp + 1 < ny;
      return row0 + (long long)up * ny + jp;
    }
  }
};

template <typename F, typename IN, bool ODD>
struct RowSrc {
  const FF_GLB IN* src;
  int nz;
  RowLines<ODD> rows;
  struct Line {
    const FF_GLB IN* p;
    int nz;
    bool two;
    __device__ __forceinline__ cx<F> operator()(int pos) const {
      if constexpr (!ODD) {
        const cx<IN> v = ((const FF_GLB cx<IN>*)p)[pos];
        return cx<F>{F(v.x), F(v.y)};
      } else {
        return cx<F>{F(p[pos]), two ? F(p[nz + pos]) : F(0)};
      }
    }
  };
  __device__ __forceinline__ Line at(int line) const {
    Line l;
    l.p = src + rows.row(line, l.two) * nz;
    l.nz = nz;
    return l;
  }
};

template <typename F, typename IN, bool ODD>
__global__ __launch_bounds__(kMixThreads) void k_mix_r2c(const RowArgs a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cx<F>* lds = reinterpret_cast<cx<F>*>(smem_raw);
  const MixPlanPtr mp = (MixPlanPtr)(a.mix);
  const PassInst io = inst_of(a);
  const int n = mp->n, T = a.T, pitch = a.pitch, stride = T * pitch;
  const long long line0 = (long long)xcd_remap(blockIdx.x, a.nblocks) * T;
  const RowLines<ODD> rows(a, line0);
  cx<F>* tab = lds + 2 * stride;
  load_tables(mp, a.mix, tab);
  const FF_GLB cx<F>* tw = glb<const cx<F>>(a.tw);
  const RowSrc<F, IN, ODD> src{glb<const IN>(io.src), a.nz, rows};
  int b = 0;
  const int p = mix_first<-1, F, true>(mp, lds, b, stride, T, 0, pitch, tw, tab, src);
  // the spectrum, in natural order, in the buffer the last stage does not read
  const int out = ((mp->np - 1 - p) & 1 ? b ^ 1 : b) ^ 1;
  const MixTile<F, true> z = mix_tile<F, true>(lds, out, stride, T, 0, pitch, tab);
  const LdsSnk<-1, F, true> to{z, NextTw{0, 1, 1, 0, 0, 0}, tw};
  mix_stages<-1, F, true>(mp, p, lds, b, stride, T, 0, pitch, tw, tab, to);
  __syncthreads();
  const FF_GLB cx<F>* twp = glb<const cx<F>>(a.twpost);
  // the half spectra: outputs k and n - k of an even row come from the same two
  // values
  each_line(T, ODD ? a.nh : n / 2 + 1, a.Linv, [&](int line, int k) {
    if (!rows.have(line)) return;
    bool two;
    const long long row = rows.row(line, two);
    FF_GLB cx<F>* dst = glb<cx<F>>(io.dst) + row * a.nh;
    const cx<F>* zl = z.buf + line * pitch;
    const cx<F> zk = zl[k], zn = zl[k ? n - k : 0];
    if constexpr (!ODD) {
      auto half = [](cx<F> p, cx<F> q, cx<F> w) {
        const cx<F> m = conj(q);
        const cx<F> ev = {F(0.5) * (p.x + m.x), F(0.5) * (p.y + m.y)};
        const cx<F> od = {F(0.5) * (p.y - m.y), F(-0.5) * (p.x - m.x)};
        return ev + twmul<-1>(od, w);
      };
      dst[k] = half(zk, zn, cx<F>(twp[k]));
      if (k == 0) dst[n] = cx<F>{zk.x - zk.y, F(0)};
      else if (k != n - k) dst[n - k] = half(zn, zk, cx<F>(twp[n - k]));
    } else {
      const cx<F> zm = conj(zn);
      dst[k] = cx<F>{F(0.5) * (zk.x + zm.x), F(0.5) * (zk.y + zm.y)};
      if (two) dst[a.nh + k] = cx<F>{F(0.5) * (zk.y - zm.y), F(-0.5) * (zk.x - zm.x)};
    }
  });
}

// The z inverse's epilogue at position pos of a line.
template <typename OUT, bool ODD, int EPI>
struct RowSnk {
  FF_GLB OUT* out;
  const FF_GLB double* f;
  int nz;
  RowLines<ODD> rows;
  double scale, shift;
  template <typename F>
  __device__ __forceinline__ void operator()(int line, int pos, cx<F> v) const {
    if (!rows.have(line)) return;
    bool two;
    const long long off = rows.row(line, two) * nz;
    const FF_GLB double* fr = EPI == EPI_RESIDUAL ? f + off : f;
    if constexpr (!ODD) {
      c2r_out2<EPI, OUT>(out + off, fr, pos, double(v.x), double(v.y), scale, shift);
    } else {
      c2r_out1<EPI, OUT>(out + off, fr, pos, double(v.x), scale, shift);
      if (two) c2r_out1<EPI, OUT>(out + off, fr, nz + pos, double(v.y), scale, shift);
    }
  }
};

template <typename F, typename OUT, bool ODD, int EPI>
__global__ __launch_bounds__(kMixThreads) void k_mix_c2r(const RowArgs a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cx<F>* lds = reinterpret_cast<cx<F>*>(smem_raw);
  const MixPlanPtr mp = (MixPlanPtr)(a.mix);
  const PassInst io = inst_of(a);
  const int n = mp->n, T = a.T, pitch = a.pitch, stride = T * pitch, nh = a.nh, ny = a.ny;
  const long long line0 = (long long)xcd_remap(blockIdx.x, a.nblocks) * T;
  const RowLines<ODD> rows(a, line0);
  cx<F>* tab = lds + 2 * stride;
  load_tables(mp, a.mix, tab);
  const FF_GLB cx<F>* tw = glb<const cx<F>>(a.tw);
  const FF_GLB cx<F>* src = glb<const cx<F>>(io.src);
  // the packed lines merged from the half spectra into buffer 0: positions k
  // and n - k from the entries k and n - k of an even row, or the entries k of
  // the two rows of a pair (a missing second row is zero).  Im of the DC and
  // Nyquist terms is ignored.
  const FF_GLB cx<F>* twp = glb<const cx<F>>(a.twpost);
  struct Two {
    cx<F> a, b;
  };
  const int per = ODD ? nh : n / 2 + 1;
  const int lgKT = a.spec.lgKT, KT = lgKT < 30 ? 1 << lgKT : 0;
  auto entry = [&](long long row, int k) -> cx<F> {
    if (lgKT >= 30) return src[row * nh + k];
    if (lgKT == 0) {
      const long long i = row / ny;
      return src[i * a.spec.fo + (row - i * ny) * a.spec.fr + (long long)k * a.spec.KS];
    }
    const int kb = k >> lgKT;
    return src[(long long)kb * a.spec.KS + row * (kb == a.spec.nb - 1 ? a.spec.Wlast : KT) + (k & (KT - 1))];
  };
  // lanes run along a plain row, and along the lines of a strided or blocked
  // spectrum, whose rows are contiguous for each kh
  const int lgT = a.lgT;
  const uint32_t perinv = a.Linv;
  auto where = [&](int it, int& line) {
    if (lgKT < 30) {
      line = it & (T - 1);
      return it >> lgT;
    }
    line = div_by(it, per, perinv);
    return it - line * per;
  };
  copy_items(
      per * T,
      [&](int it) {
        int line;
        const int k = where(it, line);
        bool two;
        const long long row = rows.row(line, two);
        Two v{entry(row, k), cx<F>{F(0), F(0)}};
        if constexpr (!ODD) v.b = entry(row, n - k);
        else if (two) v.b = entry(row + 1, k);
        return v;
      },
      [&](int it, Two v) {
        int line;
        const int k = where(it, line);
        cx<F>* zl = lds + line * pitch;
        if (k == 0) v.a.y = F(0), v.b.y = F(0);
        if constexpr (!ODD) {
          auto merge = [](cx<F> xk, cx<F> xm, cx<F> w) {
            const cx<F> cm = conj(xm);
            const cx<F> A = xk + cm;
            const cx<F> B = twmul<+1>(xk - cm, w);
            return cx<F>{A.x - B.y, A.y + B.x};
          };
          zl[k] = merge(v.a, v.b, cx<F>(twp[k]));
          if (k && k != n - k) zl[n - k] = merge(v.b, v.a, cx<F>(twp[n - k]));
        } else {
          zl[k] = cx<F>{v.a.x - v.b.y, v.a.y + v.b.x};
          if (k) zl[n - k] = cx<F>{v.a.x + v.b.y, v.b.x - v.a.y};
        }
      });
  __syncthreads();
  int b = 0;
  const int p = 0;
  const double shift = io.shiftp ? a.shift * *glb<const double>(io.shiftp) : a.shift;
  const RowSnk<OUT, ODD, EPI> snk{glb<OUT>(io.dst), glb<const double>(io.aux), a.nz, rows, a.scale, shift};
  // the last stage into LDS, then the rows whole
  const int out = ((mp->np - 1 - p) & 1 ? b ^ 1 : b) ^ 1;
  const MixTile<F, true> z = mix_tile<F, true>(lds, out, stride, T, 0, pitch, tab);
  const LdsSnk<+1, F, true> to{z, NextTw{0, 1, 1, 0, 0, 0}, tw};
  mix_stages<+1, F, true>(mp, p, lds, b, stride, T, 0, pitch, tw, tab, to);
  __syncthreads();
  each_line(T, n, mp->ninv, [&](int line, int pos) { snk(line, pos, z.buf[line * pitch + pos]); });
}

// ---------------------------------------------------------------------------
// Launchers.

[[maybe_unused]] static hipError_t mix_launch(const void* fn, const Launch& l, const void* args) {
  if (!fn) return hipErrorInvalidValue;
  if (l.lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l.lds);
    if (e != hipSuccess) return e;
  }
  void* argv[] = {const_cast<void*>(args)};
  return hipLaunchKernel(fn, l.grid, l.block, argv, l.lds, l.stream);
}

#if FF_MIX_PART == 0
const void* mix_col_f64(int mode) {
  switch (mode) {
    case COL_FWD: return (const void*)&k_mix_col<double, COL_FWD>;
    case COL_INV: return (const void*)&k_mix_col<double, COL_INV>;
    default: return nullptr;
  }
}
#elif FF_MIX_PART == 1
const void* mix_col_f64x(int mode) {
  switch (mode) {
    case COL_FILTER: return (const void*)&k_mix_col<double, COL_FILTER>;
    case COL_SYMBOL: return (const void*)&k_mix_col<double, COL_SYMBOL>;
    case COL_FILTER_FD: return (const void*)&k_mix_col<double, COL_FILTER_FD>;
    default: return nullptr;
  }
}
#elif FF_MIX_PART == 2
const void* mix_col_f32(int mode) {
  switch (mode) {
    case COL_FWD: return (const void*)&k_mix_col<float, COL_FWD>;
    case COL_INV: return (const void*)&k_mix_col<float, COL_INV>;
    case COL_FILTER: return (const void*)&k_mix_col<float, COL_FILTER>;
    case COL_FILTER_FD: return (const void*)&k_mix_col<float, COL_FILTER_FD>;
    default: return nullptr;
  }
}
#elif FF_MIX_PART == 3
template <bool ODD>
static const void* r2c_of(int f32, int in_f32) {
  if (!f32) return in_f32 ? nullptr : (const void*)&k_mix_r2c<double, double, ODD>;
  return in_f32 ? (const void*)&k_mix_r2c<float, float, ODD> : (const void*)&k_mix_r2c<float, double, ODD>;
}
hipError_t mix_r2c(int f32, int in_f32, int odd, const Launch& l, const RowArgs& a) {
  return mix_launch(odd ? r2c_of<true>(f32, in_f32) : r2c_of<false>(f32, in_f32), l, &a);
}
#elif FF_MIX_PART == 4
template <bool ODD>
static const void* c2r_of(int f32, int out_kind, int epi) {
  if (!f32) {
    if (epi == EPI_STORE && out_kind == 0) return (const void*)&k_mix_c2r<double, double, ODD, EPI_STORE>;
    if (epi == EPI_RESIDUAL && out_kind == 1) return (const void*)&k_mix_c2r<double, float, ODD, EPI_RESIDUAL>;
    if (epi == EPI_RESIDUAL && out_kind == 0) return (const void*)&k_mix_c2r<double, double, ODD, EPI_RESIDUAL>;
    return nullptr;
  }
  if (epi == EPI_STORE && out_kind == 0) return (const void*)&k_mix_c2r<float, double, ODD, EPI_STORE>;
  if (epi == EPI_ACCUM && out_kind == 0) return (const void*)&k_mix_c2r<float, double, ODD, EPI_ACCUM>;
  return nullptr;
}
hipError_t mix_c2r(int f32, int out_kind, int odd, int epi, const Launch& l, const RowArgs& a) {
  return mix_launch(odd ? c2r_of<true>(f32, out_kind, epi) : c2r_of<false>(f32, out_kind, epi), l, &a);
}
#else
const void* mix_col_f64(int mode);
const void* mix_col_f64x(int mode);
const void* mix_col_f32(int mode);
hipError_t mix_col(int f32, int mode, const Launch& l, const ColArgs& a) {
  const bool x = mode != COL_FWD && mode != COL_INV;
  return mix_launch(f32 ? mix_col_f32(mode) : x ? mix_col_f64x(mode) : mix_col_f64(mode), l, &a);
}
#endif

}  // namespace ff
