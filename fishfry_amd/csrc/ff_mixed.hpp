// Line transforms of lengths with prime factors above 5, and of odd-length
// rows in pairs: plan and launchers of the mixed-radix pass kernels
// (ff_mixed.hip).
//
// The register engine (ff_fft.hpp) needs every radix to divide its elements
// per thread, so it takes lengths 2^a 3^b 5^c only and every other one as a
// convolution of at least twice the length (Bluestein).  Here a line
// stays in LDS and every stage is a Stockham pass of its own radix R: n/R
// butterflies, spread over the workgroup's threads, read from one LDS buffer
// and written autosorted to the other.  Radices up to 13 are butterflies
// in registers; a prime factor D above 13 is a dense stage, the DFT matrix of
// length D on the matrix cores.
#pragma once

#include <vector>

#include "ff_kernels.hpp"

namespace ff {

struct LineCfg;

constexpr int kMixStages = 10;
constexpr int kMixThreads = 256;

struct MixStage {
  int R;            // radix
  int dense;        // the DFT matrix of length R on the matrix cores
  int ns;           // product of the radices before
  int cnt;          // n / R butterflies per line
  uint32_t nsinv;   // ceil(2^32 / ns) (ns > 1): exact j / ns for j, ns < 2^16
  uint32_t cntinv;  // ceil(2^32 / cnt) (cnt > 1)
  int twstep;       // n / (ns * R)
  int twnext;       // the next stage is dense: this one multiplies its outputs by that stage's twiddles
  int ktiles;       // dense: 16-row tiles over k = 0 .. (R-1)/2
  uint32_t rinv;    // dense: ceil(2^32 / R)
  int ltab;         // dense: offset of its (cos, sin)(2 pi t / R), t < R, in the tables
};

struct MixPlan {
  int n, np;
  uint32_t ninv;  // ceil(2^32 / n)
  int ntab;       // complex entries of the dense stages' tables
  int tables;     // their byte offset from the plan
  MixStage st[kMixStages];  // ascending ns; dense stages last
};

// A pass over lines of n: lines per workgroup, LDS buffers and bytes.
struct MixCfg {
  const void* plan = nullptr;  // MixPlan in device memory; null: the pass runs the register engine
  const void* tw = nullptr;    // W_n, t < n
  int n = 0, T = 0, lgT = 0, bufs = 0;
  size_t lds = 0;
};

// The number of LDS buffers a pass ping-pongs between: one where a single
// exchange separates its stages.
constexpr int mix_buffers(int exchanges) { return exchanges > 1 ? 2 : 1; }

// Row buffers hold a line, or the half spectra staged for it, at a pitch that
// is odd in complex elements.
constexpr int mix_row_pitch(int n) { return (n + 2) | 1; }

// Largest dense radix: its n^2 work against Bluestein's two transforms of 2n and
// more, for rows in pairs twice as many of those (measured on MI355X, whole
// solves with one such axis, register engine / here: FP64 199 1.06-1.21, 251
// 0.92-0.95, 509 0.55-0.8, in pairs 283 1.31, 307 0.72; FP32 283 1.4-1.6, 307
// 0.8-0.9, in pairs 401 1.9, 509 1.14).
constexpr int mix_max_dense(int prec, bool pairs) { return pairs ? (prec ? 420 : 300) : (prec ? 300 : 200); }
constexpr int kMixMaxDense = 420;
// The stages' radices of length n, the fewest, dense ones last; empty where
// there are none: n < 2, or a prime factor above kMixMaxDense.
std::vector<int> mix_radices(int n);
// The plan and tile of a pass of kind 1 (y columns), 2 (x columns), 0 (z forward
// rows) or 3 (z inverse rows) over lines of n, with its tables resident on the
// current device; ncols: the lines of a plane (columns); pairs: rows of odd nz,
// two to a line; lines: all the lines of the pass; engine: the register engine's
// line.  False where the length has no plan, no tile fits the LDS, the engine is the
// faster one, or a table could not be allocated.
bool mix_cfg(int n, int prec, int kind, int ncols, bool pairs, long long lines, const LineCfg& engine, MixCfg& out);

hipError_t mix_col(int f32, int mode, const Launch& l, const ColArgs& a);
hipError_t mix_r2c(int f32, int in_f32, int odd, const Launch& l, const RowArgs& a);
hipError_t mix_c2r(int f32, int out_kind, int odd, int epi, const Launch& l, const RowArgs& a);

}  // namespace ff
