// Host side of the mixed-radix passes: radices, device plans with their dense
// tables, and tiles.
#include <algorithm>
#include <cstring>

#include "ff_internal.hpp"
#include "ff_mixed.hpp"

namespace ff {

namespace {

constexpr int kMixRadices[] = {13, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// The fewest stages for m (prime factors up to 13), largest radices first.
int fewest_stages(int m, std::vector<int>& best) {
  if (m == 1) {
    best.clear();
    return 0;
  }
  int found = 1 << 20;
  for (int R : kMixRadices) {
    if (m % R) continue;
    std::vector<int> rest;
    const int k = fewest_stages(m / R, rest) + 1;
    if (k < found) {
      found = k;
      best = rest;
      best.push_back(R);
    }
  }
  return found;
}

uint32_t magic(int v) { return v > 1 ? (uint32_t)(((1ull << 32) + (uint64_t)v - 1) / (uint64_t)v) : 0u; }

}  // namespace

std::vector<int> mix_radices(int n) {
  if (n < 2) return {};
  // factors up to 13 are butterflies; what is left once they are out has only prime
  // factors from 17 on, which trial division finds in ascending order
  std::vector<int> dense, small;
  int m = 1, rest = n;
  for (int p : {2, 3, 5, 7, 11, 13}) {
    while (rest % p == 0) {
      rest /= p;
      m *= p;
    }
  }
  for (int p = 17; (long long)p * p <= rest; p += 2) {
    while (rest % p == 0) {
      dense.push_back(p);
      rest /= p;
    }
  }
  if (rest > 1) dense.push_back(rest);
  if (!dense.empty() && dense.back() > kMixMaxDense) return {};
  fewest_stages(m, small);
  std::sort(small.begin(), small.end(), [](int a, int b) { return a > b; });
  small.insert(small.end(), dense.begin(), dense.end());
  if ((int)small.size() > kMixStages) small.clear();
  return small;
}

static void build_plan(int n, int prec, std::vector<unsigned char>& buf) {
  const std::vector<int> rs = mix_radices(n);
  MixPlan mp;
  memset(&mp, 0, sizeof mp);
  mp.n = n;
  mp.np = (int)rs.size();
  mp.ninv = magic(n);
  buf.assign((sizeof(MixPlan) + 255) / 256 * 256, 0);
  mp.tables = (int)buf.size();
  int ns = 1;
  for (int p = 0; p < mp.np; ++p) {
    MixStage& s = mp.st[p];
    s.R = rs[p];
    s.dense = rs[p] > 13;
    s.ns = ns;
    s.cnt = n / rs[p];
    s.nsinv = magic(ns);
    s.cntinv = magic(s.cnt);
    s.twstep = n / (ns * rs[p]);
    s.twnext = p + 1 < mp.np && rs[p + 1] > 13;
    if (s.dense) {
      const int R = s.R;
      s.ktiles = ((R - 1) / 2 + 16) / 16;  // k = 0 .. (R-1)/2
      s.rinv = magic(R);
      s.ltab = mp.ntab;
      mp.ntab += (R + 15) / 16 * 16;  // (swizzled in blocks of 16)
      const size_t elem = prec ? 8 : 16;
      const size_t base = buf.size();
      buf.resize(base + (size_t)(R + 15) / 16 * 16 * elem);
      for (int t = 0; t < R; ++t) {
        long double c, sn;
        twiddle_ld(t, R, c, sn);
        const size_t at = base + (size_t)(t ^ ((t >> 4) & 15)) * elem;  // tab_at of ff_mixed.hip
        if (prec) {
          const float v[2] = {(float)c, (float)-sn};
          memcpy(&buf[at], v, sizeof v);
        } else {
          const double v[2] = {(double)c, (double)-sn};
          memcpy(&buf[at], v, sizeof v);
        }
      }
    }
    ns *= rs[p];
  }
  memcpy(buf.data(), &mp, sizeof mp);
}

// Whether Bluestein's transforms in the register engine (line e) are the faster ones
// for a pass of so many tiles.  A tile's own time counts where the tiles do not fill
// the chip: eight lines by 256 threads take n * (radices) steps, the engine's up
// to 512 threads and more the same few passes for every n up to the next engine length.
// Measured (MI355X; engine and mixed radices; about 150 tiles, and 1000 or more):
//   FP32 + 1 step 969x20x60  271 and 387 us, 566 213 and 270, 493 177 and 221, 731 303 and 304;
//     at 64x256 columns 493 and 566 are 0.6-0.9 of the engine, 969 1.15 of it
//   FP64 y passes 398  15.3 and 20.7 us, 501 16.1 and 24.9 (large: 0.3-1.1 of the engine),
//     969 200 and 251 us at 64x256
//   FP64 odd rows 283 of 768 rows  12.8 and 18.6 us, of 12288 0.4 of the engine.
static bool engine_faster(int n, int prec, int kind, bool pairs, long long tiles, const std::vector<int>& rs,
                          const LineCfg& e) {
  const int D = rs.back();
  if (D <= 13) return false;
  const bool few = tiles < 256, rows = kind == 0 || kind == 3;
  const bool two = rs.size() > 1 && rs[rs.size() - 2] > 13;  // dense stages
  if (two && n >= 965 && !rows) return true;
  if (!few) return false;
  if (two && n >= 480 && prec) return !pairs || e.lp.n <= 1296;
  if (pairs) return !prec && D > 200;
  if (prec) {
    const double cost = (double)e.lp.n * (e.lp.np + 0.04 * e.E) / n;  // (as plan_line's)
    return (n > 864 && !rows) || (D > 200 && n >= 2 * D && cost < 8.7);
  }
  return kind == 1 && D >= 130 && n >= 2 * D && e.E <= 16 && e.lp.n <= 1024;
}

bool mix_cfg(int n, int prec, int kind, int ncols, bool pairs, long long lines, const LineCfg& engine, MixCfg& out) {
  out = MixCfg{};
  const std::vector<int> rs = mix_radices(n);
  const bool rows = kind == 0 || kind == 3;
  if (rs.empty() || rs.back() > mix_max_dense(prec, rows && pairs)) return false;
  const bool dense = rs.back() > 13;
  const int eb = prec ? 8 : 16;
  // exchanges: a column pass keeps its last stage's output in registers, the x
  // pass runs two transforms, the row passes end (and the inverse begins) in LDS
  const int np = (int)rs.size(), first = np > 1 && rs[0] <= 13 ? 1 : 0;
  const int bufs = kind == 1 ? mix_buffers(np - first) : 2;
  int ntab = 0;
  for (int R : rs) ntab += R > 13 ? (R + 15) / 16 * 16 : 0;
  auto bytes = [&](int T) { return ((size_t)bufs * T * (rows ? mix_row_pitch(n) : n) + ntab) * eb; };
  // about 2048 (FP64) or 4096 (FP32) values per buffer; a column tile's row
  // segments at least 64 bytes; a dense stage's 8 lines (16 real columns) where
  // two such workgroups fit a CU's LDS
  const int tmin = rows ? 1 : 64 / eb;
  int T = rows ? 256 : 64;
  while (T > tmin && T * n > 32768 / eb) T /= 2;
  if (dense)
    while (T < 8) T *= 2;
  // (narrower where the grid would leave CUs without a tile)
  while (T > std::max(tmin, dense ? 8 : 1) && lines / T < 256) T /= 2;
  while (T > tmin && bytes(T) > 80 * 1024) T /= 2;
  while (T > 1 && bytes(T) > 160 * 1024) T /= 2;
  while (!rows && T > 1 && T / 2 >= ncols) T /= 2;
  if (bytes(T) > 160 * 1024) return false;
  if (engine_faster(n, prec, kind, pairs, (lines + T - 1) / T, rs, engine)) return false;
  // (the index divisions are exact below 2^16)
  if ((long long)T * (n + 2) >= 65536) return false;
  out.T = T;
  while ((1 << out.lgT) < T) out.lgT++;
  out.lds = bytes(T);
  out.bufs = bufs;
  out.n = n;
  out.tw = table_twiddle(n, prec);
  if (out.tw) out.plan = table_built(4, n, prec, [&](std::vector<unsigned char>& b) { build_plan(n, prec, b); });
  return out.plan != nullptr;
}

}  // namespace ff
