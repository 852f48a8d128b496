// The kernels of the kLdsCols and kLdsRows lines: the line plan compiled in, twiddles in
// LDS (ff_kernels.hpp).  The build compiles this file once per part, FF_LINES, each with
// every kLdsParts-th line of the two tables.
#include <type_traits>

#include "ff_kernels.hpp"

#ifndef FF_LINES
#error "FF_LINES must be defined"
#endif

namespace ff {

template <typename F, int N, int E, int MODE>
static const void* col_of() {
  constexpr LdsShape s = lds_shape(N, E, std::is_same<F, float>::value, MODE != COL_FWD && MODE != COL_INV);
  return (const void*)&k_col<F, E, MODE, s.split != 0, 1, false, N, s.T, s.waves, true>;
}

template <typename F, int N, int E>
static const void* col_modes(int mode) {
  switch (mode) {
    case COL_FWD: return col_of<F, N, E, COL_FWD>();
    case COL_INV: return col_of<F, N, E, COL_INV>();
    case COL_FILTER: return col_of<F, N, E, COL_FILTER>();
    case COL_FILTER_FD: return col_of<F, N, E, COL_FILTER_FD>();
    case COL_SYMBOL:
      if constexpr (std::is_same<F, double>::value) return col_of<F, N, E, COL_SYMBOL>();
      return nullptr;
    default: return nullptr;
  }
}

template <int K>
static const void* col_line_of(int f32, int mode, int n, int E) {
  if constexpr (K < kNumLdsCols) {
    constexpr LdsLine c = kLdsCols[K];
    if (c.n == n && c.E == E) return f32 ? col_modes<float, c.n, c.E>(mode) : col_modes<double, c.n, c.E>(mode);
    return col_line_of<K + kLdsParts>(f32, mode, n, E);
  } else {
    return nullptr;
  }
}

template <int K>
static const void* r2c_line_of(int f32, int in_f32, int M, int E) {
  if constexpr (K < kNumLdsRows) {
    constexpr LdsLine c = kLdsRows[K];
    if (c.n == M && c.E == E) {
      if (!f32) return in_f32 ? nullptr : (const void*)&k_r2c_line<double, double, c.E, c.n>;
      return in_f32 ? (const void*)&k_r2c_line<float, float, c.E, c.n>
                    : (const void*)&k_r2c_line<float, double, c.E, c.n>;
    }
    return r2c_line_of<K + kLdsParts>(f32, in_f32, M, E);
  } else {
    return nullptr;
  }
}

template <int K>
static const void* c2r_line_of(int f32, int out_kind, int epi, int M, int E) {
  if constexpr (K < kNumLdsRows) {
    constexpr LdsLine c = kLdsRows[K];
    if (c.n == M && c.E == E) {
#define FF_C2R(F, OUT, EPI) return (const void*)&k_c2r_line<F, OUT, c.E, EPI, c.n>
      if (!f32) {
        if (epi == EPI_STORE && out_kind == 0) FF_C2R(double, double, EPI_STORE);
        if (epi == EPI_RESIDUAL && out_kind == 1) FF_C2R(double, float, EPI_RESIDUAL);
        if (epi == EPI_RESIDUAL && out_kind == 0) FF_C2R(double, double, EPI_RESIDUAL);
        return nullptr;
      }
      if (epi == EPI_STORE && out_kind == 0) FF_C2R(float, double, EPI_STORE);
      if (epi == EPI_ACCUM && out_kind == 0) FF_C2R(float, double, EPI_ACCUM);
#undef FF_C2R
      return nullptr;
    }
    return c2r_line_of<K + kLdsParts>(f32, out_kind, epi, M, E);
  } else {
    return nullptr;
  }
}

template <>
const void* lds_col_part<FF_LINES>(int f32, int mode, int n, int E) {
  return col_line_of<FF_LINES>(f32, mode, n, E);
}
template <>
const void* lds_r2c_part<FF_LINES>(int f32, int in_f32, int M, int E) {
  return r2c_line_of<FF_LINES>(f32, in_f32, M, E);
}
template <>
const void* lds_c2r_part<FF_LINES>(int f32, int out_kind, int epi, int M, int E) {
  return c2r_line_of<FF_LINES>(f32, out_kind, epi, M, E);
}

#if FF_LINES == 0
template <int P>
static const void* col_any(int f32, int mode, int n, int E) {
  if constexpr (P < kLdsParts) {
    const void* fn = lds_col_part<P>(f32, mode, n, E);
    return fn ? fn : col_any<P + 1>(f32, mode, n, E);
  } else {
    return nullptr;
  }
}
template <int P>
static const void* r2c_any(int f32, int in_f32, int M, int E) {
  if constexpr (P < kLdsParts) {
    const void* fn = lds_r2c_part<P>(f32, in_f32, M, E);
    return fn ? fn : r2c_any<P + 1>(f32, in_f32, M, E);
  } else {
    return nullptr;
  }
}
template <int P>
static const void* c2r_any(int f32, int out_kind, int epi, int M, int E) {
  if constexpr (P < kLdsParts) {
    const void* fn = lds_c2r_part<P>(f32, out_kind, epi, M, E);
    return fn ? fn : c2r_any<P + 1>(f32, out_kind, epi, M, E);
  } else {
    return nullptr;
  }
}
const void* lds_col_kernel(int f32, int mode, int n, int E) { return col_any<0>(f32, mode, n, E); }
const void* lds_r2c_kernel(int f32, int in_f32, int odd, int M, int E) {
  return odd ? nullptr : r2c_any<0>(f32, in_f32, M, E);
}
const void* lds_c2r_kernel(int f32, int out_kind, int odd, int epi, int M, int E) {
  return odd ? nullptr : c2r_any<0>(f32, out_kind, epi, M, E);
}
#endif

}  // namespace ff
