// Shared host-side helpers of the rnsmx library: error reporting and small
// integer utilities.  Device arithmetic lives in rnsmx_arith.hpp.
#pragma once

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <string>

#include "rnsmx.h"

namespace rnsmx {

// Thread-local last-error text behind rnsmx_last_error().
void set_error(const char *fmt, ...) __attribute__((format(printf, 1, 2)));
void clear_error();

inline int32_t fail(int32_t code, const char *what) {
  set_error("%s", what);
  return code;
}

inline int64_t round_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

// Whether [a, a + an) and [b, b + bn) share a byte: a kernel that writes one
// while its other workgroups still read the other needs them apart.
inline bool ranges_meet(const void *a, int64_t an, const void *b, int64_t bn) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return x < y + static_cast<uintptr_t>(bn) && y < x + static_cast<uintptr_t>(an);
}

// Largest |centered residue| of the set: floor(max(m) / 2).
inline int32_t max_half(const rnsmx_moduli_t &mods) {
  int32_t h = 0;
  for (int i = 0; i < mods.channels; ++i)
    if (mods.moduli[i] / 2 > h) h = mods.moduli[i] / 2;
  return h;
}

// Per-channel int32 accumulators of centered residues cannot overflow when
// K * max_half^2 <= 2^31 - 1 (the bound of cuda_backend.py:210-214, 240).
inline bool accumulator_fits(const rnsmx_moduli_t &mods, int64_t k) {
  const int64_t h = max_half(mods);
  return k * h * h <= 0x7FFFFFFFLL;
}

// The same bound when A enters the MFMA as raw int8 (|a| <= 128) against
// centered weight residues: K * 128 * max_half <= 2^31 - 1.
inline bool raw_accumulator_fits(const rnsmx_moduli_t &mods, int64_t k) {
  return k * 128 * static_cast<int64_t>(max_half(mods)) <= 0x7FFFFFFFLL;
}

// Packed weights: two products of centered residues (|.| <= max_half) by
// weight bytes (|.| <= 128) per K index, plus a per-row term below 256:
// 2 * K * 128 * max_half + 255 <= 2^31 - 1.
inline bool packed_accumulator_fits(const rnsmx_moduli_t &mods, int64_t k) {
  return k * 256 * static_cast<int64_t>(max_half(mods)) + 255 <= 0x7FFFFFFFLL;
}

// Constants of the fractional reconstruction (frac_sum, rnsmx_gemm.hpp) of a
// set of up to 6 moduli: k_c = (P_p / m_c)^-1 mod m_c, centered, for the
// prefix of the first p channels, as bytes (kprefix[p], channel c in byte
// c % 4 of word c / 4), and k_c / m_c of the full set in rows: row 0 to
// multiples of 2^-20, then either the rest to 53 bits (rest1), or row 1 to
// multiples of 2^-40 and the rest after it to 53 bits (rest2).
struct FracSet {
  double row0[6], rest1[6], row1[6], rest2[6];
  double p, half, turn;  // P, (P - 1) >> 1 and (half + 1/4) / P of the set
  uint32_t kprefix[7][2];
};
// Kept per thread for the set last asked for, compared by value: the inverses
// would cost every launch a few hundred nanoseconds.
const FracSet &frac_set(const rnsmx_moduli_t &mods);

}  // namespace rnsmx
