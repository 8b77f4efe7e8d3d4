// Host-only part of the rnsmx C ABI: error text, moduli constants, LUT.
#include <cmath>
#include <cstring>

#include "rnsmx_common.hpp"

namespace rnsmx {

static thread_local char g_error[512] = {0};

void set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

void clear_error() { g_error[0] = 0; }

static int64_t gcd64(int64_t a, int64_t b) {
  while (b) {
    const int64_t t = a % b;
    a = b;
    b = t;
  }
  return a;
}

// Modular inverse of a modulo m (m <= 255, gcd(a, m) = 1) by search over the
// residues: at most 254 trials, host-side, once per moduli set.
static uint32_t inverse_mod(int64_t a, int64_t m) {
  const int64_t r = ((a % m) + m) % m;
  for (int64_t x = 1; x < m; ++x)
    if ((r * x) % m == 1) return static_cast<uint32_t>(x);
  return m == 1 ? 0u : 0xFFFFFFFFu;
}

// Inverse of a modulo m, 0 < a < m <= 255 coprime, by Euclid's algorithm.
static int inverse_euclid(int a, int m) {
  int r0 = m, r1 = a, t0 = 0, t1 = 1;
  while (r1 != 0) {
    const int q = r0 / r1;
    const int r = r0 - q * r1, t = t0 - q * t1;
    r0 = r1;
    r1 = r;
    t0 = t1;
    t1 = t;
  }
  return t0 < 0 ? t0 + m : t0;
}

static FracSet make_frac_set(const rnsmx_moduli_t &mods) {
  FracSet s{};
  const int channels = mods.channels;
  if (channels < 1 || channels > 6) return s;
  // a set that rnsmx_moduli_init has not filled: no constants, and no division by zero
  for (int c = 0; c < channels; ++c)
    if (mods.moduli[c] < 2) return s;
  for (int p = 1; p <= channels; ++p) {
    for (int c = 0; c < p; ++c) {
      const int m = mods.moduli[c];
      int rest = 1;  // P_p / m_c mod m_c
      for (int j = 0; j < p; ++j)
        if (j != c) rest = rest * (mods.moduli[j] % m) % m;
      int k = inverse_euclid(rest, m);
      if (2 * k > m) k -= m;
      s.kprefix[p][c / 4] |= (static_cast<uint32_t>(k) & 0xFFu) << (8 * (c % 4));
      if (p == channels) {
        const double md = m, kd = k, s20 = 1048576.0, s40 = 1048576.0 * 1048576.0;
        s.row0[c] = std::rint(kd / md * s20) / s20;
        const double r1 = std::fma(-s.row0[c], md, kd);  // exact
        s.rest1[c] = r1 / md;
        s.row1[c] = std::rint(r1 / md * s40) / s40;
        s.rest2[c] = std::fma(-s.row1[c], md, r1) / md;
      }
    }
  }
  const int64_t p = mods.prefix[channels];  // below 2^48
  s.p = static_cast<double>(p);
  s.half = static_cast<double>((p - 1) >> 1);
  s.turn = (s.half + 0.25) / s.p;
  return s;
}

const FracSet &frac_set(const rnsmx_moduli_t &mods) {
  static thread_local int32_t channels = 0;
  static thread_local int32_t moduli[RNSMX_MAX_CHANNELS] = {};
  static thread_local FracSet set{};
  const size_t bytes = sizeof(int32_t) * static_cast<size_t>(mods.channels);
  if (mods.channels != channels || std::memcmp(moduli, mods.moduli, bytes) != 0) {
    set = make_frac_set(mods);
    std::memcpy(moduli, mods.moduli, bytes);
    channels = mods.channels;
  }
  return set;
}

}  // namespace rnsmx

extern "C" {

const char *rnsmx_last_error(void) { return rnsmx::g_error; }

int32_t rnsmx_abi_version(void) { return 5; }

int32_t rnsmx_moduli_init(const int32_t *moduli, int32_t channels,
                          rnsmx_moduli_t *out) {
  using namespace rnsmx;
  clear_error();
  if (!moduli || !out) return fail(RNSMX_EINVAL, "null argument");
  if (channels < 1) return fail(RNSMX_EINVAL, "moduli must not be empty");
  if (channels > RNSMX_MAX_CHANNELS) {
    set_error("at most %d channels are supported, got %d", RNSMX_MAX_CHANNELS,
              channels);
    return RNSMX_EINVAL;
  }
  for (int i = 0; i < channels; ++i)
    if (moduli[i] < 2 || moduli[i] > 255)
      return fail(RNSMX_EINVAL, "every modulus must be in [2, 255]");
  for (int i = 0; i < channels; ++i)
    for (int j = i + 1; j < channels; ++j)
      if (gcd64(moduli[i], moduli[j]) != 1) {
        set_error("moduli are not pairwise coprime: %d, %d", moduli[i],
                  moduli[j]);
        return RNSMX_EINVAL;
      }

  rnsmx_moduli_t r;
  std::memset(&r, 0, sizeof(r));
  r.channels = channels;
  // prefix[i] = prod_{j<i} m_j, checked against int64 overflow.
  r.prefix[0] = 1;
  for (int i = 0; i < channels; ++i) {
    const int64_t m = moduli[i];
    if (r.prefix[i] > INT64_MAX / m)
      return fail(RNSMX_ERANGE, "moduli product must fit signed int64");
    r.prefix[i + 1] = r.prefix[i] * m;
  }
  for (int i = 0; i < channels; ++i) {
    const int64_t m = moduli[i];
    r.moduli[i] = moduli[i];
    r.magic[i] = static_cast<uint32_t>((1ULL << 32) / static_cast<uint64_t>(m));
    r.c31[i] = static_cast<uint32_t>((1LL << 31) % m);
    const int64_t p_mod = r.prefix[i] % m;
    r.qinv[i] = inverse_mod(p_mod, m);
    // the Garner digit of channel i straight from its int32 sum v = a2 2^16 +
    // a1 2^8 + a0: v qinv_i = a2 qk16_i + a1 qk8_i + a0 qinv_i (mod m_i)
    const int64_t k16 = (65536 % m) * static_cast<int64_t>(r.qinv[i]) % m;
    r.qk16[i] = static_cast<int32_t>(2 * k16 > m ? k16 - m : k16);
    r.qk8[i] = static_cast<uint32_t>((256 % m) * static_cast<int64_t>(r.qinv[i]) % m);
    for (int j = 0; j < i; ++j) {
      const int64_t pj = r.prefix[j] % m;
      const int64_t t = (pj * static_cast<int64_t>(r.qinv[i])) % m;
      r.ucoef[j][i] = static_cast<uint32_t>((m - t) % m);
    }
  }
  *out = r;
  return RNSMX_OK;
}

int32_t rnsmx_compact_lut(const rnsmx_moduli_t *mods, int16_t *lut) {
  using namespace rnsmx;
  clear_error();
  if (!mods || !lut) return fail(RNSMX_EINVAL, "null argument");
  for (int c = 0; c < mods->channels; ++c) {
    const int64_t m = mods->moduli[c];
    int64_t weight = 1;  // 256^p mod m
    for (int p = 0; p < 4; ++p) {
      for (int b = 0; b < 256; ++b)
        lut[(c * 4 + p) * 256 + b] = static_cast<int16_t>((b * weight) % m);
      weight = (weight * 256) % m;
    }
  }
  return RNSMX_OK;
}

}  // extern "C"
