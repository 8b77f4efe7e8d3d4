// The byte-product kernels for packed weights (rnsmx_bytes.hpp) and their
// launcher.
#include "rnsmx_bytes.hpp"

namespace rnsmx {

template <int AB, int WM, int WN, int MI, int NJ>
static void launch_lds_tile(GemmArgsK<kBytesCap> g, hipStream_t st) {
  using T = BytesTile<AB, WM, WN, MI, NJ>;
  g.tiles_m = (g.m + T::BM - 1) / T::BM;
  g.tiles_n = (g.n + T::BN - 1) / T::BN;
  const dim3 grid(static_cast<unsigned>(g.split_from + (g.tiles_m * g.tiles_n - g.split_from) * g.splits));
  hipLaunchKernelGGL((bytes_lds_kernel<AB, WM, WN, MI, NJ>), grid, dim3(64 * T::NW), 0, st, g);
}

template <int AB>
static bool launch_ab(const GemmArgsK<kBytesCap> &args, const GemmChoice &c, hipStream_t st) {
  GemmArgsK<kBytesCap> g = args;
  if (c.kind == kBytesRows) {
    if (c.ks < 1 || c.ks > 4) return false;
    g.tiles_m = 1;
    g.tiles_n = (g.n + 15) / 16;
    g.threads = 64 * c.ks;
    const dim3 grid(static_cast<unsigned>(g.tiles_n)), block(64 * c.ks);
    switch (c.mb) {
      case 1: hipLaunchKernelGGL((bytes_rows_kernel<AB, 1>), grid, block, 0, st, g); return true;
      case 2: hipLaunchKernelGGL((bytes_rows_kernel<AB, 2>), grid, block, 0, st, g); return true;
      case 4: hipLaunchKernelGGL((bytes_rows_kernel<AB, 4>), grid, block, 0, st, g); return true;
      default: return false;
    }
  }
  if (c.mb == 8)
    launch_lds_tile<AB, 2, 4, 4, 3>(g, st);
  else if (c.mb == 4)
    launch_lds_tile<AB, 2, 2, 2, 3>(g, st);
  else
    return false;
  return true;
}

bool launch_bytes(const GemmArgs &g, int ab, const GemmChoice &c, hipStream_t st) {
  const GemmArgsK<kBytesCap> k = compact_args<kBytesCap>(g);
  return ab == 2 ? launch_ab<2>(k, c, st) : launch_ab<1>(k, c, st);
}

}  // namespace rnsmx
