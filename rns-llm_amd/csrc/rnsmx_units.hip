// Residue-plane products by channel units: a workgroup computes one channel of
// one output tile, and the last of a tile's channels to finish reconstructs it.
#include "rnsmx_gemm.hpp"

namespace rnsmx {

// A workgroup of 2 x 4 waves owns 32 MI rows x 64 NJ columns of one channel,
// each wave 16 MI x 16 NJ.  A wave that holds every channel of its elements
// (mfma_kernel, lds_planes_kernel) issues R times the MFMAs per K step on a
// tile that registers keep small, so a product of few tiles runs long steps on
// part of the chip; units are R times as many and their steps 1/R as long.
// What bounds them is the latency of a step (load, barrier, LDS read, MFMA:
// about 0.3 us): the waves wait 73 % of their time at one workgroup per CU (matrix
// cores busy 2 %) and 51 % at two (20 %).  The exchange writes and reads a byte per
// channel and element.  Units are ordered channel by channel, so the
// workgroups that run together on an XCD share the planes of one channel.
// With the encode of the activations, 6 channels: 128 x 4096 x 4096 32 us
// (lds_planes_kernel 49), 640 x 2048 x 2048 36 (mfma_kernel 66).  Tiles of
// 256 x 192 and 256 x 256 were slower than lds_planes_kernel but for single
// sizes.  Staging and waits as lds_wide_kernel (A by pairs of K steps as whole
// 128-byte row segments two steps ahead, B three ahead, one barrier per step);
// the fragments of the next step are read during this one into a second set of
// registers.
// A finished unit writes its canonical residues to the exchange area, four rows
// of a column per word, under the ticket protocol of split_exchange: the wave
// that draws the last ticket of its part of the tile reads every channel's
// residues and reconstructs.  Units of channels past an adaptive prefix end at
// once.
// Wave grid 2 x 4; MI a multiple of 2, B fragments 4 NJ per step over 8 waves
// (rounded up: the loads past the tile repeat its last fragments).
template <int RCAP, int MI, int NJ>
struct UnitTile {
  static constexpr int WM = 2, WN = 4, NW = 8, S = 4;
  static constexpr int BM = 16 * WM * MI, BN = 16 * WN * NJ, NB = BN / 16;
  static constexpr int BLKS = BM / 8;             // 8-row blocks (1 KB per pair of steps)
  static constexpr int AU = BLKS / NW;            // A loads per wave per pair
  static constexpr int BL = (NB + NW - 1) / NW;   // B loads per wave per step
  static constexpr int PAIR = BM * 128;
  static constexpr int BSTAGE = BL * NW * 1024;
  static constexpr int BAREA = 2 * PAIR;
  static constexpr int LDS = BAREA + S * BSTAGE;
};

template <int RCAP, int MI, int NJ>
__global__ __launch_bounds__(512) void units_kernel(const GemmArgsK<RCAP> args) {
  using T = UnitTile<RCAP, MI, NJ>;
  constexpr int NW = T::NW, BM = T::BM, BN = T::BN, NB = T::NB, S = T::S, AU = T::AU, BL = T::BL;
  constexpr int PAIR = T::PAIR, BSTAGE = T::BSTAGE, BAREA = T::BAREA, WN = T::WN;
  static_assert(T::BLKS % NW == 0 && MI >= NJ, "A loads split evenly; B reads ride on the rows");
  static_assert(S * BSTAGE <= 65536, "immediate read offsets");
  KArgs<RCAP> &g = kernel_args<GemmArgsK<RCAP>>();
  prefetch_kernel_args<kGemmArgBytes<RCAP>>();
  __shared__ __attribute__((aligned(1024))) int8_t smem[T::LDS];
  // the adaptive check's slots lie in the last B stage, first written by the
  // loads of step 0, two barriers after every wave has read the count
  int8_t *spare = smem + T::LDS - BSTAGE;
  const int c_act =
      active_channels<RCAP>(g, reinterpret_cast<int64_t *>(spare), reinterpret_cast<int *>(spare + 64), 512);
  const int tiles = g.tiles_m * g.tiles_n;
  const int u = xcd_order(blockIdx.x, tiles * g.mods.channels);
  const int ch = u / tiles, tile = u - ch * tiles;
  if (ch >= c_act) return;
  // groups of 4 row tiles per column tile, as planes_work
  int mt, nt;
  {
    constexpr int RG = 4;
    const int grouped = g.tiles_m / RG * RG;
    if (tile < grouped * g.tiles_n) {
      const int r = tile % (RG * g.tiles_n);
      nt = r / RG;
      mt = tile / (RG * g.tiles_n) * RG + r % RG;
    } else {
      const int r = tile - grouped * g.tiles_n, h = g.tiles_m - grouped;
      nt = r / h;
      mt = grouped + r % h;
    }
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = mt * BM, n0 = nt * BN;
  const int nk = g.kp >> 6;

  const int8_t *abase = g.a + static_cast<int64_t>(ch) * g.a_cs;
  uint32_t aoff[AU];
  static_for<AU>([&](auto U) {
    const int r = min(m0 + (wave + NW * decltype(U)::value) * 8 + (lane >> 3), g.m - 1);
    aoff[decltype(U)::value] = static_cast<uint32_t>(r * g.a_ld + ((lane & 7) ^ (lane >> 3)) * 16);
  });
  const int nblk = (g.n + 15) >> 4;
  const int8_t *bbase[BL];
  static_for<BL>([&](auto U) {
    const int q = min(wave + NW * decltype(U)::value, NB - 1);
    const int jb = min((n0 >> 4) + q, nblk - 1);
    bbase[decltype(U)::value] = g.b + static_cast<int64_t>(ch) * g.b_cs + static_cast<int64_t>(jb) * g.b_ld;
  });
  const uint32_t boff = static_cast<uint32_t>(lane * 16);
  const uint32_t sbase = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) int8_t *)(smem))) +
      wave * 1024);
  // loads past K load the last step or pair again, into stages never read; the
  // second half of an odd last pair lies in the next row (after the last row
  // of the last plane: in the row norms that follow the planes, 256 bytes at
  // least) and is not read either
  auto dma_b = [&](auto ST, auto L, int ks) {
    constexpr int st = decltype(ST)::value, l = decltype(L)::value;
    lds_dma16<BAREA + st * BSTAGE + NW * l * 1024>(bbase[l] + static_cast<int64_t>(min(ks, nk - 1)) * 1024, boff, sbase);
  };
  auto dma_a = [&](auto ST, auto U, int ks) {
    constexpr int st = decltype(ST)::value, uu = decltype(U)::value;
    lds_dma16<(st / 2) * PAIR + NW * uu * 1024>(abase + min(ks, (nk - 1) & ~1) * 64, aoff[uu], sbase);
  };
  i32x4 fa[2][MI], fb[2][NJ];
  const int8_t *rabase[2][2];  // [pair slot][step parity]
  static_for<2>([&](auto Q) {
    static_for<2>([&](auto P) {
      constexpr int q = decltype(Q)::value, p = decltype(P)::value;
      rabase[q][p] = smem + q * PAIR + (2 * wm * MI + ((lane >> 3) & 1)) * 1024 +
                     ((lane & 7) * 8 + ((4 * p + (lane >> 4)) ^ (lane & 7))) * 16;
    });
  });
  const int8_t *rbbase = smem + BAREA + wn * NJ * 1024 + lane * 16;
  auto read_a = [&](auto H, auto BUF, auto I) {
    constexpr int h = decltype(H)::value, i = decltype(I)::value;
    fa[decltype(BUF)::value][i] = *reinterpret_cast<const i32x4 *>(rabase[h / 2][h & 1] + 2 * i * 1024);
  };
  auto read_b = [&](auto H, auto BUF, auto J) {
    constexpr int h = decltype(H)::value, j = decltype(J)::value;
    fb[decltype(BUF)::value][j] = *reinterpret_cast<const i32x4 *>(rbbase + h * BSTAGE + j * 1024);
  };
  i32x4 acc[MI][NJ];
  constexpr std::integral_constant<int, 0> k0{};
  constexpr std::integral_constant<int, 1> k1{};

  auto step = [&](auto H, int k) {
    constexpr int h = decltype(H)::value, buf = h & 1;
    constexpr std::integral_constant<int, (h + 1) % S> H1{};
    constexpr std::integral_constant<int, buf ^ 1> B1{};
    constexpr int nl = (h & 1) ? BL : AU + BL;
    if (k >= nk) return;
    wait_vmcnt<BL>();
    __builtin_amdgcn_s_barrier();
    static_for<MI>([&](auto I) {
      constexpr int i = decltype(I)::value;
      static_for<nl>([&](auto L) {
        constexpr int l = decltype(L)::value;
        if constexpr ((l * MI) / nl == i) {
          if constexpr (!(h & 1) && l < AU)
            dma_a(std::integral_constant<int, (h + 2) % S>{}, std::integral_constant<int, l>{}, k + 2);
          else
            dma_b(std::integral_constant<int, (h + S - 1) % S>{},
                  std::integral_constant<int, (h & 1) ? l : l - AU>{}, k + S - 1);
        }
      });
      read_a(H1, B1, I);
      if constexpr (i < NJ) read_b(H1, B1, I);
      static_for<NJ>([&](auto J) {
        constexpr int j = decltype(J)::value;
        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[buf][i], fb[buf][j], acc[i][j], 0, 0, 0);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  static_for<AU>([&](auto U) { dma_a(k0, U, 0); });
  static_for<BL>([&](auto L) { dma_b(k0, L, 0); });
  static_for<BL>([&](auto L) { dma_b(k1, L, 1); });
  static_for<BL>([&](auto L) { dma_b(std::integral_constant<int, 2>{}, L, 2); });
  static_for<MI>([&](auto I) {
    static_for<NJ>([&](auto J) { acc[decltype(I)::value][decltype(J)::value] = acc_zero(); });
  });
  wait_vmcnt<2 * BL>();
  __builtin_amdgcn_s_barrier();
  static_for<MI>([&](auto I) { read_a(k0, k0, I); });
  static_for<NJ>([&](auto J) { read_b(k0, k0, J); });
  __builtin_amdgcn_sched_barrier(0);
  for (int ks0 = 0; ks0 < nk; ks0 += S) {
    static_for<S>([&](auto H) { step(H, ks0 + decltype(H)::value); });
  }
  wait_vmcnt<0>();

  // residues out: word (i, j) of a wave holds rows 16 i + 4 (lane >> 4) + 0..3
  // of column 16 j + (lane & 15)
  KArgs<RCAP> &late = args_from_here<RCAP>(g);
  uint32_t m = late.mods.moduli[0], magic = late.mods.magic[0];
  static_for<RCAP - 1>([&](auto C) {
    constexpr int c = decltype(C)::value + 1;
    if (ch == c) {
      m = late.mods.moduli[c];
      magic = late.mods.magic[c];
    }
  });
  const FastMod fm = fast_mod_of(m, magic);
  constexpr int CH = MI * NJ;
  const int channels = late.mods.channels;
  const int64_t slot = static_cast<int64_t>(tile) * NW + wave;
  int8_t *xbase = late.xchg + slot * channels * CH * 256 + lane * 4;
  static_for<MI>([&](auto I) {
    static_for<NJ>([&](auto J) {
      constexpr int i = decltype(I)::value, j = decltype(J)::value;
      uint32_t w = 0;
      static_for<4>([&](auto TT) { w |= canon_fast(acc[i][j][decltype(TT)::value], fm) << (8 * decltype(TT)::value); });
      __hip_atomic_store(reinterpret_cast<uint32_t *>(xbase + (static_cast<int64_t>(ch) * CH + i * NJ + j) * 256), w,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    });
  });
  wait_vm_all();
  uint32_t old = 0;
  if (lane == 0) old = __hip_atomic_fetch_add(late.tickets + slot, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  old = __builtin_amdgcn_readfirstlane(old);
  if (old != static_cast<uint32_t>(c_act - 1)) return;
  asm volatile("" ::: "memory");
  if (lane == 0) __hip_atomic_store(late.tickets + slot, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  Epi<RCAP> e;
  load_epi<RCAP>(late, e, c_act);
  pin_epi<RCAP>(e);
  const int m_lim = late.m, n_lim = late.n;
  const int rw0 = m0 + wm * (MI * 16), cw0 = n0 + wn * (NJ * 16);
  if (rw0 >= m_lim || cw0 >= n_lim) return;
  ColScale cs[NJ];
  static_for<NJ>([&](auto J) {
    cs[decltype(J)::value] = col_scale<RCAP>(e, cw0 + decltype(J)::value * 16 + (lane & 15), n_lim);
  });
  const bool interior = rw0 + 16 * MI <= m_lim && cw0 + 16 * NJ <= n_lim;
  const bool pairs = interior && e.out_dtype == RNSMX_INT64 && (e.out_ld & 1) == 0 &&
                     (reinterpret_cast<uintptr_t>(e.out) & 15) == 0;
  const bool quads = interior && float_quads_fit<RCAP>(e);
  auto run = [&](auto DT) __attribute__((always_inline)) {
    constexpr int dt = decltype(DT)::value;
    static_for<MI / 2>([&](auto G) {
      // two rows of blocks in flight: every channel's word of each
      uint32_t w[2][NJ][RCAP];
      static_for<2>([&](auto I) {
        static_for<NJ>([&](auto J) {
          static_for<RCAP>([&](auto C) {
            constexpr int i = 2 * decltype(G)::value + decltype(I)::value, j = decltype(J)::value, c = decltype(C)::value;
            uint32_t x = 0;
            if (c < c_act)
              x = __hip_atomic_load(reinterpret_cast<uint32_t *>(xbase + (static_cast<int64_t>(c) * CH + i * NJ + j) * 256),
                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            w[decltype(I)::value][j][c] = x;
          });
        });
      });
      static_for<2>([&](auto I) {
        constexpr int i = 2 * decltype(G)::value + decltype(I)::value;
        static_for<NJ>([&](auto J) {
          constexpr int j = decltype(J)::value;
          double t[4];
          static_for<4>([&](auto TT) {
            int32_t v[RCAP];
            static_for<RCAP>([&](auto C) {
              v[decltype(C)::value] = static_cast<int32_t>(byte_of(w[decltype(I)::value][j][decltype(C)::value], decltype(TT)::value));
            });
            t[decltype(TT)::value] = frac_sum<RCAP>(e, v);
          });
          const int64_t idx = static_cast<int64_t>(rw0 + i * 16 + 4 * (lane >> 4)) * e.out_ld + cw0 + j * 16;
          if constexpr (dt == RNSMX_INT64) {
            if (pairs) {
              int64_t y[4];
              static_for<4>([&](auto TT) { y[decltype(TT)::value] = frac_int<RCAP>(t[decltype(TT)::value]); });
              store_int64_pairs(y, as_global<int64_t>(e.out) + idx + (lane & 14), e.out_ld);
              return;
            }
          } else {
            if (quads) {
              float f[4];
              static_for<4>([&](auto TT) { f[decltype(TT)::value] = frac_float<RCAP>(t[decltype(TT)::value]); });
              store_float_quads<RCAP, dt>(e, f, cs[j], idx + (lane & 3) * e.out_ld + (lane & 12));
              return;
            }
          }
          static_for<4>([&](auto TT) {
            constexpr int tt = decltype(TT)::value;
            const int row = rw0 + i * 16 + 4 * (lane >> 4) + tt, col = cw0 + j * 16 + (lane & 15);
            if (row < m_lim && col < n_lim) {
              const int64_t at = idx + tt * e.out_ld + (lane & 15);
              if constexpr (dt == RNSMX_INT64)
                store_value<RCAP, kOutInt64>(e, frac_int<RCAP>(t[tt]), at, cs[j]);
              else
                store_float<RCAP>(e, frac_float<RCAP>(t[tt]), at, cs[j]);
            }
          });
        });
      });
    });
  };
  if (e.out_dtype == RNSMX_INT64)
    run(std::integral_constant<int, RNSMX_INT64>{});
  else
    with_float_type<RCAP>(e, run);
}

template <int RCAP, int MI, int NJ>
static void launch_tile(const GemmArgs &host, hipStream_t st) {
  using T = UnitTile<RCAP, MI, NJ>;
  GemmArgsK<RCAP> g = compact_args<RCAP>(host);
  g.tiles_m = (g.m + T::BM - 1) / T::BM;
  g.tiles_n = (g.n + T::BN - 1) / T::BN;
  const dim3 grid(static_cast<unsigned>(g.tiles_m * g.tiles_n * g.mods.channels));
  hipLaunchKernelGGL((units_kernel<RCAP, MI, NJ>), grid, dim3(512), 0, st, g);
}

bool launch_units(const GemmArgs &g, const GemmChoice &c, hipStream_t st) {
  if (c.mb == 4 && c.nb == 2)
    launch_tile<6, 4, 2>(g, st);
  else if (c.mb == 2 && c.nb == 1)
    launch_tile<6, 2, 1>(g, st);
  else
    return false;
  return true;
}

}  // namespace rnsmx
