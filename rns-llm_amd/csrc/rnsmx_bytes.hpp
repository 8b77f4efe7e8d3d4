// Packed weights against int8 or int16 activations by byte products.
//
// A packed weight is v = 256 hi + lo + 128 with signed bytes hi and lo
// (rnsmx_gemm.hpp); an int16 activation splits the same way, a = 256 ah + al
// + 128, and an int8 activation is one byte already.  The product of every
// channel is then the residue of one integer,
//   sum_k a v = 2^16 sum ah hi + 2^8 (sum ah lo + sum al hi) + sum al lo
//               + 128 sum_k a + 128 (2^8 sum hi + sum lo),
// four int8 MFMAs per 16 x 16 x 64 block (two for int8 activations: 2^8 sum a
// hi + sum a lo + 128 sum_k a) whatever the number of channels, where the
// channel form (residues of the activations against both bytes) runs 2 R.
// The kernels sum it exactly: each int32 accumulator holds at most two byte
// products per K index (K below 2^16), the weighted sum stays below 2^47 and
// is formed in double, exactly.  What the residues of the active channels
// would reconstruct to is that integer taken to the centered range of their
// product P (the integer itself unless the set is undersized): centered_mod.
#pragma once

#include "rnsmx_gemm.hpp"

namespace rnsmx {

// Constants for the prefix of c_act channels: the moduli block of capacity 6
// serves every set packed weights take.
constexpr int kBytesCap = 6;

// K (padded) for which two byte products per K index fit int32.
constexpr int kBytesMaxKp = 65472;

__device__ __forceinline__ void load_bytes_epi(KArgs<kBytesCap> &g, Epi<kBytesCap> &e, int c_act) {
  const int64_t p = prefix_at<kBytesCap>(g.mods, c_act);
  e.p = static_cast<double>(p);
  e.turn = (static_cast<double>((p - 1) >> 1) + 0.25) / e.p;
  e.f[0][0] = 1.0 / e.p;
  e.out_dtype = g.out_dtype;
  e.out_ld = g.out_ld;
  e.out = g.out;
  e.w_scale = g.w_scale;
  e.bias_ptr = g.bias;
  e.a_scale = g.out_dtype != RNSMX_INT64 ? *g.a_scale : 0.0f;
}

// The integer x (|x| < 2^47, as a double) taken to the centered range of P:
// x - P n with n = floor(x / P + turn), turn = (h + 1/4) / P, h = (P - 1) >> 1
// (frac_sum).  x / P + turn misses (y + h + 1/4) / P + n by less than 2^-5 / P
// (one rounding of 1 / P, one of the fma, both relative to |x| / P), under the
// 1 / (4 P) that keeps the floor; the last fma is exact.
__device__ __forceinline__ double centered_mod(const Epi<kBytesCap> &e, double x) {
  const double n = __builtin_floor(__builtin_fma(x, e.f[0][0], e.turn));
  return __builtin_fma(-n, e.p, x);
}

template <int OUT>
__device__ __forceinline__ void bytes_store(const Epi<kBytesCap> &e, double x, int64_t idx, ColScale cs) {
  const double y = centered_mod(e, x);
  if constexpr (OUT == kOutInt64)
    store_value<kBytesCap, OUT>(e, frac_int<kBytesCap>(y + kRoundMagic), idx, cs);
  else
    store_float<kBytesCap>(e, static_cast<float>(y), idx, cs);
}

__device__ __forceinline__ i32x4 mfma_i8(i32x4 a, i32x4 b, i32x4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// Decode (few tokens): a workgroup owns 16 columns and every token, its waves
// split K (chunks of U steps, the halves in turn, as rows_packed_kernel).  The
// activations are read as they are (int16 or int8 rows, 16-byte aligned): no
// encoding launch, and a fragment's 16 rows hold the high and the low bytes
// of 8 tokens (rows 0-7 and 8-15; two byte permutes and an XOR per dword), or
// 16 int8 tokens.  Per K step and fragment two MFMAs (against hi and lo) and
// one against ones for the row sums; two more for the column sums of the
// weight bytes (int16 only).  Bound by the weight stream: 4 tokens against K =
// 4096, N = 12288 (100.7 MB) take 20.3 us, 5.0 TB/s, where encoding them and
// the channel rows (two blocks of 2 tokens) took 28.9.
// ---------------------------------------------------------------------------
template <int AB, int NF>
constexpr int bytes_rows_u() {
  // K steps per chunk: 8 registers of weights and 4 AB NF of activations a
  // step, three waves per SIMD
  constexpr int per = 8 + 4 * AB * NF;
  return per <= 16 ? 8 : per <= 24 ? 4 : 2;
}

template <int AB, int NF>
__global__ __launch_bounds__(256) void bytes_rows_kernel(const GemmArgsK<kBytesCap> args) {
  constexpr int RCAP = kBytesCap;
  KArgs<RCAP> &g = kernel_args<GemmArgsK<RCAP>>();
  prefetch_kernel_args<kGemmHotArgBytes>();
  constexpr int TPF = 16 / AB;  // tokens per fragment
  constexpr int U = bytes_rows_u<AB, NF>();
  __shared__ __attribute__((aligned(16))) int32_t sums[NF][2][16][16];
  __shared__ int32_t rsums[NF][16], csums[2][16];
  __shared__ int64_t red[4];
  __shared__ int bcast;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nthreads = g.threads, ks_n = nthreads >> 6;
  const int c_act = active_channels<RCAP>(g, red, &bcast, nthreads);
  const int n0 = blockIdx.x * 16;
  const int nk = g.kp >> 6, a_k = g.a_k;
  const int8_t *bp = g.b + static_cast<int64_t>(blockIdx.x) * g.b_ld + lane * 16;
  const int kofs = (lane >> 4) * 16;
  const int row = lane & 15;
  const int8_t *ap[NF];
  bool rowv[NF];
  static_for<NF>([&](auto F) {
    constexpr int f = decltype(F)::value;
    const int token = f * TPF + row % TPF;
    rowv[f] = token < g.m;
    ap[f] = g.a + static_cast<int64_t>(min(token, g.m - 1)) * g.a_ld * AB;
  });
  // byte selectors and sign flips of a lane's row: the odd bytes of each int16
  // pair (high) or the even ones (low, as signed: flipped)
  const uint32_t sel = row < 8 ? 0x07050301u : 0x06040200u;
  const uint32_t flip = row < 8 ? 0u : 0x80808080u;
  const i32x4 ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};

  i32x4 acch[NF], accl[NF], accr[NF], ccol[2];
  static_for<NF>([&](auto F) {
    acch[F] = acc_zero();
    accl[F] = acc_zero();
    accr[F] = acc_zero();
  });
  ccol[0] = acc_zero();
  ccol[1] = acc_zero();

  i32x4 fh[U], fl[U], ra[U][NF][AB];
  auto load_part = [&](int q, auto P0, auto P1) {
    static_for<U>([&](auto UU) {
      constexpr int u = decltype(UU)::value;
      if constexpr (u >= decltype(P0)::value && u < decltype(P1)::value) {
        const int ks = min(q + u, nk - 1);
        fh[u] = load16_nt(bp + ks * 1024);
        fl[u] = load16_nt(bp + g.b_cs + ks * 1024);
        static_for<NF>([&](auto F) {
          constexpr int f = decltype(F)::value;
          static_for<AB>([&](auto H) {
            constexpr int h = decltype(H)::value;
            // values [k, k + 16 / AB) of the row; a_k is a multiple of 16 / AB
            const int k = ks * 64 + kofs + h * (16 / AB);
            i32x4 x = {0, 0, 0, 0};
            if (rowv[f] && k < a_k) x = load16(ap[f] + k * AB);
            ra[u][f][h] = x;
          });
        });
      }
    });
  };
  auto mfma_part = [&](int q, auto P0, auto P1) {
    static_for<U>([&](auto UU) {
      constexpr int u = decltype(UU)::value;
      if constexpr (u >= decltype(P0)::value && u < decltype(P1)::value) {
        if (q + u >= nk) return;
        static_for<NF>([&](auto F) {
          constexpr int f = decltype(F)::value;
          i32x4 fa;
          if constexpr (AB == 2) {
            static_for<4>([&](auto D) {
              constexpr int d = decltype(D)::value;
              const i32x4 &w = ra[u][f][d / 2];
              fa[d] = static_cast<int32_t>(
                  __builtin_amdgcn_perm(static_cast<uint32_t>(w[2 * (d % 2) + 1]), static_cast<uint32_t>(w[2 * (d % 2)]), sel) ^
                  flip);
            });
          } else {
            fa = ra[u][f][0];
          }
          acch[f] = mfma_i8(fa, fh[u], acch[f]);
          accl[f] = mfma_i8(fa, fl[u], accl[f]);
          accr[f] = mfma_i8(fa, ones, accr[f]);
        });
        if constexpr (AB == 2) {
          ccol[0] = mfma_i8(ones, fh[u], ccol[0]);
          ccol[1] = mfma_i8(ones, fl[u], ccol[1]);
        }
      }
    });
  };
  constexpr std::integral_constant<int, 0> h0{};
  constexpr std::integral_constant<int, U / 2> h1{};
  constexpr std::integral_constant<int, U> h2{};
  int q = wave * U;
  load_part(q, h0, h1);
  load_part(q, h1, h2);
  for (int i = threadIdx.x; i < NF * 512; i += nthreads) (&sums[0][0][0][0])[i] = 0;
  for (int i = threadIdx.x; i < NF * 16; i += nthreads) (&rsums[0][0])[i] = 0;
  for (int i = threadIdx.x; i < 32; i += nthreads) (&csums[0][0])[i] = 0;
  if (q < nk) {
    for (;;) {
      const int qn = q + ks_n * U;
      mfma_part(q, h0, h1);
      if (qn < nk) load_part(qn, h0, h1);
      mfma_part(q, h1, h2);
      if (qn >= nk) break;
      load_part(qn, h1, h2);
      q = qn;
    }
  }
  Epi<RCAP> e;
  load_bytes_epi(g, e, c_act);
  __syncthreads();
  static_for<NF>([&](auto F) {
    constexpr int f = decltype(F)::value;
    static_for<4>([&](auto T) {
      constexpr int t = decltype(T)::value;
      const int r = 4 * (lane >> 4) + t;
      atomicAdd(&sums[f][0][r][lane & 15], acch[f][t]);
      atomicAdd(&sums[f][1][r][lane & 15], accl[f][t]);
      if ((lane & 15) == 0) atomicAdd(&rsums[f][r], accr[f][t]);
    });
  });
  if (AB == 2 && lane < 16) {
    atomicAdd(&csums[0][lane], ccol[0][0]);
    atomicAdd(&csums[1][lane], ccol[1][0]);
  }
  __syncthreads();

  const int m_lim = g.m, n_lim = g.n;
  auto finish = [&](auto OUT) {
    for (int x = threadIdx.x; x < m_lim * 16; x += nthreads) {
      const int token = x >> 4, j = x & 15, col = n0 + j;
      if (col >= n_lim) continue;
      const int f = token / TPF, r = token % TPF;
      double v;
      if constexpr (AB == 2) {
        // int64 in parts that a double holds: every term is an integer below 2^47
        const double hh = sums[f][0][r][j], mid = static_cast<double>(sums[f][1][r][j]) + sums[f][0][r + 8][j];
        const double ll = sums[f][1][r + 8][j];
        const double rc = 256.0 * (static_cast<double>(rsums[f][r]) + csums[0][j]) +
                          (static_cast<double>(rsums[f][r + 8]) + csums[1][j]);
        v = 65536.0 * hh + 256.0 * mid + ll + 128.0 * rc + 16384.0 * (nk * 64);
      } else {
        v = 256.0 * sums[f][0][r][j] + static_cast<double>(sums[f][1][r][j]) + 128.0 * rsums[f][r];
      }
      bytes_store<decltype(OUT)::value>(e, v, static_cast<int64_t>(token) * e.out_ld + col,
                                        col_scale<RCAP>(e, col, n_lim));
    }
  };
  if (e.out_dtype == RNSMX_INT64)
    finish(std::integral_constant<int, kOutInt64>{});
  else
    finish(std::integral_constant<int, kOutFloat>{});
}

// ---------------------------------------------------------------------------
// More tokens: tiles of 16 WM MI rows x 16 WN NJ columns, WM x WN waves, the
// activations as byte planes (bytes_planes_kernel: ah | al, or the int8 rows;
// [AB][M][a_ld], a_ld a multiple of 128, followed by the row terms 128 sum_k a
// as doubles).  Staging and waits are lds_wide_kernel's: a pair of K steps of
// A as whole 128-byte row segments (XOR-swizzled), loaded at even steps two
// steps ahead, B fragments three steps ahead, by direct-to-LDS loads, one
// barrier per step.  Per step a wave reads 2 MI + 2 NJ fragments for its 4 MI
// NJ MFMAs (64 x 48 per wave: 14 KB per 48), in four phases of MI NJ MFMAs
//   ah hi -> s0    (reads lo, al)         ah lo -> s1
//   al lo -> s2    (reads the next ah)    al hi -> s1  (reads the next hi)
// so every read has a phase to land; the accumulators take 12 MI NJ registers.
// The column sums of the weight bytes are dot products on the VALU, beside the
// MFMAs, one wave row taking even steps and the other odd ones.
// K split: partial sums are doubles (exact integers), exchanged in two words
// under the protocol of split_exchange: each split's column sums cover its own
// steps, and the row term, of the whole K, is added once, by the wave that
// finishes the tile.
// K = 4096, N = 12288, 512 tokens (256 tiles of 128 x 192, one round): 87 us,
// 2.4 POP/s of byte products, bound as lds_wide_kernel is by the staging and
// the MFMAs together; the channel form's 2 R = 12 MFMAs per block took 312.
// ---------------------------------------------------------------------------
template <int AB, int WM_, int WN_, int MI_, int NJ_>
struct BytesTile {
  static constexpr int WM = WM_, WN = WN_, MI = MI_, NJ = NJ_, NW = WM * WN;
  static constexpr int BM = 16 * WM * MI, BN = 16 * WN * NJ, NB = BN / 16;
  static constexpr int S = 4;
  static constexpr int PAIR = AB * BM * 128;  // A bytes of a pair of steps
  static constexpr int BSTAGE = 2 * NB * 1024;
  static constexpr int BAREA = 2 * PAIR;
  static constexpr int LDS = BAREA + S * BSTAGE;
};

template <int AB, int WM, int WN, int MI, int NJ>
__global__ __launch_bounds__(64 * WM * WN) void bytes_lds_kernel(const GemmArgsK<kBytesCap> args) {
  constexpr int RCAP = kBytesCap;
  using T = BytesTile<AB, WM, WN, MI, NJ>;
  constexpr int NW = T::NW, BM = T::BM, BN = T::BN, NB = T::NB, S = T::S;
  constexpr int PAIR = T::PAIR, BSTAGE = T::BSTAGE, BAREA = T::BAREA;
  constexpr int BLKS = BM / 8;             // 8-row blocks (1 KB per pair) of one A plane
  constexpr int AU = AB * BLKS / NW;       // A loads per wave per pair
  constexpr int BU = 2 * NB / NW;          // B loads per wave per step
  constexpr int NS = AB == 2 ? 3 : 2;      // accumulators per block: weights 2^16, 2^8, 1 (2^8, 1)
  constexpr int PH = 2 * AB;               // phases of MI NJ MFMAs per step
  static_assert(AB * BLKS % NW == 0 && 2 * NB % NW == 0, "loads split evenly over the waves");
  static_assert(WM == 2, "the column sums alternate between two wave rows");
  static_assert(2 * PAIR <= 65536 && 2 * BSTAGE <= 65536, "immediate read offsets");
  KArgs<RCAP> &g = kernel_args<GemmArgsK<RCAP>>();
  prefetch_kernel_args<kGemmArgBytes<RCAP>>();
  __shared__ __attribute__((aligned(1024))) int8_t smem[T::LDS];
  // the adaptive check's slots lie in the last B stage, first written by the
  // loads of step 0, two barriers after every wave has read the count
  int8_t *spare = smem + T::LDS - BSTAGE;
  const int c_act =
      active_channels<RCAP>(g, reinterpret_cast<int64_t *>(spare), reinterpret_cast<int *>(spare + 64), 64 * NW);
  const WorkUnit wu = planes_work(g);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = wu.mt * BM, n0 = wu.nt * BN;
  const KRange kr = k_range(g, wu.split);
  const int nk = kr.nk;

  // A block q = wave + NW u of a pair: plane q / BLKS, rows 8 (q % BLKS) .. +8
  // of the tile; lane l loads row (l >> 3), bytes 16 ((l & 7) ^ (l >> 3)) of the
  // 128-byte segment into chunk l
  const int8_t *abase[AU];
  uint32_t aoff[AU];
  static_for<AU>([&](auto U) {
    constexpr int u = decltype(U)::value;
    const int q = wave + NW * u, plane = q / BLKS;
    const int r = min(m0 + (q % BLKS) * 8 + (lane >> 3), g.m - 1);
    abase[u] = g.a + plane * g.a_cs + kr.ks0 * 64;
    aoff[u] = static_cast<uint32_t>(r * g.a_ld + ((lane & 7) ^ (lane >> 3)) * 16);
  });
  const int nblk = (g.n + 15) >> 4;
  const int8_t *bbase[BU];
  static_for<BU>([&](auto U) {
    constexpr int u = decltype(U)::value;
    const int q = wave + NW * u, plane = q / NB;
    const int jb = min((n0 >> 4) + q % NB, nblk - 1);
    bbase[u] = g.b + plane * g.b_cs + static_cast<int64_t>(jb) * g.b_ld + kr.ks0 * 1024;
  });
  const uint32_t boff = static_cast<uint32_t>(lane * 16);
  const uint32_t sbase = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) int8_t *)(smem))) +
      wave * 1024);
  // loads past K (near the end) load the last step or pair again, into
  // stages that are never read
  auto dma_b = [&](auto ST, auto L, int ks) {
    constexpr int st = decltype(ST)::value, l = decltype(L)::value;
    const int kc = min(ks, nk - 1);
    lds_dma16<BAREA + st * BSTAGE + NW * l * 1024>(bbase[l] + static_cast<int64_t>(kc) * 1024, boff, sbase);
  };
  auto dma_a = [&](auto ST, auto U, int ks) {  // ks even: the pair (ks, ks + 1) into the pair slot of stage ST
    constexpr int st = decltype(ST)::value, u = decltype(U)::value;
    const int kc = min(ks, (nk - 1) & ~1);
    lds_dma16<(st / 2) * PAIR + NW * u * 1024>(abase[u] + kc * 64, aoff[u], sbase);
  };

  i32x4 fa[AB][MI], fbh[2][NJ], fbl[NJ];
  const int8_t *rabase[2];
  static_for<2>([&](auto P) {
    constexpr int p = decltype(P)::value;
    rabase[p] = smem + (2 * wm * MI + ((lane >> 3) & 1)) * 1024 +
                ((lane & 7) * 8 + ((4 * p + (lane >> 4)) ^ (lane & 7))) * 16;
  });
  const int8_t *rbbase[2];
  static_for<2>([&](auto P) {
    rbbase[decltype(P)::value] = smem + BAREA + decltype(P)::value * 2 * BSTAGE + wn * NJ * 1024 + lane * 16;
  });
  auto read_a = [&](auto H, auto PL, auto I) {
    constexpr int h = decltype(H)::value, pl = decltype(PL)::value, i = decltype(I)::value;
    fa[pl][i] = *reinterpret_cast<const i32x4 *>(rabase[h & 1] + (h / 2) * PAIR + (pl * BLKS + 2 * i) * 1024);
  };
  auto read_b = [&](auto H, auto PL, auto J) {
    constexpr int h = decltype(H)::value, pl = decltype(PL)::value, j = decltype(J)::value;
    const i32x4 v = *reinterpret_cast<const i32x4 *>(rbbase[h >> 1] + (h & 1) * BSTAGE + (pl * NB + j) * 1024);
    if constexpr (pl == 0)
      fbh[AB == 2 ? (h & 1) : 0][j] = v;
    else
      fbl[j] = v;
  };
  constexpr std::integral_constant<int, 0> k0{};
  constexpr std::integral_constant<int, 1> k1{};

  i32x4 acc[NS][MI][NJ];
  int32_t csum[2][NJ];

  auto step = [&](auto H, int k) {
    constexpr int h = decltype(H)::value, nxt = (h + 1) % S;
    constexpr std::integral_constant<int, h> H0{};
    constexpr std::integral_constant<int, nxt> H1{};
    constexpr int bufh = AB == 2 ? (h & 1) : 0;
    constexpr int nl = (h & 1) ? BU : AU + BU;
    constexpr int slots = PH * MI;
    if (k >= nk) return;
    wait_vmcnt<BU>();
    __builtin_amdgcn_s_barrier();
    static_for<PH>([&](auto P) {
      constexpr int p = decltype(P)::value;
      constexpr int apl = p < 2 ? 0 : 1;               // ah, ah, al, al
      constexpr bool low = p == 1 || p == 2;           // hi, lo, lo, hi
      constexpr int sum = AB == 1 ? p : p == 0 ? 0 : p == 2 ? 2 : 1;
      if constexpr (p == 0) static_for<NJ>([&](auto J) { read_b(H0, k1, J); });
      if constexpr (AB == 2 && p == 3) {
        static_for<NJ>([&](auto J) { read_b(H1, k0, J); });
        // column sums of this step's weight bytes
        if (wm == (h & 1)) {
          static_for<NJ>([&](auto J) {
            static_for<4>([&](auto D) {
              csum[0][J] = __builtin_amdgcn_sdot4(fbh[bufh][J][decltype(D)::value], 0x01010101, csum[0][J], false);
              csum[1][J] = __builtin_amdgcn_sdot4(fbl[J][decltype(D)::value], 0x01010101, csum[1][J], false);
            });
          });
        }
      }
      static_for<MI>([&](auto I) {
        constexpr int i = decltype(I)::value, slot = p * MI + i;
        static_for<nl>([&](auto L) {
          constexpr int l = decltype(L)::value;
          if constexpr ((l * slots) / nl == slot) {
            if constexpr (!(h & 1) && l < AU)
              dma_a(std::integral_constant<int, (h + 2) % S>{}, std::integral_constant<int, l>{}, k + 2);
            else
              dma_b(std::integral_constant<int, (h + S - 1) % S>{},
                    std::integral_constant<int, (h & 1) ? l : l - AU>{}, k + S - 1);
          }
        });
        static_for<NJ>([&](auto J) {
          constexpr int j = decltype(J)::value;
          if constexpr (low)
            acc[sum][i][j] = mfma_i8(fa[apl][i], fbl[j], acc[sum][i][j]);
          else
            acc[sum][i][j] = mfma_i8(fa[apl][i], fbh[bufh][j], acc[sum][i][j]);
        });
        if constexpr (AB == 2) {
          if constexpr (p == 0) read_a(H0, k1, I);
          if constexpr (p == 2) read_a(H1, k0, I);
        } else {
          if constexpr (p == 1) read_a(H1, k0, I);
        }
        // keep the reads where they are (see lds_wide_kernel)
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (AB == 1 && p == 0) static_for<NJ>([&](auto J) { read_b(H1, k0, J); });
    });
  };

  // prologue: the A pair (0, 1) and B of steps 0 .. 2 in flight
  static_for<AU>([&](auto U) { dma_a(k0, U, 0); });
  static_for<BU>([&](auto L) { dma_b(k0, L, 0); });
  static_for<BU>([&](auto L) { dma_b(k1, L, 1); });
  static_for<BU>([&](auto L) { dma_b(std::integral_constant<int, 2>{}, L, 2); });
  static_for<NS>([&](auto C) {
    static_for<MI>([&](auto I) { static_for<NJ>([&](auto J) { acc[C][I][J] = acc_zero(); }); });
  });
  static_for<2>([&](auto C) { static_for<NJ>([&](auto J) { csum[C][J] = 0; }); });
  wait_vmcnt<2 * BU>();
  __builtin_amdgcn_s_barrier();
  static_for<MI>([&](auto I) { read_a(k0, k0, I); });
  static_for<NJ>([&](auto J) { read_b(k0, k0, J); });
  __builtin_amdgcn_sched_barrier(0);

  for (int ks0 = 0; ks0 < nk; ks0 += S) {
    static_for<S>([&](auto H) { step(H, ks0 + decltype(H)::value); });
  }
  // the loads issued for steps past K land before their LDS is used again
  wait_vmcnt<0>();

  KArgs<RCAP> &late = args_from_here<RCAP>(g);
  // column terms: a lane's sums cover its 16 of 64 K bytes and its wave row's steps
  int32_t *cs = reinterpret_cast<int32_t *>(smem);  // [WM][2][BN]
  double cterm[NJ];
  if constexpr (AB == 2) {
    __syncthreads();
    static_for<2>([&](auto C) {
      static_for<NJ>([&](auto J) {
        int32_t v = csum[C][J];
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        if (lane < 16) cs[(wm * 2 + decltype(C)::value) * BN + (wn * NJ + decltype(J)::value) * 16 + lane] = v;
      });
    });
    __syncthreads();
    static_for<NJ>([&](auto J) {
      const int at = (wn * NJ + decltype(J)::value) * 16 + (lane & 15);
      const int32_t hi = cs[at] + cs[2 * BN + at], lo = cs[BN + at] + cs[3 * BN + at];
      cterm[J] = 128.0 * (256.0 * hi + lo);
    });
  } else {
    static_for<NJ>([&](auto J) { cterm[J] = 0.0; });
  }
  Epi<RCAP> e;
  load_bytes_epi(late, e, c_act);
  const int m_lim = late.m, n_lim = late.n;
  const int rw0 = m0 + wm * (MI * 16), cw0 = n0 + wn * (NJ * 16);
  const double *rterm = reinterpret_cast<const double *>(late.a + AB * late.a_cs) + rw0 + 4 * (lane >> 4);
  // the whole sum of one element, without its row term
  auto value = [&](auto I, auto J, auto TT) -> double {
    constexpr int i = decltype(I)::value, j = decltype(J)::value, t = decltype(TT)::value;
    double x = static_cast<double>(acc[NS - 1][i][j][t]);
    x = __builtin_fma(256.0, static_cast<double>(acc[NS - 2][i][j][t]), x);
    if constexpr (AB == 2) x = __builtin_fma(65536.0, static_cast<double>(acc[0][i][j][t]), x);
    return x + cterm[j];
  };
  ColScale cscale[NJ];
  static_for<NJ>([&](auto J) {
    cscale[J] = col_scale<RCAP>(e, cw0 + decltype(J)::value * 16 + (lane & 15), n_lim);
  });

  const int splits = late.splits;
  const bool parted = wu.split >= 0;
  const int64_t slot = static_cast<int64_t>(wu.split_tile) * NW + wave;
  constexpr int CH = MI * NJ * 2;  // 1 KB blocks per wave and split: two words per element
  int8_t *xbase = late.xchg + slot * splits * CH * 1024 + lane * 4;
  auto block = [&](int s, int c) { return xbase + (static_cast<int64_t>(s) * CH + c) * 1024; };
  if (parted) {
    static_for<MI>([&](auto I) {
      static_for<NJ>([&](auto J) {
        i32x4 w0, w1;
        static_for<4>([&](auto TT) {
          const uint64_t bits = __builtin_bit_cast(uint64_t, value(I, J, TT));
          w0[decltype(TT)::value] = static_cast<int32_t>(static_cast<uint32_t>(bits));
          w1[decltype(TT)::value] = static_cast<int32_t>(static_cast<uint32_t>(bits >> 32));
        });
        constexpr int c = (decltype(I)::value * NJ + decltype(J)::value) * 2;
        store_coherent(block(wu.split, c), w0);
        store_coherent(block(wu.split, c + 1), w1);
      });
    });
    wait_vm_all();
    uint32_t old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(late.tickets + slot, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    old = __builtin_amdgcn_readfirstlane(old);
    if (old != static_cast<uint32_t>(splits - 1)) return;
    asm volatile("" ::: "memory");
    if (lane == 0) __hip_atomic_store(late.tickets + slot, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  auto run = [&](auto OUT, auto DT) __attribute__((always_inline)) {
    const bool interior = rw0 + 16 * MI <= m_lim && cw0 + 16 * NJ <= n_lim;
    const bool pairs = decltype(OUT)::value == kOutInt64 && interior && (e.out_ld & 1) == 0 &&
                       (reinterpret_cast<uintptr_t>(e.out) & 15) == 0;
    const bool quads = interior && float_quads_fit<RCAP>(e);
    static_for<MI>([&](auto I) {
      constexpr int i = decltype(I)::value;
      double rt[4];
      static_for<4>([&](auto TT) { rt[TT] = rterm[i * 16 + decltype(TT)::value]; });
      static_for<NJ>([&](auto J) {
        constexpr int j = decltype(J)::value;
        double x[4];
        static_for<4>([&](auto TT) { x[TT] = value(I, J, TT) + rt[TT]; });
        if (parted) {
          for (int s = 0; s < splits; ++s) {
            if (s == wu.split) continue;
            const i32x4 w0 = load_coherent(block(s, (i * NJ + j) * 2)), w1 = load_coherent(block(s, (i * NJ + j) * 2 + 1));
            static_for<4>([&](auto TT) {
              const uint64_t bits = (static_cast<uint64_t>(static_cast<uint32_t>(w1[decltype(TT)::value])) << 32) |
                                    static_cast<uint32_t>(w0[decltype(TT)::value]);
              x[TT] += __builtin_bit_cast(double, bits);
            });
          }
        }
        const int64_t idx = static_cast<int64_t>(rw0 + i * 16 + 4 * (lane >> 4)) * e.out_ld + cw0 + j * 16;
        if (pairs) {
          int64_t y[4];
          static_for<4>([&](auto TT) { y[TT] = frac_int<RCAP>(centered_mod(e, x[TT]) + kRoundMagic); });
          store_int64_pairs(y, as_global<int64_t>(e.out) + idx + (lane & 14), e.out_ld);
        } else if (quads) {
          if constexpr (decltype(OUT)::value == kOutFloat) {
            float f[4];
            static_for<4>([&](auto TT) { f[decltype(TT)::value] = static_cast<float>(centered_mod(e, x[TT])); });
            store_float_quads<RCAP, decltype(DT)::value>(e, f, cscale[j], idx + (lane & 3) * e.out_ld + (lane & 12));
          }
        } else {
          static_for<4>([&](auto TT) {
            constexpr int t = decltype(TT)::value;
            const int row = rw0 + i * 16 + 4 * (lane >> 4) + t, col = cw0 + j * 16 + (lane & 15);
            if (interior || (row < m_lim && col < n_lim))
              bytes_store<decltype(OUT)::value>(e, x[t], idx + t * e.out_ld + (lane & 15), cscale[j]);
          });
        }
      });
    });
  };
  if (e.out_dtype == RNSMX_INT64)
    run(std::integral_constant<int, kOutInt64>{}, std::integral_constant<int, RNSMX_INT64>{});
  else
    with_float_type<RCAP>(e, [&](auto DT) __attribute__((always_inline)) {
      run(std::integral_constant<int, kOutFloat>{}, DT);
    });
}

}  // namespace rnsmx
