// Decode in one launch: a few rows of float activations quantized inside the
// weight-streaming product (RNSLinear.forward), and a few requests' rows read
// where they lie (continuous batching).
#include "rnsmx_gemm.hpp"
#include "rnsmx_quant.hpp"

namespace rnsmx {

// The product's arguments first: kernel_args reads them in place.
struct LinearRowsArgs {
  GemmArgsK<4> g;  // m rows of a_k = K values, b, the epilogue
  QuantArgs q;     // x, vec, qmax, rcp
};

// A workgroup of 4 waves (3 where K holds no more chunks) owns 16 columns and
// every row (up to 16), the waves splitting K as in stream_kernel.  The first
// weight chunk is in flight before anything else; while it travels the
// workgroup reads all the activations (at most kLinearRowsValues, from L2 after
// the first), takes their maximum, quantizes them and leaves the int8 rows in
// LDS (rows of kp + 16 bytes, zero past K, so a fragment's 16 rows do not share
// banks), from where every K step takes its A fragment.  The next chunk is
// loaded while one computes.  Quantizing once per workgroup costs less than the
// launch it saves: the layer at 768 x 2304, 1 row, spent 2.6 of its 13 us on the
// quantizer's kernel and 3 on its launch.
// NT: weights with the streaming hint (long K, as stream_kernel).
constexpr int kLinearRowsMax = 16;
constexpr int kLinearRowsValues = 8192;

template <typename T, bool NT>
__global__ __launch_bounds__(256) void linear_rows_kernel(const LinearRowsArgs args) {
  constexpr int RCAP = 4, U = 4;
  using R = QuantRaw<T>;
  constexpr int V = 16 / sizeof(R);
  constexpr int IT = (kLinearRowsValues / V + 191) / 192;  // vectors per thread (3 waves at least)
  KArgs<RCAP> &g = kernel_args<GemmArgsK<RCAP>>();
  const QuantArgs &qa = args.q;
  prefetch_kernel_args<static_cast<int>(sizeof(LinearRowsArgs))>();
  __shared__ int32_t sums[RCAP][256];
  __shared__ float wmax[4];
  extern __shared__ __attribute__((aligned(16))) int8_t rows_q[];  // [m][kp + 16]

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nthreads = g.threads, ks_n = nthreads >> 6;
  const int n0 = blockIdx.x * 16, nk = g.kp >> 6, k = g.a_k, m = g.m;
  const int ldk = g.kp + 16;
  const int8_t *bp = g.b + static_cast<int64_t>(blockIdx.x) * g.b_ld + lane * 16;
  const int64_t b_cs = g.b_cs;

  i32x4 fb[2][U][RCAP];
  auto load_chunk = [&](auto BUF, int q) {
    static_for<U>([&](auto UU) {
      const int ks = min(q + decltype(UU)::value, nk - 1);
      static_for<RCAP>([&](auto C) {
        const int8_t *p = bp + decltype(C)::value * b_cs + ks * 1024;
        fb[decltype(BUF)::value][decltype(UU)::value][decltype(C)::value] = NT ? load16_nt(p) : load16(p);
      });
    });
  };
  constexpr std::integral_constant<int, 0> b0{};
  constexpr std::integral_constant<int, 1> b1{};
  int q = wave * U;
  const int stride = ks_n * U;
  load_chunk(b0, q);

  // activations: 16-byte vectors kept in registers where rows hold whole ones
  const R *x = static_cast<const R *>(qa.x);
  const int count = m * k;
  const bool vec = qa.vec != 0 && k % V == 0;
  const int kv = k / V, nvec = m * kv;
  R v[IT][V];
  float amax = 0.0f;
  bool nan = false;
  auto visit = [&](float f) {
    amax = fmaxf(amax, fabsf(f));
    nan |= f != f;
  };
  if (vec) {
    static_for<IT>([&](auto I) {
      const int i = tid + decltype(I)::value * nthreads;
      uint4 w = {0u, 0u, 0u, 0u};
      if (i < nvec) w = reinterpret_cast<const uint4 *>(x)[i];
      *reinterpret_cast<uint4 *>(v[decltype(I)::value]) = w;
    });
  }
  for (int i = tid; i < RCAP * 256; i += nthreads) (&sums[0][0])[i] = 0;
  for (int i = tid * 4; i < m * ldk; i += nthreads * 4) *reinterpret_cast<uint32_t *>(rows_q + i) = 0;
  if (vec) {
    static_for<IT>([&](auto I) {
      static_for<V>([&](auto E) { visit(QuantIn<T>::get(v[decltype(I)::value][decltype(E)::value])); });
    });
  } else {
    for (int i = tid; i < count; i += nthreads) visit(QuantIn<T>::get(x[i]));
  }
  amax = nan ? __builtin_nanf("") : amax;
  for (int off = 32; off > 0; off >>= 1) amax = max_nan(amax, __shfl_xor(amax, off, 64));
  if (lane == 0) wmax[wave] = amax;
  __syncthreads();
  amax = wmax[0];
  for (int w = 1; w < ks_n; ++w) amax = max_nan(amax, wmax[w]);
  const float s = quant_scale(amax, qa.rcp), qmax = qa.qmax;
  auto quant = [&](R raw) {
    return static_cast<uint32_t>(static_cast<int32_t>(quant_value(QuantIn<T>::get(raw), s, qmax))) & 0xFFu;
  };
  if (vec) {
    static_for<IT>([&](auto I) {
      const int i = tid + decltype(I)::value * nthreads;
      if (i < nvec) {
        const int row = i / kv, c = i - row * kv;
        uint32_t w[V / 4];
        static_for<V / 4>([&](auto W) {
          constexpr int e = 4 * decltype(W)::value;
          const R *r = v[decltype(I)::value];
          w[decltype(W)::value] = quant(r[e]) | (quant(r[e + 1]) << 8) | (quant(r[e + 2]) << 16) | (quant(r[e + 3]) << 24);
        });
        uint32_t *to = reinterpret_cast<uint32_t *>(rows_q + row * ldk + c * V);
        static_for<V / 4>([&](auto W) { to[decltype(W)::value] = w[decltype(W)::value]; });
      }
    });
  } else {
    for (int i = tid; i < count; i += nthreads) {
      const int row = i / k;
      rows_q[row * ldk + (i - row * k)] = static_cast<int8_t>(quant(x[i]));
    }
  }
  Epi<RCAP> e;
  load_epi<RCAP>(g, e, g.mods.channels);
  e.a_scale = s;
  const int n_lim = g.n;
  const ColScale cs = col_scale<RCAP>(e, n0 + (tid & 15), n_lim);
  __syncthreads();

  i32x4 acc[RCAP];
  static_for<RCAP>([&](auto C) { acc[decltype(C)::value] = acc_zero(); });
  const int8_t *ap = rows_q + min(lane & 15, m - 1) * ldk + (lane >> 4) * 16;
  auto mfma_chunk = [&](auto BUF, int at) {
    static_for<U>([&](auto UU) {
      constexpr int u = decltype(UU)::value;
      if (at + u >= nk) return;
      const i32x4 fa = *reinterpret_cast<const i32x4 *>(ap + (at + u) * 64);
      static_for<RCAP>([&](auto C) {
        constexpr int c = decltype(C)::value;
        acc[c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa, fb[decltype(BUF)::value][u][c], acc[c], 0, 0, 0);
      });
    });
  };
  while (q < nk) {
    if (q + stride < nk) load_chunk(b1, q + stride);
    mfma_chunk(b0, q);
    q += stride;
    if (q >= nk) break;
    if (q + stride < nk) load_chunk(b0, q + stride);
    mfma_chunk(b1, q);
    q += stride;
  }
  static_for<RCAP>([&](auto C) {
    static_for<4>([&](auto TT) {
      constexpr int c = decltype(C)::value, t = decltype(TT)::value;
      const int r = 4 * (lane >> 4) + t;
      if (r < m) atomicAdd(&sums[c][r * 16 + (lane & 15)], acc[c][t]);
    });
  });
  __syncthreads();
  // one element per thread, two trips where three waves serve more than 12 rows
  for (int at = tid; at < m * 16; at += nthreads) {
    const int col = n0 + (at & 15);
    if (col >= n_lim) continue;
    int32_t sum[RCAP];
    static_for<RCAP>([&](auto C) { sum[decltype(C)::value] = sums[decltype(C)::value][at]; });
    store_float<RCAP>(e, frac_float<RCAP>(frac_sum<RCAP>(e, sum)), static_cast<int64_t>(at >> 4) * e.out_ld + col, cs);
  }
}

template <typename T>
static void launch_linear_t(const LinearRowsArgs &a, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>((a.g.n + 15) / 16)), block(static_cast<unsigned>(a.g.threads));
  const size_t lds = static_cast<size_t>(a.g.m) * (a.g.kp + 16);
  if (a.g.kp >= 4096)
    hipLaunchKernelGGL((linear_rows_kernel<T, true>), grid, block, lds, st, a);
  else
    hipLaunchKernelGGL((linear_rows_kernel<T, false>), grid, block, lds, st, a);
}

// ---------------------------------------------------------------------------
// Continuous batching: the rows of several requests (int8, up to 16 rows in
// all) against one prepared weight, each row read through its own pointer, so
// nothing is concatenated first.  Workgroups and waves as above; A fragments
// come straight from the rows with the weight loads of their chunk.  The rows
// are also copied to the staging buffer (a row per workgroup), which a caller
// finds filled as after a concatenation.
// 4 requests of 1 row, 768 x 768: 4.7 us of a call's 19 were the concatenation.
// ---------------------------------------------------------------------------
struct RequestRowsArgs {
  GemmArgsK<4> g;
  const int8_t *row[kLinearRowsMax];
  int8_t *staging;  // [m][K]
};

template <bool NT>
__global__ __launch_bounds__(256) void request_rows_kernel(const RequestRowsArgs args) {
  constexpr int RCAP = 4, U = 4;
  KArgs<RCAP> &g = kernel_args<GemmArgsK<RCAP>>();
  RNSMX_KARG(RequestRowsArgs) &all = kernel_args<RequestRowsArgs>();
  prefetch_kernel_args<static_cast<int>(sizeof(RequestRowsArgs))>();
  __shared__ int32_t sums[RCAP][256];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nthreads = g.threads, ks_n = nthreads >> 6;
  const int n0 = blockIdx.x * 16, nk = g.kp >> 6, a_k = g.a_k, m = g.m;
  const int8_t *bp = g.b + static_cast<int64_t>(blockIdx.x) * g.b_ld + lane * 16;
  const int64_t b_cs = g.b_cs;
  const int mine = min(lane & 15, m - 1);
  const int8_t *ap = all.row[0];
  static_for<kLinearRowsMax - 1>([&](auto I) {
    constexpr int i = decltype(I)::value + 1;
    if (mine == i) ap = all.row[i];
  });
  const int kofs = (lane >> 4) * 16;

  i32x4 fa[2][U], fb[2][U][RCAP];
  auto load_chunk = [&](auto BUF, int q) {
    static_for<U>([&](auto UU) {
      constexpr int buf = decltype(BUF)::value, u = decltype(UU)::value;
      const int ks = min(q + u, nk - 1);
      const int ka = ks * 64 + kofs;
      fa[buf][u] = load16(ap + min(ka, a_k - 16));  // past K: zeroed at its use
      static_for<RCAP>([&](auto C) {
        const int8_t *p = bp + decltype(C)::value * b_cs + ks * 1024;
        fb[buf][u][decltype(C)::value] = NT ? load16_nt(p) : load16(p);
      });
    });
  };
  constexpr std::integral_constant<int, 0> b0{};
  constexpr std::integral_constant<int, 1> b1{};
  int q = wave * U;
  const int stride = ks_n * U;
  load_chunk(b0, q);
  for (int i = tid; i < RCAP * 256; i += nthreads) (&sums[0][0])[i] = 0;
  for (int r = blockIdx.x; r < m; r += gridDim.x) {
    const int8_t *from = all.row[0];
    static_for<kLinearRowsMax - 1>([&](auto I) {
      constexpr int i = decltype(I)::value + 1;
      if (r == i) from = all.row[i];
    });
    int8_t *to = all.staging + static_cast<int64_t>(r) * a_k;
    for (int i = tid * 16; i < a_k; i += nthreads * 16) *reinterpret_cast<i32x4 *>(to + i) = load16(from + i);
  }
  Epi<RCAP> e;
  load_epi<RCAP>(g, e, g.mods.channels);
  const int n_lim = g.n;
  i32x4 acc[RCAP];
  static_for<RCAP>([&](auto C) { acc[decltype(C)::value] = acc_zero(); });
  auto mfma_chunk = [&](auto BUF, int at) {
    static_for<U>([&](auto UU) {
      constexpr int buf = decltype(BUF)::value, u = decltype(UU)::value;
      if (at + u >= nk) return;
      const i32x4 a = select16((at + u) * 64 + kofs < a_k, fa[buf][u]);
      static_for<RCAP>([&](auto C) {
        constexpr int c = decltype(C)::value;
        acc[c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, fb[buf][u][c], acc[c], 0, 0, 0);
      });
    });
  };
  while (q < nk) {
    if (q + stride < nk) load_chunk(b1, q + stride);
    mfma_chunk(b0, q);
    q += stride;
    if (q >= nk) break;
    if (q + stride < nk) load_chunk(b0, q + stride);
    mfma_chunk(b1, q);
    q += stride;
  }
  __syncthreads();
  static_for<RCAP>([&](auto C) {
    static_for<4>([&](auto TT) {
      constexpr int c = decltype(C)::value, t = decltype(TT)::value;
      const int r = 4 * (lane >> 4) + t;
      if (r < m) atomicAdd(&sums[c][r * 16 + (lane & 15)], acc[c][t]);
    });
  });
  __syncthreads();
  for (int at = tid; at < m * 16; at += nthreads) {
    const int col = n0 + (at & 15);
    if (col >= n_lim) continue;
    int32_t sum[RCAP];
    static_for<RCAP>([&](auto C) { sum[decltype(C)::value] = sums[decltype(C)::value][at]; });
    store_value<RCAP, kOutInt64>(e, frac_int<RCAP>(frac_sum<RCAP>(e, sum)),
                                 static_cast<int64_t>(at >> 4) * e.out_ld + col, ColScale{0.0f, 0.0f});
  }
}

bool request_rows_fits(int64_t rows, int64_t k, const rnsmx_moduli_t &mods, int32_t a_dtype) {
  return a_dtype == RNSMX_INT8 && mods.channels == 4 && rows >= 1 && rows <= kLinearRowsMax && k % 16 == 0 &&
         raw_accumulator_fits(mods, k);
}

void launch_request_rows(const GemmArgs &g, const int8_t *const *row, int8_t *staging, hipStream_t st) {
  RequestRowsArgs a{};
  a.g = compact_args<4>(g);
  for (int i = 0; i < kLinearRowsMax; ++i) a.row[i] = row[i < g.m ? i : 0];
  a.staging = staging;
  const int chunks = (g.kp / 64 + 3) / 4;
  a.g.threads = 64 * (chunks < 4 ? 3 : 4);
  const dim3 grid(static_cast<unsigned>((g.n + 15) / 16)), block(static_cast<unsigned>(a.g.threads));
  if (g.kp >= 4096)
    hipLaunchKernelGGL(request_rows_kernel<true>, grid, block, 0, st, a);
  else
    hipLaunchKernelGGL(request_rows_kernel<false>, grid, block, 0, st, a);
}

// Every workgroup quantizes all M K values, so the launches saved pay for M K N
// up to a line: against the quantizer's kernels and the product, float16
// (device time), 4 x 768 x 8192 9.6 -> 9.2 us but 8 x 768 x 4571 8.0 -> 8.4;
// from K = 1024, where those spend longer, 4 x 2048 x 4571 14.0 -> 11.3 but
// 8 x 1024 x 8192 11.8 -> 12.1; N = 12288, 1 row, 768 11.1 -> 11.6.  Values that
// are not read 16 bytes at a time (K no multiple of 16, or the first off a
// 16-byte boundary) cost more each: 4 x 1001 x 8192 16.5 -> 14.7 us, 8 x 662 x
// 2304 10.4 -> 11.3.
bool linear_rows_fits(int64_t rows, int64_t k, int64_t n, const rnsmx_moduli_t &mods, int32_t quant_bits,
                      bool adaptive, bool aligned) {
  if (quant_bits != 8 || adaptive || mods.channels != 4 || rows < 1 || rows > kLinearRowsMax || n < 1 || n > 8192 ||
      rows * k > kLinearRowsValues || !raw_accumulator_fits(mods, k))
    return false;
  if (!aligned || k % 16 != 0) return rows * k <= kLinearRowsValues / 2;
  return k < 1024 ? rows * k * n <= 24 << 20 : rows * k * n < 64 << 20;
}

void launch_linear_rows(const GemmArgs &g, const QuantArgs &q, int32_t x_dtype, hipStream_t st) {
  LinearRowsArgs a{compact_args<4>(g), q};
  const int chunks = (g.kp / 64 + 3) / 4;
  a.g.threads = 64 * (chunks < 4 ? 3 : 4);
  switch (x_dtype) {
    case RNSMX_FLOAT16: launch_linear_t<__half>(a, st); break;
    case RNSMX_BFLOAT16: launch_linear_t<Bf16Bits>(a, st); break;
    default: launch_linear_t<float>(a, st); break;
  }
}

}  // namespace rnsmx
