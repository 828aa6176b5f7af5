// Kernel choice and launches of the GEMM family for one storage type; gemm_bf16.hip, gemm_f16.hip
// and gemm_f32.hip instantiate it (a translation unit per type, so that they compile side by side).
#pragma once

#include <type_traits>

#include "gemm_mfma.h"
#include "gemm_ring.h"
#include "gemm_stream64.h"
#include "gemm_f32.h"
#include "gemm_plan.h"

namespace tmb {

// ---------------------------------------------------------------------------
// SIMT fallback: any dtype / stride / alignment. 64x64 tile, BK = 16, 4x4 per thread.
// ---------------------------------------------------------------------------
template <typename T, int EPI>
__global__ __launch_bounds__(256) void gemm_simt_kernel(
    T* __restrict__ c, const T* __restrict__ a, const T* __restrict__ b,
    const T* __restrict__ bias, int64_t m, int64_t n, int64_t k, int64_t sa_m, int64_t sa_k,
    int64_t sb_k, int64_t sb_n, int64_t ldc, int64_t stride_a, int64_t stride_b,
    int64_t stride_c, int64_t tiles_n, bool twice) {
  constexpr int TM = 64, TN = 64, TK = 16;
  __shared__ float As[TK][TM + 4];
  __shared__ float Bs[TK][TN + 4];
  const int64_t batch = blockIdx.y;
  const int64_t tile = blockIdx.x;
  const int64_t tm = tile / tiles_n, tn = tile - tm * tiles_n;
  const int64_t m0 = tm * TM, n0 = tn * TN;
  a += batch * stride_a;
  b += batch * stride_b;
  c += batch * stride_c;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  float acc[4][4] = {};
  for (int64_t k0 = 0; k0 < k; k0 += TK) {
    // A tile: 64 rows x 16 k = 1024 elements, 4 per thread.
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = threadIdx.x + i * 256;
      int r, kk;
      if (sa_k == 1) { r = e >> 4; kk = e & 15; } else { r = e & 63; kk = e >> 6; }
      const int64_t gm = m0 + r, gk = k0 + kk;
      As[kk][r] = (gm < m && gk < k) ? to_f32(a[gm * sa_m + gk * sa_k]) : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = threadIdx.x + i * 256;
      int cidx, kk;
      if (sb_k == 1) { cidx = e >> 4; kk = e & 15; } else { cidx = e & 63; kk = e >> 6; }
      const int64_t gn = n0 + cidx, gk = k0 + kk;
      Bs[kk][cidx] = (gn < n && gk < k) ? to_f32(b[gk * sb_k + gn * sb_n]) : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; ++kk) {
      float av[4], bv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) bv[j] = Bs[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(av[i], bv[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t gm = m0 + ty * 4 + i;
    if (gm >= m) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t gn = n0 + tx * 4 + j;
      if (gn >= n) continue;
      float v = acc[i][j];
      if (bias != nullptr) v += to_f32(bias[gn]);
      c[gm * ldc + gn] = finish<T, EPI>(v, twice);
    }
  }
}

// Tile choice. 256x256 has the best reuse per byte staged through LDS, but it runs one workgroup
// per CU; narrow outputs and short-K products (attention's q.k^T and att.v) are load/store bound
// and want more, smaller workgroups in flight.
template <typename T, bool B_KMAJOR, int EPI>
static int mfma_pick_tile(const GemmArgs& g, int64_t batch, hipStream_t stream) {
  auto tiles = [&](int64_t bm, int64_t bn) { return ((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn) * batch; };
  // Direct-to-LDS ring kernel for long enough K. 256x256 (8 waves, 64-deep stages: every row
  // of a K-major operand is fetched as one whole 128-byte line) has the best steady state; it
  // is used when its tiles fill the 256 CUs in nearly whole rounds, otherwise smaller tiles cut
  // the idle tail. N-major B is staged in whole 16-byte column chunks, so N must be a multiple
  // of 8 there (nothing past column N-1 is ever read).
  if (g.k >= 256 && g.n > 64 && (B_KMAJOR || g.n % 8 == 0)) {
    const int64_t t256 = tiles(256, 256);
    // One partial round of 256 x 256 tiles (at least 144 of the 256 CUs busy) still beats smaller
    // tiles in several rounds: 16384 x 768 x 3072 runs in 66-72 us so, against 76-88 us with the
    // best smaller tile. (The 16x16x32 MFMA helps there from K = 2048 on with K-major B and from
    // K = 8192 on with N-major B: 16384 x 768 x 50304 runs in 1.05 against 1.14 ms.)
    if (g.k % 64 == 0 && t256 >= 144 && t256 <= 256 && t256 * 10 < 256 * 9) {
      if (g.k >= (B_KMAJOR ? 2048 : 8192))
        return launch_ring<T, 256, 256, 64, 2, 4, 2, B_KMAJOR, EPI, false, false, true>(g, batch, stream);
      return launch_ring<T, 256, 256, 64, 2, 4, 2, B_KMAJOR, EPI, false, false, false>(g, batch, stream);
    }
    // Short K: the prologue and epilogue of a tile weigh as much as its main loop, so rings that
    // leave room for two workgroups per CU (72 KB of LDS each) win by overlapping them.
    if (g.k % 32 == 0) {
      // (with the 16x16x32 MFMA and one fragment slot: four waves per SIMD, +2-4 %)
      if (!B_KMAJOR && g.k < 4096 && tiles(128, 256) >= 256)
        return launch_ring<T, 128, 256, 32, 2, 4, 3, B_KMAJOR, EPI, false, false, true>(g, batch, stream);
      // (K not a multiple of 64 only: the 64-deep form of this tile below is 5-10 % faster)
      if (B_KMAJOR && g.k % 64 != 0 && g.k <= 1024 && g.n <= 2304 && tiles(256, 128) >= 512)
        return launch_ring<T, 256, 128, 32, 4, 2, 3, B_KMAJOR, EPI>(g, batch, stream);
    }
    if (g.k % 64 == 0) {
      const int64_t rounds = (t256 + 255) / 256;
      if (t256 >= 768 || t256 * 10 >= rounds * 256 * 9) {
        // (the 16x16x32 MFMA: +3-6 % at long K, +2-4 % at K = 768 .. 3072; a short-K product
        // whose output streams to memory, as the 50257-wide vocabulary projection, loses 4 %)
        const bool streamed = g.m * g.n * batch * 2 >= (int64_t{256} << 20);
        if (g.k >= 4096 || !streamed)
          return launch_ring<T, 256, 256, 64, 2, 4, 2, B_KMAJOR, EPI, false, false, true>(g, batch, stream);
        return launch_ring<T, 256, 256, 64, 2, 4, 2, B_KMAJOR, EPI, false, false, false>(g, batch, stream);
      }
      // (from three quarters of a round on: 8192 x 768 x 3072 runs in 39-42 us here against
      // 50-55 us with 128 x 128 tiles)
      if (tiles(256, 128) >= 192)
        return launch_ring<T, 256, 128, 64, 4, 2, 3, B_KMAJOR, EPI>(g, batch, stream);
    }
    // (K that ends inside a stage: 1203 x 1024 x 2000 31.9 -> 17.5 us, N-major 36.7 -> 15.1, 700 x 3000 x 1416, N-major, 95
    // -> 17, 8192 x 8192 x 2024 428 -> 378; many K-major tiles run faster from registers, 9000 x 2304 x 1000 72 and 79)
    if (g.k % 64 == 0 || (g.k % 32 != 0 && (!B_KMAJOR || tiles(64, 128) <= 1024)) || tiles(256, 128) < 192) {
      switch (ring_one_round(batch, g.m, g.n, (g.k + 63) / 64 * 64, 0)) {
        case kRing64x128:
          return launch_ring<T, 64, 128, 64, 2, 4, 4, B_KMAJOR, EPI, false, false, true, true, true>(g, batch, stream);
        case kRing128x128:
          return launch_ring<T, 128, 128, 64, 2, 4, 3, B_KMAJOR, EPI, false, false, true, true, true>(g, batch, stream);
        default:  // (6800 x 768 x 3072, N-major: 55 us, 52 below)
          if (B_KMAJOR || g.k <= 1536 || g.k % 32 != 0 || tiles(64, 128) <= 512)
            return launch_ring<T, 64, 128, 64, 2, 4, 3, B_KMAJOR, EPI, false, false, true, false, true>(g, batch, stream);
      }
    }
    if (g.k % 32 == 0 && tiles(128, 128) >= 32) {
      // (16x16x32 MFMA, one k-step per 32-deep stage: +5-7 % for K-major B once the launch has
      // a few rounds of tiles; level or behind for small launches and for N-major B, whose
      // fragments need twice the LDS instructions; the 32-deep configurations that run four
      // waves per SIMD have no registers for its fragments at all)
      if constexpr (B_KMAJOR) {
        if (tiles(128, 128) >= 512)
          return launch_ring<T, 128, 128, 32, 2, 2, 4, B_KMAJOR, EPI, false, false, true>(g, batch, stream);
      }
      return launch_ring<T, 128, 128, 32, 2, 2, 4, B_KMAJOR, EPI>(g, batch, stream);
    }
  }
  // Up to 64 columns: the register-staged 256 x 64 tiles only where they give every CU one (32768 x 64 x 768 27 us on 128 of
  // them, 15.4 on 64 x 64 rings; 192 x 512 x 64 x 512 25 on 384, 32 on the rings). N-major columns that are not whole 64
  // never: 32768 x 48 x 768 66 and 15 us, 192 x 1024 x 32 x 1024 172 and 88.
  if (g.n <= 64 && g.k % 64 == 0 && g.k >= 256 && (B_KMAJOR || g.n % 8 == 0) &&
      (tiles(256, 64) <= 256 || (!B_KMAJOR && g.n % 64 != 0))) {
    if constexpr (B_KMAJOR) return launch_ring<T, 64, 64, 64, 2, 2, 4, true, EPI, false, false, true, true>(g, batch, stream);
    else return launch_ring<T, 64, 128, 64, 2, 4, 3, false, EPI>(g, batch, stream);
  }
  // Register-staged kernel for the rest (short K, K not a multiple of 32, ragged N-major N).
  if (g.n <= 64) return launch_mfma<T, 256, 64, 4, 1, B_KMAJOR, EPI>(g, batch, stream);
  if (g.k <= 128 || tiles(128, 128) >= 128)
    return launch_mfma<T, 128, 128, 2, 2, B_KMAJOR, EPI>(g, batch, stream);
  return launch_mfma<T, 64, 64, 2, 2, B_KMAJOR, EPI>(g, batch, stream);
}

template <typename T, int EPI>
static int launch_simt(const GemmArgs& g, int64_t batch, int trans_a, int trans_b,
                       hipStream_t stream) {
  const int64_t tiles_m = (g.m + 63) / 64, tiles_n = (g.n + 63) / 64;
  const int64_t tiles = tiles_m * tiles_n;
  if (tiles >= (int64_t{1} << 31) || batch > 65535) return TMB_ERR_UNSUPPORTED;
  const int64_t sa_m = trans_a ? 1 : g.lda, sa_k = trans_a ? g.lda : 1;
  const int64_t sb_k = trans_b ? 1 : g.ldb, sb_n = trans_b ? g.ldb : 1;
  gemm_simt_kernel<T, EPI><<<dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(batch)), dim3(256), 0, stream>>>(
      static_cast<T*>(g.c), static_cast<const T*>(g.a), static_cast<const T*>(g.b),
      static_cast<const T*>(g.bias), g.m, g.n, g.k, sa_m, sa_k, sb_k, sb_n, g.ldc, g.stride_a,
      g.stride_b, g.stride_c, tiles_n, g.round_like_unfused != 0);
  return check_launch();
}

// A stored [K, M] with B stored [K, N] (both "k-outer": the weight-gradient product dy^T x):
// the ring kernel stages A the way it stages N-major B. Needs whole 16-byte chunks along m and n
// and enough K for the ring.
template <typename T>
static int mfma_transposed_a(const GemmArgs& g, int64_t batch, hipStream_t stream) {
  const int64_t t256 = ((g.m + 255) / 256) * ((g.n + 255) / 256) * batch;
  // When the last round of 256 x 256 tiles would leave more than a fifth of the launch's slots
  // empty, 128 x 256 tiles on two workgroups per CU end with a shorter tail: the weight gradient
  // of a vocabulary projection, 50304 x 768 x 16384, runs in 1.11 against 1.23 ms.
  const int64_t rounds = (t256 + 255) / 256;
  const int64_t t128x256 = ((g.m + 127) / 128) * ((g.n + 255) / 256) * batch;
  if (t256 * 5 < rounds * 256 * 4 && t128x256 >= 512)
    return launch_ring<T, 128, 256, 32, 2, 4, 3, false, TMB_EPI_NONE, true, false, true>(g, batch, stream);
  if (g.k % 64 == 0 && t256 >= 192)
    return launch_ring<T, 256, 256, 64, 2, 4, 2, false, TMB_EPI_NONE, true>(g, batch, stream);
  // (from K = 2048 on in place of split launches: short chains, 4 .. 8 % of the time, 3072 x 768 x 2048 17.9 and 18.7 us)
  if (ring_one_round(batch, g.m, g.n, g.k, 1) != 0)
    return g.k >= 2048 ? launch_ring<T, 128, 128, 64, 4, 2, 3, false, TMB_EPI_NONE, true, false, false, true>(g, batch, stream)
                       : launch_ring<T, 128, 128, 64, 4, 2, 3, false, TMB_EPI_NONE, true, false, false>(g, batch, stream);
  return launch_ring<T, 128, 128, 32, 2, 2, 4, false, TMB_EPI_NONE, true>(g, batch, stream);
}

template <typename T, int EPI>
static int launch_splitk(const GemmArgs& g, const SplitKPlan& plan, int trans_a, int trans_b,
                         float* workspace, hipStream_t stream) {
  GemmArgs part = g;
  part.c = workspace;
  part.bias = nullptr;
  part.residual = nullptr;
  part.ldc = g.n;
  part.stride_c = g.m * g.n;
  part.stride_a = 0;
  part.stride_b = 0;
  part.splits = plan.splits;
  int rc;
  if (plan.tile == 256) {
    // (a split's run of K is short: the 32x32x16 MFMA, as for short unsplit products)
    if (trans_a)
      rc = launch_ring<T, 256, 256, 64, 2, 4, 2, false, TMB_EPI_NONE, true, true, false>(part, plan.splits, stream);
    else if (trans_b)
      rc = launch_ring<T, 256, 256, 64, 2, 4, 2, true, TMB_EPI_NONE, false, true, false>(part, plan.splits, stream);
    else
      rc = launch_ring<T, 256, 256, 64, 2, 4, 2, false, TMB_EPI_NONE, false, true, false>(part, plan.splits, stream);
  } else if (splitk_eight_waves(((g.m + 127) / 128) * ((g.n + 127) / 128), g.k, plan.splits)) {
    if (trans_a)
      rc = launch_ring<T, 128, 128, 64, 4, 2, 3, false, TMB_EPI_NONE, true, true, false>(part, plan.splits, stream);
    else if (trans_b)
      rc = launch_ring<T, 128, 128, 64, 4, 2, 3, true, TMB_EPI_NONE, false, true, false>(part, plan.splits, stream);
    else
      rc = launch_ring<T, 128, 128, 64, 4, 2, 3, false, TMB_EPI_NONE, false, true, false>(part, plan.splits, stream);
  } else if (trans_a) {
    rc = launch_ring<T, 128, 128, 32, 2, 2, 4, false, TMB_EPI_NONE, true, true>(part, plan.splits, stream);
  } else if (trans_b) {
    rc = launch_ring<T, 128, 128, 32, 2, 2, 4, true, TMB_EPI_NONE, false, true>(part, plan.splits, stream);
  } else {
    rc = launch_ring<T, 128, 128, 32, 2, 2, 4, false, TMB_EPI_NONE, false, true>(part, plan.splits, stream);
  }
  if (rc != 0) return rc;
  launch_splitk_reduce<T, EPI>(g.c, workspace, static_cast<const T*>(g.bias), g.m, g.n, g.ldc, plan.splits,
                               epilogue_args<T>(g, 0), stream);
  return check_launch();
}

template <int EPI>
static int launch_f32_shared(const GemmArgs& g, int64_t batch, int tile, int trans_a, int trans_b, hipStream_t stream) {
  if (g.k <= kF32SplitK) return launch_f32_tile<32, 32, 4, EPI, false>(g, batch, trans_a, trans_b, stream);
  switch (tile) {
    case 0:
      return ((g.m + 31) / 32) * ((g.n + 31) / 32) * batch <= 256
                 ? launch_f32_tile<32, 32, 8, EPI, true>(g, batch, trans_a, trans_b, stream)
                 : launch_f32_tile<32, 32, 4, EPI, true>(g, batch, trans_a, trans_b, stream);
    case 1: return launch_f32_tile<32, 64, 4, EPI, true>(g, batch, trans_a, trans_b, stream);
    case 2: return launch_f32_tile<64, 64, 4, EPI, true>(g, batch, trans_a, trans_b, stream);
    default: return launch_f32_tile<64, 64, 8, EPI, true>(g, batch, trans_a, trans_b, stream);
  }
}

// A split launch of `launch` into `workspace` and the reduction that adds bias, epilogue and residual.
template <typename T, int EPI, typename Launch>
static int launch_split(const GemmArgs& g, int splits, hipStream_t stream, void* workspace, const Launch& launch) {
  GemmArgs part = g;
  part.c = workspace;
  part.bias = nullptr;
  part.residual = nullptr;
  part.ldc = g.n;
  part.stride_c = g.m * g.n;
  part.splits = splits;
  const int rc = launch(part);
  if (rc != 0) return rc;
  launch_splitk_reduce<T, EPI>(g.c, static_cast<const float*>(workspace), static_cast<const T*>(g.bias), g.m, g.n,
                               g.ldc, splits, epilogue_args<T>(g, 0), stream);
  return check_launch();
}

template <typename T, int EPI>
static int gemm_typed(const GemmArgs& g, int64_t batch, int trans_a, int trans_b, hipStream_t stream, void* workspace,
                      size_t workspace_bytes) {
  const size_t scratch = workspace != nullptr ? workspace_bytes : 0;
  if constexpr (__is_same(T, float)) {
    const GemmRoute r = route_f32(g, batch, trans_a, trans_b, scratch);
    switch (r.kernel) {
      case TMB_GEMM_F32_WIDE:
        if (r.splits == 0) return launch_f32_wide<EPI>(g, batch, trans_a, trans_b, stream);
        return launch_split<T, EPI>(g, r.splits, stream, workspace, [&](const GemmArgs& part) {
          return launch_f32_wide<TMB_EPI_NONE>(part, r.splits, trans_a, trans_b, stream);
        });
      case TMB_GEMM_F32:
        if (r.splits == 0) return launch_f32_shared<EPI>(g, batch, r.tile, trans_a, trans_b, stream);
        return launch_split<T, EPI>(g, r.splits, stream, workspace, [&](const GemmArgs& part) {
          return launch_f32_shared<TMB_EPI_NONE>(part, r.splits, r.tile, trans_a, trans_b, stream);
        });
      case TMB_GEMM_SIMT: return launch_simt<T, EPI>(g, batch, trans_a, trans_b, stream);
      default: return TMB_ERR_UNSUPPORTED;
    }
  } else {
    constexpr bool BF16 = __is_same(T, bf16_t);
    const GemmRoute r = route_16bit(g, batch, trans_a, trans_b, EPI, scratch);
    switch (r.kernel) {
      case TMB_GEMM_SMALL: return gemm_small(g, batch, r.tile, trans_b, BF16, EPI, stream);
      case TMB_GEMM_SPLITK:
        return launch_splitk<T, EPI>(g, SplitKPlan{r.splits, r.tile == 1 ? 256 : 128, 0.0}, trans_a, trans_b,
                                     static_cast<float*>(workspace), stream);
      case TMB_GEMM_TRANSPOSED_A:
        if constexpr (EPI == TMB_EPI_NONE) return mfma_transposed_a<T>(g, batch, stream);
        // (the tile of one round, K >= 2048: no other form is asked for a GELU)
        else return launch_ring<T, 128, 128, 64, 4, 2, 3, false, EPI, true, false, false, true>(g, batch, stream);
      case TMB_GEMM_ANY:
        if (r.splits == 0) return gemm_any(g, batch, r.tile, trans_a, trans_b, BF16, EPI, stream);
        return launch_split<T, EPI>(g, r.splits, stream, workspace, [&](const GemmArgs& part) {
          return gemm_any(part, r.splits, r.tile, trans_a, trans_b, BF16, TMB_EPI_NONE, stream);
        });
      case TMB_GEMM_STREAM64:
        return trans_b ? launch_stream64<T, true>(g, batch, stream) : launch_stream64<T, false>(g, batch, stream);
      case TMB_GEMM_RING:
        return trans_b ? mfma_pick_tile<T, true, EPI>(g, batch, stream) : mfma_pick_tile<T, false, EPI>(g, batch, stream);
      case TMB_GEMM_SIMT: return launch_simt<T, EPI>(g, batch, trans_a, trans_b, stream);
      default: return TMB_ERR_UNSUPPORTED;
    }
  }
}

template <typename T>
int gemm_epi(const GemmArgs& g, int64_t batch, int ta, int tb, int epilogue,
                    hipStream_t stream, void* ws, size_t ws_bytes) {
  switch (epilogue) {
    case TMB_EPI_NONE: return gemm_typed<T, TMB_EPI_NONE>(g, batch, ta, tb, stream, ws, ws_bytes);
    case TMB_EPI_GELU_TANH: return gemm_typed<T, TMB_EPI_GELU_TANH>(g, batch, ta, tb, stream, ws, ws_bytes);
    case TMB_EPI_GELU_ERF: return gemm_typed<T, TMB_EPI_GELU_ERF>(g, batch, ta, tb, stream, ws, ws_bytes);
    default: return TMB_ERR_INVALID_ARGUMENT;
  }
}

}  // namespace tmb
