// MFMA GEMM for products that leave most of the chip idle in the ring kernels (16-bit storage,
// A [M, K] with K contiguous): a few hundred rows or fewer, as in a decode step, a short prompt or
// the layers of a small batch.
//
// What bounds such a product is latency: a 128 x 128 tile walks its K alone, stage after stage,
// each behind a workgroup barrier, on a handful of CUs. Here a workgroup owns a small tile
// (BM x BN, 16 .. 64 each way) and its WAVES waves share K between them: wave w multiplies the
// 64-deep slices w, w + WAVES, ... of the whole tile, so a wave has all its operands in flight at
// once and no barrier stands between a load and its MFMAs. The fp32 partial tiles meet in LDS once,
// are added pairwise in wave order (the result depends on the shape only) and leave through one epilogue
// (bias, GELU, residual), which also spares these shapes the second launch of a split-K product.
//
// A wave brings its slices in as whole 128-byte lines (eight lanes to a line), lays them into a
// wave-private part of LDS and reads the MFMA operands from there; the LDS works in order per wave,
// so no workgroup barrier is needed, only a point the compiler moves no LDS access across. (Loading operand fragments straight into registers, 16 rows of
// 64 bytes per instruction, ran 20-25 % slower at K = 3072: half-line requests.) B stored [K, N] is
// laid down as it lies in memory and read back transposed with ds_read_b64_tr_b16.
#pragma once

#include "gemm_mfma.h"

namespace tmb {

// LDS of one wave. A line of a K-major operand takes 144 bytes (the 16 rows of a fragment read then
// lie on 16 distinct bank groups), a k-row of an N-major B 16 bytes more than its columns (which
// spreads the four rows of a transposed read, and the groups of lanes eight rows apart).
template <int BM, int BN, bool B_KMAJOR>
struct SmallLds {
  static constexpr int LINE = 128 + 16;
  static constexpr int PITCH = B_KMAJOR ? LINE : BN * 2 + 16;
  static constexpr int A_BYTES = BM * LINE;
  static constexpr int SLICE = A_BYTES + (B_KMAJOR ? BN : 64) * PITCH;
};

template <typename T, int EPI>
__device__ __forceinline__ void small_epilogue4(const float (&sum)[4], const GemmArgs& g, const EpilogueArgs& ep,
                                                int64_t batch, int64_t row, int64_t col) {
  const T* __restrict__ bias = static_cast<const T*>(g.bias);
  const u32x2_t b4 = load_bias4<T>(bias, col, g.n);
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = sum[e] + unpack_elem<T>(b4, e);
  const bool whole = col + 4 <= g.n;
  const int64_t at = batch * g.stride_c + row * g.ldc + col;
  if (EPI == TMB_EPI_NONE && ep.wide()) {  // wave-uniform: fp32 up to the one cast
    const int64_t rat = row * ep.ldr + col;
    if (ep.resid_f32) {
      const float* r = static_cast<const float*>(ep.residual) + rat;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (whole || col + e < g.n) v[e] += r[e];
    } else {
      const T* r = static_cast<const T*>(ep.residual) + rat;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (whole || col + e < g.n) v[e] += to_f32(r[e]);
    }
    if (ep.out_f32) {
      float* c = static_cast<float*>(g.c) + at;
      if (whole) {
        const f32x4_unaligned_t o = {v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4_unaligned_t*>(c) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < g.n) c[e] = v[e];
      }
      return;
    }
  }
  u32x2_t out;
  if (EPI == TMB_EPI_NONE && ep.wide()) {
    out[0] = pack2<T>(v[0], v[1]);
    out[1] = pack2<T>(v[2], v[3]);
  } else {
    out[0] = finish2<T, EPI>(v[0], v[1], ep.twice);
    out[1] = finish2<T, EPI>(v[2], v[3], ep.twice);
    if (ep.residual != nullptr) {  // rounded after every step: T(T(epilogue) + residual)
      const T* r = static_cast<const T*>(ep.residual) + row * ep.ldr + col;
      u32x2_t r4 = {0u, 0u};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (whole || col + e < g.n)
          r4[e >> 1] |= static_cast<uint32_t>(__builtin_bit_cast(unsigned short, r[e])) << (16 * (e & 1));
      out[0] = add_pair<T>(out[0], r4[0]);
      out[1] = add_pair<T>(out[1], r4[1]);
    }
  }
  T* c = static_cast<T*>(g.c) + at;
  if (whole) {
    *reinterpret_cast<u32x2_unaligned_t*>(c) = out;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < g.n) c[e] = __builtin_bit_cast(T, static_cast<unsigned short>(out[e >> 1] >> (16 * (e & 1))));
  }
}

template <typename T, int BM, int BN, int WAVES, bool B_KMAJOR, int EPI>
__global__ __launch_bounds__(WAVES * 64) void gemm_small_kernel(GemmArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  using L = SmallLds<BM, BN, B_KMAJOR>;
  constexpr int KS = 64;                     // depth of a slice: one 128-byte line
  constexpr int TM = BM / 16, TN = BN / 16;
  constexpr int BROWS = 512 / BN;            // k-rows one 16-byte load per lane covers (N-major B)
  constexpr int ALOADS = BM / 8, BLOADS = BN / 8;
  constexpr int RP = BN + 4;                 // floats per row of a partial tile in LDS
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int tile_m, tile_n;
  tile_of_block(blockIdx.x, g.tiles_m, g.tiles_n, tile_m, tile_n);
  const int64_t m0 = static_cast<int64_t>(tile_m) * BM, n0 = static_cast<int64_t>(tile_n) * BN;
  const int64_t batch = blockIdx.y;
  const int64_t M = g.m, N = g.n, K = g.k;
  const unsigned char* a_base = reinterpret_cast<const unsigned char*>(static_cast<const T*>(g.a) + batch * g.stride_a);
  const unsigned char* b_base = reinterpret_cast<const unsigned char*>(static_cast<const T*>(g.b) + batch * g.stride_b);

  // Lane offsets from the operand's base; rows past the edge re-read the last one (never stored).
  const int line = lane >> 3, chunk = lane & 7;
  uint32_t a_off[ALOADS], b_off[BLOADS];
#pragma unroll
  for (int i = 0; i < ALOADS; ++i) {
    int64_t row = m0 + i * 8 + line;
    row = row < M ? row : M - 1;
    a_off[i] = static_cast<uint32_t>((row * g.lda + chunk * 8) * 2);
  }
#pragma unroll
  for (int j = 0; j < BLOADS; ++j) {
    if constexpr (B_KMAJOR) {
      int64_t row = n0 + j * 8 + line;
      row = row < N ? row : N - 1;
      b_off[j] = static_cast<uint32_t>((row * g.ldb + chunk * 8) * 2);
    } else {
      const int64_t krow = j * BROWS + lane / (BN / 8);
      int64_t col = n0 + (lane % (BN / 8)) * 8;
      col = col < N ? col : n0;
      b_off[j] = static_cast<uint32_t>((krow * g.ldb + col) * 2);
    }
  }
  const int64_t b_kstep = B_KMAJOR ? 2 : g.ldb * 2;  // bytes per unit of k

  f32x4v_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4v_t{0.0f, 0.0f, 0.0f, 0.0f};

  u32x4_t a_reg[ALOADS], b_reg[BLOADS];
  auto load = [&](int64_t slice) {
    const int64_t k0 = slice * KS;
    const unsigned char* ak = a_base + k0 * 2;
    const unsigned char* bk = b_base + k0 * b_kstep;
    if (k0 + KS <= K) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < ALOADS; ++i) a_reg[i] = *reinterpret_cast<const u32x4_t*>(ak + a_off[i]);
#pragma unroll
      for (int j = 0; j < BLOADS; ++j) b_reg[j] = *reinterpret_cast<const u32x4_t*>(bk + b_off[j]);
    } else {  // the last slice of a K that is no multiple of 64: zeros past K (K % 8 == 0)
      const u32x4_t zero4 = {0u, 0u, 0u, 0u};
      const bool in = k0 + chunk * 8 < K;
#pragma unroll
      for (int i = 0; i < ALOADS; ++i) a_reg[i] = in ? *reinterpret_cast<const u32x4_t*>(ak + a_off[i]) : zero4;
#pragma unroll
      for (int j = 0; j < BLOADS; ++j) {
        const bool b_in = B_KMAJOR ? in : k0 + j * BROWS + lane / (BN / 8) < K;
        b_reg[j] = b_in ? *reinterpret_cast<const u32x4_t*>(bk + b_off[j]) : zero4;
      }
    }
  };
  lds_byte_t* mine = (lds_byte_t*)smem + wave * L::SLICE;
  const int fr = lane & 15, fq = lane >> 4;  // row of a fragment, which eight of its 32 k
  auto lay_down = [&]() {
#pragma unroll
    for (int i = 0; i < ALOADS; ++i) *(lds_u32x4v_t*)(mine + (i * 8 + line) * L::LINE + chunk * 16) = a_reg[i];
#pragma unroll
    for (int j = 0; j < BLOADS; ++j) {
      const int at = B_KMAJOR ? (j * 8 + line) * L::PITCH + chunk * 16
                              : (j * BROWS + lane / (BN / 8)) * L::PITCH + (lane % (BN / 8)) * 16;
      *(lds_u32x4v_t*)(mine + L::A_BYTES + at) = b_reg[j];
    }
  };
  auto multiply = [&]() {
    typedef short i16x4s_t __attribute__((ext_vector_type(4)));
    typedef short i16x8s_t __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) i16x4s_t lds_i16x4s_t;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4_t af[TM];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[i] = *(const lds_u32x4v_t*)(mine + (i * 16 + fr) * L::LINE + h * 64 + fq * 16);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        u32x4_t bf;
        if constexpr (B_KMAJOR) {
          bf = *(const lds_u32x4v_t*)(mine + L::A_BYTES + (j * 16 + fr) * L::PITCH + h * 64 + fq * 16);
        } else {
          lds_byte_t* src = mine + L::A_BYTES + (h * 32 + fq * 8 + (fr >> 2)) * L::PITCH + (fr & 3) * 8 + j * 32;
          const i16x4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4s_t*)(src));
          const i16x4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4s_t*)(src + 4 * L::PITCH));
          bf = __builtin_bit_cast(u32x4_t, i16x8s_t(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)));
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[i][j] = Mfma16<T>::run(bf, af[i], acc[i][j]);
      }
    }
  };

  const int64_t slices = (K + KS - 1) / KS;
  if (wave < slices) load(wave);
  for (int64_t at = wave; at < slices; at += WAVES) {
    lay_down();
    wave_lds_point();
    if (at + WAVES < slices) load(at + WAVES);
    multiply();
    wave_lds_point();
  }

  // A lane holds row lane % 16 and four consecutive columns of each 16 x 16 result.
  __syncthreads();  // the partial tiles overlay the slices
  float* part = reinterpret_cast<float*>(smem) + wave * (BM * RP);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      *reinterpret_cast<f32x4v_t*>(part + (i * 16 + fr) * RP + j * 16 + fq * 4) = acc[i][j];
  __syncthreads();
  const EpilogueArgs ep = epilogue_args<T>(g, batch);
  const float* all = reinterpret_cast<const float*>(smem);
#pragma unroll
  for (int p = 0; p < (BM * BN / 4 + WAVES * 64 - 1) / (WAVES * 64); ++p) {
    const int idx = p * WAVES * 64 + tid;
    if ((BM * BN / 4) % (WAVES * 64) != 0 && idx >= BM * BN / 4) break;
    const int r = idx / (BN / 4), c = (idx % (BN / 4)) * 4;
    const int64_t row = m0 + r, col = n0 + c;
    if (row >= M || col >= N) continue;
    // pairwise: a short chain of adds, and the rounding of log2(WAVES) of them instead of WAVES
    f32x4v_t v[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v[w] = *reinterpret_cast<const f32x4v_t*>(all + w * (BM * RP) + r * RP + c);
#pragma unroll
    for (int step = 1; step < WAVES; step *= 2)
#pragma unroll
      for (int w = 0; w < WAVES; w += 2 * step)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[w][e] += v[w + step][e];
    const float sum[4] = {v[0][0], v[0][1], v[0][2], v[0][3]};
    small_epilogue4<T, EPI>(sum, g, ep, batch, row, col);
  }
#endif
}

template <typename T, int BM, int BN, int WAVES, bool B_KMAJOR, int EPI>
static int launch_small(const GemmArgs& base, int64_t batch, hipStream_t stream) {
  constexpr int PARTS = WAVES * BM * (BN + 4) * 4;
  constexpr int STAGED = WAVES * SmallLds<BM, BN, B_KMAJOR>::SLICE;
  constexpr int SMEM = PARTS > STAGED ? PARTS : STAGED;
  static_assert(SMEM <= 160 * 1024, "LDS of one CU");
  auto kernel = gemm_small_kernel<T, BM, BN, WAVES, B_KMAJOR, EPI>;
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
    if (e != hipSuccess) return static_cast<int>(e);
    configured = true;
  }
  GemmArgs g = base;
  g.tiles_m = static_cast<int>((g.m + BM - 1) / BM);
  g.tiles_n = static_cast<int>((g.n + BN - 1) / BN);
  const int64_t tiles = static_cast<int64_t>(g.tiles_m) * g.tiles_n;
  if (tiles >= (int64_t{1} << 31) || batch > 65535) return TMB_ERR_UNSUPPORTED;
  kernel<<<dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(batch)), dim3(WAVES * 64), SMEM, stream>>>(g);
  return check_launch();
}

}  // namespace tmb
