// 16-bit MFMA GEMM that takes its operands as they lie: any of the four layouts (A [M, K] or [K, M],
// B [N, K] or [K, N]), any row pitch, any 2-byte aligned address, any extents of eight or more along
// the contiguous directions.
//
// The ring and small kernels move operands in aligned 16-byte vectors; a vocabulary of 50257, 750 rows
// of a ragged batch as the K of a weight gradient, or 1001 classes had to be copied into padded buffers
// first, which for all but the largest products takes longer than the product. The structure is the
// small kernel's (gemm_small.h): a workgroup owns a BM x BN tile, its WAVES waves take every WAVES-th
// 64-deep slice of K each, through registers and a wave-private part of LDS, and the fp32 partial tiles
// meet in LDS once, added pairwise in wave order (the result depends on the shape only). What bounds it
// is the rate at which L2 serves 16-byte pieces that straddle its lines.
//
// Measured against padded copies and the ring kernels (or, below 2^26 multiply-adds, the any-layout vector
// kernel): 12 x 273 x 7011 904 -> 5.5 us, 43 x 3065 x 478 72 -> 4.8, 768 x 768 x 750 with both operands
// K-outer 21 -> 9, 511 x 3174 x 1396 48 -> 26, 1001 x 1500 x 1999 (a weight gradient) 61 -> 33. Large
// products stay with the copies (4099^3 197 us, here 348): gemm_plan.h compares the two.
//
// An operand with K contiguous is laid down as lines of 64 k and read back 16 bytes a lane; one with its
// M or N extent contiguous is laid down as k-rows and read back transposed (ds_read_b64_tr_b16).
#pragma once

#include "gemm_small.h"

namespace tmb {

typedef u32x4_t __attribute__((aligned(2))) u32x4_half_aligned_t;

// Halves sh .. 7 of x moved to the front, zeros behind them (sh >= 8: all zeros).
__device__ __forceinline__ u32x4_t half_shift(u32x4_t x, int sh) {
  const int dw = sh >> 1;
  uint32_t d[5];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    d[e] = 0u;
#pragma unroll
    for (int k = 3 - e; k >= 0; --k) d[e] = dw == k ? x[e + k] : d[e];
  }
  d[4] = 0u;
  u32x4_t r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = (sh & 1) ? (d[e] >> 16) | (d[e + 1] << 16) : d[e];
  return r;
}

// One operand's slice: ROWS rows (m or n) by 64 k, as 16-byte pieces along its contiguous direction. A
// piece that reaches past the operand's edge is read from the last eight elements that exist (so at
// least eight must) and moved into place on its way into LDS: no access outside the operand.
template <int ROWS, bool K_CONTIGUOUS>
struct HalfSlice {
  static constexpr int KS = 64;
  // bytes per LDS line / k-row: 16 more than the data spread the rows of a fragment read over the banks
  static constexpr int PITCH = (K_CONTIGUOUS ? KS : ROWS) * 2 + 16;
  static constexpr int BYTES = (K_CONTIGUOUS ? ROWS : KS) * PITCH;
  static constexpr int LOADS = ROWS / 8;                   // pieces per lane and slice
  static constexpr int LPL = K_CONTIGUOUS ? 8 : ROWS / 8;  // lanes per line
  u32x4_t v[LOADS];
  uint32_t off[LOADS];  // bytes from eight elements in front of the tile's first one (a tile of fewer than
                        // eight columns is read from in front of it: offsets stay unsigned that way)
  int shift;            // how far this lane's pieces reach past the last row (MN-contiguous operands)

  static __device__ __forceinline__ int line_of(int i, int lane) { return i * (64 / LPL) + lane / LPL; }
  // `rows`: how many of the operand's rows exist from the tile's first one on (lines past the edge of a
  // K-contiguous operand re-read the last one: computed, never stored)
  __device__ __forceinline__ void plan(int64_t ld, int64_t rows, int lane) {
    const int c = (lane % LPL) * 8;
    const int last = rows > ROWS ? ROWS : static_cast<int>(rows);
    const int at = K_CONTIGUOUS || c + 8 <= last ? c : last - 8;
    shift = c - at;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int line = line_of(i, lane);
      if constexpr (K_CONTIGUOUS) line = line < last ? line : last - 1;
      off[i] = static_cast<uint32_t>((line * ld + at + 8) * 2);
    }
  }
  // first: the tile's first row at this slice's first k. `k_left`: how many k exist from there on.
  __device__ __forceinline__ void load(const unsigned char* first, int64_t ld, int64_t k_left, int lane) {
    const unsigned char* base = first - 16;
    if (k_left >= KS) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < LOADS; ++i) v[i] = *reinterpret_cast<const u32x4_half_aligned_t*>(base + off[i]);
    } else {
      const int left = static_cast<int>(k_left), c = (lane % LPL) * 8;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        int64_t at = off[i];
        if constexpr (K_CONTIGUOUS) {
          if (c + 8 > left) at += (left - 8 - c) * 2;
        } else {
          const int line = line_of(i, lane);
          if (line >= left) at -= (line - left + 1) * ld * 2;
        }
        v[i] = *reinterpret_cast<const u32x4_half_aligned_t*>(base + at);
      }
    }
  }
  __device__ __forceinline__ void lay_down(lds_byte_t* lds, int64_t k_left, bool edge, int lane) {
    const int c = (lane % LPL) * 8;
    if (K_CONTIGUOUS ? k_left < KS : (edge || k_left < KS)) {  // wave-uniform
      const int left = k_left < KS ? static_cast<int>(k_left) : KS;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        if constexpr (K_CONTIGUOUS) v[i] = half_shift(v[i], c + 8 > left ? c - (left - 8) : 0);
        else v[i] = half_shift(v[i], line_of(i, lane) < left ? shift : 8);
      }
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i) *(lds_u32x4v_t*)(lds + line_of(i, lane) * PITCH + c * 2) = v[i];
  }
  // Rows 16 tile + lane % 16, the eight k from 32 h + 8 (lane / 16) on.
  static __device__ __forceinline__ u32x4_t fragment(lds_byte_t* lds, int tile, int h, int lane) {
    const int fr = lane & 15, fq = lane >> 4;
    if constexpr (K_CONTIGUOUS) {
      return *(const lds_u32x4v_t*)(lds + (tile * 16 + fr) * PITCH + h * 64 + fq * 16);
    } else {
      typedef short i16x4a_t __attribute__((ext_vector_type(4)));
      typedef short i16x8a_t __attribute__((ext_vector_type(8)));
      typedef __attribute__((address_space(3))) i16x4a_t lds_i16x4a_t;
      lds_byte_t* src = lds + (h * 32 + fq * 8 + (fr >> 2)) * PITCH + (fr & 3) * 8 + tile * 32;
      const i16x4a_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4a_t*)(src));
      const i16x4a_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4a_t*)(src + 4 * PITCH));
      return __builtin_bit_cast(u32x4_t, i16x8a_t(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)));
    }
  }
};

template <int BM, int BN, int WAVES, bool A_MMAJOR, bool B_KMAJOR>
struct AnyLds {
  static constexpr int SLICE = HalfSlice<BM, !A_MMAJOR>::BYTES + HalfSlice<BN, B_KMAJOR>::BYTES;
  static constexpr int PARTS = WAVES * BM * (BN + 4) * 4;
  static constexpr int BYTES = WAVES * SLICE > PARTS ? WAVES * SLICE : PARTS;
};

// (the epilogue is chosen at run time: it runs once per tile, and a kernel per epilogue would be
// another hundred of them)
template <typename T, int BM, int BN, int WAVES, bool A_MMAJOR, bool B_KMAJOR>
__global__ __launch_bounds__(WAVES * 64) void gemm_any_kernel(GemmArgs g, int epilogue) {
#if defined(__HIP_DEVICE_COMPILE__)
  using SliceA = HalfSlice<BM, !A_MMAJOR>;
  using SliceB = HalfSlice<BN, B_KMAJOR>;
  using L = AnyLds<BM, BN, WAVES, A_MMAJOR, B_KMAJOR>;
  constexpr int KS = 64, TM = BM / 16, TN = BN / 16;
  constexpr int RP = BN + 4;  // floats per row of a partial tile in LDS
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int tile_m, tile_n;
  tile_of_block(blockIdx.x, g.tiles_m, g.tiles_n, tile_m, tile_n);
  // a split launch (g.splits > 0): blockIdx.y is the split, which multiplies its run of slices and
  // stores fp32 partials [splits][M][N]
  const int64_t split = g.splits > 0 ? blockIdx.y : 0;
  const int64_t batch = g.splits > 0 ? 0 : blockIdx.y;
  const int64_t m0 = static_cast<int64_t>(tile_m) * BM, n0 = static_cast<int64_t>(tile_n) * BN;
  const int64_t M = g.m, N = g.n, K = g.k;
  const unsigned char* A = reinterpret_cast<const unsigned char*>(
      static_cast<const T*>(g.a) + batch * g.stride_a + (A_MMAJOR ? m0 : m0 * g.lda));
  const unsigned char* B = reinterpret_cast<const unsigned char*>(
      static_cast<const T*>(g.b) + batch * g.stride_b + (B_KMAJOR ? n0 * g.ldb : n0));
  const int64_t a_k = (A_MMAJOR ? g.lda : 1) * 2, b_k = (B_KMAJOR ? 1 : g.ldb) * 2;  // bytes per unit of k

  f32x4v_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4v_t{0.0f, 0.0f, 0.0f, 0.0f};

  SliceA sa;
  SliceB sb;
  sa.plan(g.lda, M - m0, lane);
  sb.plan(g.ldb, N - n0, lane);
  lds_byte_t* la = (lds_byte_t*)smem + wave * L::SLICE;
  lds_byte_t* lb = la + SliceA::BYTES;
  int64_t first = 0, slices = (K + KS - 1) / KS;
  if (g.splits > 0) {
    first = slices * split / g.splits;
    slices = slices * (split + 1) / g.splits;
  }
  const bool a_edge = M - m0 < BM, b_edge = N - n0 < BN;
  auto load = [&](int64_t s) {
    const int64_t k0 = s * KS;
    sa.load(A + k0 * a_k, g.lda, K - k0, lane);
    sb.load(B + k0 * b_k, g.ldb, K - k0, lane);
  };
  if (first + wave < slices) load(first + wave);
  for (int64_t s = first + wave; s < slices; s += WAVES) {
    sa.lay_down(la, K - s * KS, a_edge, lane);
    sb.lay_down(lb, K - s * KS, b_edge, lane);
    wave_lds_point();
    if (s + WAVES < slices) load(s + WAVES);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4_t af[TM];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = SliceA::fragment(la, i, h, lane);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const u32x4_t bf = SliceB::fragment(lb, j, h, lane);
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[i][j] = Mfma16<T>::run(bf, af[i], acc[i][j]);
      }
    }
    wave_lds_point();
  }

  // A lane holds row lane % 16 and four consecutive columns of each 16 x 16 result.
  __syncthreads();  // the partial tiles overlay the slices
  float* part = reinterpret_cast<float*>(smem) + wave * (BM * RP);
  const int fr = lane & 15, fq = lane >> 4;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      *reinterpret_cast<f32x4v_t*>(part + (i * 16 + fr) * RP + j * 16 + fq * 4) = acc[i][j];
  __syncthreads();
  const EpilogueArgs ep = epilogue_args<T>(g, batch);
  const float* all = reinterpret_cast<const float*>(smem);
#pragma unroll 1
  for (int idx = tid; idx < BM * BN / 4; idx += WAVES * 64) {
    const int r = idx / (BN / 4), c = (idx % (BN / 4)) * 4;
    const int64_t row = m0 + r, col = n0 + c;
    if (row >= M || col >= N) continue;
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
    if (g.splits > 0) {
      float* dst = static_cast<float*>(g.c) + split * g.stride_c + row * g.ldc + col;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < N) dst[e] = sum[e];
    } else if (epilogue == TMB_EPI_NONE) {
      small_epilogue4<T, TMB_EPI_NONE>(sum, g, ep, batch, row, col);
    } else if (epilogue == TMB_EPI_GELU_TANH) {
      small_epilogue4<T, TMB_EPI_GELU_TANH>(sum, g, ep, batch, row, col);
    } else {
      small_epilogue4<T, TMB_EPI_GELU_ERF>(sum, g, ep, batch, row, col);
    }
  }
#endif
}

template <typename T, int BM, int BN, int WAVES, bool A_MMAJOR, bool B_KMAJOR>
static int launch_any_tile(const GemmArgs& base, int64_t batch, int epilogue, hipStream_t stream) {
  constexpr int SMEM = AnyLds<BM, BN, WAVES, A_MMAJOR, B_KMAJOR>::BYTES;
  static_assert(SMEM <= 160 * 1024, "LDS of one CU");
  auto kernel = gemm_any_kernel<T, BM, BN, WAVES, A_MMAJOR, B_KMAJOR>;
  static const hipError_t configured = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
  if (configured != hipSuccess) return static_cast<int>(configured);
  GemmArgs g = base;
  g.tiles_m = static_cast<int>((g.m + BM - 1) / BM);
  g.tiles_n = static_cast<int>((g.n + BN - 1) / BN);
  const int64_t tiles = static_cast<int64_t>(g.tiles_m) * g.tiles_n;
  if (tiles >= (int64_t{1} << 31) || batch > 65535) return TMB_ERR_UNSUPPORTED;
  kernel<<<dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(batch)), dim3(WAVES * 64), SMEM, stream>>>(
      g, epilogue);
  return check_launch();
}

}  // namespace tmb
