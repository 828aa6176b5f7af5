// fp32 GEMM on the matrix cores (v_mfma_f32_32x32x2_f32: true fp32 products, fp32 accumulation), any
// of the four operand layouts, any extents and any row pitch.
//
// A workgroup owns a BM x BN tile of C and its WAVES waves share K: wave w multiplies the 32-deep
// slices w, w + WAVES, ... of the whole tile and the partial tiles meet in LDS once, at the end, where
// they are added pairwise in wave order (the result depends on the shape only). An fp32 MFMA takes
// 64 cycles for two 4-byte operands per lane, so the matrix cores bound all but the smallest launches,
// and what has to be right is the division of the work: tiles small enough to give every CU the same
// amount (1332 x 3072 x 768 is 264 tiles of 128 x 128, i.e. two rounds of the 256 CUs for 1.03 rounds
// of work), and no workgroup barrier in the main loop. Sharing K instead of the tile halves what a wave
// reads from LDS per MFMA against the same tile cut into quarters, and lets a 32 x 32 tile, of which
// even a small product has hundreds, keep all four SIMDs busy.
//
// A wave brings a slice in through registers (the next slice travels while this one is multiplied) and
// a wave-private part of LDS, which works in order per wave. An operand stored with K contiguous
// (A [M, K], B [N, K]) is kept as lines of 32 floats; a lane takes four consecutive k with one 16-byte
// read and feeds four MFMAs with them (lanes 0-31 the first four of a group of eight, lanes 32-63 the
// others: the order in which the k of a slice are added is free as long as A and B agree). An operand
// stored with its M or N extent contiguous (A [K, M], B [K, N]) is kept as k-rows.
//
// The MFMA gets the B fragment first, so a lane ends up with one row m of C and four consecutive
// columns per register quad.
#pragma once

#include "gemm_mfma.h"

namespace tmb {

constexpr int kF32KS = 32;  // depth of a slice: one 128-byte line

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Elements sh .. 3 of x moved to the front, zeros behind them (sh >= 4: all zeros).
__device__ __forceinline__ f32x4_t f32_shift(f32x4_t x, int sh) {
  f32x4_t r;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float y = 0.0f;
#pragma unroll
    for (int k = 3 - e; k >= 0; --k) y = sh == k ? x[e + k] : y;
    r[e] = y;
  }
  return r;
}

// One operand's slice: ROWS rows (m or n) by 32 k, as 16-byte pieces along its contiguous direction.
// A piece that reaches past the operand's edge is read from the last four elements that exist (so at
// least four must) and moved into place on its way into LDS: no access outside the operand, and no
// divergent code in the way of the full slices.
template <int ROWS, bool K_CONTIGUOUS>
struct F32Slice {
  // floats per LDS line / k-row: four more than the data keep 16-byte alignment and spread the rows
  // of a fragment read over the banks
  static constexpr int PITCH = K_CONTIGUOUS ? kF32KS + 4 : ROWS + 4;
  static constexpr int FLOATS = K_CONTIGUOUS ? ROWS * PITCH : kF32KS * PITCH;
  static constexpr int LOADS = ROWS / 8;                   // pieces per lane and slice
  static constexpr int LPL = K_CONTIGUOUS ? 8 : ROWS / 4;  // lanes per line
  f32x4_t v[LOADS];
  uint32_t off[LOADS];  // bytes from four elements in front of the tile's first one (a tile of fewer than
                        // four columns is read from in front of it: offsets stay unsigned that way)
  int shift;            // how far this lane's pieces reach past the last row (MN-contiguous operands)

  static __device__ __forceinline__ int line_of(int i, int lane) { return i * (64 / LPL) + lane / LPL; }
  // `rows`: how many of the operand's rows exist from the tile's first one on (lines past the edge of
  // a K-contiguous operand re-read the last one: computed, never stored)
  __device__ __forceinline__ void plan(int64_t ld, int64_t rows, int lane) {
    const int c = (lane % LPL) * 4;
    const int last = rows > ROWS ? ROWS : static_cast<int>(rows);
    const int at = K_CONTIGUOUS || c + 4 <= last ? c : last - 4;
    shift = c - at;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int line = line_of(i, lane);
      if constexpr (K_CONTIGUOUS) line = line < last ? line : last - 1;
      off[i] = static_cast<uint32_t>((line * ld + at + 4) * 4);
    }
  }
  // first: the tile's first row at this slice's first k. `k_left`: how many k exist from there on.
  __device__ __forceinline__ void load(const char* __restrict__ first, int64_t ld, int64_t k_left, int lane) {
    const char* __restrict__ base = first - 16;
    if (k_left >= kF32KS) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < LOADS; ++i) v[i] = *reinterpret_cast<const f32x4_unaligned_t*>(base + off[i]);
    } else {
      const int left = static_cast<int>(k_left), c = (lane % LPL) * 4;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        int64_t at = off[i];
        if constexpr (K_CONTIGUOUS) {
          if (c + 4 > left) at += (left - 4 - c) * 4;
        } else {
          const int line = line_of(i, lane);
          if (line >= left) at -= (line - left + 1) * ld * 4;
        }
        v[i] = *reinterpret_cast<const f32x4_unaligned_t*>(base + at);
      }
    }
  }
  __device__ __forceinline__ void lay_down(float* __restrict__ lds, int64_t k_left, bool edge, int lane) {
    const int c = (lane % LPL) * 4;
    if (K_CONTIGUOUS ? k_left < kF32KS : (edge || k_left < kF32KS)) {  // wave-uniform
      const int left = k_left < kF32KS ? static_cast<int>(k_left) : kF32KS;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        if constexpr (K_CONTIGUOUS) v[i] = f32_shift(v[i], c + 4 > left ? c - (left - 4) : 0);
        else v[i] = f32_shift(v[i], line_of(i, lane) < left ? shift : 4);
      }
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i) *reinterpret_cast<f32x4_t*>(lds + line_of(i, lane) * PITCH + c) = v[i];
  }
  // The four k that lane half `lk` takes of group `g` (eight k) in row `row`.
  static __device__ __forceinline__ f32x4_t fragment(const float* __restrict__ lds, int row, int g, int lk) {
    if constexpr (K_CONTIGUOUS) {
      return *reinterpret_cast<const f32x4_t*>(lds + row * PITCH + g * 8 + lk * 4);
    } else {
      const float* p = lds + (g * 8 + lk * 4) * PITCH + row;
      return f32x4_t{p[0], p[PITCH], p[2 * PITCH], p[3 * PITCH]};
    }
  }
};

template <int BM, int BN, int WAVES, int EPI, bool A_MMAJOR, bool B_KMAJOR>
__global__ __launch_bounds__(WAVES * 64, BM * BN <= 4096 ? 2 : 1) void gemm_f32_kernel(const GemmArgs g) {
  using SliceA = F32Slice<BM, !A_MMAJOR>;
  using SliceB = F32Slice<BN, B_KMAJOR>;
  constexpr int TM = BM / 32, TN = BN / 32;
  constexpr int WAVE_FLOATS = SliceA::FLOATS + SliceB::FLOATS;
  constexpr int RP = BN + 4;  // floats per row of a partial tile
  extern __shared__ __attribute__((aligned(16))) float f32_lds[];

  int tm, tn;
  tile_of_block(blockIdx.x, g.tiles_m, g.tiles_n, tm, tn);
  // a split launch (g.splits > 0): blockIdx.y is the split, which multiplies its run of slices and
  // stores fp32 partials [splits][M][N]
  const int64_t split = g.splits > 0 ? blockIdx.y : 0;
  const int64_t batch = g.splits > 0 ? 0 : blockIdx.y;
  const int64_t m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * BN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lk = lane >> 5;
  const int64_t M = g.m, N = g.n, K = g.k;
  const float* A = static_cast<const float*>(g.a) + batch * g.stride_a + (A_MMAJOR ? m0 : m0 * g.lda);
  const float* B = static_cast<const float*>(g.b) + batch * g.stride_b + (B_KMAJOR ? n0 * g.ldb : n0);
  const int64_t a_k = A_MMAJOR ? g.lda : 1, b_k = B_KMAJOR ? 1 : g.ldb;  // floats per unit of k

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  SliceA sa;
  SliceB sb;
  sa.plan(g.lda, M - m0, lane);
  sb.plan(g.ldb, N - n0, lane);
  float* la = f32_lds + wave * WAVE_FLOATS;
  float* lb = la + SliceA::FLOATS;
  int64_t first = 0, slices = (K + kF32KS - 1) / kF32KS;
  if (g.splits > 0) {
    first = slices * split / g.splits;
    slices = slices * (split + 1) / g.splits;
  }
  const bool a_edge = M - m0 < BM, b_edge = N - n0 < BN;
  auto load = [&](int64_t s) {
    const int64_t k0 = s * kF32KS;
    sa.load(reinterpret_cast<const char*>(A + k0 * a_k), g.lda, K - k0, lane);
    sb.load(reinterpret_cast<const char*>(B + k0 * b_k), g.ldb, K - k0, lane);
  };
  if (first + wave < slices) load(first + wave);
  for (int64_t s = first + wave; s < slices; s += WAVES) {
    sa.lay_down(la, K - s * kF32KS, a_edge, lane);
    sb.lay_down(lb, K - s * kF32KS, b_edge, lane);
    wave_lds_point();
    if (s + WAVES < slices) load(s + WAVES);
#pragma unroll
    for (int grp = 0; grp < kF32KS / 8; ++grp) {
      f32x4_t af[TM], bf[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = SliceA::fragment(la, i * 32 + lr, grp, lk);
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[j] = SliceB::fragment(lb, j * 32 + lr, grp, lk);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(bf[j][e], af[i][e], acc[i][j], 0, 0, 0);
    }
    wave_lds_point();
  }

  // Lane holds row lr of each 32 x 32 result and columns 8q + 4 * lk + {0..3}.
  __syncthreads();  // the partial tiles overlay the slices
  float* part = f32_lds + wave * (BM * RP);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        *reinterpret_cast<f32x4_t*>(part + (i * 32 + lr) * RP + j * 32 + 8 * q + 4 * lk) = v;
      }
  __syncthreads();
  const float* __restrict__ bias = static_cast<const float*>(g.bias);
  const float* __restrict__ resid = g.residual == nullptr
                                        ? nullptr
                                        : static_cast<const float*>(g.residual) + batch * g.stride_r;
  float* __restrict__ C = static_cast<float*>(g.c) + (batch + split) * g.stride_c;
#pragma unroll
  for (int p = 0; p < (BM * BN / 4 + WAVES * 64 - 1) / (WAVES * 64); ++p) {
    const int idx = p * WAVES * 64 + tid;
    if ((BM * BN / 4) % (WAVES * 64) != 0 && idx >= BM * BN / 4) break;
    const int r = idx / (BN / 4), c = (idx % (BN / 4)) * 4;
    const int64_t row = m0 + r, col = n0 + c;
    if (row >= M || col >= N) continue;
    f32x4_t v[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v[w] = *reinterpret_cast<const f32x4_t*>(f32_lds + w * (BM * RP) + r * RP + c);
#pragma unroll
    for (int step = 1; step < WAVES; step *= 2)
#pragma unroll
      for (int w = 0; w < WAVES; w += 2 * step)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[w][e] += v[w + step][e];
    const bool whole = col + 4 <= N;
    float out[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x = v[0][e];
      if (bias != nullptr && (whole || col + e < N)) x += bias[col + e];
      x = finish<float, EPI>(x, false);
      if (resid != nullptr && (whole || col + e < N)) x += resid[row * g.ldr + col + e];
      out[e] = x;
    }
    float* dst = C + row * g.ldc + col;
    if (whole) {
      const f32x4_unaligned_t o = {out[0], out[1], out[2], out[3]};
      if (g.stream_c) __builtin_nontemporal_store(o, reinterpret_cast<f32x4_unaligned_t*>(dst));
      else *reinterpret_cast<f32x4_unaligned_t*>(dst) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < N) dst[e] = out[e];
    }
  }
}

template <int BM, int BN, int WAVES, int EPI>
static int launch_f32_tile(const GemmArgs& base, int64_t batch, int trans_a, int trans_b, hipStream_t stream) {
  GemmArgs g = base;
  g.tiles_m = static_cast<int>((g.m + BM - 1) / BM);
  g.tiles_n = static_cast<int>((g.n + BN - 1) / BN);
  g.stream_c = batch * g.m * g.n * 4 > (int64_t{256} << 20);
  const int64_t tiles = static_cast<int64_t>(g.tiles_m) * g.tiles_n;
  if (tiles >= (int64_t{1} << 31) || batch > 65535) return TMB_ERR_UNSUPPORTED;
  const dim3 grid(static_cast<unsigned>(tiles), static_cast<unsigned>(batch));
  auto go = [&](auto a_mmajor, auto b_kmajor) {
    constexpr bool AM = decltype(a_mmajor)::value, BK = decltype(b_kmajor)::value;
    constexpr int SLICES = WAVES * (F32Slice<BM, !AM>::FLOATS + F32Slice<BN, BK>::FLOATS) * 4;
    constexpr int PARTS = WAVES * BM * (BN + 4) * 4;
    constexpr int SMEM = SLICES > PARTS ? SLICES : PARTS;
    static_assert(SMEM <= 160 * 1024, "LDS of one CU");
    auto kernel = gemm_f32_kernel<BM, BN, WAVES, EPI, AM, BK>;
    static bool configured = false;
    if (!configured) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
      if (e != hipSuccess) return static_cast<int>(e);
      configured = true;
    }
    kernel<<<grid, WAVES * 64, SMEM, stream>>>(g);
    return check_launch();
  };
  if (trans_a) return trans_b ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
  return trans_b ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
}

}  // namespace tmb
