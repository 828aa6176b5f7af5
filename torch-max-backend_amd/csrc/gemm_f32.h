// fp32 GEMM on the bf16 matrix cores, any of the four operand layouts, any extents and any row pitch.
//
// An fp32 MFMA takes 64 cycles for what a bf16 one does in four. So each operand element is taken apart into three bf16
// whose sum it is, exactly (F32Pair), and a product is eight of the nine partial products, all but the one below 2^-33 of
// it, added up in fp32 by v_mfma_f32_16x16x32_bf16: 32 cycles of matrix core for 64. The large partial products and the
// small ones are summed apart and joined by a rounded addition: a product that stands alone is off by 1.01 half units at
// most (with the small ones in one chain, 3.8: the MFMA aligns addends to the largest and cuts), and a sum is rounded once
// in 32 k instead of at every k. Against fp32 MFMAs the error of dense operands is 0.1 .. 1.0 of what it was over K 129 ..
// 50257, of rows with a single term the same, of rows with 4 .. 16 terms 0.6 .. 1.13 (each product is rounded before it is
// added, and the order of the sum is another); operands of exponents 2^-20 .. 2^20 0.3 .. 1.03.
// 1332 x 768 x 3072 68 -> 57 us, 1332 x 3072 x 768 70 -> 58, 750 x 2304 x 768 36 -> 29.
//
// A workgroup owns a BM x BN tile of C and its WAVES waves share K: wave w multiplies the 32-deep
// slices w, w + WAVES, ... of the whole tile and the partial tiles meet in LDS once, at the end, where
// they are added pairwise in wave order (the result depends on the shape only): no workgroup barrier in the main loop,
// and tiles small enough to give every CU the same amount. What bounds it is the vector units, which take the operands
// apart (44 instructions for a fragment of 16 rows, of which two hide behind an MFMA), and the matrix cores.
//
// A wave brings a slice in through registers (the next slice travels while this one is multiplied) and
// a wave-private part of LDS, which works in order per wave; a lane of a fragment takes eight consecutive k of a row.
// The split of a column block is scheduled between the MFMAs of the block before it.
//
// The MFMA gets the B fragment first, so a lane ends up with one row m of C and four consecutive
// columns.
#pragma once

#include "gemm_mfma.h"

namespace tmb {

constexpr int kF32KS = 32;  // depth of a slice: one 128-byte line
// Up to here products are fp32 ones: a wave has a slice at most, and the larger code and register file of the split kernel
// cost more than its matrix cores save (64 x 64 tiles 1.06 of the time at K = 128, 0.93 at 160; 32 x 32 1.07 up to 256, where
// the split ones are kept for half the error).
constexpr int64_t kF32SplitK = 128;

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

// One operand's slice: ROWS rows (m or n) by 32 k, kept in LDS as lines of 32 k.
//
// K contiguous in memory: 16-byte pieces of lines. A piece that reaches past K is read from the last four
// elements that exist (so at least four must) and moved into place on its way into LDS: no access outside the operand,
// and no divergent code in the way of the full slices.
template <int ROWS, bool K_CONTIGUOUS>
struct F32Slice {
  // floats per LDS line: four more than the data keep 16-byte alignment and spread the rows of a fragment read
  // over the banks
  static constexpr int PITCH = kF32KS + 4;
  static constexpr int FLOATS = ROWS * PITCH;
  static constexpr int LOADS = ROWS / 8;  // pieces per lane and slice
  f32x4_t v[LOADS];
  uint32_t off[LOADS];  // bytes from four elements in front of the tile's first one (a tile of fewer than
                        // four columns is read from in front of it: offsets stay unsigned that way)

  static __device__ __forceinline__ int line_of(int i, int lane) { return i * 8 + lane / 8; }
  // `rows`: how many of the operand's rows exist from the tile's first one on (lines past the edge re-read the last
  // one: computed, never stored)
  __device__ __forceinline__ void plan(int64_t ld, int64_t rows, int lane) {
    const int c = (lane % 8) * 4;
    const int last = rows > ROWS ? ROWS : static_cast<int>(rows);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int line = line_of(i, lane) < last ? line_of(i, lane) : last - 1;
      off[i] = static_cast<uint32_t>((line * ld + c + 4) * 4);
    }
  }
  // first: the tile's first row at this slice's first k. `k_left`: how many k exist from there on.
  __device__ __forceinline__ void load(const char* __restrict__ first, int64_t, int64_t k_left, int lane) {
    const char* __restrict__ base = first - 16;
    if (k_left >= kF32KS) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < LOADS; ++i) v[i] = *reinterpret_cast<const f32x4_unaligned_t*>(base + off[i]);
    } else {
      const int left = static_cast<int>(k_left), c = (lane % 8) * 4;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        int64_t at = off[i];
        if (c + 4 > left) at += (left - 4 - c) * 4;
        v[i] = *reinterpret_cast<const f32x4_unaligned_t*>(base + at);
      }
    }
  }
  __device__ __forceinline__ void lay_down(float* __restrict__ lds, int64_t k_left, int lane) {
    const int c = (lane % 8) * 4;
    if (k_left < kF32KS) {  // wave-uniform
      const int left = static_cast<int>(k_left);
#pragma unroll
      for (int i = 0; i < LOADS; ++i) v[i] = f32_shift(v[i], c + 4 > left ? c - (left - 4) : 0);
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i) *reinterpret_cast<f32x4_t*>(lds + line_of(i, lane) * PITCH + c) = v[i];
  }
  // The eight k that lane quarter `lq` takes of row `row`: 8 * lq .. 8 * lq + 7.
  static __device__ __forceinline__ void fragment(const float* __restrict__ lds, int row, int lq, f32x4_t (&x)[2]) {
    const float* p = lds + row * PITCH + lq * 8;
    x[0] = *reinterpret_cast<const f32x4_t*>(p);
    x[1] = *reinterpret_cast<const f32x4_t*>(p + 4);
  }
};
// M or N contiguous, 64 rows: a lane is a row and brings its k one by one (the lanes read a k-row's neighbours), so that
// what it lays down are pieces of lines too: a fragment is two reads instead of eight (4096^3 with both operands so
// 1030 us, 1190 with the layout below, whose eight fragments at once do not fit the registers).
template <>
struct F32Slice<64, false> {
  static constexpr int ROWS = 64;
  using Lines = F32Slice<ROWS, true>;
  static constexpr int FLOATS = Lines::FLOATS, LOADS = Lines::LOADS;
  f32x4_t v[LOADS];
  uint32_t off;  // bytes: the lane's row

  __device__ __forceinline__ void plan(int64_t, int64_t rows, int lane) {
    const int last = rows > ROWS ? ROWS : static_cast<int>(rows);
    off = static_cast<uint32_t>((lane < last ? lane : last - 1) * 4);
  }
  __device__ __forceinline__ void load(const char* __restrict__ first, int64_t ld, int64_t k_left, int) {
    const int64_t step = ld * 4;
    auto at = [](const char* p) { return *reinterpret_cast<const float*>(p); };
    if (k_left >= kF32KS) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const char* __restrict__ p = first + 4 * i * step;
        v[i] = f32x4_t{at(p + off), at(p + step + off), at(p + 2 * step + off), at(p + 3 * step + off)};
      }
    } else {  // (k past the last one re-read it)
      const int most = static_cast<int>(k_left) - 1;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const char* __restrict__ p = first + off;
        auto k = [&](int e) { return (4 * i + e < most ? 4 * i + e : most) * step; };
        v[i] = f32x4_t{at(p + k(0)), at(p + k(1)), at(p + k(2)), at(p + k(3))};
      }
    }
  }
  __device__ __forceinline__ void lay_down(float* __restrict__ lds, int64_t k_left, int lane) {
    if (k_left < kF32KS) {  // wave-uniform
      const int left = static_cast<int>(k_left);
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
        v[i] = f32x4_t{4 * i < left ? v[i][0] : 0.0f, 4 * i + 1 < left ? v[i][1] : 0.0f, 4 * i + 2 < left ? v[i][2] : 0.0f,
                       4 * i + 3 < left ? v[i][3] : 0.0f};
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      *reinterpret_cast<f32x4_t*>(lds + lane * Lines::PITCH + 4 * i) = v[i];
  }
  static __device__ __forceinline__ void fragment(const float* __restrict__ lds, int row, int lq, f32x4_t (&x)[2]) {
    Lines::fragment(lds, row, lq, x);
  }
};

// M or N contiguous, 32 rows: 16-byte pieces of k-rows, kept as k-rows. A piece that reaches past the last row is read
// from the last four that exist and moved into place.
template <>
struct F32Slice<32, false> {
  static constexpr int ROWS = 32;
  static constexpr int PITCH = ROWS + 4, FLOATS = kF32KS * PITCH, LOADS = ROWS / 8, LPL = ROWS / 4;  // (lanes per k-row)
  f32x4_t v[LOADS];
  uint32_t off[LOADS];  // bytes from four elements in front of the tile's first one
  int shift;            // how far this lane's pieces reach past the last row

  static __device__ __forceinline__ int line_of(int i, int lane) { return i * (64 / LPL) + lane / LPL; }
  __device__ __forceinline__ void plan(int64_t ld, int64_t rows, int lane) {
    const int c = (lane % LPL) * 4;
    const int last = rows > ROWS ? ROWS : static_cast<int>(rows);
    const int at = c + 4 <= last ? c : last - 4;
    shift = c - at;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) off[i] = static_cast<uint32_t>((line_of(i, lane) * ld + at + 4) * 4);
  }
  __device__ __forceinline__ void load(const char* __restrict__ first, int64_t ld, int64_t k_left, int lane) {
    const char* __restrict__ base = first - 16;
    if (k_left >= kF32KS) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < LOADS; ++i) v[i] = *reinterpret_cast<const f32x4_unaligned_t*>(base + off[i]);
    } else {
      const int left = static_cast<int>(k_left);
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        int64_t at = off[i];
        const int line = line_of(i, lane);
        if (line >= left) at -= (line - left + 1) * ld * 4;
        v[i] = *reinterpret_cast<const f32x4_unaligned_t*>(base + at);
      }
    }
  }
  __device__ __forceinline__ void lay_down(float* __restrict__ lds, int64_t k_left, int lane) {
    const int left = k_left < kF32KS ? static_cast<int>(k_left) : kF32KS;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int line = line_of(i, lane);
      *reinterpret_cast<f32x4_t*>(lds + line * PITCH + (lane % LPL) * 4) = f32_shift(v[i], line < left ? shift : 4);
    }
  }
  static __device__ __forceinline__ void fragment(const float* __restrict__ lds, int row, int lq, f32x4_t (&x)[2]) {
    const float* p = lds + lq * 8 * PITCH + row;
    x[0] = f32x4_t{p[0], p[PITCH], p[2 * PITCH], p[3 * PITCH]};
    x[1] = f32x4_t{p[4 * PITCH], p[5 * PITCH], p[6 * PITCH], p[7 * PITCH]};
  }
};

// Two fp32 values, times 2^16, as three bf16 each: x = h + m + l with |m| <= 2^-8 |x|, |l| <= 2^-17 |x|. Exact: 24 bits of
// significand in three times eight, and 2^16 times the smallest fp32 number is the smallest bf16 one. (h and m are rounded
// to nearest; what h leaves has at most sixteen bits, what m leaves of those at most seven.)
struct F32Pair {
  uint32_t h, m, l;
  static constexpr float kUp = 0x1p16f, kDown = 0x1p-16f;  // each operand's factor, and what undoes it
  static __device__ __forceinline__ F32Pair of(float a, float b) {
    F32Pair r;
    a *= kUp;
    b *= kUp;
    r.h = pack2<bf16_t>(a, b);
    a -= __builtin_bit_cast(float, r.h << 16);
    b -= __builtin_bit_cast(float, r.h & 0xffff0000u);
    r.m = pack2<bf16_t>(a, b);
    a -= __builtin_bit_cast(float, r.m << 16);
    b -= __builtin_bit_cast(float, r.m & 0xffff0000u);
    r.l = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
    return r;
  }
};
struct F32Split {
  u32x4_t h, m, l;
  __device__ __forceinline__ void of(const f32x4_t (&x)[2]) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const F32Pair s = F32Pair::of(x[p >> 1][2 * (p & 1)], x[p >> 1][2 * (p & 1) + 1]);
      h[p] = s.h;
      m[p] = s.m;
      l[p] = s.l;
    }
  }
};

// SPLIT false: fp32 products (short K, kF32SplitK).
template <int BM, int BN, int WAVES, int EPI, bool A_MMAJOR, bool B_KMAJOR, bool SPLIT>
__global__ __launch_bounds__(WAVES * 64, BM * BN <= 4096 && WAVES < 8 ? 2 : 1) void gemm_f32_kernel(const GemmArgs g) {
  using SliceA = F32Slice<BM, !A_MMAJOR>;
  using SliceB = F32Slice<BN, B_KMAJOR>;
  constexpr int TM = BM / 16, TN = BN / 16;
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
  const int lr = lane & 15, lq = lane >> 4;
  const int64_t M = g.m, N = g.n, K = g.k;
  const float* A = static_cast<const float*>(g.a) + batch * g.stride_a + (A_MMAJOR ? m0 : m0 * g.lda);
  const float* B = static_cast<const float*>(g.b) + batch * g.stride_b + (B_KMAJOR ? n0 * g.ldb : n0);
  const int64_t a_k = A_MMAJOR ? g.lda : 1, b_k = B_KMAJOR ? 1 : g.ldb;  // floats per unit of k

  f32x4v_t acc[TM][TN];

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
  auto load = [&](int64_t s) {
    const int64_t k0 = s * kF32KS;
    sa.load(reinterpret_cast<const char*>(A + k0 * a_k), g.lda, K - k0, lane);
    sb.load(reinterpret_cast<const char*>(B + k0 * b_k), g.ldb, K - k0, lane);
  };
  auto multiply = [&](auto as_bf16) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4v_t{0.0f, 0.0f, 0.0f, 0.0f};
    if (first + wave < slices) load(first + wave);
    for (int64_t s = first + wave; s < slices; s += WAVES) {
      sa.lay_down(la, K - s * kF32KS, lane);
      sb.lay_down(lb, K - s * kF32KS, lane);
      wave_lds_point();
      if (s + WAVES < slices) load(s + WAVES);
      if constexpr (decltype(as_bf16)::value) {
        F32Split af[TM], bf[2];
        f32x4v_t t[TM], u[TM];  // the small products' sums, the large ones'
        f32x4_t x[2];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          SliceA::fragment(la, i * 16 + lr, lq, x);
          af[i].of(x);
        }
        SliceB::fragment(lb, lr, lq, x);
        bf[0].of(x);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          __builtin_amdgcn_sched_barrier(0);
          if (j > 0) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[i][j - 1][e] += u[i][e] + t[i][e];
          }
          if (j + 1 < TN) {
            SliceB::fragment(lb, (j + 1) * 16 + lr, lq, x);
            bf[(j + 1) & 1].of(x);
          }
          const F32Split& b = bf[j & 1];
#pragma unroll
          for (int i = 0; i < TM; ++i) t[i] = Mfma16<bf16_t>::run(b.l, af[i].m, f32x4v_t{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
          for (int i = 0; i < TM; ++i) t[i] = Mfma16<bf16_t>::run(b.m, af[i].l, t[i]);
#pragma unroll
          for (int i = 0; i < TM; ++i) t[i] = Mfma16<bf16_t>::run(b.l, af[i].h, t[i]);
#pragma unroll
          for (int i = 0; i < TM; ++i) t[i] = Mfma16<bf16_t>::run(b.h, af[i].l, t[i]);
#pragma unroll
          for (int i = 0; i < TM; ++i) t[i] = Mfma16<bf16_t>::run(b.m, af[i].m, t[i]);
#pragma unroll
          for (int i = 0; i < TM; ++i) t[i] = Mfma16<bf16_t>::run(b.m, af[i].h, t[i]);
#pragma unroll
          for (int i = 0; i < TM; ++i) t[i] = Mfma16<bf16_t>::run(b.h, af[i].m, t[i]);
#pragma unroll
          for (int i = 0; i < TM; ++i) u[i] = Mfma16<bf16_t>::run(b.h, af[i].h, f32x4v_t{0.0f, 0.0f, 0.0f, 0.0f});
          __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);  // LDS reads
#pragma unroll
          for (int i = 0; i < 8 * TM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // vector ALU
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][TN - 1][e] += u[i][e] + t[i][e];
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          f32x4_t bf[2];
          SliceB::fragment(lb, j * 16 + lr, lq, bf);
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            f32x4_t af[2];
            SliceA::fragment(la, i * 16 + lr, lq, af);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[e >> 2][e & 3], af[e >> 2][e & 3], acc[i][j], 0, 0, 0);
          }
        }
      }
      wave_lds_point();
    }
  };
  multiply(std::integral_constant<bool, SPLIT>{});
  __syncthreads();  // the partial tiles overlay the slices

  const float* __restrict__ bias = static_cast<const float*>(g.bias);
  const float* __restrict__ resid = g.residual == nullptr
                                        ? nullptr
                                        : static_cast<const float*>(g.residual) + batch * g.stride_r;
  float* __restrict__ C = static_cast<float*>(g.c) + (batch + split) * g.stride_c;
  uint32_t spoiled = 0;  // this thread's elements whose split sum is not finite
  // Joins the partial tiles and stores what is finite, or (AGAIN) what was not. `down`: what undoes the operands' factors,
  // once per wave and once for their sum: it is rounded once among subnormals, and stays in range.
  auto join = [&](auto again, float down) {
    constexpr bool AGAIN = decltype(again)::value;
    // Lane holds row lr of each 16 x 16 result and columns 4 * lq + {0..3}.
    float* part = f32_lds + wave * (BM * RP);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        *reinterpret_cast<f32x4_t*>(part + (i * 16 + lr) * RP + j * 16 + 4 * lq) =
            f32x4_t{acc[i][j][0] * down, acc[i][j][1] * down, acc[i][j][2] * down, acc[i][j][3] * down};
    __syncthreads();
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
      uint32_t mine = 15;
      if constexpr (SPLIT) {
        if constexpr (AGAIN) {
          mine = spoiled >> (4 * p) & 15;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) mine &= ~((__builtin_fabsf(v[0][e]) < HUGE_VALF ? 0u : 1u) << e);
          spoiled |= (mine ^ 15) << (4 * p);
        }
      }
      float out[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x = v[0][e] * down;
        if (bias != nullptr && (whole || col + e < N)) x += bias[col + e];
        x = finish<float, EPI>(x, false);
        if (resid != nullptr && (whole || col + e < N)) x += resid[row * g.ldr + col + e];
        out[e] = x;
      }
      float* dst = C + row * g.ldc + col;
      if (whole && mine == 15) {
        const f32x4_unaligned_t o = {out[0], out[1], out[2], out[3]};
        if (g.stream_c) __builtin_nontemporal_store(o, reinterpret_cast<f32x4_unaligned_t*>(dst));
        else *reinterpret_cast<f32x4_unaligned_t*>(dst) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < N && (mine >> e & 1) != 0) dst[e] = out[e];
      }
    }
  };
  join(std::false_type{}, SPLIT ? F32Pair::kDown : 1.0f);
  if constexpr (SPLIT) {
    // An element whose sum is not finite (an operand or the result is not, or is beyond what the operands' factor leaves
    // room for) is formed again from fp32 products; its neighbours keep theirs, so a row's bits do not depend on others.
    // (1332 x 768 x 3072 with a NaN in one row 118 us for 64.)
    __shared__ int wave_spoiled[WAVES];
    const uint64_t any = __ballot(spoiled != 0);
    if (lane == 0) wave_spoiled[wave] = any != 0;
    __syncthreads();  // (the slices overlay the partial tiles)
    bool again = false;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) again |= wave_spoiled[w] != 0;
    if (again) {
      multiply(std::false_type{});
      __syncthreads();
      join(std::true_type{}, 1.0f);
    }
  }
}

template <int BM, int BN, int WAVES, int EPI, bool SPLIT>
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
    auto kernel = gemm_f32_kernel<BM, BN, WAVES, EPI, AM, BK, SPLIT>;
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
