// fp32 GEMM on the bf16 matrix cores, for products of many tiles: each fp32 operand element is three bf16
// (F32Pair, gemm_f32.h) and a product is eight of their nine products.
//
// One workgroup of 2 x 4 waves owns a 128 x 128 tile of C, each wave a 64 x 32 part, and walks K in stages of 32. The
// workgroup splits each element once, on its way into LDS: stage s + 2 travels from global memory into registers while
// stage s + 1 is taken apart and laid down in one LDS buffer and stage s is multiplied out of the other; one barrier
// closes the stage. The vector units that do the splitting are the second bound after the matrix cores (five vector
// instructions hide behind a 32 x 32 x 16 MFMA, two behind a 16 x 16 x 32 one; measured), hence the large tile and the
// large MFMA.
//
// 4096^3 890 us (154 TFLOP/s: 1230 of bf16 products, where the clock falls to what the matrix cores' power leaves), 2048^3
// 117, 1332 x 50257 x 768 820; fp32 MFMAs took 1110, 169 and 870.
//
// LDS: three planes (high, middle, low parts) of four chunks of eight k; a chunk holds 16 bytes per row, so that both the
// fragment reads (32 rows of one chunk per half wave) and the eight-byte stores run without bank conflicts.
//
// The MFMA gets the B fragment first, so a lane ends up with one row m of C and four consecutive
// columns per register quad: 16-byte stores after bias and epilogue.
#pragma once

#include "gemm_f32_short.h"

namespace tmb {

constexpr int kF32Wide = 128, kF32WideThreads = 512;

// One operand's share of a stage: 128 rows by 32 k, of which a thread brings four consecutive k of two rows.
template <bool K_CONTIGUOUS>
struct F32Staged {
  static constexpr int ROWS = kF32Wide, ITEMS = ROWS / 64;
  static constexpr int CHUNK = ROWS * 16 + 64;  // bytes; the pad spreads the chunks that a store goes to over the banks
  static constexpr int PLANE = 4 * CHUNK, BYTES = 3 * PLANE;
  f32x4_t v[ITEMS];
  const float* at[ITEMS];  // K-contiguous: this thread's four k of stage 0; otherwise its column in the first k-row
  int64_t ld;
  int k4;      // which four of the stage's k
  int write;   // byte offset of item 0 in a plane

  // base: the operand's first row of the tile. `rows`: how many rows exist from there on (rows past the edge re-read
  // the last one: computed, never stored).
  __device__ __forceinline__ void plan(const float* base, int64_t ld_, int64_t rows, int wave, int lane) {
    ld = ld_;
    const int row = K_CONTIGUOUS ? wave * 8 + lane / 8 : lane;
    k4 = K_CONTIGUOUS ? lane % 8 : wave;
    write = (k4 >> 1) * CHUNK + row * 16 + (k4 & 1) * 8;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int64_t r = row + 64 * i < rows ? row + 64 * i : rows - 1;
      at[i] = K_CONTIGUOUS ? base + r * ld + 4 * k4 : base + r;
    }
  }
  // Item i of a stage that lies inside K and begins at k0.
  __device__ __forceinline__ void load(int i, int64_t k0) {
    if constexpr (K_CONTIGUOUS) {
      v[i] = *reinterpret_cast<const f32x4_unaligned_t*>(at[i] + k0);
    } else {
      const float* p = at[i] + (k0 + 4 * k4) * ld;
      v[i] = f32x4_t{p[0], p[ld], p[2 * ld], p[3 * ld]};
    }
  }
  // Any stage; elements past K are zeros.
  __device__ __forceinline__ void load_stage(int64_t k0, int64_t K) {
    if (k0 + 32 <= K) {
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) load(i, k0);
    } else {
      const int64_t left = K - k0 - 4 * k4;
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        const float* p = K_CONTIGUOUS ? at[i] + k0 : at[i] + (k0 + 4 * k4) * ld;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] = e < left ? p[K_CONTIGUOUS ? e : e * ld] : 0.0f;
      }
    }
  }
  // Half `p` (two k) of item i taken apart, and the whole item laid down.
  __device__ __forceinline__ void split(int i, int p, u32x2_t& h, u32x2_t& m, u32x2_t& l) const {
    const F32Pair s = F32Pair::of(v[i][2 * p], v[i][2 * p + 1]);
    h[p] = s.h;
    m[p] = s.m;
    l[p] = s.l;
  }
  __device__ __forceinline__ void lay_down(unsigned char* __restrict__ lds, int i, u32x2_t h, u32x2_t m, u32x2_t l) const {
    unsigned char* dst = lds + write + i * 64 * 16;
    *reinterpret_cast<u32x2_t*>(dst) = h;
    *reinterpret_cast<u32x2_t*>(dst + PLANE) = m;
    *reinterpret_cast<u32x2_t*>(dst + 2 * PLANE) = l;
  }
  __device__ __forceinline__ void lay_down_all(unsigned char* __restrict__ lds) const {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      u32x2_t h, m, l;
      split(i, 0, h, m, l);
      split(i, 1, h, m, l);
      lay_down(lds, i, h, m, l);
    }
  }
  // The stage as it is, rows of 32 k (four more floats spread them over the banks), and four k of a row of it.
  static constexpr int RAW_PITCH = 36, RAW_FLOATS = ROWS * RAW_PITCH;
  __device__ __forceinline__ void lay_down_raw(float* __restrict__ lds, int wave, int lane) const {
    const int row = K_CONTIGUOUS ? wave * 8 + lane / 8 : lane;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) *reinterpret_cast<f32x4_t*>(lds + (row + 64 * i) * RAW_PITCH + 4 * k4) = v[i];
  }
  static __device__ __forceinline__ f32x4_t raw_fragment(const float* __restrict__ lds, int row, int quad) {
    return *reinterpret_cast<const f32x4_t*>(lds + row * RAW_PITCH + 4 * quad);
  }
  // The eight k of chunk `chunk` in row `row`, part `part` (0 high, 1 middle, 2 low).
  static __device__ __forceinline__ u32x4_t fragment(const unsigned char* __restrict__ lds, int part, int row, int chunk) {
    return *reinterpret_cast<const u32x4_t*>(lds + part * PLANE + chunk * CHUNK + row * 16);
  }
};

template <int EPI, bool A_MMAJOR, bool B_KMAJOR>
__global__ __launch_bounds__(kF32WideThreads) void gemm_f32_wide_kernel(const GemmArgs g) {
  using StagedA = F32Staged<!A_MMAJOR>;
  using StagedB = F32Staged<B_KMAJOR>;
  constexpr int WAVES_N = 4, TM = 2;
  constexpr int STAGE = StagedA::BYTES + StagedB::BYTES;
  extern __shared__ __attribute__((aligned(16))) unsigned char f32_wide_lds[];

  int tm, tn;
  tile_of_block(blockIdx.x, g.tiles_m, g.tiles_n, tm, tn);
  // a split launch (g.splits > 0): blockIdx.y is the split, which multiplies its run of stages and
  // stores fp32 partials [splits][M][N]
  const int64_t split = g.splits > 0 ? blockIdx.y : 0;
  const int64_t batch = g.splits > 0 ? 0 : blockIdx.y;
  const int64_t m0 = static_cast<int64_t>(tm) * kF32Wide, n0 = static_cast<int64_t>(tn) * kF32Wide;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 31, lk = lane >> 5;
  const int row0 = wave / WAVES_N * 64, col0 = wave % WAVES_N * 32;  // the wave's part of the tile
  const int64_t M = g.m, N = g.n, K = g.k;
  const float* A = static_cast<const float*>(g.a) + batch * g.stride_a + (A_MMAJOR ? m0 : m0 * g.lda);
  const float* B = static_cast<const float*>(g.b) + batch * g.stride_b + (B_KMAJOR ? n0 * g.ldb : n0);
  int64_t first = 0, last = (K + 31) / 32;
  if (g.splits > 0) {
    const int64_t stages = last;
    first = stages * split / g.splits;
    last = stages * (split + 1) / g.splits;
  }
  StagedA sa;
  StagedB sb;
  sa.plan(A, g.lda, M - m0, wave, lane);
  sb.plan(B, g.ldb, N - n0, wave, lane);
  f32x16_t acc[TM], t[TM], u[TM];  // the sum; a run of stages' small products, and its large ones

  auto close_stage = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  u32x4_t a[2][TM][3], b[2][3];
  auto read_b = [&](const unsigned char* stage, int half, int part) {
    b[half][part] = StagedB::fragment(stage + StagedA::BYTES, part, col0 + lr, 2 * half + lk);
  };
  auto read_a = [&](const unsigned char* stage, int half, int i, int part) {
    a[half][i][part] = StagedA::fragment(stage, part, row0 + i * 32 + lr, 2 * half + lk);
  };
  auto read_first_half = [&](const unsigned char* stage) {
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      read_b(stage, 0, 2 - part);
#pragma unroll
      for (int i = 0; i < TM; ++i) read_a(stage, 0, i, part);
    }
  };
  // A stage's products, added to u (high part times high part) and t (the others, 2^-8 and less of them: in a sum of
  // their own their bits are not lost to the MFMA's alignment, and a single product is rounded once). A run of stages'
  // u + t is joined to the sum in one addition per element; runs of about the square root of the stages make the errors of
  // the two levels least (K = 768, positive operands: 5.0e-8, joined every stage 7.6e-8; K = 6000 7.9e-8 against 1.06e-7
  // in runs of four). A step is two MFMAs, the reading of a fragment that comes later and a share of
  // the next stage's splitting; nothing moves between steps, so that the vector instructions stand behind the MFMAs.
  // The barrier that closes the stage is in front of the last steps, which hide the reading of the next stage's first
  // fragments: by then every wave has read all it needs of this stage and laid down its part of the next.
  auto multiply = [&](const unsigned char* cur, unsigned char* next, int64_t k_after, auto splits_next) {
    constexpr bool NEXT = decltype(splits_next)::value;
    constexpr int TERMS = 8, STEPS = 2 * TERMS, CLOSE = STEPS - 3, PAIRS = 2 * (StagedA::ITEMS + StagedB::ITEMS);
    static_assert(PAIRS < CLOSE, "laid down before the barrier");
    constexpr int kPartA[TERMS] = {1, 2, 0, 2, 1, 0, 1, 0}, kPartB[TERMS] = {2, 1, 2, 0, 1, 1, 0, 0};  // (smallest first)
    u32x2_t h, m, l;
#pragma unroll
    for (int step = 0; step < STEPS; ++step) {
      const int half = step / TERMS, term = step % TERMS;
      if (NEXT && step == CLOSE) {
        close_stage();
        read_first_half(next);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        f32x16_t& sum = term == TERMS - 1 ? u[i] : t[i];
        sum = Mfma<bf16_t>::run(b[half][kPartB[term]], a[half][i][kPartA[term]], sum);
      }
      if (half == 0 && term < 6) {
        if (term < 3) read_b(cur, 1, 2 - term);
        read_a(cur, 1, term & 1, term >> 1);
      }
      if (NEXT && step < PAIRS) {
        const int item = step >> 1;
        if (item < StagedA::ITEMS) sa.split(item, step & 1, h, m, l);
        else sb.split(item - StagedA::ITEMS, step & 1, h, m, l);
        if ((step & 1) != 0) {
          if (item < StagedA::ITEMS) {
            sa.lay_down(next, item, h, m, l);
            sa.load(item, k_after);
          } else {
            sb.lay_down(next + StagedA::BYTES, item - StagedA::ITEMS, h, m, l);
            sb.load(item - StagedA::ITEMS, k_after);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto join = [&] {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[i][e] += u[i][e] + t[i][e];
        t[i][e] = u[i][e] = 0.0f;
      }
  };

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = t[i][e] = u[i][e] = 0.0f;
  if (first < last) {
    sa.load_stage(first * 32, K);
    sb.load_stage(first * 32, K);
    sa.lay_down_all(f32_wide_lds);
    sb.lay_down_all(f32_wide_lds + StagedA::BYTES);
    if (first + 1 < last) {
      sa.load_stage((first + 1) * 32, K);
      sb.load_stage((first + 1) * 32, K);
    }
    close_stage();
    read_first_half(f32_wide_lds);
    int run = 1;
    while (run < 16 && 4 * run * run <= last - first) run *= 2;
    int buffer = 0;
    for (int64_t s = first; s + 1 < last; ++s) {
      // (an element's register is loaded again as soon as it has been taken apart: a stage's time for the way from
      // memory. Where there is no stage s + 2 or it ends past K, what is loaded is not used.)
      const bool whole = s + 2 < last && (s + 3) * 32 <= K;
      multiply(f32_wide_lds + buffer * STAGE, f32_wide_lds + (buffer ^ 1) * STAGE, (whole ? s + 2 : first) * 32,
               std::true_type{});
      if (!whole && s + 2 < last) {
        sa.load_stage((s + 2) * 32, K);
        sb.load_stage((s + 2) * 32, K);
      }
      if (((s - first) & (run - 1)) == run - 1) join();
      buffer ^= 1;
    }
    multiply(f32_wide_lds + buffer * STAGE, nullptr, 0, std::false_type{});
    join();
  }

  // Sums that are not finite (an operand or a result that is not, or one beyond what the factor leaves room for) are
  // formed again from fp32 products; their neighbours keep theirs, so a row's bits do not depend on others. (4096^3 with a NaN
  // in one row 1630 us for 910, in every row 2020; each wave by itself, two k at a time from memory: 2400 and 6010.)
  __shared__ int wave_spoiled[kF32WideThreads / 64];
  uint32_t spoiled = 0;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      spoiled |= (__builtin_fabsf(acc[i][e]) < HUGE_VALF ? 0u : 1u) << (16 * i + e);
      acc[i][e] *= F32Pair::kDown * F32Pair::kDown;
    }
  const uint64_t any = __ballot(spoiled != 0);
  if (lane == 0) wave_spoiled[wave] = any != 0;
  __syncthreads();
  bool again = false;
#pragma unroll
  for (int w = 0; w < kF32WideThreads / 64; ++w) again |= wave_spoiled[w] != 0;
  if (again) {
    float* ra = reinterpret_cast<float*>(f32_wide_lds);
    float* rb = ra + StagedA::RAW_FLOATS;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) t[i][e] = 0.0f;
    sa.load_stage(first * 32, K);
    sb.load_stage(first * 32, K);
#pragma unroll 1
    for (int64_t s = first; s < last; ++s) {
      sa.lay_down_raw(ra, wave, lane);
      sb.lay_down_raw(rb, wave, lane);
      __syncthreads();
      if (s + 1 < last) {
        sa.load_stage((s + 1) * 32, K);
        sb.load_stage((s + 1) * 32, K);
      }
#pragma unroll
      for (int k8 = 0; k8 < 4; ++k8) {
        const f32x4_t bf = StagedB::raw_fragment(rb, col0 + lr, 2 * k8 + lk);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const f32x4_t af = StagedA::raw_fragment(ra, row0 + i * 32 + lr, 2 * k8 + lk);
#pragma unroll
          for (int e = 0; e < 4; ++e) t[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(bf[e], af[e], t[i], 0, 0, 0);
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][e] = (spoiled >> (16 * i + e) & 1) != 0 ? t[i][e] : acc[i][e];
  }

  // Lane holds row lr of each 32 x 32 result and columns 8q + 4 * lk + {0..3}.
  const float* __restrict__ bias = static_cast<const float*>(g.bias);
  float* __restrict__ C = static_cast<float*>(g.c) + (batch + split) * g.stride_c;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t row = m0 + row0 + i * 32 + lr;
    if (row >= M) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t col = n0 + col0 + 8 * q + 4 * lk;
      if (col >= N) continue;
      float* dst = C + row * g.ldc + col;
      float out[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = acc[i][4 * q + e];
        if (bias != nullptr && col + e < N) v += bias[col + e];
        out[e] = finish<float, EPI>(v, false);
      }
      if (col + 4 <= N) {
        const f32x4_unaligned_t v = {out[0], out[1], out[2], out[3]};
        if (g.stream_c) __builtin_nontemporal_store(v, reinterpret_cast<f32x4_unaligned_t*>(dst));
        else *reinterpret_cast<f32x4_unaligned_t*>(dst) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < N) dst[e] = out[e];
      }
    }
  }
}

// 16-byte loads need whole, aligned chunks along each operand's contiguous direction.
static inline bool f32_mfma_eligible(const GemmArgs& g, int64_t batch, int trans_a, int trans_b) {
  if (g.m < 1 || g.n < 1 || g.k < 1) return false;
  if (g.lda % 4 != 0 || g.ldb % 4 != 0) return false;
  if ((reinterpret_cast<uintptr_t>(g.a) & 15) != 0 || (reinterpret_cast<uintptr_t>(g.b) & 15) != 0)
    return false;
  if (batch > 1 && (g.stride_a % 4 != 0 || g.stride_b % 4 != 0)) return false;
  if (trans_a ? g.m % 4 != 0 : g.k % 4 != 0) return false;
  if (trans_b ? g.k % 4 != 0 : g.n % 4 != 0) return false;
  const int64_t tiles_m = (g.m + 127) / 128, tiles_n = (g.n + 127) / 128;
  return tiles_m * tiles_n < (int64_t{1} << 30) && tiles_m < (1 << 24) && tiles_n < (1 << 24);
}

template <int EPI>
static int launch_f32_wide(GemmArgs g, int64_t batch, int trans_a, int trans_b, hipStream_t stream) {
  g.tiles_m = static_cast<int>((g.m + kF32Wide - 1) / kF32Wide);
  g.tiles_n = static_cast<int>((g.n + kF32Wide - 1) / kF32Wide);
  if (g.k <= kF32SplitK) return launch_f32_mfma<EPI>(g, batch, trans_a, trans_b, stream);
  g.stream_c = batch * g.m * g.n * 4 > (int64_t{256} << 20);
  const dim3 grid(static_cast<unsigned>(g.tiles_m * g.tiles_n), static_cast<unsigned>(batch));
  auto go = [&](auto a_mmajor, auto b_kmajor) {
    constexpr bool AM = decltype(a_mmajor)::value, BK = decltype(b_kmajor)::value;
    constexpr int SMEM = 2 * (F32Staged<!AM>::BYTES + F32Staged<BK>::BYTES);
    static_assert(SMEM <= 160 * 1024, "LDS of one CU");
    auto kernel = gemm_f32_wide_kernel<EPI, AM, BK>;
    static bool configured = false;
    if (!configured) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
      if (e != hipSuccess) return static_cast<int>(e);
      configured = true;
    }
    kernel<<<grid, kF32WideThreads, SMEM, stream>>>(g);
    return check_launch();
  };
  if (trans_a) return trans_b ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
  return trans_b ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
}

}  // namespace tmb
