// Fused float32 attention for gfx950, forward and backward, heads of 64: out = softmax(scale * q k^T
// [+ causal mask]) v and its gradients without the [batch, heads, q_len, kv_len] scores in memory.
//
// fp32 MFMAs (32 x 32 x 2: 4096 operations in 64 cycles of a SIMD) set the pace, and at that pace
// nothing needs LDS on its way in: a wave multiplies 32 x 32 pieces of the score matrix and takes
// both operands straight from memory (L2) into registers, 48 loads against 64 MFMAs of the forward.
// A lane keeps one COLUMN of a piece (its own query, or key in the dK/dV kernel), so the row
// statistics are in-lane sums plus one exchange between lanes l and l^32, and the exponentials lie in
// registers the way the next product takes its B operand.
//
// The k index of an MFMA is free to stand for any dimension as long as A and B agree: lanes 0..31 hold the even
// quads of a row's dimensions, lanes 32..63 the odd ones, as 16-byte loads deliver them. The transposed operands
// (V^T, K^T, Q^T, dout^T) are loaded as rows too: register r of a piece is row 8 (r / 4) + 4 (lane / 32) + r % 4, and
// a lane takes dimensions 2 (lane % 32) and 2 (lane % 32) + 1 of it, one for each of its two 32 x 32 tiles.
//
// Four waves share 32 queries (keys): each walks every fourth block of 32 keys (queries) with
// statistics and sums of its own, and LDS is where the four meet at the end, in wave order: results
// do not depend on scheduling. That makes 4 * batch * heads * ceil(len / 32) waves, enough for the
// 1024 SIMDs at 4 sequences of 333, and shortens each sum.
//
// Sums of 64 products and of many keys run as short chains that are then added, so that no result is further off
// float64 than the op-by-op chain's (relative error of out, dq, dk, dv over 4 x 12 heads x 333 tokens 1.34, 1.81,
// 1.89, 1.50e-7 against 1.44, 2.10, 2.16, 1.52e-7; x 1024 1.44, 1.87, 1.98, 1.65 against 2.26, 2.77, 2.85, 2.35;
// x 64 1.17, 1.82, 1.86, 1.32 against 1.35, 1.86, 1.98, 1.58).
//
// What bounds it: the MFMAs (62-68 % of the SIMDs' time without a mask) and, one after the other with them on a
// SIMD, some 6 vector instructions per MFMA; under a causal mask also workgroups of unequal length on 512 places.
// Against the op-by-op chain (two products, copies, softmax), 12 heads, us forward / forward and backward: 4 x 333
// 93 -> 20 / 208 -> 78, 3 x 250 58 -> 13 / 124 -> 51, 4 x 1024 266 -> 82 / 729 -> 349, 1 x 128 23 -> 8 / 52 -> 30,
// 1 x 16 20 -> 7 / 44 -> 24.
//
// Scores are rounded to float32 before and after the scale, as a product and a multiplication store them, and the
// exponential is exp_f32 of the difference to the row's maximum: what a separate softmax computes.
//
// Infinities and NaN: what a query sees reaches it as through a softmax and two products. What the mask hides from it is
// multiplied by its probability of 0 only within its own block of 32, by the MFMAs: an infinite or NaN value (in dq: key;
// in dk, dv: query, dout) that is hidden from all of a block does not reach the block, where a product with the whole
// score matrix would give NaN, and one that part of a block sees leaves NaN in the rest of that block too.
#include "tmb_common.h"

namespace tmb {

typedef float af32x16_t __attribute__((ext_vector_type(16)));
typedef float af32x4_t __attribute__((ext_vector_type(4)));
typedef float af32x2_t __attribute__((ext_vector_type(2)));

constexpr int kF32Block = 32;    // queries and keys of one piece
constexpr int kF32Waves = 4;     // waves that share a workgroup's queries (keys)
constexpr int kF32Pitch = 68;    // floats per row of the LDS the waves meet in (64 + padding)
constexpr int kF32Chunk = 64;    // heads whose K and V (Q and dout) the L2s hold at a time

struct AttnF32Strides {
  int64_t b, h, t;  // elements: batch, head, token (head_dim is contiguous)
};

struct AttnF32Args {
  float* out;
  float* stats;  // may be null: [batch, heads, q_len, 2], maximum of the scaled, masked scores and sum of exponentials
  const float* q;
  const float* k;
  const float* v;
  AttnF32Strides qs, ks, vs, os;
  int heads, bh, q_len, kv_len;
  float scale;
  int causal;
};

struct AttnF32BwdArgs {
  float* dq;
  float* dk;
  float* dv;
  const float* dout;
  const float* q;
  const float* k;
  const float* v;
  const float* out;
  const float* stats;
  af32x4_t* rows;  // workspace [batch, heads, q_len], from the dq kernel: maximum, 1 / sum, sum of dout * out, 0
  AttnF32Strides qs, ks, vs, os, gs, dqs, dks, dvs;
  int heads, bh, q_len, kv_len;
  float scale;
  int causal;
};

__device__ __forceinline__ float f32_other_half(float x, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, x)));
}

// exp of a difference to a maximum (<= 0, -inf, or NaN): exp_f32 without what only larger arguments need
__device__ __forceinline__ float f32_exp_nonpositive(float x) {
#pragma clang fp contract(off)
  constexpr float kLog2eHi = 1.44269502162933349609375f, kLog2eLo = 1.92596299112661746e-08f;
  constexpr float kLn2 = 0.693147180559945309417f;
  const float c = x < -200.0f ? -200.0f : x;  // 2^-288 is 0, and keeps -inf out of the correction
  const float hi = c * kLog2eHi;
  const float lo = __builtin_fmaf(c, kLog2eHi, -hi) + c * kLog2eLo;
  const float e = __builtin_amdgcn_exp2f(hi);
  return __builtin_fmaf(e, lo * kLn2, e);
}

// A scaled score, rounded by itself wherever it is formed: the backward takes the forward's maximum off the same number
__device__ __forceinline__ float f32_scaled(float score, float scale) {
#pragma clang fp contract(off)
  return score * scale;
}

__device__ __forceinline__ void f32_clear(af32x16_t& x) {
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = 0.0f;
}

// The rows of one (batch, head): 32-bit byte offsets from its first element, and rows past the last read as 0 (the
// buffer ends there), so no block needs a bounds check or a clamp of its own.
struct F32Rows {
  __amdgpu_buffer_rsrc_t buf;
  uint32_t pitch;  // bytes
};
__device__ __forceinline__ F32Rows f32_rows(const float* base, int64_t stride, int len) {
  const uint32_t bytes = static_cast<uint32_t>(((len - 1) * stride + 64) * 4);
  return {__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, static_cast<int>(bytes), 0x00020000),
          static_cast<uint32_t>(stride) * 4u};
}

// A lane's 32 floats of an operand row: 8 loads of 16 bytes, the two lanes of a row side by side. Four loads in a
// row then take up the 32 lines they touch whole (with 128 contiguous bytes per lane eight loads of 64 lines
// each, whose lines the L1 had dropped by the time the last were read).
__device__ __forceinline__ void f32_load_row(af32x4_t (&r)[8], const F32Rows& rows, int row0, int lane) {
  const uint32_t off = static_cast<uint32_t>(row0 + (lane & 31)) * rows.pitch + (lane >> 5) * 16u;
#pragma unroll
  for (int j = 0; j < 8; ++j)
    r[j] = __builtin_bit_cast(af32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rows.buf, off + 32 * j, 0, 0));
}

// The transposed operand of a block of 32 rows from `row0`: register r is row 8 (r / 4) + 4 half + r % 4, two
// dimensions per lane.
__device__ __forceinline__ void f32_load_tr(af32x2_t (&r)[16], const F32Rows& rows, int row0, int lane) {
  const uint32_t off = static_cast<uint32_t>(row0 + (lane >> 5) * 4) * rows.pitch + (lane & 31) * 8u;
#pragma unroll
  for (int i = 0; i < 16; ++i)
    r[i] = __builtin_bit_cast(af32x2_t, __builtin_amdgcn_raw_buffer_load_b64(
                                            rows.buf, off + (8 * (i >> 2) + (i & 3)) * rows.pitch, 0, 0));
}

__device__ __forceinline__ af32x16_t f32_mfma(float a, float b, af32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Operand rows that all waves of a workgroup share, in LDS as the lanes read them
typedef af32x4_t F32Shared[8][kWave];
__device__ __forceinline__ const af32x4_t& f32_part(const af32x4_t (&b)[8], int j, int) { return b[j]; }
__device__ __forceinline__ af32x4_t f32_part(const F32Shared& b, int j, int lane) { return b[j][lane]; }

// rows(a) x rows(b)^T over the 64 dimensions in chains of 8 * CHAIN products that are then added; element r of the result: row 8 (r / 4) + 4 half + r % 4 of a, row
// lane % 32 of b
template <int CHAIN = 2, typename B>
__device__ __forceinline__ af32x16_t f32_scores(const af32x4_t (&a)[8], const B& b, int lane) {
  af32x16_t total;
#pragma unroll
  for (int c = 0; c < 8; c += CHAIN) {
    af32x16_t acc;
    f32_clear(acc);
#pragma unroll
    for (int j = c; j < c + CHAIN; ++j) {
      const af32x4_t x = f32_part(b, j, lane);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = f32_mfma(a[j][e], x[e], acc);
    }
    total = c == 0 ? acc : total + acc;
    __builtin_amdgcn_sched_barrier(0);
  }
  return total;
}

// acc[dt] += tr^T x p over the block's 32 rows, 16 products a chain; element r of tile dt: dimension 2 (8 (r / 4) + 4 half + r % 4) + dt
__device__ __forceinline__ void f32_apply(af32x16_t (&acc)[2], const af32x2_t (&tr)[16], const af32x16_t& p) {
#pragma unroll
  for (int dt = 0; dt < 2; ++dt) {
    af32x16_t lo, hi;
    f32_clear(lo);
    f32_clear(hi);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      lo = f32_mfma(tr[r][dt], p[r], lo);
      hi = f32_mfma(tr[r + 8][dt], p[r + 8], hi);
    }
    acc[dt] += lo + hi;
    __builtin_amdgcn_sched_barrier(0);
  }
}

// A wave's [32 columns x 64 dimensions] accumulator as rows of LDS: row = lane % 32, dimensions in order.
__device__ __forceinline__ void f32_store_acc(float* rows, const af32x16_t (&acc)[2], int lane) {
  float* dst = rows + (lane & 31) * kF32Pitch + (lane >> 5) * 8;
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      af32x4_t x;
      x[0] = acc[0][4 * g + 2 * i];
      x[1] = acc[1][4 * g + 2 * i];
      x[2] = acc[0][4 * g + 2 * i + 1];
      x[3] = acc[1][4 * g + 2 * i + 1];
      *reinterpret_cast<af32x4_t*>(dst + 16 * g + 4 * i) = x;
    }
}

// Which block of which (batch, head) a workgroup takes. Workgroup i runs on XCD i % 8: with the heads innermost a
// head's workgroups meet on one or two XCDs, and its K and V in their L2s. A causal block's cost
// grows with its index (dq) or falls with it (dkv); the dear ones go first. `kF32Chunk` heads at a time, so that
// a large batch still finds its operands in the L2s (8 heads of 1024 tokens each: 4 MB).
__device__ __forceinline__ void f32_unit(int id, int bh, int blocks, int& head, int& block) {
  const int chunk = id / (kF32Chunk * blocks);
  const int rem = id - chunk * (kF32Chunk * blocks);
  const int left = bh - chunk * kF32Chunk;
  const int n = left < kF32Chunk ? left : kF32Chunk;
  block = rem / n;
  head = chunk * kF32Chunk + rem % n;
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attention_f32_fwd_kernel(
    AttnF32Args a) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) float sums[kF32Waves * kF32Block * kF32Pitch];
  __shared__ float wave_m[kF32Waves * kF32Block], wave_l[kF32Waves * kF32Block];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5;
  const int n_qb = (a.q_len + kF32Block - 1) / kF32Block;
  int bh, rev;
  f32_unit(blockIdx.x, a.bh, n_qb, bh, rev);
  const int b = bh / a.heads, h = bh % a.heads;
  const int q0 = (n_qb - 1 - rev) * kF32Block;
  const int qi = q0 + (lane & 31);
  const float neg_inf = -__builtin_inff();
  const F32Rows kr = f32_rows(a.k + b * a.ks.b + h * a.ks.h, a.ks.t, a.kv_len);
  const F32Rows vr = f32_rows(a.v + b * a.vs.b + h * a.vs.h, a.vs.t, a.kv_len);

  af32x4_t qf[8];
  f32_load_row(qf, f32_rows(a.q + b * a.qs.b + h * a.qs.h, a.qs.t, a.q_len), q0, lane);

  int n_kb = (a.kv_len + kF32Block - 1) / kF32Block;
  if (a.causal) {
    const int need = q0 / kF32Block + 1;
    n_kb = n_kb < need ? n_kb : need;
  }

  af32x16_t acc_o[2];
  f32_clear(acc_o[0]);
  f32_clear(acc_o[1]);
  float m_run = neg_inf, l_run = 0.0f;
  af32x4_t kf[8];
  if (wave < n_kb) f32_load_row(kf, kr, wave * kF32Block, lane);
  for (int blk = wave; blk < n_kb; blk += kF32Waves) {
    const int k0 = blk * kF32Block;
    af32x2_t vf[16];
    f32_load_tr(vf, vr, k0, lane);                 // arrives while the scores are formed
    __builtin_amdgcn_sched_barrier(0);
    af32x16_t s = f32_scores(kf, qf, lane);
    __builtin_amdgcn_sched_barrier(0);
    const int next = blk + kF32Waves < n_kb ? blk + kF32Waves : blk;
    f32_load_row(kf, kr, next * kF32Block, lane);  // arrives while the values are multiplied
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = f32_scaled(s[r], a.scale);
    if ((a.causal && k0 + kF32Block - 1 > q0) || k0 + kF32Block > a.kv_len) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + 8 * (r >> 2) + 4 * half + (r & 3);
        s[r] = (a.causal && key > qi) || key >= a.kv_len ? neg_inf : s[r];
      }
    }
    float m_blk = neg_inf;
#pragma unroll
    for (int r = 0; r < 16; ++r) m_blk = fmaxf(m_blk, s[r]);
    m_blk = fmaxf(m_blk, f32_other_half(m_blk, lane));
    const float m_new = fmaxf(m_run, m_blk);
    const float m_use = m_new == neg_inf ? 0.0f : m_new;  // nothing visible yet: keep the difference defined
    const float alpha = f32_exp_nonpositive(m_run - m_use);
    float l_blk = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = f32_exp_nonpositive(s[r] - m_use);
      l_blk += s[r];
    }
    l_run = l_run * alpha + l_blk;  // (of this half's keys: the halves meet at the end)
    m_run = m_new;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc_o[dt][e] *= alpha;
    f32_apply(acc_o, vf, s);
  }
  l_run += f32_other_half(l_run, lane);
  if (half == 0) {
    wave_m[wave * kF32Block + lane] = m_run;
    wave_l[wave * kF32Block + lane] = l_run;
  }
  f32_store_acc(sums + wave * kF32Block * kF32Pitch, acc_o, lane);
  __syncthreads();

  // 8 dimensions of one query per thread, the waves in order
  const int qr = tid >> 3, d0 = (tid & 7) * 8;
  float m_all = neg_inf;
#pragma unroll
  for (int w = 0; w < kF32Waves; ++w) m_all = fmaxf(m_all, wave_m[w * kF32Block + qr]);
  const float m_use = m_all == neg_inf ? 0.0f : m_all;
  float l = 0.0f, o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = 0.0f;
#pragma unroll
  for (int w = 0; w < kF32Waves; ++w) {
    if (w >= n_kb) break;  // no block, nothing to add
    const float f = f32_exp_nonpositive(wave_m[w * kF32Block + qr] - m_use);
    l += f * wave_l[w * kF32Block + qr];
    const float* src = sums + (w * kF32Block + qr) * kF32Pitch + d0;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] += f * src[e];
  }
  const int64_t query = q0 + qr;
  if (query < a.q_len) {
    const float inv = 1.0f / l;
    float* dst = a.out + b * a.os.b + h * a.os.h + query * a.os.t + d0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      af32x4_t x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = o[4 * i + e] * inv;
      *reinterpret_cast<af32x4_t*>(dst + 4 * i) = x;
    }
    if (a.stats != nullptr && d0 == 0) {
      float* st = a.stats + (static_cast<int64_t>(bh) * a.q_len + query) * 2;
      st[0] = m_use;
      st[1] = l;
    }
  }
#endif
}

// dq: as the forward, a lane owning a query. dS^T = P^T (dP^T - delta) scale with P from the forward's maximum and
// sum; delta = sum of dout * out is formed first and left, beside them, for the second launch. The operand rows
// of the queries are the same for the four waves and stay in LDS (registers would hold 64 more): 16 reads of 16
// bytes against 96 MFMAs.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attention_f32_bwd_dq_kernel(
    AttnF32BwdArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) float sums[kF32Waves * kF32Block * kF32Pitch];
  __shared__ F32Shared q_rows, g_rows;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5;
  const int n_qb = (a.q_len + kF32Block - 1) / kF32Block;
  int bh, rev;
  f32_unit(blockIdx.x, a.bh, n_qb, bh, rev);
  const int b = bh / a.heads, h = bh % a.heads;
  const int q0 = (n_qb - 1 - rev) * kF32Block;
  const int qi = q0 + (lane & 31);
  const int64_t qr = qi < a.q_len ? qi : a.q_len - 1;
  const F32Rows kr = f32_rows(a.k + b * a.ks.b + h * a.ks.h, a.ks.t, a.kv_len);
  const F32Rows vr = f32_rows(a.v + b * a.vs.b + h * a.vs.h, a.vs.t, a.kv_len);

  float delta = 0.0f;
  {
    af32x4_t gf[8], of[8];
    f32_load_row(gf, f32_rows(a.dout + b * a.gs.b + h * a.gs.h, a.gs.t, a.q_len), q0, lane);
    f32_load_row(of, f32_rows(a.out + b * a.os.b + h * a.os.h, a.os.t, a.q_len), q0, lane);
    af32x4_t part = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[e] = __builtin_fmaf(gf[j][e], of[j][e], part[e]);
    delta = (part[0] + part[1]) + (part[2] + part[3]);
    delta += f32_other_half(delta, lane);
    if (wave == 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) g_rows[j][lane] = gf[j];
    } else if (wave == 1) {
      f32_load_row(of, f32_rows(a.q + b * a.qs.b + h * a.qs.h, a.qs.t, a.q_len), q0, lane);
#pragma unroll
      for (int j = 0; j < 8; ++j) q_rows[j][lane] = of[j];
    }
  }
  const af32x2_t st = *reinterpret_cast<const af32x2_t*>(a.stats + (static_cast<int64_t>(bh) * a.q_len + qr) * 2);
  const float m = st[0], inv_l = 1.0f / st[1];
  if (wave == 0 && half == 0 && qi < a.q_len) {
    af32x4_t x;
    x[0] = m;
    x[1] = inv_l;
    x[2] = delta;
    x[3] = 0.0f;
    a.rows[static_cast<int64_t>(bh) * a.q_len + qi] = x;
  }

  int n_kb = (a.kv_len + kF32Block - 1) / kF32Block;
  if (a.causal) {
    const int need = q0 / kF32Block + 1;
    n_kb = n_kb < need ? n_kb : need;
  }

  af32x16_t acc[2];
  f32_clear(acc[0]);
  f32_clear(acc[1]);
  af32x4_t kf[8], vf[8];
  if (wave < n_kb) {
    f32_load_row(kf, kr, wave * kF32Block, lane);
    f32_load_row(vf, vr, wave * kF32Block, lane);
  }
  __syncthreads();  // the shared rows
  for (int blk = wave; blk < n_kb; blk += kF32Waves) {
    const int k0 = blk * kF32Block;
    const int next = blk + kF32Waves < n_kb ? blk + kF32Waves : blk;
    af32x16_t s = f32_scores(kf, q_rows, lane);
    __builtin_amdgcn_sched_barrier(0);
    af32x2_t kt[16];
    f32_load_tr(kt, kr, k0, lane);
    __builtin_amdgcn_sched_barrier(0);
    af32x16_t dp = f32_scores<1>(vf, g_rows, lane);
    __builtin_amdgcn_sched_barrier(0);
    f32_load_row(kf, kr, next * kF32Block, lane);
    f32_load_row(vf, vr, next * kF32Block, lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 16; ++r)
      s[r] = f32_exp_nonpositive(f32_scaled(s[r], a.scale) - m) * inv_l * (dp[r] - delta) * a.scale;
    if ((a.causal && k0 + kF32Block - 1 > q0) || k0 + kF32Block > a.kv_len) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + 8 * (r >> 2) + 4 * half + (r & 3);
        s[r] = (a.causal && key > qi) || key >= a.kv_len ? 0.0f : s[r];
      }
    }
    f32_apply(acc, kt, s);
  }
  f32_store_acc(sums + wave * kF32Block * kF32Pitch, acc, lane);
  __syncthreads();
  const int row = tid >> 3, d0 = (tid & 7) * 8;
  if (q0 + row < a.q_len) {
    float* dst = a.dq + b * a.dqs.b + h * a.dqs.h + static_cast<int64_t>(q0 + row) * a.dqs.t + d0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      af32x4_t x = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int w = 0; w < kF32Waves; ++w)
        if (w < n_kb) x += *reinterpret_cast<const af32x4_t*>(sums + (w * kF32Block + row) * kF32Pitch + d0 + 4 * i);
      *reinterpret_cast<af32x4_t*>(dst + 4 * i) = x;
    }
  }
#endif
}

// dk, dv: a lane owns a key, and the waves share the query blocks that see the workgroup's 32 keys, whose operand
// rows stay in LDS as the queries' do above. A block's statistics (a lane holds scores of 16 queries) come in with
// its rows, one query per lane, and reach the other lanes through LDS of the wave's own.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attention_f32_bwd_dkv_kernel(
    AttnF32BwdArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) float sums[kF32Waves * kF32Block * kF32Pitch];
  __shared__ F32Shared k_rows, v_rows;
  __shared__ af32x4_t row_stats[kF32Waves][kF32Block];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5;
  const int n_kb = (a.kv_len + kF32Block - 1) / kF32Block;
  int bh, block;
  f32_unit(blockIdx.x, a.bh, n_kb, bh, block);
  const int b = bh / a.heads, h = bh % a.heads;
  const int k0 = block * kF32Block;
  const int ki = k0 + (lane & 31);
  const F32Rows qr = f32_rows(a.q + b * a.qs.b + h * a.qs.h, a.qs.t, a.q_len);
  const F32Rows gr = f32_rows(a.dout + b * a.gs.b + h * a.gs.h, a.gs.t, a.q_len);
  const af32x4_t* rows = a.rows + static_cast<int64_t>(bh) * a.q_len;
  if (wave < 2) {
    af32x4_t x[8];
    f32_load_row(x, wave == 0 ? f32_rows(a.k + b * a.ks.b + h * a.ks.h, a.ks.t, a.kv_len)
                              : f32_rows(a.v + b * a.vs.b + h * a.vs.h, a.vs.t, a.kv_len), k0, lane);
#pragma unroll
    for (int j = 0; j < 8; ++j) (wave == 0 ? k_rows : v_rows)[j][lane] = x[j];
  }
  __syncthreads();

  const int n_qb = (a.q_len + kF32Block - 1) / kF32Block;
  const int first = (a.causal ? block : 0) + wave;  // (keys past the last query: no block at all)
  const int last_query = a.q_len - 1;

  af32x16_t acc_k[2], acc_v[2];
#pragma unroll
  for (int dt = 0; dt < 2; ++dt) {
    f32_clear(acc_k[dt]);
    f32_clear(acc_v[dt]);
  }
  for (int blk = first; blk < n_qb; blk += kF32Waves) {
    const int q0 = blk * kF32Block;
    af32x4_t qf[8], gf[8];
    f32_load_row(qf, qr, q0, lane);
    f32_load_row(gf, gr, q0, lane);
    row_stats[wave][lane & 31] = rows[q0 + (lane & 31) < last_query ? q0 + (lane & 31) : last_query];  // (lanes l and l + 32 write the same)
    af32x16_t s = f32_scores(qf, k_rows, lane);
    __builtin_amdgcn_sched_barrier(0);
    af32x2_t gt[16];
    f32_load_tr(gt, gr, q0, lane);
    __builtin_amdgcn_sched_barrier(0);
    af32x16_t ds = f32_scores<1>(gf, v_rows, lane);
    __builtin_amdgcn_sched_barrier(0);
    af32x2_t qt[16];
    f32_load_tr(qt, qr, q0, lane);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // row_stats: this wave's own writes
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const af32x4_t st = row_stats[wave][8 * (r >> 2) + 4 * half + (r & 3)];
      s[r] = f32_exp_nonpositive(f32_scaled(s[r], a.scale) - st[0]) * st[1];
      ds[r] = s[r] * (ds[r] - st[2]) * a.scale;
      if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (all the statistics at once would be 64 registers)
    }
    if ((a.causal && k0 + kF32Block - 1 > q0) || k0 + kF32Block > a.kv_len || q0 + kF32Block > a.q_len) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int query = q0 + 8 * (r >> 2) + 4 * half + (r & 3);
        const bool hidden = (a.causal && ki > query) || ki >= a.kv_len || query >= a.q_len;
        s[r] = hidden ? 0.0f : s[r];
        ds[r] = hidden ? 0.0f : ds[r];
      }
    }
    f32_apply(acc_v, gt, s);
    f32_apply(acc_k, qt, ds);
  }
  const int row = tid >> 3, d0 = (tid & 7) * 8;
  auto merge = [&](const af32x16_t (&acc)[2], float* base, const AttnF32Strides& s) {
    f32_store_acc(sums + wave * kF32Block * kF32Pitch, acc, lane);
    __syncthreads();
    if (k0 + row < a.kv_len) {
      float* dst = base + b * s.b + h * s.h + static_cast<int64_t>(k0 + row) * s.t + d0;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        af32x4_t x = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < kF32Waves; ++w)
          x += *reinterpret_cast<const af32x4_t*>(sums + (w * kF32Block + row) * kF32Pitch + d0 + 4 * i);
        *reinterpret_cast<af32x4_t*>(dst + 4 * i) = x;
      }
    }
  };
  merge(acc_v, a.dv, a.dvs);
  __syncthreads();
  merge(acc_k, a.dk, a.dks);
#endif
}

// 16-byte accesses of every row, and 32-bit byte offsets from the first to the end of the last block of rows
static bool f32_layout(const void* p, const int64_t* s, int64_t len) {
  return aligned16(p) && s[0] % 4 == 0 && s[1] % 4 == 0 && s[2] % 4 == 0 && s[0] >= 0 && s[1] >= 0 && s[2] >= 0 &&
         s[2] < (int64_t{1} << 30) / (len + kF32Block);
}
static AttnF32Strides f32_strides(const int64_t* s) { return {s[0], s[1], s[2]}; }

static int64_t f32_blocks(int64_t len) { return (len + kF32Block - 1) / kF32Block; }

// (a grid has less than 2^32 threads, and a chunk of heads times its blocks is a 32-bit number in the kernels)
static bool f32_fits(int64_t bh, int64_t len) {
  return len < (int64_t{1} << 28) && bh < (int64_t{1} << 24) && bh * f32_blocks(len) < (int64_t{1} << 24);
}

}  // namespace tmb

extern "C" int tmb_attention_f32_fwd(void* out, void* stats, const void* q, const void* k, const void* v,
                                     int64_t batch, int64_t heads, int64_t q_len, int64_t kv_len, int64_t head_dim,
                                     const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                     const int64_t* out_strides, float scale, int causal, void* stream) {
  using namespace tmb;
  if (batch < 0 || heads < 0 || q_len < 0 || kv_len < 0) return TMB_ERR_INVALID_ARGUMENT;
  if (head_dim != 64) return TMB_ERR_UNSUPPORTED;
  if (!(scale == scale)) return TMB_ERR_INVALID_ARGUMENT;
  if (!(scale > 0.0f) || scale > 3.0e38f) return TMB_ERR_UNSUPPORTED;
  if (batch == 0 || heads == 0 || q_len == 0) return TMB_OK;
  if (kv_len == 0) return TMB_ERR_UNSUPPORTED;  // every row empty: left to the caller
  if (!out || !q || !k || !v || !q_strides || !k_strides || !v_strides || !out_strides)
    return TMB_ERR_INVALID_ARGUMENT;
  if (stats != nullptr && (reinterpret_cast<uintptr_t>(stats) & 7)) return TMB_ERR_INVALID_ARGUMENT;
  if (batch >= (int64_t{1} << 31) || heads >= (int64_t{1} << 31) || !f32_fits(batch * heads, q_len) ||
      !f32_fits(batch * heads, kv_len) || !f32_layout(q, q_strides, q_len) ||
      !f32_layout(k, k_strides, kv_len) || !f32_layout(v, v_strides, kv_len) || !f32_layout(out, out_strides, q_len))
    return TMB_ERR_UNSUPPORTED;
  AttnF32Args a{static_cast<float*>(out), static_cast<float*>(stats), static_cast<const float*>(q),
                static_cast<const float*>(k), static_cast<const float*>(v), f32_strides(q_strides),
                f32_strides(k_strides), f32_strides(v_strides), f32_strides(out_strides), static_cast<int>(heads),
                static_cast<int>(batch * heads), static_cast<int>(q_len), static_cast<int>(kv_len), scale,
                causal ? 1 : 0};
  const dim3 grid(static_cast<unsigned>(batch * heads * f32_blocks(q_len)));
  attention_f32_fwd_kernel<<<grid, dim3(256), 0, static_cast<hipStream_t>(stream)>>>(a);
  return check_launch();
}

extern "C" int64_t tmb_attention_f32_bwd_workspace_bytes(int64_t batch, int64_t heads, int64_t q_len) {
  if (batch < 0 || heads < 0 || q_len < 0) return 0;
  return batch * heads * q_len * static_cast<int64_t>(sizeof(tmb::af32x4_t));
}

extern "C" int tmb_attention_f32_bwd(void* dq, void* dk, void* dv, const void* dout, const void* q, const void* k,
                                     const void* v, const void* out, const void* stats, void* workspace,
                                     int64_t batch, int64_t heads, int64_t q_len, int64_t kv_len, int64_t head_dim,
                                     const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                     const int64_t* out_strides, const int64_t* dout_strides,
                                     const int64_t* dq_strides, const int64_t* dk_strides,
                                     const int64_t* dv_strides, float scale, int causal, void* stream) {
  using namespace tmb;
  if (batch < 0 || heads < 0 || q_len < 0 || kv_len < 0) return TMB_ERR_INVALID_ARGUMENT;
  if (head_dim != 64) return TMB_ERR_UNSUPPORTED;
  if (!(scale == scale)) return TMB_ERR_INVALID_ARGUMENT;
  if (!(scale > 0.0f) || scale > 3.0e38f) return TMB_ERR_UNSUPPORTED;
  if (batch == 0 || heads == 0 || (q_len == 0 && kv_len == 0)) return TMB_OK;
  if (q_len == 0 || kv_len == 0) return TMB_ERR_UNSUPPORTED;  // zero gradients: left to the caller
  const int64_t* all[] = {q_strides, k_strides, v_strides, out_strides, dout_strides, dq_strides, dk_strides, dv_strides};
  for (const int64_t* s : all)
    if (!s) return TMB_ERR_INVALID_ARGUMENT;
  if (!dq || !dk || !dv || !dout || !q || !k || !v || !out || !stats || !workspace) return TMB_ERR_INVALID_ARGUMENT;
  if ((reinterpret_cast<uintptr_t>(stats) & 7) || (reinterpret_cast<uintptr_t>(workspace) & 15))
    return TMB_ERR_INVALID_ARGUMENT;
  if (batch >= (int64_t{1} << 31) || heads >= (int64_t{1} << 31) || !f32_fits(batch * heads, q_len) ||
      !f32_fits(batch * heads, kv_len))
    return TMB_ERR_UNSUPPORTED;
  const void* ptrs[] = {q, k, v, out, dout, dq, dk, dv};
  const int64_t lens[] = {q_len, kv_len, kv_len, q_len, q_len, q_len, kv_len, kv_len};
  for (int i = 0; i < 8; ++i)
    if (!f32_layout(ptrs[i], all[i], lens[i])) return TMB_ERR_UNSUPPORTED;
  AttnF32BwdArgs a{static_cast<float*>(dq), static_cast<float*>(dk), static_cast<float*>(dv),
                   static_cast<const float*>(dout), static_cast<const float*>(q), static_cast<const float*>(k),
                   static_cast<const float*>(v), static_cast<const float*>(out), static_cast<const float*>(stats),
                   static_cast<af32x4_t*>(workspace), f32_strides(q_strides), f32_strides(k_strides),
                   f32_strides(v_strides), f32_strides(out_strides), f32_strides(dout_strides),
                   f32_strides(dq_strides), f32_strides(dk_strides), f32_strides(dv_strides), static_cast<int>(heads),
                   static_cast<int>(batch * heads), static_cast<int>(q_len), static_cast<int>(kv_len), scale,
                   causal ? 1 : 0};
  hipStream_t s = static_cast<hipStream_t>(stream);
  attention_f32_bwd_dq_kernel<<<dim3(static_cast<unsigned>(batch * heads * f32_blocks(q_len))), dim3(256), 0, s>>>(a);
  attention_f32_bwd_dkv_kernel<<<dim3(static_cast<unsigned>(batch * heads * f32_blocks(kv_len))), dim3(256), 0, s>>>(a);
  return check_launch();
}
