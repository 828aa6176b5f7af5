// GEMM family (mm / addmm / bmm / linear) for gfx950.
//
// MFMA path (bf16 / fp16 storage, fp32 accumulation): each 256-thread workgroup (4 waves as
// 2x2) owns a BM x BN tile of C and walks K in steps of 64. Tiles of A and B are staged through
// double-buffered LDS in a K-major layout (one 128-byte line of 64 K-values per matrix row),
// with the 16-byte chunks of every line XOR-swizzled by the row number so that both the
// workgroup's stores and the waves' ds_read_b128 operand fetches are bank-conflict free.
// Every wave computes a (BM/2) x (BN/2) sub-tile with v_mfma_f32_32x32x16 instructions.
// B may be stored K-major ([N,K] rows: the `weight.t()` view of a Linear layer) or N-major
// ([K,N] rows); the N-major case is transposed in registers on its way into LDS.
// The epilogue adds the bias in fp32, applies the optional GELU, casts once and stores.
// Workgroups are numbered so that the 32 tiles resident on one XCD form a compact patch of
// C and share A/B panels through that XCD's L2.
//
// 16-bit operands that are not whole aligned 16-byte vectors: gemm_any.h.
//
// Fallback path: a 64x64 SIMT tile kernel that takes any dtype, strides and alignment.
//
// Arithmetic contract: fp32 accumulate, bias added in fp32 before the single down-cast
// (torch_mojo_backend/eager_kernels/matmul_ops.mojo:2651-2720).
#include "gemm_plan.h"

namespace tmb {

// Fills C with epilogue(bias) (or zeros) when k == 0.
template <typename T, int EPI>
__global__ void gemm_k0_kernel(T* c, const T* bias, int64_t m, int64_t n, int64_t ldc,
                               int64_t stride_c, bool twice) {
  T* cb = c + static_cast<int64_t>(blockIdx.y) * stride_c;
  const int64_t total = m * n;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = i / n, col = i - r * n;
    const float v = bias != nullptr ? to_f32(bias[col]) : 0.0f;
    cb[r * ldc + col] = finish<T, EPI>(v, twice);
  }
}

}  // namespace tmb

static int gemm_entry(void* c, const void* a, const void* b, const void* bias,
                      const void* residual, int64_t batch, int64_t m, int64_t n, int64_t k,
                      int64_t lda, int64_t ldb, int64_t ldc, int64_t ldr, int64_t stride_a,
                      int64_t stride_b, int64_t stride_c, int64_t stride_r, int trans_a,
                      int trans_b, int dtype, int epilogue_flags, void* stream,
                      void* workspace = nullptr, size_t workspace_bytes = 0,
                      int residual_dtype = -1, int out_dtype = -1) {
  using namespace tmb;
  if (batch < 0 || m < 0 || n < 0 || k < 0) return TMB_ERR_INVALID_ARGUMENT;
  if (epilogue_flags < 0 || (epilogue_flags & ~(0xff | TMB_EPI_ROUND_LIKE_UNFUSED)) != 0)
    return TMB_ERR_INVALID_ARGUMENT;
  const int epilogue = epilogue_flags & 0xff;
  const bool twice = (epilogue_flags & TMB_EPI_ROUND_LIKE_UNFUSED) != 0;
  if (epilogue < TMB_EPI_NONE || epilogue > TMB_EPI_GELU_ERF) return TMB_ERR_INVALID_ARGUMENT;
  if (dtype != TMB_F32 && dtype != TMB_F16 && dtype != TMB_BF16) return TMB_ERR_UNSUPPORTED;
  if (residual_dtype < 0) residual_dtype = dtype;
  if (out_dtype < 0) out_dtype = dtype;
  if ((residual_dtype != dtype && residual_dtype != TMB_F32) ||
      (out_dtype != dtype && out_dtype != TMB_F32))
    return TMB_ERR_UNSUPPORTED;
  const bool resid_f32 = residual != nullptr && residual_dtype == TMB_F32 && dtype != TMB_F32;
  const bool out_f32 = out_dtype == TMB_F32 && dtype != TMB_F32;
  if (batch == 0 || m == 0 || n == 0) return TMB_OK;
  if (c == nullptr) return TMB_ERR_INVALID_ARGUMENT;
  if (k > 0 && (a == nullptr || b == nullptr)) return TMB_ERR_INVALID_ARGUMENT;
  // Leading dimensions must cover the stored row of each operand.
  if (ldc < n) return TMB_ERR_INVALID_ARGUMENT;
  if (k > 0) {
    if (lda < (trans_a ? m : k)) return TMB_ERR_INVALID_ARGUMENT;
    if (ldb < (trans_b ? k : n)) return TMB_ERR_INVALID_ARGUMENT;
  }
  if (batch > 65535) return TMB_ERR_UNSUPPORTED;
  hipStream_t s = static_cast<hipStream_t>(stream);
  GemmArgs g{c, a, b, bias, m, n, k, lda, ldb, ldc, stride_a, stride_b, stride_c, 0, 0, 0, residual, ldr, stride_r};
  g.round_like_unfused = twice ? 1 : 0;
  g.resid_f32 = resid_f32 ? 1 : 0;
  g.out_f32 = out_f32 ? 1 : 0;
  if (out_f32 && residual == nullptr) return TMB_ERR_UNSUPPORTED;  // fp32 C exists for the residual form only
  if (residual != nullptr) {
    // only the MFMA kernels carry the second epilogue step; the caller adds separately otherwise
    if (k == 0 || ldr < n || (dtype != TMB_F32 && !mfma_eligible(g, batch, trans_a, trans_b) &&
                              !any_eligible(m, n, k, lda, ldb, trans_a, trans_b)))
      return TMB_ERR_UNSUPPORTED;
    // fp32 operands of the epilogue and an epilogue that stays in fp32 exist without GELU only
    if ((resid_f32 || out_f32 || !twice) && epilogue != TMB_EPI_NONE) return TMB_ERR_UNSUPPORTED;
    if ((resid_f32 || out_f32) && twice) return TMB_ERR_INVALID_ARGUMENT;
  }
  if (k == 0) {
    const unsigned blocks = static_cast<unsigned>((m * n + 255) / 256 > 4096 ? 4096 : (m * n + 255) / 256);
    dim3 grid(blocks, static_cast<unsigned>(batch));
#define TMB_K0(T)                                                                                   \
  switch (epilogue) {                                                                               \
    case TMB_EPI_NONE: gemm_k0_kernel<T, TMB_EPI_NONE><<<grid, 256, 0, s>>>((T*)c, (const T*)bias, m, n, ldc, stride_c, twice); break; \
    case TMB_EPI_GELU_TANH: gemm_k0_kernel<T, TMB_EPI_GELU_TANH><<<grid, 256, 0, s>>>((T*)c, (const T*)bias, m, n, ldc, stride_c, twice); break; \
    default: gemm_k0_kernel<T, TMB_EPI_GELU_ERF><<<grid, 256, 0, s>>>((T*)c, (const T*)bias, m, n, ldc, stride_c, twice); break; \
  }
    if (dtype == TMB_F32) { TMB_K0(float) } else if (dtype == TMB_F16) { TMB_K0(f16_t) } else { TMB_K0(bf16_t) }
#undef TMB_K0
    return check_launch();
  }
  switch (dtype) {
    case TMB_F32: return gemm_epi<float>(g, batch, trans_a, trans_b, epilogue, s, workspace, workspace_bytes);
    case TMB_F16: return gemm_epi<f16_t>(g, batch, trans_a, trans_b, epilogue, s, workspace, workspace_bytes);
    default: return gemm_epi<bf16_t>(g, batch, trans_a, trans_b, epilogue, s, workspace, workspace_bytes);
  }
}

extern "C" int tmb_gemm(void* c, const void* a, const void* b, const void* bias, int64_t batch,
                        int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, int64_t ldc,
                        int64_t stride_a, int64_t stride_b, int64_t stride_c, int trans_a,
                        int trans_b, int dtype, int epilogue, void* stream) {
  return gemm_entry(c, a, b, bias, nullptr, batch, m, n, k, lda, ldb, ldc, 0, stride_a, stride_b,
                    stride_c, 0, trans_a, trans_b, dtype, epilogue, stream);
}

extern "C" size_t tmb_gemm_workspace_bytes(int64_t batch, int64_t m, int64_t n, int64_t k,
                                           int dtype) {
  using namespace tmb;
  if (dtype != TMB_F32 && dtype != TMB_F16 && dtype != TMB_BF16) return 0;
  if (batch < 1 || m < 1 || n < 1 || k < 1 || m * n >= (int64_t{1} << 31)) return 0;
  int splits = 0;
  if (dtype == TMB_F32) {
    for (int layout = 0; layout < 4; ++layout) {
      const int here = f32_most_splits(batch, m, n, k, layout >> 1, layout & 1);
      splits = here > splits ? here : splits;
    }
  } else {
    splits = splitk_plan(batch, m, n, k).splits;
  }
  return static_cast<size_t>(splits) * static_cast<size_t>(m) * static_cast<size_t>(n) * 4;
}

extern "C" size_t tmb_gemm_layout_workspace_bytes(int64_t batch, int64_t m, int64_t n, int64_t k, int trans_a,
                                                  int trans_b, int dtype) {
  if (dtype == TMB_F32) {
    if (batch < 1 || m < 1 || n < 1 || k < 1 || m * n >= (int64_t{1} << 31)) return 0;
    return static_cast<size_t>(tmb::f32_most_splits(batch, m, n, k, trans_a, trans_b)) * m * n * 4;
  }
  // the kernel for small products needs none (operands it cannot take run unsplit then)
  if (!trans_a && (trans_b || n % 8 == 0) && k % 8 == 0 && tmb::small_applies(batch, m, n, k)) return 0;
  return tmb_gemm_workspace_bytes(batch, m, n, k, dtype);
}

extern "C" int64_t tmb_gemm_in_place_workspace_bytes(int64_t batch, int64_t m, int64_t n, int64_t k, int64_t lda,
                                                     int64_t ldb, int a_aligned, int b_aligned, int trans_a,
                                                     int trans_b, int plain, int dtype) {
  if ((dtype != TMB_F16 && dtype != TMB_BF16) || batch < 1 || batch > 65535) return -1;
  if (!tmb::any_eligible(m, n, k, lda, ldb, trans_a, trans_b)) return -1;
  const tmb::AnyPlan plan = tmb::any_plan(batch, m, n, k, true);
  double cost = plan.cost;
  if (plan.splits == 0 && k > 2048)  // (runs of K this long no longer stay in L2: 597 x 5159 x 7235 166 us, not 131)
    cost *= 1.0 + 0.1 * static_cast<double>(k - 2048) / 2048.0;
  tmb::GemmArgs g{};
  g.m = m, g.n = n, g.k = k;
  if (tmb::simt_instead_of_any(g, batch, plan)) cost = tmb::simt_cost(false, batch, m, n, k);
  if (cost > tmb::padded_cost(batch, m, n, k, lda, ldb, a_aligned != 0, b_aligned != 0, trans_a, trans_b,
                                   plain != 0))
    return -1;
  return static_cast<int64_t>(plan.splits) * m * n * 4;
}

extern "C" int tmb_gemm_f32_padding_pays(int64_t batch, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
                                         int a_aligned, int b_aligned, int trans_a, int trans_b) {
  using namespace tmb;
  if (batch < 1 || m < 1 || n < 1 || k < 1) return 0;
  GemmArgs g{};
  g.m = m, g.n = n, g.k = k, g.lda = lda, g.ldb = ldb;
  if (!f32_shared_eligible(g, trans_a, trans_b)) return 1;
  const F32Plan plan = f32_plan(batch, m, n, k, 16);
  double here = plan.cost;
  if (k >= kF32WideUnalignedK) here = std::fmin(here, f32_wide_plan(batch, m, n, k, plan).cost);
  if (k <= 48 && plan.splits == 0) here = std::fmin(here, simt_cost(true, batch, m, n, k));
  return f32_padded_cost(batch, m, n, k, lda, ldb, a_aligned != 0, b_aligned != 0, trans_a, trans_b) < here;
}

extern "C" int64_t tmb_gemm_route(int64_t batch, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
                                  int64_t stride_a, int64_t stride_b, int a_aligned, int b_aligned, int trans_a,
                                  int trans_b, int dtype, int epilogue_flags, int with_residual,
                                  size_t workspace_bytes) {
  using namespace tmb;
  if (batch < 1 || m < 1 || n < 1 || k < 1 || lda < (trans_a ? m : k) || ldb < (trans_b ? k : n))
    return TMB_ERR_INVALID_ARGUMENT;
  if ((dtype != TMB_F32 && dtype != TMB_F16 && dtype != TMB_BF16) || batch > 65535) return TMB_ERR_UNSUPPORTED;
  // addresses that are never read: only their alignment is looked at
  auto at = [](int aligned) { return reinterpret_cast<const void*>(static_cast<uintptr_t>(aligned ? 16 : 18)); };
  GemmArgs g{};
  g.a = at(a_aligned);
  g.b = at(b_aligned);
  g.m = m, g.n = n, g.k = k, g.lda = lda, g.ldb = ldb, g.ldc = n;
  g.stride_a = stride_a, g.stride_b = stride_b, g.stride_c = m * n;
  g.residual = with_residual ? at(1) : nullptr;
  g.ldr = n;
  g.round_like_unfused = (epilogue_flags & TMB_EPI_ROUND_LIKE_UNFUSED) != 0;
  const GemmRoute r = dtype == TMB_F32
                          ? route_f32(g, batch, trans_a, trans_b, workspace_bytes)
                          : route_16bit(g, batch, trans_a, trans_b, epilogue_flags & 0xff, workspace_bytes);
  if (r.kernel < 0) return r.kernel;
  return r.kernel | static_cast<int64_t>(r.tile) << 8 | static_cast<int64_t>(r.splits) << 16;
}

extern "C" int tmb_gemm_ws(void* c, const void* a, const void* b, const void* bias, int64_t batch,
                           int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, int64_t ldc,
                           int64_t stride_a, int64_t stride_b, int64_t stride_c, int trans_a,
                           int trans_b, int dtype, int epilogue, void* workspace,
                           size_t workspace_bytes, void* stream) {
  return gemm_entry(c, a, b, bias, nullptr, batch, m, n, k, lda, ldb, ldc, 0, stride_a, stride_b,
                    stride_c, 0, trans_a, trans_b, dtype, epilogue, stream, workspace,
                    workspace_bytes);
}

extern "C" int tmb_gemm_residual(void* c, const void* a, const void* b, const void* bias,
                                 const void* residual, int64_t batch, int64_t m, int64_t n,
                                 int64_t k, int64_t lda, int64_t ldb, int64_t ldc, int64_t ldr,
                                 int64_t stride_a, int64_t stride_b, int64_t stride_c,
                                 int64_t stride_r, int trans_a, int trans_b, int dtype,
                                 int residual_dtype, int out_dtype, int epilogue, void* stream) {
  return tmb_gemm_residual_ws(c, a, b, bias, residual, batch, m, n, k, lda, ldb, ldc, ldr, stride_a, stride_b,
                              stride_c, stride_r, trans_a, trans_b, dtype, residual_dtype, out_dtype, epilogue,
                              nullptr, 0, stream);
}

extern "C" int tmb_gemm_residual_ws(void* c, const void* a, const void* b, const void* bias, const void* residual,
                                    int64_t batch, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
                                    int64_t ldc, int64_t ldr, int64_t stride_a, int64_t stride_b, int64_t stride_c,
                                    int64_t stride_r, int trans_a, int trans_b, int dtype, int residual_dtype,
                                    int out_dtype, int epilogue, void* workspace, size_t workspace_bytes,
                                    void* stream) {
  if (residual == nullptr) return TMB_ERR_INVALID_ARGUMENT;
  if (residual_dtype < 0 || out_dtype < 0) return TMB_ERR_INVALID_ARGUMENT;
  return gemm_entry(c, a, b, bias, residual, batch, m, n, k, lda, ldb, ldc, ldr, stride_a,
                    stride_b, stride_c, stride_r, trans_a, trans_b, dtype, epilogue, stream, workspace,
                    workspace_bytes, residual_dtype, out_dtype);
}
