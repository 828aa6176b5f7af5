// Instantiations and launch of the kernel for small products (gemm_small.h).
#include "gemm_small.h"
#include "gemm_plan.h"

namespace tmb {

template <typename T, bool B_KMAJOR, int EPI>
static int small_launch(const GemmArgs& g, int64_t batch, int tile, hipStream_t stream) {
  switch (tile) {
    case 0: return launch_small<T, 16, 16, 8, B_KMAJOR, EPI>(g, batch, stream);
    case 1: return launch_small<T, 16, 32, 8, B_KMAJOR, EPI>(g, batch, stream);
    case 2: return launch_small<T, 32, 32, 8, B_KMAJOR, EPI>(g, batch, stream);
    case 3: return launch_small<T, 32, 32, 4, B_KMAJOR, EPI>(g, batch, stream);
    case 4: return launch_small<T, 32, 64, 8, B_KMAJOR, EPI>(g, batch, stream);
    default: return launch_small<T, 64, 64, 8, B_KMAJOR, EPI>(g, batch, stream);
  }
}

template <typename T, bool B_KMAJOR>
static int small_epi(const GemmArgs& g, int64_t batch, int tile, int epilogue, hipStream_t stream) {
  switch (epilogue) {
    case TMB_EPI_NONE: return small_launch<T, B_KMAJOR, TMB_EPI_NONE>(g, batch, tile, stream);
    case TMB_EPI_GELU_TANH: return small_launch<T, B_KMAJOR, TMB_EPI_GELU_TANH>(g, batch, tile, stream);
    case TMB_EPI_GELU_ERF: return small_launch<T, B_KMAJOR, TMB_EPI_GELU_ERF>(g, batch, tile, stream);
    default: return TMB_ERR_INVALID_ARGUMENT;
  }
}

int gemm_small(const GemmArgs& g, int64_t batch, int tile, int trans_b, bool bf16, int epilogue, hipStream_t stream) {
  if (bf16) return trans_b ? small_epi<bf16_t, true>(g, batch, tile, epilogue, stream)
                           : small_epi<bf16_t, false>(g, batch, tile, epilogue, stream);
  return trans_b ? small_epi<f16_t, true>(g, batch, tile, epilogue, stream)
                 : small_epi<f16_t, false>(g, batch, tile, epilogue, stream);
}

}  // namespace tmb
