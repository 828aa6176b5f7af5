// Instantiations and launch of the kernel for operands of any layout and alignment (gemm_any.h).
#include "gemm_any.h"
#include "gemm_plan.h"

namespace tmb {

template <typename T, bool A_MMAJOR, bool B_KMAJOR>
static int any_launch(const GemmArgs& g, int64_t batch, int tile, int epilogue, hipStream_t stream) {
  switch (tile) {
    case 0: return launch_any_tile<T, 16, 16, 8, A_MMAJOR, B_KMAJOR>(g, batch, epilogue, stream);
    case 1: return launch_any_tile<T, 16, 32, 8, A_MMAJOR, B_KMAJOR>(g, batch, epilogue, stream);
    case 2: return launch_any_tile<T, 32, 32, 8, A_MMAJOR, B_KMAJOR>(g, batch, epilogue, stream);
    case 3: return launch_any_tile<T, 32, 32, 4, A_MMAJOR, B_KMAJOR>(g, batch, epilogue, stream);
    default: return launch_any_tile<T, 64, 64, 4, A_MMAJOR, B_KMAJOR>(g, batch, epilogue, stream);
  }
}

template <typename T>
static int any_layout(const GemmArgs& g, int64_t batch, int tile, int trans_a, int trans_b, int epilogue,
                      hipStream_t stream) {
  if (trans_a) return trans_b ? any_launch<T, true, true>(g, batch, tile, epilogue, stream)
                              : any_launch<T, true, false>(g, batch, tile, epilogue, stream);
  return trans_b ? any_launch<T, false, true>(g, batch, tile, epilogue, stream)
                 : any_launch<T, false, false>(g, batch, tile, epilogue, stream);
}

int gemm_any(const GemmArgs& g, int64_t batch, int tile, int trans_a, int trans_b, bool bf16, int epilogue,
             hipStream_t stream) {
  return bf16 ? any_layout<bf16_t>(g, batch, tile, trans_a, trans_b, epilogue, stream)
              : any_layout<f16_t>(g, batch, tile, trans_a, trans_b, epilogue, stream);
}

}  // namespace tmb
