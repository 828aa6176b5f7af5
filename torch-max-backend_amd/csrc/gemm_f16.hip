#include "gemm_typed.h"

template int tmb::gemm_epi<tmb::f16_t>(const tmb::GemmArgs&, int64_t, int, int, int, hipStream_t, void*, size_t);
