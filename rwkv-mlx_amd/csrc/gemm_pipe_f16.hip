// The pipelined GEMM tiles of gemm_pipe.h for fp16.
#include "gemm_pipe.h"

namespace rwkvmoe {
template hipError_t pipe_run<f16>(const GemmParams<f16>& p, int cfg, int epi, int mode, hipStream_t s);
}  // namespace rwkvmoe
