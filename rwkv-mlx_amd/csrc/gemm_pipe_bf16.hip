// The pipelined GEMM tiles of gemm_pipe.h for bf16.
#include "gemm_pipe.h"

namespace rwkvmoe {
template hipError_t pipe_run<bf16>(const GemmParams<bf16>& p, int cfg, int epi, int mode, hipStream_t s);
}  // namespace rwkvmoe
