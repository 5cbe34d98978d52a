// The 128x128 lock-step variants' kernels (kSmall, and kSmall64 at BK = 64:
// bf16/f16 operands, with and without reductions).  One variant per translation unit so that the library's kernels
// compile in parallel.
#include "gemm_epilogue_kernel.h"

FUSEML_GEMM_INSTANTIATE_ROWS(fuseml_gemm::kSmall, false)
FUSEML_GEMM_INSTANTIATE_ROWS(fuseml_gemm::kSmall, true)
FUSEML_GEMM_INSTANTIATE_ROWS(fuseml_gemm::kSmall64, false)
FUSEML_GEMM_INSTANTIATE_ROWS(fuseml_gemm::kSmall64, true)
