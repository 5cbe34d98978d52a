// The large tile variant's kernels (kLarge: bf16/f16 operands, with and without
// reductions).  One variant per translation unit so that the library's kernels
// compile in parallel.
#include "gemm_epilogue_kernel.h"

FUSEML_GEMM_INSTANTIATE(fuseml_gemm::kLarge)
FUSEML_GEMM_INSTANTIATE_ANY(fuseml_gemm::kLarge, _Float16, false, fuseml_gemm::kChainGeneric, false)
FUSEML_GEMM_INSTANTIATE_ANY(fuseml_gemm::kLarge, _Float16, true, fuseml_gemm::kChainGeneric, false)
