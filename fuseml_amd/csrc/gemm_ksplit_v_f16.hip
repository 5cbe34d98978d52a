// The K-split kernel's tiles for fp16 GEMM operands.
#include "gemm_ksplit.h"

template hipError_t fuseml_gemm::launch_ksplit<_Float16>(const fuseml_gemm_desc&, int, hipStream_t);
