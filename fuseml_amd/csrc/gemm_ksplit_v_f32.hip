// The K-split kernel's tiles for fp32 GEMM operands.
#include "gemm_ksplit.h"

template hipError_t fuseml_gemm::launch_ksplit<float>(const fuseml_gemm_desc&, int, hipStream_t);
