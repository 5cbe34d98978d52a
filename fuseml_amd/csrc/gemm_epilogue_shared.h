// gemm_epilogue_shared.h — what the host side of the GEMM+epilogue kernels
// (gemm_epilogue.hip) and the kernel template (gemm_epilogue_kernel.h) both
// need: the host-derived operand flags, the tile variants, and the kernel's
// declaration.  The kernels are instantiated one variant per translation
// unit (gemm_epilogue_v_*.hip), so the library builds in parallel.
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "fuseml_hip.h"
#include "ksplit_rule.h"

namespace fuseml_gemm {

// Host-derived flags kept in the `reserved` field of operands and outputs.
constexpr int kFlagVec4 = 1;   // unit stride along N, rows 4-element aligned: 8/16-byte vectors
constexpr int kFlagStage = 2;  // 16-bit, unit stride along N, N >= 8: LDS-staged tile
constexpr int kFlagAligned = 8;  // a staged tile's rows are whole 16-byte chunks at 16-byte addresses
constexpr int kFlagAux = 4;    // row ([N]) or column ([M]) vector staged as fp32 in LDS slot (bits 8-9)
constexpr int kAuxSlots = 4;   // vector operands staged per launch

struct TileConfig {
  int bm, bn, bk, stages, wm, wn;
  int sched;  // K-loop schedule (kernel template parameter SCHED)
  constexpr int lds_bytes() const {
    return stages * (bm + bn) * bk * 2 + kAuxSlots * (bm > bn ? bm : bn) * 4;
  }
};

constexpr TileConfig kLarge = {256, 256, 32, 4, 2, 4, 1};  // 8 waves ping-pong, 132 KB LDS, 1 WG/CU
constexpr TileConfig kDeep = {256, 256, 64, 2, 2, 2, 3};   // 4 waves (1/SIMD), BK=64 x 2 stages, 132 KB LDS
constexpr TileConfig kSmall = {128, 128, 32, 4, 2, 2, 0};  // 4 waves lock-step, 66 KB LDS, 2 WG/CU
constexpr TileConfig kDeep3 = {256, 256, 64, 2, 2, 2, 6};  // as kDeep, whole-stage fragments; K % 64 == 0
constexpr TileConfig kNarrow64 = {64, 128, 64, 3, 2, 2, 0};  // 4 waves lock-step (wave tile 32x64), 74 KB LDS, 2 WG/CU
constexpr TileConfig kNarrow32 = {32, 128, 64, 3, 1, 4, 0};  // 4 waves lock-step (wave tile 32x32), 62 KB LDS, 2 WG/CU
constexpr TileConfig kLarge128 = {256, 128, 32, 4, 4, 2, 1};  // 8 waves ping-pong (wave tile 64x64), 100 KB LDS, 1 WG/CU
constexpr TileConfig kSmall64 = {128, 128, 64, 4, 2, 2, 0};  // kSmall at BK = 64: 130 KB LDS, 1 WG/CU

// Whether a variant has a kernel of its own for aligned rows (parameter ANY): the
// tiles below 256x256, whose prologue and epilogue are the larger share.  Without the
// code for ragged rows they take (M x N x K, bf16, us, one kernel -> two)
// 2048x1024x4096 bias+residual 30.35 -> 29.93, 2048x1024x1024 bias+GELU 12.39 ->
// 12.25, 2048x2048x1024 bias+residual 17.98 -> 17.87, 2048x1024x1024 ReLU + three row
// reductions 13.93 -> 13.73.  The 256x256 ping-pong kernel has one for fp16 alone:
// 689x11288x576 bias+GELU, scale, add 27.74 -> 26.98 (26.93 before ragged rows were
// staged), its other chains 0.99-1.01; in bf16 that chain had lost nothing, and
// bias+GELU would lose 1% (28.59 -> 28.87 at 4096x4096x576).
template <typename T>
constexpr bool splits_rows(const TileConfig& c) {
  return c.bm * c.bn < 256 * 256 || (c.sched == kLarge.sched && std::is_same<T, _Float16>::value);
}

// Launch tile `index` of kKsplit; T: __bf16, _Float16 or float GEMM operands
// (gemm_ksplit_v_*.hip).
template <typename T>
hipError_t launch_ksplit(const fuseml_gemm_desc& d, int index, hipStream_t stream);

// Epilogue chains compiled into kernels of their own (template parameter CH
// of the kernel).  kChainGeneric runs the descriptor's op list through the
// runtime op loop; every other value is one fixed op sequence, matched on the
// host (operand kinds included) and compiled as straight-line code with no
// per-op dispatch.  "row" is a [N] vector operand in an LDS slot, "tile" the
// LDS-staged 2-D operand of the GEMM operands' type; ADD keeps its alpha from the descriptor.
enum FixedChain : int {
  kChainGeneric = 0,
  kChainNone = 1,          // (no ops)
  kChainBias = 2,          // add(row)
  kChainBiasGeluErf = 3,   // add(row), gelu(approximate='none')
  kChainBiasGeluTanh = 4,  // add(row), gelu(approximate='tanh')
  kChainBiasRelu = 5,      // add(row), relu
  kChainBiasTile = 6,      // add(row), add(tile)           (bias + residual)
  kChainActHeavy = 7,      // add(row), relu, mul(tile), sigmoid, add(row)
  kChainRelu = 8,          // relu                          (also with reductions)
  kChainBiasGeluScale = 9,  // add(row), gelu(approximate='none'), scale, add_scalar
  kNumChains = 10,
};

// The kernel (defined in gemm_epilogue_kernel.h).  SCHED selects the K-loop
// schedule, T the GEMM operand type (__bf16 or _Float16), RED whether the
// launch has reductions, CH the epilogue chain (FixedChain).
template <int BM, int BN, int BK, int S, int WM, int WN, int SCHED, typename T, bool RED, int CH, bool ANY>
__global__ void gemm_epilogue_kernel(const fuseml_gemm_desc d_arg);

}  // namespace fuseml_gemm
