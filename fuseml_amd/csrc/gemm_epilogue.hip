// gemm_epilogue.hip — host side of the gfx950 fused GEMM+epilogue kernel
// family: validation, variant choice, launch, and the C ABI.  The kernel
// template is gemm_epilogue_kernel.h, instantiated one tile variant per
// translation unit (gemm_epilogue_v_*.hip).
//
// What one launch computes (one fusion group):
//   acc = A[M,K] @ B[K,N] in fp32 on bf16/f16 MFMA (v_mfma_f32_32x32x16_*),
//   v   = epilogue op chain applied to acc in registers,
//   out = cast(v) stored once, plus optional escape stores and fused row/column
//         sum/amax/mean reductions.
// This replaces the generated Triton kernel of the reference
// (fuseml/codegen/kernel_generator.py: K-loop 1454-1542, bias 881-901,
// epilogue emitters 1599-1903, store 1544-1593, reductions 1909-2018) and the
// cuBLASLt epilogue extension (fuseml/codegen/cublas_epilogue.py:355-557).
//
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>

#include "fuseml_hip.h"
#include "gemm_epilogue_shared.h"

using namespace fuseml_gemm;

namespace {

thread_local char g_last_error[512];

void set_error(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
}

// Initialise reduction buffers: sum/mean to 0, amax to -inf.
__global__ void reduce_fill_kernel(float* sum, float* amax, float* mean, int len) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= len) return;
  if (sum) sum[i] = 0.0f;
  if (amax) amax[i] = -INFINITY;
  if (mean) mean[i] = 0.0f;
}

// ---------------------------------------------------------------------------
// Host side: validation, variant table, launch
// ---------------------------------------------------------------------------

constexpr int64_t kMaxBytes = (int64_t)1 << 31;
constexpr int64_t kTileSpan = 256;  // largest tile edge of any variant

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Pinned variant: 0 automatic, else 1 + index into {large, deep, deep3, small,
// deep3-generic, narrow64, narrow32, large128, small64} (deep3-generic: deep3
// with the generic op loop even where a fixed chain matches).  Initialised once per process from FUSEML_HIP_TILE, changed
// only through fuseml_gemm_epilogue_force_variant.
constexpr const char* kVariantNames[] = {"large", "deep", "deep3", "small", "deep3-generic", "narrow64", "narrow32",
                                         "large128", "small64"};
constexpr int kNumVariantNames = 9;
constexpr int kForcedDeep3Generic = 5;
std::atomic<int> g_forced_variant{-1};  // -1: environment not read yet

int variant_code(const char* name) {
  if (name == nullptr || name[0] == '\0' || !strcmp(name, "auto")) return 0;
  for (int i = 0; i < kNumVariantNames; ++i)
    if (!strcmp(name, kVariantNames[i])) return i + 1;
  return -1;
}

int forced_variant() {
  int v = g_forced_variant.load(std::memory_order_relaxed);
  if (v < 0) {
    const int e = variant_code(getenv("FUSEML_HIP_TILE"));
    int expected = -1;
    g_forced_variant.compare_exchange_strong(expected, e < 0 ? 0 : e, std::memory_order_relaxed);
    v = g_forced_variant.load(std::memory_order_relaxed);
  }
  return v;
}

int match_fixed_chain(const fuseml_gemm_desc& d);

// Below one round of 256x256 tiles: the 128x128, 64x128 or 32x128 lock-step
// tile (4 waves, two workgroups per CU) or the 256x128 ping-pong tile (8
// waves, one per CU), whichever gives its busiest CU the least K-loop work:
// ceil(tiles / CUs) x (BM + BN) operand rows per unit of K, weighted by how
// fast a CU moves them: 5 for the lock-step tiles with two workgroups on some
// CU, 8 with at most one (one wave per SIMD hides less of the LDS DMA's
// latency and none of the epilogue; 7 for K > 2048), 6 for the ping-pong
// tile; the first of the list on a tie.  Also for M <= 128 at any N, where a
// 256-row tile is at least half padding.  Each CU moves its tiles' A and W
// rows through the LDS DMA at a roughly fixed rate (37-48 GB/s measured,
// whatever the tile), so below two 128x128 tiles per CU a narrower tile
// spreads the same K over more CUs or more waves.  Measured
// (bias + GELU or bias + residual, M x N x K, us): 128x1024x256 9.6 -> 5.9 and
// 1024x1024x1024 16.8 -> 9.9 on 32x128 tiles; 2048x1024x4096 44.7 -> 31.7,
// 2048x2048x1024 20.0 -> 17.7 and 8192x512x2048 31.5 -> 28.8 on 64x128 tiles;
// 2048x4096x1024 33.0 -> 29.0 and 4096x2048x1024 31.8 -> 29.5 on 256x128
// ping-pong tiles (64x128 tiles there: 35.0 and 33.2); 128x32768x4096 stays on
// 128x128 tiles (58.2; 64x128 63.8); 64x65536x4096 138.7 -> 125,
// 16x65536x1024 36.0 -> 23.0, 128x65536x1024 38.7 -> 31.9 and 128x65536x4096
// 151.9 -> 136.1 on lock-step tiles instead of 256x256 ones.
TileConfig choose_partial_round(const fuseml_gemm_desc& d, int cus, int64_t* least = nullptr) {
  struct Cand {
    const TileConfig* c;
    int w_one, w_two;  // weight with at most one / with two workgroups on a CU
  };
  // One lock-step workgroup per CU costs less beside a long K loop, where the
  // pipeline runs in its steady state longer than the epilogue takes.
  const int one = d.K > 2048 ? 7 : 8;
  const Cand cand[4] = {{&kSmall, one, 5}, {&kNarrow64, one, 5}, {&kNarrow32, one, 5}, {&kLarge128, 6, 6}};
  const TileConfig* best = cand[0].c;
  int64_t best_work = 0;
  for (const Cand& k : cand) {
    const int64_t tiles = cdiv(d.M, k.c->bm) * cdiv(d.N, k.c->bn);
    const int64_t work = cdiv(tiles, cus) * (k.c->bm + k.c->bn) * (tiles <= cus ? k.w_one : k.w_two);
    if (k.c == cand[0].c || work < best_work) {
      best = k.c;
      best_work = work;
    }
  }
  if (least != nullptr) *least = best_work;
  return *best;
}

// Decode-sized M against a wide weight: a 128-column tile per CU or more.
bool weight_streaming(const fuseml_gemm_desc& d, int cus) { return d.M <= 128 && cdiv(d.N, 128) >= cus; }

// `cus`: the device's CU count (the 256-wide variants run one workgroup per CU).
// `d` has its flags derived (derive_flags).
TileConfig choose_config(const fuseml_gemm_desc& d, int cus) {
  // A pinned variant (tuning sweeps and the per-variant parity tests; deep3
  // falls back to deep when K % 64 != 0).
  switch (forced_variant()) {
    case 1: return kLarge;
    case 2: return kDeep;
    case 3: return d.K % 64 == 0 ? kDeep3 : kDeep;
    case 4: return kSmall;
    case kForcedDeep3Generic: return d.K % 64 == 0 ? kDeep3 : kDeep;
    case 6: return kNarrow64;
    case 7: return kNarrow32;
    case 8: return kLarge128;
    case 9: return kSmall64;
    default: break;
  }
  // A 256x256 tile keeps the LDS traffic per MFMA low enough for the MFMA pipe
  // to stay busy; below one full wave of 256-tile work the 128x128 variant
  // fills more CUs.  Of the 256x256 schedules, the one-wave-per-SIMD ones have
  // the faster K loop but the slower epilogue (no second wave on a SIMD to
  // overlap its latencies).  The whole-stage one's fixed-chain kernels win from
  // K = 1024, on full rounds and on a partial one (136 to 224 tiles) alike: bf16
  // ReLU, residual and act-heavy chains 0.94-1.01 of the ping-pong kernel's time
  // at K = 1024 and 0.91-0.96 at K = 4096, fp16 ones 0.92-1.00 and 0.89-0.95
  // (8192x4096x4096 bias+residual, fp16, 260 -> 231 us).  The GELU(erf) chains,
  // those with the most VALU work, only from K = 2048 (0.94-1.02 there, 0.92-0.97
  // at K = 4096; 1.00-1.06 at K = 1024), or with 7/8 of a round from K = 1536
  // (0.95-0.99) and fp16 from K = 1024 (0.98-1.00).  Its generic op loop loses
  // 3-17% below K = 2048 and below 224 tiles, and wins from K = 2048 with at
  // least 7/8 of a round (0.94-1.00 at 224 tiles) or from K = 8192.  With K % 64
  // != 0 the two-stage one takes over from K = 8192.
  // Below one round of 256x256 tiles (2 x large_tiles <= cus) the smaller
  // tiles (choose_partial_round): at 128 large tiles on 256 CUs the 128x128
  // one was 7-17% faster than 256x256 (bias+GELU at K = 512-1024), from 144
  // on the 256x256 ones are.
  // Decode-sized M against a wide weight (a 128-column tile per CU or more):
  // the GEMM streams the weight from HBM, so one row of tiles (the smallest
  // BM >= M: the weight read once) in K stages of 64 (128 contiguous bytes of
  // each weight row per stage where 32 fetch 64).  128x65536x8192 251.9 ->
  // 215.8 us and 128x32768x4096 59.6 -> 53.6 on the 128x128 tile at BK = 64
  // instead of 32 (eager 219.9 and 57.3); 64 and 16 rows: 113.0 and 41.8 on
  // 64x128 and 32x128 tiles (eager 134.2, 44.4).
  if (weight_streaming(d, cus)) return d.M <= 32 ? kNarrow32 : d.M <= 64 ? kNarrow64 : kSmall64;
  const int64_t large_tiles = cdiv(d.M, 256) * cdiv(d.N, 256);
  if (2 * large_tiles <= cus || d.M <= 128) return choose_partial_round(d, cus);
  if (d.K % 64 == 0 && (d.K >= 8192 || (d.K >= 2048 && 8 * large_tiles >= 7 * cus))) return kDeep3;
  if (d.K % 64 == 0 && d.K >= 1024) {
    const int ch = match_fixed_chain(d);
    const bool gelu = ch == kChainBiasGeluErf || ch == kChainBiasGeluScale;
    const int64_t gelu_k = 8 * large_tiles < 7 * cus ? 2048 : d.ab_dtype == FUSEML_F16 ? 1024 : 1536;
    if (ch != kChainGeneric && (!gelu || d.K >= gelu_k)) return kDeep3;
  }
  return d.K >= 8192 ? kDeep : kLarge;
}

// The K-split tile (index into kKsplit) a launch of `d` runs on, or -1 for the
// tiled family.  Both sides are priced in microseconds by what was measured on
// 1400 shapes of 1 to 2048 rows, 128 to 16384 columns and K = 64 to 16384, most of
// them ragged (bf16: bias + residual, bias + GELU, ReLU + three row or column
// reductions), where the tiled family would run one of its tiles below a round:
//   K-split  3.5 + r (0.6 to 1.2 + 0.36 (mb + nb) K / 1024), r the rounds of a tile
//            per CU: launch, first loads, partials and epilogue, then operand bytes.
//            Whole rounds, since the CU with the most tiles ends last: 257 tiles
//            take nearly as long as 512.  The 96 KB rings of the 32x64 and 64x32
//            tiles leave one workgroup per CU, so a further round overlaps nothing:
//            1 + r (5.1 + ..).
//   tiled    -3 + work (5.05 + 3.6 K / 1024) / 160, work as choose_partial_round
//            weighs it.
//   both     fused reductions (reduction_us).
// The K-split price is within 17% of the measurement on average, so that kernel runs
// where it is priced at 0.9 of the other or less: 1097 of the 1400 shapes, 1.9x
// faster there (geometric mean), 2 of them slower than the tiled family by more than
// 2% (353x192x64 with row reductions 7.9 -> 9.4, 1371x720x5728 36.7 -> 39.9); e.g.
// 8x4096x16384 107.7 -> 27.0, 64x4096x4096 31.4 -> 14.3, 128x256x1024 10.3 -> 5.1.  With tiles /
// CUs for r, 0.32 and 0.85 it took 1150, 34 of them slower: 182x2944x1024 10.8 ->
// 14.6, 1808x416x4728 30.8 -> 39.5, 1069x992x7600 51.9 -> 76.9.
// Not at 1024x1024x1024 (11.0 tiled, 13.0 here: operands shared by more waves
// win) nor where the weight streams through a full row of tiles
// (16x65536x1024 28.5 against 30.7).
int choose_ksplit(const fuseml_gemm_desc& d, int cus) {
  if (forced_variant() != 0 || d.K <= 0 || weight_streaming(d, cus)) return -1;
  if (d.M > 128 && 2 * cdiv(d.M, 256) * cdiv(d.N, 256) > cus) return -1;
  double cost = 0.0;
  const int best = cheapest_ksplit(d.M, d.N, d.K, cus, kKsplitPerK, &cost);
  int64_t work = 0;
  choose_partial_round(d, cus, &work);
  double tiled = -3.0 + (double)work / (5.0 * 160.0) * (5.05 + 3.6 * (double)d.K / 1024.0);
  if (d.reduce_mask != 0) {
    cost += reduction_us(d.reduce_axis == 1, d.M, d.N, kKsplit[best].bn());
    tiled += reduction_us(d.reduce_axis == 1, d.M, d.N, 128);
  }
  return cost < kKsplitMargin * tiled ? best : -1;
}

int choose_ksplit_f32(const fuseml_gemm_desc& d, int cus) { return ksplit_f32(d.M, d.N, d.K, cus); }

bool check_output(const fuseml_output& o, const fuseml_gemm_desc& d, const char* what) {
  if (o.ptr == nullptr) return true;
  if (o.dtype < FUSEML_BF16 || o.dtype > FUSEML_F32) {
    set_error("%s: unknown dtype %d", what, o.dtype);
    return false;
  }
  if (o.ld < d.N) {
    set_error("%s: row stride %lld < N %lld", what, (long long)o.ld, (long long)d.N);
    return false;
  }
  return true;
}

// `f32`: fp32 GEMM operands (fuseml_gemm_epilogue_f32) instead of 16-bit ones.
int validate(const fuseml_gemm_desc* dp, bool f32 = false) {
  if (dp == nullptr) {
    set_error("null descriptor");
    return FUSEML_EINVAL;
  }
  const fuseml_gemm_desc& d = *dp;
  if (d.M <= 0 || d.N <= 0 || d.K < 0) {
    set_error("bad problem size M=%lld N=%lld K=%lld", (long long)d.M, (long long)d.N,
              (long long)d.K);
    return FUSEML_EINVAL;
  }
  if (d.M >= ((int64_t)1 << 30) || d.N >= ((int64_t)1 << 30) || d.K >= ((int64_t)1 << 30)) {
    set_error("problem dimension exceeds 2^30");
    return FUSEML_EUNSUPPORTED;
  }
  if (f32 && d.ab_dtype != FUSEML_F32) {
    set_error("GEMM operand dtype %d: fp32 only", d.ab_dtype);
    return FUSEML_EUNSUPPORTED;
  }
  if (!f32 && d.ab_dtype != FUSEML_BF16 && d.ab_dtype != FUSEML_F16) {
    set_error("GEMM operand dtype %d has no MFMA variant (bf16/f16 only)", d.ab_dtype);
    return FUSEML_EUNSUPPORTED;
  }
  if (d.K > 0 && (d.a == nullptr || d.b == nullptr)) {
    set_error("null GEMM operand");
    return FUSEML_EINVAL;
  }
  const int eb = f32 ? 4 : 2, unit = 16 / eb;  // a 16-byte piece of a row
  if (d.K > 0 && (d.K % unit != 0 || d.lda % unit != 0 || d.ldb % unit != 0 || ((uintptr_t)d.a & 15) ||
      ((uintptr_t)d.b & 15))) {
    set_error("GEMM operands need K, lda, ldb multiples of %d and 16-byte aligned bases "
              "(K=%lld lda=%lld ldb=%lld)",
              unit, (long long)d.K, (long long)d.lda, (long long)d.ldb);
    return FUSEML_EUNSUPPORTED;
  }
  if (d.K > 0 && (d.lda < d.K || d.ldb < d.K)) {
    set_error("row stride smaller than K");
    return FUSEML_EINVAL;
  }
  // Buffer resources are based at each tile's origin: the rows one tile reads
  // must span less than 2 GiB (the whole operand may be larger).
  const int64_t tm = d.M < kTileSpan ? d.M : kTileSpan, tn = d.N < kTileSpan ? d.N : kTileSpan;
  if (d.K > 0 && (((tm - 1) * d.lda + d.K) * eb >= kMaxBytes || ((tn - 1) * d.ldb + d.K) * eb >= kMaxBytes)) {
    set_error("GEMM operand rows of one tile span 2 GiB or more (lda=%lld ldb=%lld)", (long long)d.lda,
              (long long)d.ldb);
    return FUSEML_EUNSUPPORTED;
  }
  if (d.n_ops < 0 || d.n_ops > FUSEML_MAX_OPS || d.n_operands < 0 ||
      d.n_operands > FUSEML_MAX_OPERANDS || d.n_extra < 0 || d.n_extra > FUSEML_MAX_EXTRA_OUT) {
    set_error("op/operand/extra counts out of range");
    return FUSEML_EINVAL;
  }
  for (int i = 0; i < d.n_operands; ++i) {
    const fuseml_operand& op = d.operands[i];
    if (op.ptr == nullptr || op.dtype < FUSEML_BF16 || op.dtype > FUSEML_F32 || op.stride_m < 0 ||
        op.stride_n < 0 || op.extent <= 0) {
      set_error("operand %d malformed", i);
      return FUSEML_EINVAL;
    }
    const int64_t need = (d.M - 1) * op.stride_m + (d.N - 1) * op.stride_n + 1;
    if (op.extent < need) {
      set_error("operand %d extent %lld < reachable %lld", i, (long long)op.extent,
                (long long)need);
      return FUSEML_EINVAL;
    }
    if (((tm - 1) * op.stride_m + (tn - 1) * op.stride_n + 1) * (op.dtype == FUSEML_F32 ? 4 : 2) >= kMaxBytes) {
      set_error("operand %d: one tile's elements span 2 GiB or more", i);
      return FUSEML_EUNSUPPORTED;
    }
  }
  for (int i = 0; i < d.n_ops; ++i) {
    const fuseml_epi_op& o = d.ops[i];
    if (o.kind < FUSEML_OP_ADD || o.kind > FUSEML_OP_MUL_SELF) {
      set_error("op %d: unknown kind %d", i, o.kind);
      return FUSEML_EINVAL;
    }
    if ((o.kind == FUSEML_OP_ADD || o.kind == FUSEML_OP_MUL) &&
        (o.operand < 0 || o.operand >= d.n_operands)) {
      set_error("op %d: operand index %d out of range", i, o.operand);
      return FUSEML_EINVAL;
    }
    if (o.kind == FUSEML_OP_STORE &&
        (o.operand < 0 || o.operand >= d.n_extra || d.extra[o.operand].ptr == nullptr)) {
      set_error("op %d: extra output %d missing", i, o.operand);
      return FUSEML_EINVAL;
    }
  }
  if (!check_output(d.out, d, "out")) return FUSEML_EINVAL;
  for (int i = 0; i < d.n_extra; ++i)
    if (!check_output(d.extra[i], d, "extra")) return FUSEML_EINVAL;
  if (d.reduce_mask & ~7u) {
    set_error("unknown reduction bits 0x%x", d.reduce_mask);
    return FUSEML_EINVAL;
  }
  if (d.reduce_mask) {
    if (d.reduce_axis != 0 && d.reduce_axis != 1) {
      set_error("reduce_axis must be 0 or 1");
      return FUSEML_EINVAL;
    }
    for (int b = 0; b < 3; ++b)
      if ((d.reduce_mask & (1u << b)) && d.reduce_out[b] == nullptr) {
        set_error("reduction output %d missing", b);
        return FUSEML_EINVAL;
      }
  }
  if (d.out.ptr == nullptr && d.reduce_mask == 0 && d.n_extra == 0) {
    set_error("descriptor produces no output");
    return FUSEML_EINVAL;
  }
  return FUSEML_OK;
}

// A chain that has no main output and ends in an escape store writes that
// store as the main output: through the LDS staging tile as whole rows, not
// from the accumulator layout (32 rows per store instruction).  The values and
// the reductions after the chain are unchanged.
void fold_final_store(fuseml_gemm_desc& d) {
  if (d.out.ptr != nullptr || d.n_ops == 0) return;
  const fuseml_epi_op& last = d.ops[d.n_ops - 1];
  if (last.kind != FUSEML_OP_STORE) return;
  d.out = d.extra[last.operand];
  d.n_ops -= 1;
}

// Fill in the host-derived access-path flags (kept in the `reserved` fields).
void derive_flags(fuseml_gemm_desc& d) {
  for (int i = 0; i < d.n_operands; ++i) {
    fuseml_operand& op = d.operands[i];
    const int eb = op.dtype == FUSEML_F32 ? 4 : 2;
    const bool vec = op.stride_n == 1 && (op.stride_m % 4 == 0) && (d.N % 4 == 0) &&
                     ((uintptr_t)op.ptr % (4 * eb) == 0);
    const bool stage = eb == 2 && op.stride_n == 1 && op.stride_m != 0 && d.N >= 8;
    const bool aligned = op.stride_m % 8 == 0 && d.N % 8 == 0 && (uintptr_t)op.ptr % 16 == 0;
    op.reserved = (vec ? kFlagVec4 : 0) | (stage ? kFlagStage : 0) | (aligned ? kFlagAligned : 0);
  }
  // Vector operands of ADD/MUL ops get LDS slots, in first-use order.
  int slots = 0;
  for (int o = 0; o < d.n_ops && slots < kAuxSlots; ++o) {
    const int k = d.ops[o].kind;
    if (k != FUSEML_OP_ADD && k != FUSEML_OP_MUL) continue;
    fuseml_operand& op = d.operands[d.ops[o].operand];
    if ((op.reserved & kFlagAux) || (op.stride_m != 0 && op.stride_n != 0)) continue;
    op.reserved = (op.reserved & ~kFlagStage) | kFlagAux | (slots << 8);
    ++slots;
  }
  auto out_flags = [&](fuseml_output& o) {
    const int eb = o.dtype == FUSEML_F32 ? 4 : 2;
    const bool vec = o.ptr != nullptr && o.ld % 4 == 0 && d.N % 4 == 0 && (uintptr_t)o.ptr % (4 * eb) == 0;
    const bool stage = o.ptr != nullptr && eb == 2 && d.N >= 8;
    const bool aligned = o.ld % 8 == 0 && d.N % 8 == 0 && (uintptr_t)o.ptr % 16 == 0;
    o.reserved = (vec ? kFlagVec4 : 0) | (stage ? kFlagStage : 0) | (aligned ? kFlagAligned : 0);
  };
  out_flags(d.out);
  for (int i = 0; i < d.n_extra; ++i) out_flags(d.extra[i]);
}

// The fixed chain (FixedChain) that expresses the descriptor's epilogue, or
// kChainGeneric.  Called after derive_flags: a "row" operand is a [N] vector
// holding an LDS slot, a "tile" operand the LDS-staged 2-D operand of the GEMM
// operands' type.  Fixed chains are built for bf16 GEMM operands and for fp16
// ones with an fp16 output, no escape stores, and no reductions except after a
// lone relu (the ReLU + row/column reductions group).
int match_fixed_chain(const fuseml_gemm_desc& d) {
  if (d.n_extra != 0 || (d.ab_dtype == FUSEML_F16 && d.out.ptr != nullptr && d.out.dtype != FUSEML_F16))
    return kChainGeneric;
  auto is = [&](int o, int kind) { return o < d.n_ops && d.ops[o].kind == kind; };
  auto row = [&](int o) {
    if (!is(o, FUSEML_OP_ADD)) return false;
    const fuseml_operand& op = d.operands[d.ops[o].operand];
    return (op.reserved & kFlagAux) != 0 && op.stride_m == 0;
  };
  auto tile = [&](int o, int kind) {
    if (!is(o, kind)) return false;
    const fuseml_operand& op = d.operands[d.ops[o].operand];
    return (op.reserved & kFlagStage) != 0 && (op.reserved & kFlagAligned) != 0 && op.dtype == d.ab_dtype;
  };
  int ch = kChainGeneric;
  switch (d.n_ops) {
    case 0: ch = kChainNone; break;
    case 1:
      if (row(0)) ch = kChainBias;
      else if (is(0, FUSEML_OP_RELU)) ch = kChainRelu;
      break;
    case 2:
      if (row(0) && is(1, FUSEML_OP_GELU_ERF)) ch = kChainBiasGeluErf;
      else if (row(0) && is(1, FUSEML_OP_GELU_TANH)) ch = kChainBiasGeluTanh;
      else if (row(0) && is(1, FUSEML_OP_RELU)) ch = kChainBiasRelu;
      else if (row(0) && tile(1, FUSEML_OP_ADD)) ch = kChainBiasTile;
      break;
    case 4:
      if (row(0) && is(1, FUSEML_OP_GELU_ERF) && is(2, FUSEML_OP_SCALE) && is(3, FUSEML_OP_ADD_SCALAR))
        ch = kChainBiasGeluScale;
      break;
    case 5:
      if (row(0) && is(1, FUSEML_OP_RELU) && tile(2, FUSEML_OP_MUL) && is(3, FUSEML_OP_SIGMOID) && row(4))
        ch = kChainActHeavy;
      break;
    default: break;
  }
  if (d.reduce_mask != 0 && ch != kChainRelu) return kChainGeneric;
  return ch;
}

// `max_wg` caps the grid (0: one workgroup per tile); the kernel loops over the
// remaining tiles.
template <const TileConfig& C, typename T, bool ANY>
hipError_t launch_rows(const fuseml_gemm_desc& d, hipStream_t stream, int max_wg) {
  int64_t tiles = cdiv(d.M, C.bm) * cdiv(d.N, C.bn);
  if (max_wg > 0 && tiles > max_wg) tiles = max_wg;
  const dim3 grid((unsigned)tiles), block(C.wm * C.wn * 64);
  constexpr int G = kChainGeneric;
  if (d.reduce_mask == 0)
    hipLaunchKernelGGL((gemm_epilogue_kernel<C.bm, C.bn, C.bk, C.stages, C.wm, C.wn, C.sched, T, false, G, ANY>), grid,
                       block, 0, stream, d);
  else
    hipLaunchKernelGGL((gemm_epilogue_kernel<C.bm, C.bn, C.bk, C.stages, C.wm, C.wn, C.sched, T, true, G, ANY>), grid,
                       block, 0, stream, d);
  return hipGetLastError();
}

// Whether a launch needs the kernel's parameter ANY: a staged operand whose rows are
// not whole 16-byte chunks at 16-byte addresses, or an output that is not staged or
// has such rows.
bool needs_any(const fuseml_gemm_desc& d) {
  constexpr int kBoth = kFlagStage | kFlagAligned;
  for (int i = 0; i < d.n_operands; ++i)
    if ((d.operands[i].reserved & kBoth) == kFlagStage) return true;
  return d.out.ptr != nullptr && (d.out.reserved & kBoth) != kBoth;
}

template <const TileConfig& C, typename T>
hipError_t launch_typed(const fuseml_gemm_desc& d, hipStream_t stream, int max_wg) {
  if constexpr (splits_rows<T>(C)) {
    if (!needs_any(d)) return launch_rows<C, T, false>(d, stream, max_wg);
  }
  return launch_rows<C, T, true>(d, stream, max_wg);
}

template <const TileConfig& C>
hipError_t launch_variant(const fuseml_gemm_desc& d, hipStream_t stream, int max_wg) {
  return d.ab_dtype == FUSEML_BF16 ? launch_typed<C, __bf16>(d, stream, max_wg)
                                   : launch_typed<C, _Float16>(d, stream, max_wg);
}

// A fixed-chain kernel of variant C (reductions only with kChainRelu, as
// match_fixed_chain guarantees).
template <const TileConfig& C, typename T, int CH>
void launch_fixed_one(const fuseml_gemm_desc& d, hipStream_t stream, dim3 grid, dim3 block) {
  if constexpr (CH == kChainRelu) {
    if (d.reduce_mask != 0) {
      hipLaunchKernelGGL((gemm_epilogue_kernel<C.bm, C.bn, C.bk, C.stages, C.wm, C.wn, C.sched, T, true, CH, true>), grid,
                         block, 0, stream, d);
      return;
    }
  }
  hipLaunchKernelGGL((gemm_epilogue_kernel<C.bm, C.bn, C.bk, C.stages, C.wm, C.wn, C.sched, T, false, CH, true>), grid,
                     block, 0, stream, d);
}

template <const TileConfig& C, typename T>
hipError_t launch_fixed(const fuseml_gemm_desc& d, int ch, hipStream_t stream, int max_wg) {
  int64_t tiles = cdiv(d.M, C.bm) * cdiv(d.N, C.bn);
  if (max_wg > 0 && tiles > max_wg) tiles = max_wg;
  const dim3 grid((unsigned)tiles), block(C.wm * C.wn * 64);
  switch (ch) {
    case kChainNone: launch_fixed_one<C, T, kChainNone>(d, stream, grid, block); break;
    case kChainBias: launch_fixed_one<C, T, kChainBias>(d, stream, grid, block); break;
    case kChainBiasGeluErf: launch_fixed_one<C, T, kChainBiasGeluErf>(d, stream, grid, block); break;
    case kChainBiasGeluTanh: launch_fixed_one<C, T, kChainBiasGeluTanh>(d, stream, grid, block); break;
    case kChainBiasRelu: launch_fixed_one<C, T, kChainBiasRelu>(d, stream, grid, block); break;
    case kChainBiasTile: launch_fixed_one<C, T, kChainBiasTile>(d, stream, grid, block); break;
    case kChainActHeavy: launch_fixed_one<C, T, kChainActHeavy>(d, stream, grid, block); break;
    case kChainRelu: launch_fixed_one<C, T, kChainRelu>(d, stream, grid, block); break;
    case kChainBiasGeluScale: launch_fixed_one<C, T, kChainBiasGeluScale>(d, stream, grid, block); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// The fixed chain a launch of `d` (flags derived) on variant `c` runs, or
// kChainGeneric: fixed chains are built for the one-wave whole-stage variant.
int launch_chain(const fuseml_gemm_desc& d, const TileConfig& c) {
  if (c.sched != kDeep3.sched || forced_variant() == kForcedDeep3Generic) return kChainGeneric;
  return match_fixed_chain(d);
}

// Per-device check and CU count, queried once per device: the CU count for a
// gfx950 device, else FUSEML_EDEVICE or FUSEML_EHIP (negative; the error is set).
constexpr int kMaxDevices = 64;
std::atomic<int> g_device_cus[kMaxDevices];

int device_cus(int dev) {
  if (dev >= 0 && dev < kMaxDevices) {
    const int known = g_device_cus[dev].load(std::memory_order_relaxed);
    if (known > 0) return known;
  }
  char arch[64];
  if (fuseml_device_arch(dev, arch, sizeof(arch)) != FUSEML_OK) return FUSEML_EHIP;
  if (strncmp(arch, "gfx950", 6) != 0) {
    set_error("device %d is %s; kernels are built for gfx950 only", dev, arch);
    return FUSEML_EDEVICE;
  }
  int cus = 0;
  const hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess || cus <= 0) {
    set_error("hipDeviceGetAttribute(MultiprocessorCount): %s", hipGetErrorString(e));
    return FUSEML_EHIP;
  }
  if (dev >= 0 && dev < kMaxDevices) g_device_cus[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

// One launch of `d` (flags derived) on the kernel its size and chain choose.
hipError_t launch_one(const fuseml_gemm_desc& d, int cus, hipStream_t stream) {
  const int ks = choose_ksplit(d, cus);
  if (ks >= 0)
    return d.ab_dtype == FUSEML_BF16 ? launch_ksplit<__bf16>(d, ks, stream) : launch_ksplit<_Float16>(d, ks, stream);
  const TileConfig c = choose_config(d, cus);
  const int ch = launch_chain(d, c);
  if (ch != kChainGeneric)
    return d.ab_dtype == FUSEML_BF16 ? launch_fixed<kDeep3, __bf16>(d, ch, stream, cus)
                                     : launch_fixed<kDeep3, _Float16>(d, ch, stream, cus);
  if (c.sched == kDeep.sched) return launch_variant<kDeep>(d, stream, cus);
  if (c.sched == kLarge.sched && c.bn == kLarge128.bn) return launch_variant<kLarge128>(d, stream, cus);
  if (c.sched == kLarge.sched) return launch_variant<kLarge>(d, stream, cus);
  if (c.sched == kDeep3.sched) return launch_variant<kDeep3>(d, stream, cus);
  if (c.bm == kSmall64.bm && c.bk == kSmall64.bk) return launch_variant<kSmall64>(d, stream, 0);
  if (c.bm == kNarrow64.bm) return launch_variant<kNarrow64>(d, stream, 0);
  if (c.bm == kNarrow32.bm) return launch_variant<kNarrow32>(d, stream, 0);
  return launch_variant<kSmall>(d, stream, 0);
}

// The rows from m1 on (or the columns from n1 on) of `d` as a group of their own.
fuseml_gemm_desc rest_of(const fuseml_gemm_desc& d, int64_t m1, int64_t n1) {
  fuseml_gemm_desc r = d;
  auto advance = [](const void* p, int64_t elements, int dtype) -> void* {
    return p == nullptr ? nullptr : (char*)p + elements * (dtype == FUSEML_F32 ? 4 : 2);
  };
  r.M -= m1;
  r.N -= n1;
  r.a = advance(d.a, m1 * d.lda, d.ab_dtype);
  r.b = advance(d.b, n1 * d.ldb, d.ab_dtype);
  for (int i = 0; i < d.n_operands; ++i) {
    fuseml_operand& o = r.operands[i];
    const int64_t skip = m1 * o.stride_m + n1 * o.stride_n;
    o.ptr = advance(o.ptr, skip, o.dtype);
    o.extent -= skip;
  }
  r.out.ptr = advance(d.out.ptr, m1 * d.out.ld + n1, d.out.dtype);
  for (int i = 0; i < d.n_extra; ++i)
    r.extra[i].ptr = advance(d.extra[i].ptr, m1 * d.extra[i].ld + n1, d.extra[i].dtype);
  if (d.reduce_mask != 0)
    for (int b = 0; b < 3; ++b)
      if (d.reduce_out[b] != nullptr) r.reduce_out[b] += d.reduce_axis == 1 ? m1 : n1;
  return r;
}

// A last round of few 256x256 tiles takes nearly as long as a full one (a CU's
// time for one tile: 23 us at K = 1024 and 67 at K = 4096 behind a full round, for
// 16 to 64 tiles of 256), so it runs as a group of its own on the tiles of its
// size: `d` keeps the whole rounds, `rest` the remaining rows (or columns, where
// rows would leave more than 7% of the rounds idle).  Priced as choose_ksplit
// prices a small group, 2 us for the second launch, and only where that is 0.9 of
// the partial round or less.  Not for a mean along the split axis, whose divisor
// is the whole length.  Measured (M x N x K, us, one launch -> two): 4352x4096x1024
// bias+GELU 63.8 -> 50.4, 4608x4096x4096 bias+residual 176.9 -> 141.3, 17408x1024x4096
// 187.2 -> 142.4, 512x34000x1024 64.3 -> 50.5.
bool split_rounds(fuseml_gemm_desc& d, int cus, fuseml_gemm_desc& rest) {
  if (forced_variant() != 0 || d.K <= 0 || d.M <= 128) return false;
  const int64_t tm = cdiv(d.M, 256), tn = cdiv(d.N, 256), rounds = tm * tn / cus;
  if (rounds == 0 || tm * tn % cus == 0) return false;
  const int64_t m_tiles = rounds * cus / tn, n_tiles = rounds * cus / tm;
  const bool by_rows = m_tiles * tn >= n_tiles * tm;
  const int64_t kept = by_rows ? m_tiles * tn : n_tiles * tm;
  if (kept * 100 < rounds * cus * 93) return false;
  if ((d.reduce_mask & FUSEML_RED_MEAN) && d.reduce_axis == (by_rows ? 0 : 1)) return false;
  fuseml_gemm_desc r = rest_of(d, by_rows ? m_tiles * 256 : 0, by_rows ? 0 : n_tiles * 256);
  if (2 * cdiv(r.M, 256) * cdiv(r.N, 256) > cus) return false;
  const double k = (double)d.K / 1024.0;
  const double left = (double)(tm * tn - rounds * cus) / cus;
  const double partial = (8.3 + 14.7 * k) * (left > 0.25 ? 0.875 + 0.5 * left : 1.0);
  double small = 0.0;
  int64_t work = 0;
  choose_partial_round(r, cus, &work);
  cheapest_ksplit(r.M, r.N, r.K, cus, kKsplitPerK, &small);
  const double tiled = -3.0 + (double)work / (5.0 * 160.0) * (5.05 + 3.6 * k);
  if (small >= kKsplitMargin * tiled) small = tiled;
  if (small + 2.0 > 0.9 * partial) return false;
  derive_flags(r);
  rest = r;
  if (by_rows) d.M = m_tiles * 256; else d.N = n_tiles * 256;
  derive_flags(d);
  return true;
}

}  // namespace

namespace fuseml_detail {
// Error text for the other translation units of the library (mlp_block.hip).
void set_error_text(const char* msg) {
  strncpy(g_last_error, msg, sizeof(g_last_error) - 1);
  g_last_error[sizeof(g_last_error) - 1] = '\0';
}
}  // namespace fuseml_detail

extern "C" {

const char* fuseml_last_error(void) { return g_last_error; }

int fuseml_abi_version(void) { return FUSEML_ABI_VERSION; }

size_t fuseml_desc_size(void) { return sizeof(fuseml_gemm_desc); }

size_t fuseml_mlp_desc_size(void) { return sizeof(fuseml_mlp_desc); }

int fuseml_gemm_epilogue_supported(const fuseml_gemm_desc* desc) {
  g_last_error[0] = '\0';
  return validate(desc) == FUSEML_OK ? 1 : 0;
}

int fuseml_gemm_epilogue_config(const fuseml_gemm_desc* desc, int32_t cfg[4]) {
  g_last_error[0] = '\0';
  const int rc = validate(desc);
  if (rc != FUSEML_OK) return rc;
  // The CU count of the current device if it is known, else MI355X's.
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices) {
    const int known = g_device_cus[dev].load(std::memory_order_relaxed);
    if (known > 0) cus = known;
  }
  fuseml_gemm_desc d = *desc;
  fold_final_store(d);
  derive_flags(d);
  const TileConfig c = choose_config(d, cus);
  cfg[0] = c.bm;
  cfg[1] = c.bn;
  cfg[2] = c.wm * c.wn;
  cfg[3] = c.lds_bytes();
  return FUSEML_OK;
}

int fuseml_gemm_epilogue_ksplit(const fuseml_gemm_desc* desc, int32_t cfg[4]) {
  g_last_error[0] = '\0';
  const int rc = validate(desc);
  if (rc != FUSEML_OK) return rc;
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices) {
    const int known = g_device_cus[dev].load(std::memory_order_relaxed);
    if (known > 0) cus = known;
  }
  const int i = choose_ksplit(*desc, cus);
  if (i < 0) return 0;
  cfg[0] = kKsplit[i].bm();
  cfg[1] = kKsplit[i].bn();
  cfg[2] = kKsplit[i].waves;
  cfg[3] = kKsplit[i].lds_bytes();
  return 1;
}

int fuseml_gemm_epilogue_f32_supported(const fuseml_gemm_desc* desc) {
  g_last_error[0] = '\0';
  const int rc = validate(desc, true);
  if (rc != FUSEML_OK) return 0;
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices) {
    const int known = g_device_cus[dev].load(std::memory_order_relaxed);
    if (known > 0) cus = known;
  }
  // Under a pinned variant, fp32 groups are to run on it: as split parts.  (A
  // launch is not refused for that: its caller may have asked before the pin.)
  if (forced_variant() == 0 && choose_ksplit_f32(*desc, cus) >= 0) return 1;
  set_error("fp32 operands of this size run as bf16 parts (fuseml_split_bf16x3)");
  return 0;
}

int fuseml_gemm_epilogue_chain(const fuseml_gemm_desc* desc) {
  g_last_error[0] = '\0';
  const int rc = validate(desc);
  if (rc != FUSEML_OK) return rc;
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices) {
    const int known = g_device_cus[dev].load(std::memory_order_relaxed);
    if (known > 0) cus = known;
  }
  fuseml_gemm_desc d = *desc;
  fold_final_store(d);
  derive_flags(d);
  return launch_chain(d, choose_config(d, cus));
}

int fuseml_gemm_epilogue_force_variant(const char* name) {
  g_last_error[0] = '\0';
  const int v = variant_code(name);
  if (v < 0) {
    set_error("unknown variant '%s' (large, deep, deep3, small, deep3-generic, narrow64, narrow32, large128, small64 "
              "or auto)", name);
    return FUSEML_EINVAL;
  }
  forced_variant();  // the environment is read first, so it cannot override this later
  g_forced_variant.store(v, std::memory_order_relaxed);
  return FUSEML_OK;
}

int fuseml_device_arch(int device, char* buf, int buflen) {
  hipDeviceProp_t prop;
  const hipError_t e = hipGetDeviceProperties(&prop, device);
  if (e != hipSuccess) {
    set_error("hipGetDeviceProperties: %s", hipGetErrorString(e));
    return FUSEML_EHIP;
  }
  if (buf != nullptr && buflen > 0) {
    strncpy(buf, prop.gcnArchName, (size_t)buflen - 1);
    buf[buflen - 1] = '\0';
  }
  return FUSEML_OK;
}

// The start of a launch, common to both operand kinds: the validated descriptor
// with its derived flags, the CU count, and the reduction buffers' fill on the
// stream.  FUSEML_OK or an error code (the error is set).
static int begin_launch(const fuseml_gemm_desc* desc, bool f32, hipStream_t stream, fuseml_gemm_desc& d, int& cus) {
  g_last_error[0] = '\0';
  const int rc = validate(desc, f32);
  if (rc != FUSEML_OK) return rc;

  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error("hipGetDevice: %s", hipGetErrorString(e));
    return FUSEML_EHIP;
  }
  cus = device_cus(dev);
  if (cus <= 0) return cus < 0 ? cus : FUSEML_EHIP;

  d = *desc;
  fold_final_store(d);
  derive_flags(d);
  if (f32 && choose_ksplit_f32(d, cus) < 0) {
    set_error("fp32 operands of this size run as bf16 parts (fuseml_split_bf16x3)");
    return FUSEML_EUNSUPPORTED;
  }

  if (d.reduce_mask) {
    const int len = (int)(d.reduce_axis == 1 ? d.M : d.N);
    float* sum = (d.reduce_mask & FUSEML_RED_SUM) ? d.reduce_out[0] : nullptr;
    float* amax = (d.reduce_mask & FUSEML_RED_AMAX) ? d.reduce_out[1] : nullptr;
    float* mean = (d.reduce_mask & FUSEML_RED_MEAN) ? d.reduce_out[2] : nullptr;
    hipLaunchKernelGGL(reduce_fill_kernel, dim3((unsigned)cdiv(len, 256)), dim3(256), 0, stream,
                       sum, amax, mean, len);
    e = hipGetLastError();
    if (e != hipSuccess) {
      set_error("reduce_fill launch: %s", hipGetErrorString(e));
      return FUSEML_EHIP;
    }
  }
  return FUSEML_OK;
}

int fuseml_gemm_epilogue_f32(const fuseml_gemm_desc* desc, void* stream_ptr) {
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_ptr);
  fuseml_gemm_desc d;
  int cus = 0;
  const int rc = begin_launch(desc, true, stream, d, cus);
  if (rc != FUSEML_OK) return rc;
  const hipError_t e = launch_ksplit<float>(d, choose_ksplit_f32(d, cus), stream);
  if (e != hipSuccess) {
    set_error("gemm_ksplit launch: %s", hipGetErrorString(e));
    return FUSEML_EHIP;
  }
  return FUSEML_OK;
}

int fuseml_gemm_epilogue(const fuseml_gemm_desc* desc, void* stream_ptr) {
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_ptr);
  fuseml_gemm_desc d;
  int cus = 0;
  const int rc = begin_launch(desc, false, stream, d, cus);
  if (rc != FUSEML_OK) return rc;
  hipError_t e = hipSuccess;

  // The part of whole rounds, then the rest, each on the kernel of its own size.
  fuseml_gemm_desc rest;
  if (split_rounds(d, cus, rest)) {
    e = launch_one(d, cus, stream);
    if (e == hipSuccess) e = launch_one(rest, cus, stream);
  } else {
    e = launch_one(d, cus, stream);
  }
  if (e != hipSuccess) {
    set_error("gemm_epilogue launch: %s", hipGetErrorString(e));
    return FUSEML_EHIP;
  }
  return FUSEML_OK;
}

}  // extern "C"