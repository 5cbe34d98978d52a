// gemm_ksplit.h — the K-split GEMM+epilogue kernel for small outputs, included
// only by its instantiation units (gemm_ksplit_*.hip).
//
// The tiled family (gemm_epilogue_kernel.h) gives every workgroup the whole K
// loop of its tile and shares the tile's operands between its waves through
// LDS, one barrier per stage.  With few output tiles most CUs idle, and a CU's
// K loop is bound by the one or two stages it has in flight.  Here the waves of
// a workgroup split K instead: wave w multiplies the whole BM x BN tile over
// 128-byte chunks w, w + NW, ... of every operand row.  No operand element is
// used by two waves, so each wave streams its chunks through a ring of its own
// in LDS, DEPTH chunks ahead, with no barrier in the loop, and the tile can be
// small (16 to 64 rows and columns), so a decode-sized output still gives every
// CU a workgroup.  After the loop the waves' fp32 partials meet in LDS once, are
// added in wave order (the result does not depend on timing), and each thread
// runs the epilogue chain on runs of 4 columns.
//
// What bounds it: the bytes a CU pulls, (BM + BN) rows x K, at 60-75 GB/s per CU
// and about 4 us of launch, first loads, partials and epilogue; for a weight of
// tens of MB, HBM.  Why the ring: fragment loads straight into registers (no LDS
// at all) were measured first, at 21-24 GB/s per CU, since neighbouring lanes of
// an MFMA fragment lie in different rows and a load touches a cache line per
// lane; a DMA's neighbouring lanes read whole 128-byte lines.  Measured
// (M x N x K, bias + residual, bf16, us; tiled kernels -> registers -> ring):
// 8x4096x16384 107.7 -> 29.7 -> 27.0 (5.0 TB/s), 16x4096x1024 10.3 -> 6.1 -> 5.5,
// 64x1024x4096 23.6 -> 11.3 -> 6.9, 512x1024x4096 24.1 -> 26.4 -> 14.3.
//
// MFMA: v_mfma_f32_16x16x32, W rows as operand A, so that a lane holds one
// output row and 4 consecutive columns.
#pragma once

#include "gemm_epilogue_kernel.h"

namespace fuseml_gemm {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ f32x4_t mfma16(i32x4_t a, i32x4_t b, f32x4_t c);

template <>
__device__ __forceinline__ f32x4_t mfma16<__bf16>(i32x4_t a, i32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                 0, 0, 0);
}

template <>
__device__ __forceinline__ f32x4_t mfma16<_Float16>(i32x4_t a, i32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                0, 0);
}

// fp32 operands: 8 consecutive-in-order values of a row (two 16-byte pieces) as
// the bf16 parts of split_f32.hip: hi = bf16(x) (truncated where that would
// overflow a finite x), lo = bf16(x - hi) and 0 for inf and NaN, hf = hi with
// inf and NaN written as 0.  Parts beyond hi and lo differ from the plain
// rounding only where a value is not finite or above the largest bf16, which
// one uniform test per fragment rules out.
struct SplitFrag {
  i32x4_t hi, lo, hf;
};

__device__ __forceinline__ SplitFrag split_frag(i32x4_t p0, i32x4_t p1) {
  constexpr float kBf16Max = 3.38953139e38f;  // largest finite bf16, (2 - 2^-7) 2^127
  float x[8];
  static_for<0, 4>([&](auto e) {
    x[e] = __int_as_float(p0[(int)e]);
    x[4 + e] = __int_as_float(p1[(int)e]);
  });
  SplitFrag f;
  static_for<0, 4>([&](auto e) {
    const uint32_t h = pack_bf16x2(x[2 * e], x[2 * e + 1]);
    const float ha = __uint_as_float(h << 16), hb = __uint_as_float(h & 0xffff0000u);
    f.hi[(int)e] = (int)h;
    f.lo[(int)e] = (int)pack_bf16x2(x[2 * e] - ha, x[2 * e + 1] - hb);
  });
  f.hf = f.hi;
  float big = 0.0f;
  static_for<0, 8>([&](auto e) { big = max_nan(big, __builtin_fabsf(x[e])); });
  if (__builtin_amdgcn_ballot_w64(!(big <= kBf16Max)) != 0) {
    static_for<0, 4>([&](auto e) {
      const float a = x[2 * e], b = x[2 * e + 1];
      const bool fa = __builtin_isfinite(a), fb = __builtin_isfinite(b);
      uint32_t h = (uint32_t)f.hi[(int)e];
      if (__builtin_fabsf(a) > kBf16Max && fa) h = (h & 0xffff0000u) | (__float_as_uint(a) >> 16);
      if (__builtin_fabsf(b) > kBf16Max && fb) h = (h & 0x0000ffffu) | (__float_as_uint(b) & 0xffff0000u);
      const float ha = __uint_as_float(h << 16), hb = __uint_as_float(h & 0xffff0000u);
      f.hi[(int)e] = (int)h;
      f.lo[(int)e] = (int)pack_bf16x2(fa ? a - ha : 0.0f, fb ? b - hb : 0.0f);
      f.hf[(int)e] = (int)(h & ((fa ? 0x0000ffffu : 0u) | (fb ? 0xffff0000u : 0u)));
    });
  }
  return f;
}

// An operand's 4 values at (m, n..n+3) of the tile at (m0, n0), in two halves:
// the raw load (issued before the K loop, so that its latency lies under it)
// and the conversion to fp32.  As load_operand4.
template <typename Op>
__device__ __forceinline__ i32x4_t load_raw4(const Op& op, int m0, int n0, int m, int n, bool ok) {
  const int eb = dtype_bytes(op.dtype);
  const __amdgpu_buffer_rsrc_t r =
      make_rsrc_at(op.ptr, ((int64_t)m0 * op.stride_m + (int64_t)n0 * op.stride_n) * eb, op.extent * eb);
  const int64_t base = (int64_t)(m - m0) * op.stride_m + (int64_t)(n - n0) * op.stride_n;
  i32x4_t x = {0, 0, 0, 0};
  if (op.reserved & kFlagVec4) {
    const uint32_t off = ok ? (uint32_t)(base * eb) : kOOB;
    if (eb == 4) {
      x = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    } else {
      const i32x2_t y = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
      x.x = y.x;
      x.y = y.y;
    }
    return x;
  }
  static_for<0, 4>([&](auto e) {
    if (e == 0 || op.stride_n != 0) {
      const uint32_t off = ok ? (uint32_t)((base + (int64_t)e * op.stride_n) * eb) : kOOB;
      x[(int)e] = (eb == 4) ? (int)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0)
                            : (int)(uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
    }
  });
  return x;
}

template <typename Op>
__device__ __forceinline__ void convert_raw4(const Op& op, i32x4_t x, float v[4]) {
  const int dt = op.dtype;
  if ((op.reserved & kFlagVec4) && dt != FUSEML_F32) {
    v[0] = elem_to_f32((uint32_t)x.x & 0xffffu, dt);
    v[1] = elem_to_f32((uint32_t)x.x >> 16, dt);
    v[2] = elem_to_f32((uint32_t)x.y & 0xffffu, dt);
    v[3] = elem_to_f32((uint32_t)x.y >> 16, dt);
    return;
  }
  const bool one = !(op.reserved & kFlagVec4) && op.stride_n == 0;
  v[0] = elem_to_f32((uint32_t)x.x, dt);
  v[1] = elem_to_f32((uint32_t)(one ? x.x : x.y), dt);
  v[2] = elem_to_f32((uint32_t)(one ? x.x : x.z), dt);
  v[3] = elem_to_f32((uint32_t)(one ? x.x : x.w), dt);
}

// MB x NB blocks of 16 rows x 16 columns per tile; NW waves split K; DEPTH
// chunks of 128 bytes of every row per wave in its LDS ring.  RED: the launch has
// reductions; the others' kernels carry none of that code (3% of a 6 us launch).
template <int MB, int NB, int NW, int DEPTH, typename T, bool RED>
__global__ __launch_bounds__(NW * 64) void gemm_ksplit_kernel(const fuseml_gemm_desc d_arg) {
  constexpr int BM = 16 * MB, BN = 16 * NB, NT = NW * 64;
  constexpr int UNITS = BM * BN / 4;             // runs of 4 columns
  constexpr int UPT = (UNITS + NT - 1) / NT;     // per thread
  constexpr int EB = sizeof(T);                  // bytes per GEMM operand element
  constexpr int kPre = 2;                        // operands fetched before the K loop
  constexpr int kRing = NW * DEPTH * (BM + BN) * 128, kPart = NW * BM * BN * 4;
  __shared__ __attribute__((aligned(1024))) char smem[kRing > kPart ? kRing : kPart];

  const KDesc& d = *(const KDesc*)(__builtin_amdgcn_kernarg_segment_ptr());
  const int M = (int)d.M, N = (int)d.N;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;

  // Workgroups are dealt to the 8 XCDs round-robin: each XCD gets a contiguous
  // range of the tiles, ordered in GROUP_M-row column strips, so the tiles of an
  // XCD share W rows (and x rows) in its L2.
  const int n_tiles = gridDim.x;
  const int xcd = (int)blockIdx.x & 7, per = n_tiles >> 3, rest = n_tiles & 7;
  const int lid = xcd * per + min(xcd, rest) + ((int)blockIdx.x >> 3);
  const int strip = kGroupM * tiles_n;
  const int first_m = (lid / strip) * kGroupM;
  const int strip_h = min(tiles_m - first_m, kGroupM);
  const int m0 = (first_m + (lid % strip) % strip_h) * BM;
  const int n0 = ((lid % strip) / strip_h) * BN;

  const uint32_t k_bytes = (uint32_t)d.K * (uint32_t)EB;
  const __amdgpu_buffer_rsrc_t ra =
      make_rsrc_at(d.a, (int64_t)m0 * d.lda * EB, ((int64_t)(M - 1) * d.lda + d.K) * EB);
  const __amdgpu_buffer_rsrc_t rb =
      make_rsrc_at(d.b, (int64_t)n0 * d.ldb * EB, ((int64_t)(N - 1) * d.ldb + d.K) * EB);
  // One DMA fills 8 rows x 128 bytes: lane l's slot is physical 16-byte piece
  // l % 8 of row l / 8, which holds logical piece (l % 8) ^ swizzle(row).  Rows
  // past the edge repeat the last one (their results are not stored).
  using G = StageGeom<64>;
  const int dr = lane >> 3;
  uint32_t a_off[2 * MB], b_off[2 * NB];
  static_for<0, 2 * MB>([&](auto i) {
    a_off[i] = (uint32_t)((int64_t)min(8 * i + dr, M - 1 - m0) * d.lda * EB);
  });
  static_for<0, 2 * NB>([&](auto i) {
    b_off[i] = (uint32_t)((int64_t)min(8 * i + dr, N - 1 - n0) * d.ldb * EB);
  });
  // swizzle(8 i + dr) = (4 i + dr / 2) & 7: the same for every second i.
  const uint32_t piece0 = (uint32_t)(((lane & 7) ^ (dr >> 1)) * 16);
  const uint32_t piece1 = (uint32_t)(((lane & 7) ^ (4 + (dr >> 1))) * 16);
  constexpr int CB = (BM + BN) * 128;            // one chunk of the tile's rows
  constexpr int LPC = (BM + BN) / 8;             // DMAs per chunk
  static_assert(LPC * (DEPTH - 1) < 64, "vmcnt range");
  char* ring = smem + wave * (DEPTH * CB);
  auto load = [&](int slot, int c) {
    char* st = ring + slot * CB;
    const uint32_t kb = (uint32_t)c * 128u;
    const uint32_t k0 = kb + piece0 < k_bytes ? kb + piece0 : kOOB;
    const uint32_t k1 = kb + piece1 < k_bytes ? kb + piece1 : kOOB;
    static_for<0, 2 * NB>([&](auto i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)(st + i * 1024), 16,
                                               b_off[i] + ((i & 1) ? k1 : k0), 0, 0, 0);
    });
    static_for<0, 2 * MB>([&](auto i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(st + BN * 128 + i * 1024),
                                               16, a_off[i] + ((i & 1) ? k1 : k0), 0, 0, 0);
    });
  };

  // Units of this thread: u = tid + NT q; row u / (BN / 4), columns 4 (u % (BN / 4)).
  i32x4_t raw[UPT][kPre];
  static_for<0, UPT>([&](auto q) {
    const int u = tid + NT * q;
    const int m = m0 + u / (BN / 4), n = n0 + 4 * (u % (BN / 4));
    static_for<0, kPre>([&](auto o) {
      raw[q][o] = i32x4_t{0, 0, 0, 0};
      if (o < d.n_operands && u < UNITS) raw[q][o] = load_raw4(d.operands[o], m0, n0, m, n, m < M && n < N);
    });
  });

  const int chunks = (int)((k_bytes + 127u) >> 7);
  const int mine = chunks > wave ? (chunks - wave + NW - 1) / NW : 0;
  __builtin_amdgcn_sched_barrier(0);
  static_for<0, DEPTH>([&](auto b) { load(b, wave + NW * b); });

  f32x4_t acc[MB][NB];
  static_for<0, MB>([&](auto i) {
    static_for<0, NB>([&](auto j) { acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}; });
  });
  const int fr = (lane & 15) * 128;
  const int sw = G::swizzle(lane & 15);
  int slot = 0;
  for (int t = 0; t < mine; ++t) {
    wait_vmcnt<LPC * (DEPTH - 1)>();  // the oldest chunk of this wave's ring has landed
    __builtin_amdgcn_sched_barrier(0);
    const char* st = ring + slot * CB;
    i32x4_t fa[2][NB], fb[2][MB];
    static_for<0, 2>([&](auto s) {
      const int piece = ((4 * s + (lane >> 4)) ^ sw) << 4;
      static_for<0, NB>([&](auto i) { fa[s][i] = *reinterpret_cast<const i32x4_t*>(st + i * 2048 + fr + piece); });
      static_for<0, MB>(
          [&](auto i) { fb[s][i] = *reinterpret_cast<const i32x4_t*>(st + BN * 128 + i * 2048 + fr + piece); });
    });
    wait_lgkmcnt0();  // fragments read: the slot can be refilled
    __builtin_amdgcn_sched_barrier(0);
    load(slot, wave + NW * (t + DEPTH));
    if constexpr (EB == 4) {
      SplitFrag w[NB];
      static_for<0, NB>([&](auto j) { w[j] = split_frag(fa[0][j], fa[1][j]); });
      static_for<0, MB>([&](auto i) {
        const SplitFrag x = split_frag(fb[0][i], fb[1][i]);
        static_for<0, NB>([&](auto j) {
          acc[i][j] = mfma16<__bf16>(w[j].lo, x.hf, acc[i][j]);
          acc[i][j] = mfma16<__bf16>(w[j].hf, x.lo, acc[i][j]);
          acc[i][j] = mfma16<__bf16>(w[j].hi, x.hi, acc[i][j]);
        });
      });
    } else {
      static_for<0, 2>([&](auto s) {
        static_for<0, MB>([&](auto i) {
          static_for<0, NB>([&](auto j) { acc[i][j] = mfma16<T>(fa[s][j], fb[s][i], acc[i][j]); });
        });
      });
    }
    if (++slot == DEPTH) slot = 0;
  }
  // The DMAs still in flight (zeros past K) land before the partials overwrite
  // the rings; other waves may still read theirs.
  wait_vmcnt<0>();
  __syncthreads();

  // Partials: block (i, j) of wave w is 1 KB at ((w MB + i) NB + j) KB; lane l
  // holds row l & 15, columns 4 (l >> 4) .. +3, in slot 16 (l >> 4) + ((l & 15) ^
  // 4 (l >> 4)), which both the writes and the reads below hit without bank
  // conflicts.
  {
    const int q = lane >> 4;
    const int slot = q * 16 + ((lane & 15) ^ (4 * q));
    static_for<0, MB>([&](auto i) {
      static_for<0, NB>([&](auto j) {
        *reinterpret_cast<f32x4_t*>(smem + (((wave * MB + i) * NB + j) << 10) + slot * 16) = acc[i][j];
      });
    });
  }
  lds_barrier();

  // A unit's values into the fused reductions, one atomic per row or column of the
  // tile.  The BN / 4 units of a row are neighbouring lanes.  A thread's units all
  // lie in the same 4 columns, whose partials it keeps to the end (col_s, col_mx).
  // Elements outside [0, M) x [0, N) never enter.
  auto put = [&](int idx, float s, float mx, float inv) {
    if (d.reduce_mask & FUSEML_RED_SUM) atomicAdd(d.reduce_out[0] + idx, s);
    if (d.reduce_mask & FUSEML_RED_AMAX) atomic_max_f32(d.reduce_out[1] + idx, mx);
    if (d.reduce_mask & FUSEML_RED_MEAN) atomicAdd(d.reduce_out[2] + idx, s * inv);
  };
  static_assert(NT % (BN / 4) == 0, "a thread's units share their columns");
  float col_s[4] = {0.0f, 0.0f, 0.0f, 0.0f}, col_mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  auto reduce = [&](const float v[4], int m, int n, int nq) {
    float s[4], mx[4];
    static_for<0, 4>([&](auto e) {
      const bool in = m < M && n + e < N;
      s[e] = in ? v[e] : 0.0f;
      mx[e] = in ? v[e] : -INFINITY;
    });
    if (d.reduce_axis == 1) {
      s[0] = (s[0] + s[1]) + (s[2] + s[3]);
      mx[0] = max_nan(max_nan(mx[0], mx[1]), max_nan(mx[2], mx[3]));
#pragma unroll
      for (int sh = 1; sh < BN / 4; sh <<= 1) {
        s[0] += __shfl_xor(s[0], sh);
        mx[0] = max_nan(mx[0], __shfl_xor(mx[0], sh));
      }
      if (nq == 0 && m < M) put(m, s[0], mx[0], 1.0f / (float)N);
    } else {
      static_for<0, 4>([&](auto e) {
        col_s[e] += s[e];
        col_mx[e] = max_nan(col_mx[e], mx[e]);
      });
    }
  };

  static_for<0, UPT>([&](auto q) {
    const int u = tid + NT * q;
    if (u >= UNITS) return;
    const int ml = u / (BN / 4), nq = u % (BN / 4);
    const int m = m0 + ml, n = n0 + 4 * nq;
    const int slot = (nq & 3) * 16 + ((ml & 15) ^ (4 * (nq & 3)));
    const char* src = smem + (((ml >> 4) * NB + (nq >> 2)) << 10) + slot * 16;
    f32x4_t sum = *reinterpret_cast<const f32x4_t*>(src);
    static_for<1, NW>([&](auto w) { sum += *reinterpret_cast<const f32x4_t*>(src + ((w * MB * NB) << 10)); });
    float v[4] = {sum[0], sum[1], sum[2], sum[3]};
    for (int o = 0; o < d.n_ops; ++o) {
      const int kind = d.ops[o].kind, oi = d.ops[o].operand;
      const float sc = d.ops[o].scalar;
      if (kind == FUSEML_OP_ADD || kind == FUSEML_OP_MUL) {
        float x[4];
        if (oi == 0)
          convert_raw4(d.operands[0], raw[q][0], x);
        else if (oi == 1)
          convert_raw4(d.operands[1], raw[q][1], x);
        else
          load_operand4(d.operands[oi], m0, n0, m, n, m < M && n < N, x);
        if (kind == FUSEML_OP_ADD)
          static_for<0, 4>([&](auto e) { v[e] = fmaf(sc, x[e], v[e]); });
        else
          static_for<0, 4>([&](auto e) { v[e] = v[e] * x[e]; });
        continue;
      }
      switch (kind) {
        case FUSEML_OP_STORE: store_out4(d.extra[oi], m, n, M, N, v); break;
        case FUSEML_OP_RELU: static_for<0, 4>([&](auto e) { v[e] = max_nan(v[e], 0.0f); }); break;
        case FUSEML_OP_GELU_ERF: gelu_erf_n<4>(v); break;
        case FUSEML_OP_GELU_TANH: gelu_tanh_n<4>(v); break;
        case FUSEML_OP_SIGMOID: sigmoid_n<4>(v); break;
        case FUSEML_OP_SCALE: static_for<0, 4>([&](auto e) { v[e] = v[e] * sc; }); break;
        case FUSEML_OP_ADD_SCALAR: static_for<0, 4>([&](auto e) { v[e] = v[e] + sc; }); break;
        case FUSEML_OP_ADD_SELF: static_for<0, 4>([&](auto e) { v[e] = fmaf(sc, v[e], v[e]); }); break;
        case FUSEML_OP_MUL_SELF: static_for<0, 4>([&](auto e) { v[e] = v[e] * v[e]; }); break;
        default: break;
      }
    }
    if (d.out.ptr != nullptr) store_out4(d.out, m, n, M, N, v);
    if constexpr (RED) reduce(v, m, n, nq);
  });

  // Column partials: over the lanes of the wave that hold the same columns (BN / 4
  // apart), then over the waves through LDS, where every wave has read the K
  // partials by the first barrier.  (With one atomic per column and wave step
  // instead, M / 4 on each column at BN = 64, 824x528x4480 ReLU + three column
  // reductions took 54.6 us for 16.9, 29.1 on the tiled kernels.)
  if (RED && d.reduce_axis == 0) {
#pragma unroll
    for (int sh = BN / 4; sh < 64; sh <<= 1) {
      static_for<0, 4>([&](auto e) {
        col_s[e] += __shfl_xor(col_s[e], sh);
        col_mx[e] = max_nan(col_mx[e], __shfl_xor(col_mx[e], sh));
      });
    }
    lds_barrier();
    float* part_s = reinterpret_cast<float*>(smem);
    float* part_mx = part_s + NW * BN;
    if (lane < BN / 4) {
      static_for<0, 4>([&](auto e) {
        part_s[wave * BN + 4 * lane + e] = col_s[e];
        part_mx[wave * BN + 4 * lane + e] = col_mx[e];
      });
    }
    lds_barrier();
    if (tid < BN && n0 + tid < N) {
      float s = 0.0f, mx = -INFINITY;
      static_for<0, NW>([&](auto w) {
        s += part_s[w * BN + tid];
        mx = max_nan(mx, part_mx[w * BN + tid]);
      });
      put(n0 + tid, s, mx, 1.0f / (float)M);
    }
  }
}

template <int I, typename T>
void launch_ksplit_tile(const fuseml_gemm_desc& d, int index, hipStream_t stream) {
  if constexpr (I < kNumKsplit) {
    constexpr KsplitConfig C = kKsplit[I];
    if (index != I) return launch_ksplit_tile<I + 1, T>(d, index, stream);
    const int64_t tiles = ((d.M + C.bm() - 1) / C.bm()) * ((d.N + C.bn() - 1) / C.bn());
    const dim3 grid((unsigned)tiles), block(C.waves * 64);
    if (d.reduce_mask != 0)
      hipLaunchKernelGGL((gemm_ksplit_kernel<C.mb, C.nb, C.waves, C.depth, T, true>), grid, block, 0, stream, d);
    else
      hipLaunchKernelGGL((gemm_ksplit_kernel<C.mb, C.nb, C.waves, C.depth, T, false>), grid, block, 0, stream, d);
  }
}

template <typename T>
hipError_t launch_ksplit(const fuseml_gemm_desc& d, int index, hipStream_t stream) {
  launch_ksplit_tile<0, T>(d, index, stream);
  return hipGetLastError();
}

}  // namespace fuseml_gemm
