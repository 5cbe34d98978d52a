// ksplit_rule.h — the K-split kernel's tiles (gemm_ksplit.h) and what a launch on
// them is priced at.  Plain C++, so that the rules can be compiled on the host.
#pragma once

#include <stdint.h>

namespace fuseml_gemm {

// mb x nb blocks of 16 x 16, waves splitting K, chunks of 128 bytes per row that a
// wave's LDS ring holds.
struct KsplitConfig {
  int mb, nb, waves, depth;
  constexpr int bm() const { return 16 * mb; }
  constexpr int bn() const { return 16 * nb; }
  constexpr int lds_bytes() const {
    const int ring = waves * depth * (bm() + bn()) * 128, part = waves * bm() * bn() * 4;
    return ring > part ? ring : part;
  }
  constexpr int64_t tiles(int64_t M, int64_t N) const {
    return ((M + bm() - 1) / bm()) * ((N + bn() - 1) / bn());
  }
};

constexpr KsplitConfig kKsplit[] = {{1, 1, 8, 2}, {1, 2, 4, 2}, {2, 1, 4, 2}, {2, 2, 4, 2},
                                    {1, 4, 4, 2}, {2, 4, 4, 2}, {4, 2, 4, 2}};
constexpr int kNumKsplit = 7;

// us per block row or column of a tile and 1024 of K, 16-bit operands.
constexpr double kKsplitPerK = 0.36;
// The K-split kernel runs where it is priced at this part of the tiled family or less.
constexpr double kKsplitMargin = 0.9;

// us that fused reductions add on tiles of `bn` columns.  Over columns 2 on either
// side.  Over rows 1, and one atomic per row and column tile, of which those of 32
// rows queue on one line of the output, about 1.5 ns each (16x8128x2544 ReLU + three
// row reductions on 32 columns 17.1 us, 6.5 without).
inline double reduction_us(bool rows, int64_t M, int64_t N, int bn) {
  return rows ? 1.0 + 0.0015 * (double)((N + bn - 1) / bn) * (double)(M < 32 ? M : 32) : 2.0;
}

// The K-split tile with the least priced time (the formula is choose_ksplit's, in
// gemm_epilogue.hip), `per_k` us per block row or column and 1024 of K.
inline int cheapest_ksplit(int64_t M, int64_t N, int64_t K, int cus, double per_k, double* least) {
  int best = -1;
  for (int i = 0; i < kNumKsplit; ++i) {
    const KsplitConfig& c = kKsplit[i];
    const double r = (double)((c.tiles(M, N) + cus - 1) / cus);
    const bool alone = c.lds_bytes() > 80 * 1024;
    const double fixed = alone ? 5.1 : c.mb * c.nb == 2 ? 0.6 : 1.2;
    const double t = (alone ? 1.0 : 3.5) + r * (fixed + per_k * (c.mb + c.nb) * (double)K / 1024.0);
    if (best < 0 || t < *least) {
      best = i;
      *least = t;
    }
  }
  return best;
}

// The K-split tile for fp32 GEMM operands, or -1 where splitting them into bf16
// parts first (fuseml_split_bf16x3, three launches, 10 bytes of traffic per
// element before the GEMM) is the faster way.  The K-split kernel reads 4 bytes
// per element once and splits each fragment in registers, but every tile splits
// its rows anew, at about 0.9 us per block and 1024 of K: it wins while the
// output is small.  Measured (M x N x K, us, split passes and GEMM -> this):
// 64x2048x512 15.9 -> 6.3, 1024x1024x1024 31 -> 22, 1024x1024x4096 80 -> 64,
// 512x4096x256 23.8 -> 21.9, a tie at 2048x1024x1024 (38.0 and 39.0), and
// 2048x2048x512 38.3 -> 52.7 the other way.  Up to 32 rows no row of W is split
// more than twice, and it wins at every N and K (55 shapes of 1 to 32 rows, 256 to
// 131072 columns, K = 256 to 16384, 1.6 to 4.8 times): 1x256x16384 43.7 -> 27.7,
// 16x4096x16384 208.7 -> 44.1, 32x131072x256 106.7 -> 45.9.
// Which sizes it takes does not depend on the device (the padded size is that of the
// tile for 256 CUs, where it was measured), so a caller that asked before the device
// was known has its launch accepted; the tile does.
inline int ksplit_f32(int64_t M, int64_t N, int64_t K, int cus) {
  if (K <= 0) return -1;
  double cost = 0.0;
  const KsplitConfig& c = kKsplit[cheapest_ksplit(M, N, K, 256, 0.9, &cost)];
  const int64_t padded = c.tiles(M, N) * c.bm() * c.bn();
  if (M > 32 && padded > ((int64_t)1 << (K <= 512 ? 21 : 20))) return -1;
  return cheapest_ksplit(M, N, K, cus, 0.9, &cost);
}

}  // namespace fuseml_gemm
