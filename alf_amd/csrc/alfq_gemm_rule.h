// Which kernel a dense product runs on, from its sizes alone (no HIP in here: the rule can be compiled
// and checked by itself).
#pragma once

// direct: split-K kernel on 16 x 16 tiles without LDS staging; the others by their output tile
enum GemmKernel { GEMM_DIRECT, GEMM_TILE_64, GEMM_TILE_32, GEMM_LDS_16_32, GEMM_LDS_16 };

// Tiling policies a context may pick (its autotuner measures them): 0 the estimate-based
// default, 1 the 64 x 64 kernel from one tile per CU, 2 never the 64 x 64 kernel, 3 the
// direct-load kernel up to 512 tiles of 32 x 32.
constexpr int GEMM_POLICIES = 4;

// grid sizes of the tiling policies: direct-load kernel below direct_below tiles of 32 x 32,
// 64 x 64 tiles from big_from tiles of 64 x 64 (with 3/4 of their area inside the product)
struct TilePolicy { long long direct_below, big_from; };
constexpr TilePolicy kTilePolicy[GEMM_POLICIES] = {{256, 512}, {256, 256}, {256, 1LL << 62}, {512, 512}};

inline long long cdivl(long long a, long long b) { return (a + b - 1) / b; }

// Tile shape with the least estimated time: every SIMD of the 256 CUs holds one wave of a
// full round, and a wave's time is proportional to the K it covers (K / KS).
inline GemmKernel gemm_tile_shape(int M, int N, int K, long long b) {
  const long long slots = 256LL * 4;
  struct Opt { GemmKernel kernel; int ks; long long tm, tn; };
  const Opt opts[3] = {{GEMM_TILE_32, 1, 32, 32}, {GEMM_LDS_16_32, 2, 16, 32}, {GEMM_LDS_16, 4, 16, 16}};
  int best = 0;
  double best_cost = 0.0;
  for (int o = 0; o < 3; ++o) {
    const long long waves = 4 * b * cdivl(M, opts[o].tm) * cdivl(N, opts[o].tn);
    const double cost = (double)cdivl(waves, slots) * (double)cdivl(K > 0 ? K : 1, 16 * opts[o].ks);
    if (o == 0 || cost < best_cost) { best = o; best_cost = cost; }
  }
  return opts[best].kernel;
}

// M x N x K, b of them (batch times chains); tile: the LDS tile kernel takes the product's types,
// orders and leading dimensions
inline GemmKernel gemm_kernel_for(int M, int N, int K, long long b, int policy, bool tile) {
  const TilePolicy& p = kTilePolicy[(policy >= 0 && policy < GEMM_POLICIES) ? policy : 0];
  // too few 32 x 32 tiles to fill the device: 16 x 16 tiles, K split over up to 8 waves
  if (cdivl(M, 32) * cdivl(N, 32) * b < p.direct_below) return GEMM_DIRECT;
  // two or more 64 x 64 tiles per CU, at least 3/4 of each tile's area inside the product
  const long long tm = cdivl(M, 64), tn = cdivl(N, 64);
  if (tm * tn * b >= p.big_from && 4LL * M * N >= 3LL * (64 * tm) * (64 * tn) && tile) return GEMM_TILE_64;
  return gemm_tile_shape(M, N, K, b);
}
