// FP64 MFMA GEMM for gfx950: real x complex and complex x complex products with
// fused diagonal scalings, gathers and conjugation.
//
// Tiling: a workgroup of 4 waves computes a (16 WM) x (16 WN) complex output tile;
// the waves are arranged WM x WN x KS, so with KS > 1 the waves of one tile split
// K and their partial tiles are summed through LDS in a fixed order (the result
// does not depend on scheduling).  Each wave holds a 16 x 16 sub-tile as two
// (re, im) v_mfma_f64_16x16x4f64 accumulators (three for complex x complex).  K advances in stages of 16 KS
// through LDS, where the operands are split into real and imaginary planes so each
// MFMA consumes one plane; a complex x complex product costs 3 MFMAs per k-step of 4 (3M:
// Ar Br, Ai Bi and (Ar + Ai)(Br + Bi), combined after the K loop), a real x complex one 2.
// The host picks the tile shape per launch: at Ndim = 256 a 32 x 32 tiling leaves most of
// the 256 CUs idle, a 16 x 16 tiling with KS = 4 fills them with a quarter of the per-wave K.
//
// gemm_tile_kernel takes the same products where the grid fills the device without a K split; the
// 32 x 32 tiles here are left to real products, FP32 operands in other orders than N x N and matrices
// past 32-bit offsets.  alfq_gemm_rule.h holds the choice between the kernels.
// These kernels carry every dense product of the sweep:
//   * hopping wraps  G <- D exp(-dtau T) G exp(dtau T) D^-1       (real T: 2 MFMA/step)
//   * UDV chain      U <- D exp(-dtau T) U,  U <- exp(-dtau T) conj(D) U
//   * delayed-update flush  G += X Y^T
//   * QR trailing updates / Q formation / TRMM / CGR products
#include "alfq_chain.h"
#include "alfq_common.h"
#include "alfq_gemm_rule.h"

namespace {

constexpr int NT = 256;

// Every MFMA kernel here is bounded to two waves per SIMD at least (second argument of
// __launch_bounds__): with 256 registers or fewer the compiler keeps the accumulators in VGPRs,
// without the bound it puts them in AGPRs and moves them there and back around every K stage.

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// The two MFMA arithmetics of the kernels below (GemmArgs::prec 0 and 1).  Both take A as
// lane = row + 16 k and B as lane = column + 16 k (k = 0..3); they differ in where the
// 16 x 16 result lands:
//   FP64 v_mfma_f64_16x16x4f64: D(i, j) in lane j + 16 (i % 4), register i / 4
//   FP32 v_mfma_f32_16x16x4f32: D(i, j) in lane j + 16 (i / 4), register i % 4
// With FP32 the operands are rounded to float when staged and the products accumulate in
// float; scalings, alpha and beta are applied to the result in double.
template <bool F32> struct Mma;
template <> struct Mma<false> {
  typedef double E;
  typedef v4d Acc;
  __device__ __forceinline__ static Acc mac(E a, E b, Acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  __device__ __forceinline__ static int row(int r, int lk) { return 4 * r + lk; }
};
template <> struct Mma<true> {
  typedef float E;
  typedef v4f Acc;
  __device__ __forceinline__ static Acc mac(E a, E b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  __device__ __forceinline__ static int row(int r, int lk) { return 4 * lk + r; }
};

// moves every operand pointer to the arena of the chain bz / batch; true when the product is
// the identity slice of a chain beyond its own Ltrot (the hopping operand is the identity) and
// the workgroup can write its tile as a copy of the other operand (identity_tile)
__device__ __forceinline__ bool chain_operands(GemmArgs& g, int bz) {
  if (g.nchain <= 1) return false;
  const long long off = (long long)(bz / (g.batch > 1 ? g.batch : 1)) * g.cstride;
  auto mv = [off](auto p) { return p ? (decltype(p))((const char*)p + off) : p; };
  g.A = mv(g.A); g.B = mv(g.B); g.C = (void*)mv((const char*)g.C);
  g.rs = mv(g.rs); g.cs = mv(g.cs); g.bs = mv(g.bs); g.rs_real = mv(g.rs_real);
  g.amap = mv(g.amap); g.bmap = mv(g.bmap); g.kdev = mv(g.kdev);
  if (g.lz && g.slice >= g.lz[bz / (g.batch > 1 ? g.batch : 1)]) {
    if (g.hop_side == 1) g.A = g.ident;
    else if (g.hop_side == 2) g.B = g.ident;
    // the identity is K x K: M = K when it is opA, N = K when it is opB
    return ((g.hop_side == 1 && g.M == g.K) || (g.hop_side == 2 && g.N == g.K)) && g.batch <= 1 && !g.amap &&
           !g.bmap && !g.kdev;
  }
  return false;
}

// The tile [i0, i0 + tm) x [j0, j0 + tn) of C = alpha rs (I X) cs + beta C when the hopping
// operand is the identity: X = diag(bs) opB for hop_side 1, opA diag(bs) for hop_side 2, each element
// with the epilogue of the product.  The product's value without its MFMA work: in FP64 the
// MFMA product with an identity adds only zeros, and with FP32 operands (prec 1) the copy
// keeps the double values the product would have rounded.
__device__ void identity_tile(const GemmArgs& g, int i0, int j0, int tm, int tn, int tid, int nt) {
  cplx* C = (cplx*)g.C;
  for (int e = tid; e < tm * tn; e += nt) {
    const int i = i0 + e % tm, j = j0 + e / tm;
    if (i >= g.M || j >= g.N) continue;
    cplx v;
    if (g.hop_side == 1) {
      const long long off = (g.opB == OP_N) ? i + (long long)j * g.ldb : j + (long long)i * g.ldb;
      v = g.b_cplx ? ((const cplx*)g.B)[off] : make_double2(((const double*)g.B)[off], 0.0);
      if (g.opB == OP_C) v.y = -v.y;
      if (g.bs) v = cmul(g.bs[i], v);
    } else {
      const long long off = (g.opA == OP_N) ? i + (long long)j * g.lda : j + (long long)i * g.lda;
      v = g.a_cplx ? ((const cplx*)g.A)[off] : make_double2(((const double*)g.A)[off], 0.0);
      if (g.opA == OP_C) v.y = -v.y;
      if (g.bs) v = cmul(v, g.bs[j]);
    }
    v = cmul(g.alpha, v);
    if (g.rs) v = cmul(g.rs[i], v);
    if (g.rs_real) v = cscale(v, g.rs_real[i]);
    if (g.cs) v = cmul(v, g.cs[j]);
    const long long o = i + (long long)j * g.ldc;
    if (g.beta.x != 0.0 || g.beta.y != 0.0) v = cadd(v, cmul(g.beta, C[o]));
    C[o] = v;
  }
}

// One K stage of an LDS-tiled kernel's operands, held in registers from its global loads to
// its LDS stores.  Gather indices and row scales are read first and every data load is then
// issued back to back: no wait on one load sits between the issue of two others (a wait at
// the join of an optional map lookup would otherwise serialise the whole stage).
// Conjugation is applied when the stage is stored; the row scales of opB (one per k) go to
// an LDS vector of the stage and are applied to the B fragments at multiplication time.
template <int TM, int TN, int BK, bool A_CPLX, bool B_CPLX>
struct Stage {
  static constexpr int LA = TM * BK / NT, LB = BK * TN / NT;   // elements per thread
  static_assert(LA >= 1 && LB >= 1 && BK <= NT, "a stage covers the workgroup");
  double a_re[LA], a_im[LA], b_re[LB], b_im[LB];
  cplx scl;                 // bs(k0 + tid) for tid < BK

  __device__ __forceinline__ static void a_index(const GemmArgs& g, int tid, int p, int& i, int& kk) {
    const int idx = tid + NT * p;
    if (g.opA == OP_N) { i = idx % TM; kk = idx / TM; } else { kk = idx % BK; i = idx / BK; }
  }
  __device__ __forceinline__ static void b_index(const GemmArgs& g, int tid, int p, int& kk, int& j) {
    const int idx = tid + NT * p;
    if (g.opB == OP_N) { kk = idx % BK; j = idx / BK; } else { j = idx % TN; kk = idx / TN; }
  }

  __device__ __forceinline__ void load(const GemmArgs& g, const void* A, const void* B, int i0, int j0,
                                       int K, int k0, int tid) {
    int ka[LA], kb[LB];
#pragma unroll
    for (int p = 0; p < LA; ++p) {
      int i, kk;
      a_index(g, tid, p, i, kk);
      ka[p] = (i0 + i < g.M && k0 + kk < K) ? k0 + kk : -1;
    }
#pragma unroll
    for (int p = 0; p < LB; ++p) {
      int kk, j;
      b_index(g, tid, p, kk, j);
      kb[p] = (k0 + kk < K && j0 + j < g.N) ? k0 + kk : -1;
    }
    if (g.bs) scl = (tid < BK && k0 + tid < K) ? g.bs[k0 + tid] : make_double2(0.0, 0.0);
    if (g.amap) {
#pragma unroll
      for (int p = 0; p < LA; ++p) if (ka[p] >= 0) ka[p] = g.amap[ka[p]];
    }
    if (g.bmap) {
#pragma unroll
      for (int p = 0; p < LB; ++p) if (kb[p] >= 0) kb[p] = g.bmap[kb[p]];
    }
#pragma unroll
    for (int p = 0; p < LA; ++p) {
      int i, kk;
      a_index(g, tid, p, i, kk);
      const long long gi = i0 + i;
      double re = 0.0, im = 0.0;
      if (ka[p] >= 0) {
        const long long off = (g.opA == OP_N) ? gi + (long long)ka[p] * g.lda : ka[p] + gi * g.lda;
        if (A_CPLX) {
          const cplx v = ((const cplx*)A)[off];
          re = v.x;
          im = v.y;
        } else {
          re = ((const double*)A)[off];
        }
      }
      a_re[p] = re;
      a_im[p] = im;
    }
#pragma unroll
    for (int p = 0; p < LB; ++p) {
      int kk, j;
      b_index(g, tid, p, kk, j);
      const long long gj = j0 + j;
      double re = 0.0, im = 0.0;
      if (kb[p] >= 0) {
        const long long off = (g.opB == OP_N) ? kb[p] + gj * g.ldb : gj + (long long)kb[p] * g.ldb;
        if (g.b_cplx) {
          const cplx v = ((const cplx*)B)[off];
          re = v.x;
          im = v.y;
        } else {
          re = ((const double*)B)[off];
        }
      }
      b_re[p] = re;
      b_im[p] = im;
    }
  }

  template <typename E>
  __device__ __forceinline__ void store(const GemmArgs& g, int tid, E (*As_re)[TM + 1], E (*As_im)[TM + 1],
                                        E (*Bs_re)[TN + 1], E (*Bs_im)[TN + 1], cplx* bsl) const {
#pragma unroll
    for (int p = 0; p < LA; ++p) {
      int i, kk;
      a_index(g, tid, p, i, kk);
      As_re[kk][i] = (E)a_re[p];
      if (A_CPLX) As_im[kk][i] = (E)((g.opA == OP_C) ? -a_im[p] : a_im[p]);
    }
#pragma unroll
    for (int p = 0; p < LB; ++p) {
      int kk, j;
      b_index(g, tid, p, kk, j);
      Bs_re[kk][j] = (E)b_re[p];
      if (B_CPLX) Bs_im[kk][j] = (E)((g.opB == OP_C) ? -b_im[p] : b_im[p]);
    }
    if (g.bs && tid < BK) bsl[tid] = scl;
  }
};

// B fragment times the row scale of its k (the scales of a stage sit in LDS)
template <typename E>
__device__ __forceinline__ void scale_b(const cplx s, E& re, E& im) {
  const E r2 = re * (E)s.x - im * (E)s.y;
  im = re * (E)s.y + im * (E)s.x;
  re = r2;
}

template <bool A_CPLX, bool B_CPLX, int WM, int WN, bool F32>
__global__ __launch_bounds__(NT, 2) void gemm_kernel(GemmArgs g) {
  typedef Mma<F32> M;
  typedef typename M::E E;
  constexpr int KS = 4 / (WM * WN);
  constexpr int TM = 16 * WM, TN = 16 * WN, BK = 16 * KS;
  constexpr int LA = TM * BK / NT, LB = BK * TN / NT;   // elements per thread per stage
  static_assert(WM * WN * KS == 4 && LA >= 1 && LB >= 1, "4 waves per tile");
  __shared__ E As_re[BK][TM + 1];
  __shared__ E As_im[A_CPLX ? BK : 1][TM + 1];
  __shared__ E Bs_re[BK][TN + 1];
  __shared__ E Bs_im[B_CPLX ? BK : 1][TN + 1];
  __shared__ cplx red[KS > 1 ? KS - 1 : 1][KS > 1 ? TM * TN : 1];
  __shared__ cplx bsl[BK];

  const int tid = threadIdx.x;
  const int i0 = blockIdx.x * TM;
  const int j0 = blockIdx.y * TN;
  if (chain_operands(g, blockIdx.z)) { identity_tile(g, i0, j0, TM, TN, tid, blockDim.x); return; }
  const int z = blockIdx.z % (g.batch > 1 ? g.batch : 1);
  int K = g.K;
  if (g.kdev) {
    int kd = *g.kdev;
    K = kd < K ? kd : K;
  }
  if (K <= 0 && g.beta.x == 1.0 && g.beta.y == 0.0) return;  // nothing to add

  const long long za = g.batch > 1 ? z * g.strideA : 0, zb = g.batch > 1 ? z * g.strideB : 0;
  const void* A = A_CPLX ? (const void*)((const cplx*)g.A + za) : (const void*)((const double*)g.A + za);
  const void* B = g.b_cplx ? (const void*)((const cplx*)g.B + zb) : (const void*)((const double*)g.B + zb);
  cplx* C = (cplx*)g.C + (g.batch > 1 ? z * g.strideC : 0);

  const int wave = tid >> 6, lane = tid & 63;
  const int wm = wave % WM, wn = (wave / WM) % WN, ks = wave / (WM * WN);
  const int wr = 16 * wm, wc = 16 * wn;
  const int lr = lane & 15, lk = lane >> 4;

  typename M::Acc acc_re = {0, 0, 0, 0};
  typename M::Acc acc_im = {0, 0, 0, 0};
  typename M::Acc acc_t2 = {0, 0, 0, 0};   // complex x complex: Ai Bi (3M)

  Stage<TM, TN, BK, A_CPLX, B_CPLX> st;

  if (K > 0) st.load(g, A, B, i0, j0, K, 0, tid);
  for (int k0 = 0; k0 < K; k0 += BK) {
    st.store(g, tid, As_re, As_im, Bs_re, Bs_im, bsl);
    __syncthreads();
    if (k0 + BK < K) st.load(g, A, B, i0, j0, K, k0 + BK, tid);   // in flight during this stage's MFMAs
#pragma unroll
    for (int kq = 0; kq < 16; kq += 4) {
      const int kk = 16 * ks + kq;
      const E a_re = As_re[kk + lk][wr + lr];
      E b_re = Bs_re[kk + lk][wc + lr];
      E b_im = B_CPLX ? Bs_im[kk + lk][wc + lr] : (E)0;
      if (B_CPLX && g.bs) scale_b(bsl[kk + lk], b_re, b_im);
      acc_re = M::mac(a_re, b_re, acc_re);
      if (A_CPLX && B_CPLX) {
        // 3M: acc_t2 = Ai Bi, acc_im = (Ar + Ai)(Br + Bi), combined after the K loop
        const E a_im = As_im[kk + lk][wr + lr];
        acc_t2 = M::mac(a_im, b_im, acc_t2);
        acc_im = M::mac(a_re + a_im, b_re + b_im, acc_im);
      } else if (B_CPLX) {
        acc_im = M::mac(a_re, b_im, acc_im);
      } else if (A_CPLX) {
        const E a_im = As_im[kk + lk][wr + lr];
        acc_im = M::mac(a_im, b_re, acc_im);
      }
    }
    __syncthreads();
  }
  if (A_CPLX && B_CPLX) {
    acc_im = acc_im - acc_re - acc_t2;
    acc_re = acc_re - acc_t2;
  }

  // ---- epilogue: register r of a lane holds row wr + M::row(r, lane / 16) of column
  //      wc + lane % 16 ----
  if (KS > 1) {
    // waves ks >= 1 park their partial tiles; the ks = 0 waves add them in order ks = 1, 2, ...
    if (ks > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[ks - 1][(wr + M::row(r, lk)) + TM * (wc + lr)] = make_double2(acc_re[r], acc_im[r]);
    }
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int q = 0; q < KS - 1; ++q) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const cplx p = red[q][(wr + M::row(r, lk)) + TM * (wc + lr)];
        acc_re[r] += p.x;
        acc_im[r] += p.y;
      }
    }
  }
  const int gj = j0 + wc + lr;
  if (gj >= g.N) return;
  cplx csj = g.cs ? g.cs[gj] : make_double2(1.0, 0.0);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int gi = i0 + wr + M::row(r, lk);
    if (gi >= g.M) continue;
    cplx v = make_double2(acc_re[r], (A_CPLX || B_CPLX) ? acc_im[r] : 0.0);
    v = cmul(g.alpha, v);
    if (g.rs) v = cmul(g.rs[gi], v);
    if (g.rs_real) v = cscale(v, g.rs_real[gi]);
    if (g.cs) v = cmul(v, csj);
    const long long off = gi + (long long)gj * g.ldc;
    if (g.beta.x != 0.0 || g.beta.y != 0.0) v = cadd(v, cmul(g.beta, C[off]));
    C[off] = v;
  }
}

// Tile kernel for grids that fill the device (batched chains, large lattices): a workgroup of
// 2 x 2 waves owns a (32 MB) x (32 NB) complex tile, each wave MB x NB blocks of 16 x 16.
//
// What bounds it is the FP64 matrix rate (78.6 TF/s, reached by a loop of independent
// v_mfma_f64_16x16x4f64 whose accumulators stay in VGPRs), so everything else has to stay out of
// the K loop: the storage order of both operands and their types are template parameters, edges
// are clamped addresses instead of branches (a clamped row or column is not stored, a clamped k
// is selected to zero), and the gather maps and row scales are read one stage ahead of the data
// they serve.  K stages of 16 go global -> registers -> LDS, double-buffered, one barrier per
// stage, with the next stage's loads in flight during this stage's products.
// LDS rows hold one k of the tile, complex entries as (re, im) pairs read by one ds_read_b128;
// the row pads keep both the k-fastest stores and the fragment reads free of bank conflicts.
// The fragments enter the MFMA exchanged (opB as its first operand), so that the 16 lanes of a
// result row run along a column of C: 256-byte segments instead of 64.
//
// 256 chains of n = 256, per launch: real x complex wraps 430 -> 304 us (56 TF/s), with row scales 353
// and 382 us (49 and 45 TF/s), complex x complex 572 -> 475 us (54 TF/s of issued products), gathered
// or scaled 515 to 555; one product of n = 1024 issues at 61 TF/s.  The
// kernel this replaces chose orders, gathers and edges by branches inside the K stage.  128 x 64
// tiles, three waves per SIMD and K stages of 32 measured the same or slower.
//
// AKF / BKF: k is the fastest index in memory (opA = T, C / opB = N).  With both operands complex
// the product is three real ones (3M): Ar Br, Ai Bi, (Ar + Ai)(Br + Bi).
template <bool CPLX, bool F32> struct TileElem;
template <> struct TileElem<false, false> { typedef double T; };
template <> struct TileElem<true, false> { typedef double2 T; };
template <> struct TileElem<false, true> { typedef float T; };
template <> struct TileElem<true, true> { typedef float2 T; };

template <bool A_CPLX, bool B_CPLX, bool AKF, bool BKF, bool EXTRA, bool F32, int MB, int NB>
__global__ __launch_bounds__(NT, 2) void gemm_tile_kernel(GemmArgs g) {
  typedef Mma<F32> M;
  typedef typename M::E E;
  typedef typename TileElem<A_CPLX, F32>::T TA;
  typedef typename TileElem<B_CPLX, F32>::T TB;
  typedef typename TileElem<A_CPLX, false>::T GA;          // elements in memory
  typedef typename TileElem<B_CPLX, false>::T GB;
  constexpr int TM = 32 * MB, TN = 32 * NB, BK = 16;
  constexpr int LA = TM * BK / NT, LB = TN * BK / NT;     // elements per thread and stage
  // row pitch in elements: an odd number of 16-byte units for the 16-byte rows; for 8-byte rows
  // 16 entries more than a multiple of 32, so the two k rows of a half-wave read meet other banks
  constexpr int PA = A_CPLX ? TM + 1 : TM + (AKF ? 2 : 16), PB = B_CPLX ? TN + 1 : TN + (BKF ? 2 : 16);
  __shared__ __align__(16) TA As[2][BK][PA];
  __shared__ __align__(16) TB Bs[2][BK][PB];

  const int tid = threadIdx.x;
  int bx, by, bz;
  xcd_order(bx, by, bz);
  const int i0 = bx * TM, j0 = by * TN;
  if (chain_operands(g, bz)) { identity_tile(g, i0, j0, TM, TN, tid, blockDim.x); return; }
  const int z = bz % (g.batch > 1 ? g.batch : 1);
  int K = g.K;
  if (g.kdev) {
    const int kd = *g.kdev;
    K = kd < K ? kd : K;
  }
  if (K <= 0 && g.beta.x == 1.0 && g.beta.y == 0.0) return;  // nothing to add
  const GA* const A = (const GA*)g.A + (g.batch > 1 ? z * g.strideA : 0);
  const GB* const B = (const GB*)g.B + (g.batch > 1 ? z * g.strideB : 0);
  cplx* C = (cplx*)g.C + (g.batch > 1 ? z * g.strideC : 0);
  // the row scales of opB multiply opB, or the columns of opA when only opA is complex
  constexpr bool SCALE_A = A_CPLX && !B_CPLX;
  const double ca = g.opA == OP_C ? -1.0 : 1.0, cb = g.opB == OP_C ? -1.0 : 1.0;

  // this thread's elements of a stage: k offset and tile index of element p
  auto a_k = [&](int p) { return AKF ? tid % BK : (tid + NT * p) / TM; };
  auto a_i = [&](int p) { return AKF ? tid / BK + (NT / BK) * p : (tid + NT * p) % TM; };
  auto b_k = [&](int p) { return BKF ? tid % BK : (tid + NT * p) / TN; };
  auto b_j = [&](int p) { return BKF ? tid / BK + (NT / BK) * p : (tid + NT * p) % TN; };
  constexpr int KA = AKF ? 1 : LA, KB = BKF ? 1 : LB;     // distinct k of a thread per stage
  const int kmax = K > 0 ? K - 1 : 0;
  auto clampk = [&](int k) { return k < kmax ? k : kmax; };
  // element offsets inside a stage; the stage's own offset k0 is added to the uniform base
  // pointer, so a full stage costs no address arithmetic (tile_kernel_takes keeps them in 32 bits)
  unsigned ao[LA], bo[LB];
#pragma unroll
  for (int p = 0; p < LA; ++p) {
    const int i = i0 + a_i(p) < g.M ? i0 + a_i(p) : g.M - 1;
    ao[p] = AKF ? (unsigned)i * (unsigned)g.lda : (unsigned)i;
    if (!EXTRA) ao[p] += AKF ? (unsigned)a_k(p) : (unsigned)a_k(p) * (unsigned)g.lda;
  }
#pragma unroll
  for (int p = 0; p < LB; ++p) {
    const int j = j0 + b_j(p) < g.N ? j0 + b_j(p) : g.N - 1;
    bo[p] = BKF ? (unsigned)j * (unsigned)g.ldb : (unsigned)j;
    if (!EXTRA) bo[p] += BKF ? (unsigned)b_k(p) : (unsigned)b_k(p) * (unsigned)g.ldb;
  }
  // EXTRA: gathered k of the next stage's elements, read one stage ahead
  unsigned ka[EXTRA ? KA : 1], kb[EXTRA ? KB : 1];
  auto load_k = [&](int k0) {
    if constexpr (EXTRA) {
#pragma unroll
      for (int p = 0; p < KA; ++p) { const int k = clampk(k0 + a_k(p)); ka[p] = g.amap ? g.amap[k] : k; }
#pragma unroll
      for (int p = 0; p < KB; ++p) { const int k = clampk(k0 + b_k(p)); kb[p] = g.bmap ? g.bmap[k] : k; }
    }
  };
  GA av[LA];
  GB bv[LB];
  cplx sv[EXTRA ? (SCALE_A ? KA : KB) : 1];
  auto load = [&](int k0) {
    if constexpr (EXTRA) {
#pragma unroll
      for (int p = 0; p < LA; ++p) {
        const unsigned k = ka[AKF ? 0 : p];
        av[p] = A[AKF ? ao[p] + k : ao[p] + k * (unsigned)g.lda];
      }
#pragma unroll
      for (int p = 0; p < LB; ++p) {
        const unsigned k = kb[BKF ? 0 : p];
        bv[p] = B[BKF ? bo[p] + k : bo[p] + k * (unsigned)g.ldb];
      }
      if (g.bs) {
#pragma unroll
        for (int p = 0; p < (SCALE_A ? KA : KB); ++p) sv[p] = g.bs[clampk(k0 + (SCALE_A ? a_k(p) : b_k(p)))];
      }
    } else {
      const GA* const Ak = A + (AKF ? (long long)k0 : (long long)k0 * g.lda);
      const GB* const Bk = B + (BKF ? (long long)k0 : (long long)k0 * g.ldb);
      if (k0 + BK <= K) {
#pragma unroll
        for (int p = 0; p < LA; ++p) av[p] = Ak[ao[p]];
#pragma unroll
        for (int p = 0; p < LB; ++p) bv[p] = Bk[bo[p]];
      } else {
        const int kl = kmax - k0;                         // last k of the partial stage
#pragma unroll
        for (int p = 0; p < LA; ++p) {
          const unsigned over = a_k(p) > kl ? a_k(p) - kl : 0;
          av[p] = Ak[ao[p] - (AKF ? over : over * (unsigned)g.lda)];
        }
#pragma unroll
        for (int p = 0; p < LB; ++p) {
          const unsigned over = b_k(p) > kl ? b_k(p) - kl : 0;
          bv[p] = Bk[bo[p] - (BKF ? over : over * (unsigned)g.ldb)];
        }
      }
    }
  };
  auto store = [&](int k0, int buf) {
    if (k0 + BK > K) {
      // the partial last stage: elements beyond K are zero
#pragma unroll
      for (int p = 0; p < LA; ++p)
        if (k0 + a_k(p) >= K) av[p] = GA{};
#pragma unroll
      for (int p = 0; p < LB; ++p)
        if (k0 + b_k(p) >= K) bv[p] = GB{};
    }
#pragma unroll
    for (int p = 0; p < LA; ++p) {
      if constexpr (A_CPLX) {
        cplx v = av[p];
        if (AKF) v.y *= ca;
        if constexpr (EXTRA && SCALE_A) if (g.bs) v = cmul(v, sv[AKF ? 0 : p]);
        As[buf][a_k(p)][a_i(p)] = TA{(E)v.x, (E)v.y};
      } else {
        As[buf][a_k(p)][a_i(p)] = (E)av[p];
      }
    }
#pragma unroll
    for (int p = 0; p < LB; ++p) {
      if constexpr (B_CPLX) {
        cplx v = bv[p];
        if (!BKF) v.y *= cb;
        if constexpr (EXTRA && !SCALE_A) if (g.bs) v = cmul(v, sv[BKF ? 0 : p]);
        Bs[buf][b_k(p)][b_j(p)] = TB{(E)v.x, (E)v.y};
      } else {
        Bs[buf][b_k(p)][b_j(p)] = (E)bv[p];
      }
    }
  };

  const int wave = tid >> 6, lane = tid & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int wr = 16 * MB * (wave & 1), wc = 16 * NB * (wave >> 1);
  constexpr bool M3 = A_CPLX && B_CPLX;
  typename M::Acc acc_re[MB][NB], acc_im[MB][NB], acc_t2[M3 ? MB : 1][M3 ? NB : 1];
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      acc_re[a][b] = typename M::Acc{0, 0, 0, 0};
      acc_im[a][b] = typename M::Acc{0, 0, 0, 0};
      if (M3) acc_t2[M3 ? a : 0][M3 ? b : 0] = typename M::Acc{0, 0, 0, 0};
    }

  if (K > 0) {
    load_k(0);
    load(0);
    load_k(BK);
  }
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += BK, buf ^= 1) {
    store(k0, buf);
    __syncthreads();
    if (k0 + BK < K) {
      load(k0 + BK);
      load_k(k0 + 2 * BK);
    }
    // the fragments of the next k-step are read while this one's products issue (left to itself
    // the compiler waits for every k-step's reads in front of its first product)
    TA fa[2][MB];
    TB fb[2][NB];
    auto frag = [&](int kq) {
#pragma unroll
      for (int a = 0; a < MB; ++a) fa[(kq >> 2) & 1][a] = As[buf][kq + lk][wr + 16 * a + lr];
#pragma unroll
      for (int b = 0; b < NB; ++b) fb[(kq >> 2) & 1][b] = Bs[buf][kq + lk][wc + 16 * b + lr];
    };
    frag(0);
#pragma unroll
    for (int kq = 0; kq < BK; kq += 4) {
      const int f = (kq >> 2) & 1;
      if (kq + 4 < BK) frag(kq + 4);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          if constexpr (M3) {
            acc_re[a][b] = M::mac(fb[f][b].x, fa[f][a].x, acc_re[a][b]);
            acc_t2[a][b] = M::mac(fb[f][b].y, fa[f][a].y, acc_t2[a][b]);
            acc_im[a][b] = M::mac(fb[f][b].x + fb[f][b].y, fa[f][a].x + fa[f][a].y, acc_im[a][b]);
          } else if constexpr (B_CPLX) {
            acc_re[a][b] = M::mac(fb[f][b].x, fa[f][a], acc_re[a][b]);
            acc_im[a][b] = M::mac(fb[f][b].y, fa[f][a], acc_im[a][b]);
          } else {
            acc_re[a][b] = M::mac(fb[f][b], fa[f][a].x, acc_re[a][b]);
            acc_im[a][b] = M::mac(fb[f][b], fa[f][a].y, acc_im[a][b]);
          }
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // register r of a lane holds column M::row(r, lane / 16) and row lane % 16 of its block
#pragma unroll
  for (int a = 0; a < MB; ++a) {
    const int gi = i0 + wr + 16 * a + lr;
    if (gi >= g.M) continue;
    cplx rsi = g.rs ? g.rs[gi] : make_double2(1.0, 0.0);
    if (g.rs_real) rsi = cscale(rsi, g.rs_real[gi]);
    rsi = cmul(g.alpha, rsi);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gj = j0 + wc + 16 * b + M::row(r, lk);
        if (gj >= g.N) continue;
        double re = acc_re[a][b][r], im = acc_im[a][b][r];
        if constexpr (M3) {
          const double t2 = acc_t2[a][b][r];
          im = im - re - t2;
          re = re - t2;
        }
        cplx v = cmul(rsi, make_double2(re, im));
        if (g.cs) v = cmul(v, g.cs[gj]);
        const long long off = gi + (long long)gj * g.ldc;
        if (g.beta.x != 0.0 || g.beta.y != 0.0) v = cadd(v, cmul(g.beta, C[off]));
        C[off] = v;
      }
    }
  }
}

// Delayed-update flush G += X Y^T of rank m <= CHAIN_BLOCK_KMAX (the block kernel's round).  A
// workgroup owns a 64 x 64 tile of one chain's G; the tile itself, in the layout of the product,
// and the first 16 columns of X (for the tile's rows) and Y (for its columns) are requested at
// the start, the next 16 columns while the ones before them are multiplied, and G is written once.
// Bound by the traffic of G (2 x 16 n^2 bytes per chain): 256 chains of n = 256 take 76 us for 537 MB
// in full rounds (7.1 TB/s), 60 -> 49 us over the first sweeps of a random start.  X Y^T is three real
// products (3M) here, where the round's other products are four: with four the error of G over a
// slice of 16 x 16 is the same (8.6e-15 against 8.8e-15, mean of 16 chains; 1.8e-14 when X came from
// W = C D^T), for X and Y are of the size of G's columns and nothing large cancels.
constexpr int FL_T = 64, FL_C = 16;
__global__ __launch_bounds__(NT, 2) void flush_kernel(cplx* G, const cplx* X, const cplx* Y, const int* mdev,
                                                      int n, int kmax, long long cs) {
  typedef Mma<false> M;
  __shared__ cplx Xs[2][FL_C][FL_T + 1], Ys[2][FL_C][FL_T + 1];
  int bx, by, bz;
  xcd_order(bx, by, bz);
  G = chain_ptr_at(G, cs, bz);
  X = chain_ptr_at(X, cs, bz);
  Y = chain_ptr_at(Y, cs, bz);
  mdev = chain_ptr_at(mdev, cs, bz);
  int m = *mdev;
  m = m < kmax ? m : kmax;
  if (m <= 0) return;
  const int tid = threadIdx.x;
  const int i0 = bx * FL_T, j0 = by * FL_T;
  const int wave = tid >> 6, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int wr = 32 * (wave & 1), wc = 32 * (wave >> 1);
  const int li = tid & 63, lkb = tid >> 6;   // operand rows: index li, columns k = lkb + 4 p
  const int xi = i0 + li < n ? i0 + li : n - 1, yi = j0 + li < n ? j0 + li : n - 1;

  cplx xv[FL_C / 4], yv[FL_C / 4];
  auto load = [&](int k0) {
#pragma unroll
    for (int p = 0; p < FL_C / 4; ++p) {
      const int k = k0 + lkb + 4 * p < m ? k0 + lkb + 4 * p : m - 1;
      xv[p] = X[xi + (long long)k * n];
      yv[p] = Y[yi + (long long)k * n];
    }
  };
  load(0);
  cplx gv[2][2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gi = i0 + wr + 16 * a + lr, gj = j0 + wc + 16 * b + M::row(r, lk);
        gv[a][b][r] = make_double2(0.0, 0.0);
        if (gi < n && gj < n) gv[a][b][r] = G[gi + (long long)gj * n];
      }
  v4d acc_re[2][2], acc_im[2][2], acc_t2[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc_re[a][b] = acc_im[a][b] = acc_t2[a][b] = v4d{0, 0, 0, 0};
  int buf = 0;
  for (int k0 = 0; k0 < m; k0 += FL_C, buf ^= 1) {
#pragma unroll
    for (int p = 0; p < FL_C / 4; ++p) {
      const bool live = k0 + lkb + 4 * p < m;
      Xs[buf][lkb + 4 * p][li] = live ? xv[p] : make_double2(0.0, 0.0);
      Ys[buf][lkb + 4 * p][li] = live ? yv[p] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    if (k0 + FL_C < m) load(k0 + FL_C);
    const int kn = m - k0 < FL_C ? m - k0 : FL_C;
    for (int kq = 0; kq < kn; kq += 4) {
      cplx fa[2], fb[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) fa[a] = Xs[buf][kq + lk][wr + 16 * a + lr];
#pragma unroll
      for (int b = 0; b < 2; ++b) fb[b] = Ys[buf][kq + lk][wc + 16 * b + lr];
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          // operands exchanged: the 16 lanes of a result row run along a column of G
          acc_re[a][b] = M::mac(fb[b].x, fa[a].x, acc_re[a][b]);
          acc_t2[a][b] = M::mac(fb[b].y, fa[a].y, acc_t2[a][b]);
          acc_im[a][b] = M::mac(fb[b].x + fb[b].y, fa[a].x + fa[a].y, acc_im[a][b]);
        }
    }
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gi = i0 + wr + 16 * a + lr, gj = j0 + wc + 16 * b + M::row(r, lk);
        const double re = acc_re[a][b][r], t2 = acc_t2[a][b][r];
        if (gi < n && gj < n)
          G[gi + (long long)gj * n] =
              make_double2(gv[a][b][r].x + (re - t2), gv[a][b][r].y + (acc_im[a][b][r] - re - t2));
      }
}

inline unsigned gemm_zdim(const GemmArgs& g) {
  return (unsigned)((g.batch > 1 ? g.batch : 1) * (g.nchain > 1 ? g.nchain : 1));
}

template <int WM, int WN, bool F32>
void launch_shape_p(const GemmArgs& g, hipStream_t s) {
  dim3 grid((unsigned)cdivl(g.M, 16 * WM), (unsigned)cdivl(g.N, 16 * WN), gemm_zdim(g));
  const bool bc = g.b_cplx || g.bs != nullptr;
  if (g.a_cplx && bc) hipLaunchKernelGGL((gemm_kernel<true, true, WM, WN, F32>), grid, dim3(NT), 0, s, g);
  else if (g.a_cplx) hipLaunchKernelGGL((gemm_kernel<true, false, WM, WN, F32>), grid, dim3(NT), 0, s, g);
  else if (bc) hipLaunchKernelGGL((gemm_kernel<false, true, WM, WN, F32>), grid, dim3(NT), 0, s, g);
  else hipLaunchKernelGGL((gemm_kernel<false, false, WM, WN, F32>), grid, dim3(NT), 0, s, g);
}
template <int WM, int WN>
void launch_shape(const GemmArgs& g, hipStream_t s) {
  if (g.prec) launch_shape_p<WM, WN, true>(g, s);
  else launch_shape_p<WM, WN, false>(g, s);
}

// The tile kernel takes every product with exactly one or two complex operands whose elements
// are addressable with 32-bit offsets; FP32 operands only in the order of the hopping wraps (N x N).
bool tile_kernel_takes(const GemmArgs& g) {
  if (!g.a_cplx && !g.b_cplx) return false;
  const long long ea = (long long)g.lda * (g.opA == OP_N ? g.K : g.M), eb = (long long)g.ldb * (g.opB == OP_N ? g.N : g.K);
  if (ea >= (1LL << 27) || eb >= (1LL << 27)) return false;
  return !g.prec || (g.opA == OP_N && g.opB == OP_N);
}
template <bool A_CPLX, bool B_CPLX, bool AKF, bool BKF, bool F32, int MB, int NB>
void launch_tile_o(const GemmArgs& g, hipStream_t s) {
  dim3 grid((unsigned)cdivl(g.M, 32 * MB), (unsigned)cdivl(g.N, 32 * NB), gemm_zdim(g));
  if (g.bs || g.amap || g.bmap)
    hipLaunchKernelGGL((gemm_tile_kernel<A_CPLX, B_CPLX, AKF, BKF, true, F32, MB, NB>), grid, dim3(NT), 0, s, g);
  else
    hipLaunchKernelGGL((gemm_tile_kernel<A_CPLX, B_CPLX, AKF, BKF, false, F32, MB, NB>), grid, dim3(NT), 0, s, g);
}
template <bool A_CPLX, bool B_CPLX, int MB, int NB>
void launch_tile_p(const GemmArgs& g, hipStream_t s) {
  const bool akf = g.opA != OP_N, bkf = g.opB == OP_N;
  if (g.prec) launch_tile_o<A_CPLX, B_CPLX, false, true, true, MB, NB>(g, s);
  else if (akf && bkf) launch_tile_o<A_CPLX, B_CPLX, true, true, false, MB, NB>(g, s);
  else if (akf) launch_tile_o<A_CPLX, B_CPLX, true, false, false, MB, NB>(g, s);
  else if (bkf) launch_tile_o<A_CPLX, B_CPLX, false, true, false, MB, NB>(g, s);
  else launch_tile_o<A_CPLX, B_CPLX, false, false, false, MB, NB>(g, s);
}
template <int MB, int NB>
void launch_tile(const GemmArgs& g, hipStream_t s) {
  if (g.a_cplx && g.b_cplx) launch_tile_p<true, true, MB, NB>(g, s);
  else if (g.a_cplx) launch_tile_p<true, false, MB, NB>(g, s);
  else launch_tile_p<false, true, MB, NB>(g, s);
}

// Direct-load split-K kernel for grids that would not fill the device: a workgroup of
// NW waves owns one 16 x 16 output tile; wave w takes the w-th contiguous quarter
// (eighth, ...) of K and feeds its MFMAs straight from global memory in the
// v_mfma_f64_16x16x4f64 operand layout (lane = row + 16 k for A, column + 16 k for B),
// four or eight k-steps per batch with the next batch in flight.  The NW partial tiles are
// summed through LDS in wave order.
template <bool A_CPLX, bool B_CPLX, int NW, bool F32>
__global__ __launch_bounds__(64 * NW, 2) void gemm_direct_kernel(GemmArgs g) {
  typedef Mma<F32> M;
  typedef typename M::E E;
  __shared__ cplx red[NW > 1 ? NW - 1 : 1][256];
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int i0 = blockIdx.x * 16, j0 = blockIdx.y * 16;
  if (chain_operands(g, blockIdx.z)) { identity_tile(g, i0, j0, 16, 16, tid, blockDim.x); return; }
  const int z = blockIdx.z % (g.batch > 1 ? g.batch : 1);
  int K = g.K;
  if (g.kdev) {
    const int kd = *g.kdev;
    K = kd < K ? kd : K;
  }
  if (K <= 0 && g.beta.x == 1.0 && g.beta.y == 0.0) return;  // nothing to add
  const double* Ar = (const double*)g.A;
  const cplx* Ac = (const cplx*)g.A;
  const double* Br = (const double*)g.B;
  const cplx* Bc = (const cplx*)g.B;
  if (g.batch > 1) {
    Ar += z * g.strideA; Ac += z * g.strideA;
    Br += z * g.strideB; Bc += z * g.strideB;
  }
  cplx* C = (cplx*)g.C + (g.batch > 1 ? z * g.strideC : 0);
  // K range of this wave, in whole k-steps of 4
  const int ksteps = (K + 3) >> 2;
  const int per = (ksteps + NW - 1) / NW;
  const int kb = wave * per * 4, ke0 = (wave + 1) * per * 4;
  const int ke = ke0 < K ? ke0 : K;
  const int gi = i0 + lr, gj = j0 + lr;
  const bool row_ok = gi < g.M, col_ok = gj < g.N;

  // One batch of U k-steps in the MFMA operand layout.  Gather indices and row scales are
  // read first, then every data load is issued back to back; conjugation and scaling are
  // applied when the batch moves into the MFMA operands.
  constexpr int U = NW >= 4 ? 8 : 4;   // k-steps per batch: one batch covers a wave's K at Ndim = 256
  auto load_batch = [&](int kbase, cplx* a, cplx* b, cplx* sc) {
    int ia[U], ib[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = kbase + 4 * u + lk;
      ia[u] = (row_ok && k < ke) ? k : -1;
      ib[u] = (col_ok && k < ke) ? k : -1;
    }
    if (g.bs) {
#pragma unroll
      for (int u = 0; u < U; ++u) sc[u] = ib[u] >= 0 ? g.bs[ib[u]] : make_double2(0.0, 0.0);
    }
    if (g.amap) {
#pragma unroll
      for (int u = 0; u < U; ++u) if (ia[u] >= 0) ia[u] = g.amap[ia[u]];
    }
    if (g.bmap) {
#pragma unroll
      for (int u = 0; u < U; ++u) if (ib[u] >= 0) ib[u] = g.bmap[ib[u]];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      a[u] = make_double2(0.0, 0.0);
      if (ia[u] >= 0) {
        const long long off = (g.opA == OP_N) ? gi + (long long)ia[u] * g.lda : ia[u] + (long long)gi * g.lda;
        if (A_CPLX) a[u] = Ac[off];
        else a[u].x = Ar[off];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      b[u] = make_double2(0.0, 0.0);
      if (ib[u] >= 0) {
        const long long off = (g.opB == OP_N) ? ib[u] + (long long)gj * g.ldb : gj + (long long)ib[u] * g.ldb;
        if (g.b_cplx) b[u] = Bc[off];
        else b[u].x = Br[off];
      }
    }
  };
  auto finish = [&](cplx* a, cplx* b, const cplx* sc) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (A_CPLX && g.opA == OP_C) a[u].y = -a[u].y;
      if (g.opB == OP_C) b[u].y = -b[u].y;
      if (g.bs) b[u] = cmul(b[u], sc[u]);
    }
  };

  // complex x complex in three real products (3M): acc_re = Ar Br, acc_t2 = Ai Bi,
  // acc_im = (Ar + Ai)(Br + Bi); re = acc_re - acc_t2, im = acc_im - acc_re - acc_t2
  constexpr bool M3 = A_CPLX && B_CPLX;
  typename M::Acc acc_re = {0, 0, 0, 0}, acc_im = {0, 0, 0, 0}, acc_t2 = {0, 0, 0, 0};
  cplx av[U], bv[U], sv[U];
  load_batch(kb, av, bv, sv);
  finish(av, bv, sv);
  for (int k0 = kb; k0 < ke; k0 += 4 * U) {
    cplx an[U], bn[U], sn[U];
    load_batch(k0 + 4 * U, an, bn, sn);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (M3) {
        acc_re = M::mac((E)av[u].x, (E)bv[u].x, acc_re);
        acc_t2 = M::mac((E)av[u].y, (E)bv[u].y, acc_t2);
        acc_im = M::mac((E)(av[u].x + av[u].y), (E)(bv[u].x + bv[u].y), acc_im);
      } else {
        acc_re = M::mac((E)av[u].x, (E)bv[u].x, acc_re);
        if (B_CPLX) acc_im = M::mac((E)av[u].x, (E)bv[u].y, acc_im);
        if (A_CPLX) acc_im = M::mac((E)av[u].y, (E)bv[u].x, acc_im);
      }
    }
    finish(an, bn, sn);
#pragma unroll
    for (int u = 0; u < U; ++u) { av[u] = an[u]; bv[u] = bn[u]; }
  }
  if (M3) {
    acc_im = acc_im - acc_re - acc_t2;
    acc_re = acc_re - acc_t2;
  }
  // register r of a lane holds row M::row(r, lane / 16) of the tile
  if (NW > 1) {
    if (wave > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave - 1][M::row(r, lk) + 16 * lr] = make_double2(acc_re[r], acc_im[r]);
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < NW - 1; ++w) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const cplx p = red[w][M::row(r, lk) + 16 * lr];
        acc_re[r] += p.x;
        acc_im[r] += p.y;
      }
    }
  }
  if (!col_ok) return;
  const cplx csj = g.cs ? g.cs[gj] : make_double2(1.0, 0.0);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int ri = i0 + M::row(r, lk);
    if (ri >= g.M) continue;
    cplx v = make_double2(acc_re[r], (A_CPLX || B_CPLX) ? acc_im[r] : 0.0);
    v = cmul(g.alpha, v);
    if (g.rs) v = cmul(g.rs[ri], v);
    if (g.rs_real) v = cscale(v, g.rs_real[ri]);
    if (g.cs) v = cmul(v, csj);
    const long long off = ri + (long long)gj * g.ldc;
    if (g.beta.x != 0.0 || g.beta.y != 0.0) v = cadd(v, cmul(g.beta, C[off]));
    C[off] = v;
  }
}

template <int NW, bool F32>
void launch_direct_p(const GemmArgs& g, hipStream_t s) {
  dim3 grid((unsigned)cdivl(g.M, 16), (unsigned)cdivl(g.N, 16), gemm_zdim(g));
  const bool bc = g.b_cplx || g.bs != nullptr;
  if (g.a_cplx && bc) hipLaunchKernelGGL((gemm_direct_kernel<true, true, NW, F32>), grid, dim3(64 * NW), 0, s, g);
  else if (g.a_cplx) hipLaunchKernelGGL((gemm_direct_kernel<true, false, NW, F32>), grid, dim3(64 * NW), 0, s, g);
  else if (bc) hipLaunchKernelGGL((gemm_direct_kernel<false, true, NW, F32>), grid, dim3(64 * NW), 0, s, g);
  else hipLaunchKernelGGL((gemm_direct_kernel<false, false, NW, F32>), grid, dim3(64 * NW), 0, s, g);
}
template <int NW>
void launch_direct(const GemmArgs& g, hipStream_t s) {
  if (g.prec) launch_direct_p<NW, true>(g, s);
  else launch_direct_p<NW, false>(g, s);
}
}  // namespace

// ---- the flush of a delayed-update round -------------------------------------------------------
//   Go = Gi + X Y^T,   X = Gi(:, A) C,   Y = Yhat D,   Yhat(c, j) = delta(c, P_j) - Gi(P_j, c),
// A = (P_0 .. P_{m-1}) the round's accepted sites, CD the m x m upper triangular C and, from column
// CHAIN_BLOCK_KMAX on, D, with leading dimension CHAIN_CD_LD, m = *mdev <= CHAIN_BLOCK_KMAX.
// The products of the kernels below are four real ones: with three, the imaginary parts get the
// rounding of the real ones (flush_kernel says why it may take three).
constexpr int RF_T = 16, RF_W = (CHAIN_BLOCK_KMAX + 15) / 16, RF_K = 16 * RF_W;

// One wave's 16 rows r0 .. and columns 16 w .. 16 w + 15 of X or (isy) Y: register q of a lane holds
// column 16 w + 4 q + lane / 16 of row r0 + lane % 16, which is gr; live: the wave has columns
// below m.  Every global load is issued before the first MFMA, and the sites are read beside m so
// that the gathers wait for one load.  C and D are zero below row 16 w + 15.
struct RoundFactor {
  cplx ga[RF_K / 4], cd[RF_K / 4];
  v4d re = {0, 0, 0, 0}, im = {0, 0, 0, 0}, t = {0, 0, 0, 0};
  // (the sites' buffer holds CHAIN_KMAX >= RF_K entries)
  __device__ __forceinline__ void load(const cplx* __restrict__ G, const cplx* __restrict__ CD, const int (&pa)[RF_K / 4],
                                       int m, int n, int gr, int w, bool isy) {
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int u = 0; u < RF_K / 4; ++u) {
      const int k = 4 * u + lk;
      const bool in = 16 * w < m && k < m && u < 4 * (w + 1);
      ga[u] = (in && gr < n) ? G[isy ? pa[u] + (long long)gr * n : gr + (long long)pa[u] * n] : make_double2(0.0, 0.0);
      cd[u] = (in && 16 * w + lr < m) ? CD[k + (long long)((isy ? CHAIN_BLOCK_KMAX : 0) + 16 * w + lr) * CHAIN_CD_LD]
                                      : make_double2(0.0, 0.0);
      if (isy && in && gr < n) ga[u] = make_double2((gr == pa[u] ? 1.0 : 0.0) - ga[u].x, -ga[u].y);
    }
  }
  __device__ __forceinline__ void mul(int w) {
    typedef Mma<false> M;
#pragma unroll
    for (int u = 0; u < RF_K / 4; ++u) {
      if (u < 4 * (w + 1)) {
        re = M::mac(cd[u].x, ga[u].x, re);
        im = M::mac(cd[u].x, ga[u].y, im);
        t = M::mac(cd[u].y, ga[u].y, t);
        im = M::mac(cd[u].y, ga[u].x, im);
      }
    }
  }
  __device__ __forceinline__ cplx get(int q) const { return make_double2(re[q] - t[q], im[q]); }
};

// X and Y alone, for batches and for matrices whose tiles are too many for the kernel below: 16
// rows to a workgroup, its waves as below.  The rows A of G are gathered here, over the device, and
// not by the block kernel's one workgroup a chain.
__global__ __launch_bounds__(128 * RF_W, 2) void round_factors_kernel(const cplx* __restrict__ G,
                                                                     const cplx* __restrict__ CD,
                                                                     const int* __restrict__ amap, const int* mdev,
                                                                     cplx* __restrict__ X, cplx* __restrict__ Y,
                                                                     int n, int kmax, long long cs) {
  const int z = blockIdx.z;
  G = chain_ptr_at(G, cs, z);
  CD = chain_ptr_at(CD, cs, z);
  amap = chain_ptr_at(amap, cs, z);
  mdev = chain_ptr_at(mdev, cs, z);
  X = chain_ptr_at(X, cs, z);
  Y = chain_ptr_at(Y, cs, z);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const bool isy = wave >= RF_W;
  const int w = isy ? wave - RF_W : wave;
  const int gr = blockIdx.x * RF_T + lr;
  int pa[RF_K / 4];
#pragma unroll
  for (int u = 0; u < RF_K / 4; ++u) pa[u] = amap[4 * u + lk];
  int m = *mdev;
  m = m < kmax ? m : kmax;
  RoundFactor f;
  f.load(G, CD, pa, m, n, gr, w, isy);
  if (16 * w >= m) return;
  f.mul(w);
  cplx* const out = isy ? Y : X;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = 16 * w + 4 * q + lk;
    if (j < m && gr < n) out[gr + (long long)j * n] = f.get(q);
  }
}

// The whole flush for a few chains, in one launch.  Gi is only read and Go only written (two
// buffers), so a workgroup can gather the columns A and rows A of Gi that it needs while others
// write their tiles.  A workgroup owns a 16 x 16 tile: of its 2 RF_W waves the first half forms its
// rows of X, the second its rows of Y, 16 columns each; then RF_W waves take 16 columns of the
// rank-m product each, and the parts are added through LDS.  Latency-bound.
__global__ __launch_bounds__(128 * RF_W, 2) void round_flush_kernel(const cplx* __restrict__ Gi, cplx* __restrict__ Go,
                                                                   const cplx* __restrict__ CD,
                                                                   const int* __restrict__ amap, const int* mdev,
                                                                   int n, int kmax, long long cs) {
  typedef Mma<false> M;
  __shared__ cplx XY[2][RF_K][RF_T + 1];   // X(i0 + r, j), Y(j0 + r, j) at [j][r]
  __shared__ cplx red[RF_W - 1][RF_T * RF_T];
  const int z = blockIdx.z;
  Gi = chain_ptr_at(Gi, cs, z);
  Go = chain_ptr_at(Go, cs, z);
  CD = chain_ptr_at(CD, cs, z);
  amap = chain_ptr_at(amap, cs, z);
  mdev = chain_ptr_at(mdev, cs, z);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const bool isy = wave >= RF_W;
  const int w = isy ? wave - RF_W : wave;
  const int i0 = blockIdx.x * RF_T, j0 = blockIdx.y * RF_T;
  const int gj = j0 + lr;
  int pa[RF_K / 4];
#pragma unroll
  for (int u = 0; u < RF_K / 4; ++u) pa[u] = amap[4 * u + lk];
  int m = *mdev;
  m = m < kmax ? m : kmax;
  m = m > 0 ? m : 0;
  const bool live = 16 * w < m;
  RoundFactor f;
  f.load(Gi, CD, pa, m, n, isy ? gj : i0 + lr, w, isy);
  // the tile of Gi in the layout of the product (wave 0 adds it)
  cplx gt[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int ri = i0 + M::row(r, lk);
    gt[r] = (wave == 0 && ri < n && gj < n) ? Gi[ri + (long long)gj * n] : make_double2(0.0, 0.0);
  }
  if (live) {
    f.mul(w);
#pragma unroll
    for (int q = 0; q < 4; ++q) XY[isy][16 * w + 4 * q + lk][lr] = f.get(q);
  }
  __syncthreads();
  v4d gre = {0, 0, 0, 0}, gim = {0, 0, 0, 0}, gt2 = {0, 0, 0, 0};
  if (live && !isy) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const cplx a = XY[0][16 * w + 4 * u + lk][lr], b = XY[1][16 * w + 4 * u + lk][lr];
      gre = M::mac(a.x, b.x, gre);
      gim = M::mac(a.x, b.y, gim);
      gt2 = M::mac(a.y, b.y, gt2);
      gim = M::mac(a.y, b.x, gim);
    }
    if (w > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) red[w - 1][M::row(r, lk) + RF_T * lr] = make_double2(gre[r] - gt2[r], gim[r]);
    }
  }
  __syncthreads();
  if (wave > 0 || gj >= n) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int ri = i0 + M::row(r, lk);
    if (ri >= n) continue;
    cplx v = make_double2(gre[r] - gt2[r], gim[r]);
#pragma unroll
    for (int q = 1; q < RF_W; ++q)
      if (16 * q < m) v = cadd(v, red[q - 1][M::row(r, lk) + RF_T * lr]);
    Go[ri + (long long)gj * n] = cadd(gt[r], v);
  }
}

int round_factors_launch(const cplx* G, const cplx* CD, const int* amap, const int* mdev, cplx* X, cplx* Y, int n,
                         int kmax, int nchain, long long cs, hipStream_t s) {
  if (kmax < 1 || kmax > CHAIN_BLOCK_KMAX) { alfq_set_error("round factors: rank outside the block kernel's depth"); return ST_GENERIC; }
  if (nchain < 1 || nchain > 65535 || n < 1) { alfq_set_error("round factors: bad batch"); return ST_GENERIC; }
  hipLaunchKernelGGL(round_factors_kernel, dim3((unsigned)cdivl(n, RF_T), 1, (unsigned)nchain), dim3(128 * RF_W), 0, s,
                     G, CD, amap, mdev, X, Y, n, kmax, cs);
  HIP_OK(hipGetLastError());
  return ST_NONE;
}

int round_flush_launch(const cplx* Gi, cplx* Go, const cplx* CD, const int* amap, const int* mdev, int n, int kmax,
                       int nchain, long long cs, hipStream_t s) {
  if (kmax < 1 || kmax > CHAIN_BLOCK_KMAX) { alfq_set_error("round flush: rank outside the block kernel's depth"); return ST_GENERIC; }
  if (nchain < 1 || nchain > 65535 || n < 1) { alfq_set_error("round flush: bad batch"); return ST_GENERIC; }
  const unsigned t = (unsigned)cdivl(n, RF_T);
  hipLaunchKernelGGL(round_flush_kernel, dim3(t, t, (unsigned)nchain), dim3(128 * RF_W), 0, s, Gi, Go, CD, amap, mdev,
                     n, kmax, cs);
  HIP_OK(hipGetLastError());
  return ST_NONE;
}

int flush_launch(cplx* G, const cplx* X, const cplx* Y, const int* mdev, int n, int kmax, int nchain,
                 long long cs, hipStream_t s) {
  if (kmax < 1 || kmax > CHAIN_BLOCK_KMAX) { alfq_set_error("flush: rank outside the block kernel's depth"); return ST_GENERIC; }
  if (nchain < 1 || nchain > 65535) { alfq_set_error("flush: bad batch"); return ST_GENERIC; }
  const unsigned t = (unsigned)cdivl(n, FL_T);
  hipLaunchKernelGGL(flush_kernel, dim3(t, t, (unsigned)nchain), dim3(NT), 0, s, G, X, Y, mdev, n, kmax, cs);
  HIP_OK(hipGetLastError());
  return ST_NONE;
}

GemmArgs gemm_args(int M, int N, int K, const void* A, int lda, int opA, bool a_cplx,
                   const void* B, int ldb, int opB, bool b_cplx, void* C, int ldc,
                   cplx alpha, cplx beta) {
  GemmArgs g{};
  g.M = M; g.N = N; g.K = K; g.kdev = nullptr;
  g.A = A; g.lda = lda; g.opA = opA; g.a_cplx = a_cplx;
  g.B = B; g.ldb = ldb; g.opB = opB; g.b_cplx = b_cplx;
  g.C = C; g.ldc = ldc;
  g.alpha = alpha; g.beta = beta;
  g.batch = 1;
  g.nchain = 1;
  g.cstride = 0;
  g.prec = 0;
  g.policy = 0;
  g.lz = nullptr;
  g.slice = 0;
  g.hop_side = 0;
  g.ident = nullptr;
  return g;
}

int gemm_launch(const GemmArgs& g, hipStream_t s) {
  if (g.M <= 0 || g.N <= 0) return ST_NONE;
  if (gemm_zdim(g) > 65535) { alfq_set_error("gemm_launch: batch too large"); return ST_GENERIC; }
  switch (gemm_kernel_for(g.M, g.N, g.K, gemm_zdim(g), g.policy, tile_kernel_takes(g))) {
    case GEMM_DIRECT: {
      const int ksteps = g.K > 0 ? (g.K + 3) / 4 : 1;
      if (ksteps >= 32) launch_direct<8>(g, s);
      else if (ksteps >= 16) launch_direct<4>(g, s);
      else if (ksteps >= 8) launch_direct<2>(g, s);
      else launch_direct<1>(g, s);
      break;
    }
    case GEMM_TILE_64: launch_tile<2, 2>(g, s); break;
    case GEMM_TILE_32:
      if (tile_kernel_takes(g)) launch_tile<1, 1>(g, s);
      else launch_shape<2, 2>(g, s);
      break;
    case GEMM_LDS_16_32: launch_shape<1, 2>(g, s); break;
    default: launch_shape<1, 1>(g, s); break;
  }
  HIP_OK(hipGetLastError());
  return ST_NONE;
}
