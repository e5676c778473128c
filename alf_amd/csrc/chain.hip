// Metropolis sweep over the fields of one time slice with delayed
// Sherman-Morrison updates (the per-op loop of WRAPGRUP/WRAPGRDO with Upgrade2,
// Prog/Wrapgr_mod.F90:115-147, 198-236; Prog/upgrade_mod.F90:105-302), plus
// the diagonal-exponential vectors of a slice and the random-number stream.
//
// Delayed update: after m accepted flips the current Green's function is
//   G_cur = G + X(:, 0:m) Y(:, 0:m)^T,
//   X(:, j) = -x_j G_cur_j(:, P_j),  Y(:, j) = e_P - G_cur_j(P_j, :)^T,
// which is the rank-1 update of upgrade_mod.F90:266-269 (ZGERU) kept
// unapplied.  The block kernel decides from a submatrix of G_cur held in LDS
// and forms the columns of X and Y in bulk per block of visits; the generic
// kernel (deep delays) forms them one accepted flip at a time.  A kernel stops
// after K accepted flips; the flush G += X Y^T is an MFMA GEMM.
//
// Diagonal operator exponentials (the type-1 Op_Wrapup/Op_Wrapdo scalings,
// Operator_mod.F90:767-782, 884-899) are not applied here: for diagonal
// operators they are a similarity transform G -> D G D^-1 that commutes with
// the rank-1 update and leaves G_PP unchanged, so all of a slice's scalings are
// fused into the epilogue of the adjacent hopping GEMM.
#include <hip/hip_ext.h>

#include <mutex>
#include <type_traits>

#include "alfq_chain.h"

namespace {

__device__ inline void mulhilo(uint32_t a, uint32_t b, uint32_t& hi, uint32_t& lo) {
  const uint64_t p = (uint64_t)a * (uint64_t)b;
  hi = (uint32_t)(p >> 32);
  lo = (uint32_t)p;
}

// Philox4x32 with 10 rounds (Salmon, Moraes, Dror, Shaw, SC'11).
__device__ inline uint4 philox4x32_10(uint4 c, uint2 k) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    uint32_t hi0, lo0, hi1, lo1;
    mulhilo(0xD2511F53u, c.x, hi0, lo0);
    mulhilo(0xCD9E8D57u, c.z, hi1, lo1);
    c = make_uint4(hi1 ^ c.y ^ k.x, lo1, hi0 ^ c.w ^ k.y, lo0);
    k.x += 0x9E3779B9u;
    k.y += 0xBB67AE85u;
  }
  return c;
}

// uniform number q of a chain's Philox stream (the value philox_fill_kernel leaves at q)
__device__ inline double philox_uniform(unsigned long long q, unsigned long long seed, unsigned stream) {
  const uint4 r = philox4x32_10(make_uint4((uint32_t)q, (uint32_t)(q >> 32), stream, 0x414c4651u),
                                make_uint2((uint32_t)seed, (uint32_t)(seed >> 32)));
  return (double)((((uint64_t)r.x << 32) | r.y) >> 11) * (1.0 / 9007199254740992.0);
}

// uniforms u[q - base] for global indices q in [base, base + count), base = st->rng_pos: one
// Philox block per index, 53-bit mantissa from two words, u in [0, 1).  The window is read
// from and recorded in device memory, so a captured sweep replays with the stream's position.
__global__ void philox_fill_kernel(double* __restrict__ u, ChainState* st, long long count, long long cs) {
  u = chain_ptr(u, cs);
  st = chain_ptr(st, cs);
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned long long base = st->rng_pos, seed = st->seed;
  const unsigned stream = st->stream;
  if (i == 0) {
    st->u_base = base;
    st->u_len = count;
  }
  if (i >= count) return;
  u[i] = philox_uniform(base + (unsigned long long)i, seed, stream);
}

__device__ inline cplx wave_csum(cplx v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    v.x += __shfl_xor(v.x, o, 64);
    v.y += __shfl_xor(v.y, o, 64);
  }
  return v;
}

__device__ inline int nranf3(double u) {
  // nranf(3) = clamp(nint(3u + 0.5), 1, 3)   (random_wrap_mod.F90:159-168)
  const double x = u * 3.0 + 0.5;
  int k = (int)floor(x + 0.5);
  return k < 1 ? 1 : (k > 3 ? 3 : k);
}

__device__ inline int flip_st(int s, int k) {
  // FLIP_st(s, k) of Fields_mod.F90:287-301
  switch (s) {
    case -2: return k == 1 ? -1 : (k == 2 ? 1 : 2);
    case -1: return k == 1 ? 1 : (k == 2 ? 2 : -2);
    case 1: return k == 1 ? 2 : (k == 2 ? -2 : -1);
    default: return k == 1 ? -2 : (k == 2 ? -1 : 1);
  }
}

// One thread per visit (VisitArgs).  The block kernel would otherwise look a visit up itself, four
// dependent loads deep, each a miss in the caches a new kernel starts with: 2.9 us of a launch for
// one chain, 11 us in a batch of 256, against one load of 64 bytes.
__global__ void visit_kernel(VisitArgs a) {
  a.out = chain_ptr(a.out, a.cs);
  a.st = chain_ptr(a.st, a.cs);
  a.f = chain_ptr(a.f, a.cs);
  a.u = chain_ptr(a.u, a.cs);
  a.op_myexp = chain_ptr(a.op_myexp, a.cs);
  a.op_expalpha = chain_ptr(a.op_expalpha, a.cs);
  a.gama_ratio = chain_ptr(a.gama_ratio, a.cs);
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long long)a.n_op * a.ns) return;
  const int v = (int)(idx % a.n_op), q = (int)(idx / a.n_op);
  const int slice = a.dir > 0 ? a.s0 + q : a.s0 + a.ns - 1 - q;
  int ord = q;               // slices of the pass that the chain has visited before this one
  if (a.lz) {
    const int lz = a.lz[blockIdx.z], end = a.s0 + a.ns;
    if (slice >= lz) return;
    if (a.dir < 0 && lz < end) ord -= end - lz;
  }
  const int nop = a.dir > 0 ? v : a.n_op - 1 - v;
  const int typ = a.op_type[nop];
  const int s_old = a.f[(long long)slice * a.n_op + nop];
  const int need = a.uoff[v + 1] - a.uoff[v];
  const unsigned long long pos = a.st->rng_pos + (unsigned long long)ord * a.per + a.uoff[v];
  BVisit w;
  w.ca = make_double2(1.0, 0.0); w.cb = make_double2(0.0, 0.0); w.delta = make_double2(0.0, 0.0);
  w.thr = 2.0; w.fnew = VISIT_NONE; w.loc = 0;
  w.P = a.op_site[nop];
  double u0 = 0.0, u1 = 0.0;  // the proposal's number (type 2) and the decision's
  bool ok = true;
  if (a.u) {
    const unsigned long long ub = a.st->u_base;
    ok = !(pos < ub || pos + (unsigned long long)need > ub + (unsigned long long)a.st->u_len);
    if (ok) {
      u0 = a.u[pos - ub];
      u1 = a.u[pos - ub + need - 1];
    }
  } else {
    const unsigned long long seed = a.st->seed;
    const unsigned stream = a.st->stream;
    if (typ == 2) u0 = philox_uniform(pos, seed, stream);
    u1 = philox_uniform(pos + need - 1, seed, stream);
  }
  if (ok) {
    const int s_new = typ == 2 ? flip_st(s_old, nranf3(u0)) : -s_old;
    const int ti = nop * 25 + (s_old + 2) * 5 + (s_new + 2);
    const cplx myexp = a.op_myexp[ti], expal = a.op_expalpha[ti];
    w.delta = make_double2(myexp.x - 1.0, myexp.y);
    w.ca = cmul(expal, myexp);
    w.cb = cmul(expal, w.delta);
    w.thr = u1 / fabs(a.gama_ratio[ti]);
    w.fnew = (short)s_new;
  }
  a.out[(long long)(slice - a.s0) * a.n_op + v] = w;
}

__global__ __launch_bounds__(256) void chain_kernel(ChainArgs a) {
  __shared__ cplx s_xr[CHAIN_KMAX];
  __shared__ cplx s_yr[CHAIN_KMAX];
  __shared__ int s_acc, s_P, s_pos, s_m, s_stop;
  __shared__ cplx s_x;

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int n = a.n;
  ChainState* st = a.st;
  if (tid == 0) {
    s_pos = st->pos;
    s_m = 0;
    s_stop = 0;
  }
  __syncthreads();

  while (true) {
    const int pos = s_pos;
    const int m = s_m;
    if (pos >= a.n_op || m >= a.Kmax || s_stop) break;
    const int nop = a.dir > 0 ? pos : a.n_op - 1 - pos;
    const int P = a.op_site[nop];
    if (wave == 0) {
      cplx d = make_double2(0.0, 0.0);
      for (int j = lane; j < m; j += 64) {
        const cplx xv = a.X[P + (long long)j * n];
        const cplx yv = a.Y[P + (long long)j * n];
        s_xr[j] = xv;
        s_yr[j] = yv;
        d = cfma(xv, yv, d);
      }
      d = wave_csum(d);
      if (lane == 0) {
        const cplx gpp = cadd(a.G[P + (long long)P * n], d);
        const int typ = a.op_type[nop];
        int8_t* fp = a.f + (long long)a.slice * a.n_op + nop;
        const int s_old = *fp;
        unsigned long long q = st->rng_pos;
        const unsigned long long need = (typ == 2) ? 3ull : 2ull;
        int acc = 0;
        if (q < st->u_base || q + need > st->u_base + (unsigned long long)st->u_len) {
          st->status = 1;   // random stream exhausted: stop without touching G
          s_stop = 1;
        } else {
          const double* u = a.u + (q - st->u_base);
          int s_new, k = 0;
          if (typ == 2) { s_new = flip_st(s_old, nranf3(u[0])); k = 1; } else { s_new = -s_old; }
          // u[k]: T0_proposal = 1.5 > ranf, always taken
          const double u3 = u[k + 1];
          st->rng_pos = q + need;
          const int ti = nop * 25 + (s_old + 2) * 5 + (s_new + 2);
          const cplx myexp = a.op_myexp[ti];
          const cplx delta = make_double2(myexp.x - 1.0, myexp.y);
          const cplx dmat = csub(myexp, cmul(delta, gpp));
          const cplx ratio = cmul(dmat, a.op_expalpha[ti]);
          cplx rt = ratio;
          for (int p = 1; p < a.n_sun; ++p) rt = cmul(rt, ratio);
          rt = cscale(rt, a.gama_ratio[ti]);
          const cplx ph = st->phase;
          const double weight = fabs(cmul(ph, rt).x / ph.x);
          st->nc += 1;
          if (weight > u3) {
            acc = 1;
            st->acc += 1;
            st->phase = cmul(ph, cscale(rt, 1.0 / sqrt(cabs2(rt))));
            *fp = (int8_t)s_new;
            // x = Delta / (1 + v_P Delta), v_P = 1 - G_cur(P,P)
            const cplx vp = make_double2(1.0 - gpp.x, -gpp.y);
            const cplx den = cadd(make_double2(1.0, 0.0), cmul(vp, delta));
            s_x = cdiv(delta, den);
          }
        }
        s_acc = acc;
        s_P = P;
      }
    }
    __syncthreads();
    if (s_stop) break;
    if (s_acc) {
      const cplx x = s_x;
      const cplx mx = make_double2(-x.x, -x.y);
      for (int r = tid; r < n; r += blockDim.x) {
        cplx col = a.G[r + (long long)P * n];
        cplx row = a.G[P + (long long)r * n];
        for (int j = 0; j < m; ++j) {
          col = cfma(a.X[r + (long long)j * n], s_yr[j], col);
          row = cfma(s_xr[j], a.Y[r + (long long)j * n], row);
        }
        a.X[r + (long long)m * n] = cmul(mx, col);
        a.Y[r + (long long)m * n] = make_double2((r == P ? 1.0 : 0.0) - row.x, -row.y);
      }
    }
    __syncthreads();
    if (tid == 0) {
      s_pos = pos + 1;
      if (s_acc) s_m = m + 1;
    }
    __syncthreads();
  }
  if (tid == 0) {
    st->pos = s_pos;
    st->m = s_m;
  }
}

// ---------------------------------------------------------------------------------
// Submatrix block kernel.  The visits of a round are taken in blocks of up to SB_V
// consecutive visits.  For the sites S of a block the kernel holds g = G_cur[S, S] in
// LDS and decides each visit from g alone (G_cur(P,P) = g(p,p)).  An accepted flip is the
// rank-1 update of upgrade_mod.F90:266-269 restricted to S,
//   g += u w^T,  u = -x g(:, p),  w = e_p - g(p, :)^T.
//
// Full columns and rows of G are never formed here.  With A = (P_0, P_1, ...) the sites of
// the round's accepted flips in order, G the Green's function at the start of the round and
// Yhat(:, j) = e_{P_j} - G(P_j, :)^T, the current one is G_cur = G + X Y^T with
//   X = G(:, A) C,   Y = Yhat D,
// C and D m x m and upper triangular, kept in LDS.  A block starts from g = G[S, S] + X[S] Y[S]^T,
// X[S] = G[S, A] C, Y[S] = Yhat[S, A] D, and its flips add the columns
//   C(:, m + j) = -x_j (e_j + T2(:, p_j) + sum_{i<j} C(:, m + i) w_i(p_j)),  T2 = C Y[S]^T,
//   D(:, m + j) =        e_j - T1(p_j, :)^T - sum_{i<j} D(:, m + i) u_i(p_j), T1 = X[S] D^T
// (i, j over the block's flips).  The four products are on the matrix cores.  At the end the
// kernel leaves C, D and the site list A; the flush over the device is G += X Y^T.
// One table W = C D^T (m x m) with G_cur = G + G(:, A) W Yhat^T, extended by each block to
// W + Cn Dn^T, would save two of the block's products and one of the flush, but X and Y are of the
// size of G's columns and rows, where W's entries are some 30 times as large and cancel in what is
// formed from them: one slice's 32 flips left 7.8e-14 of G as error (C and D here and W in the
// flush 3.7e-14, C and D throughout 2.1e-14), and G after ten slices was 3 to 6 times as far off.
//
// What bounds it: the chain of decisions, so the instructions and waits per accepted flip.  One
// wave decides (no barrier inside a block), left-looking: lanes 0..31 hold column p of g, lanes
// 32..63 row p, each formed from the block-start g and the block's earlier u_i, w_i in LDS, so a
// flip costs one LDS round trip and a dot product over the block's flips instead of an update of
// all of g by four waves between barriers; lane v keeps g(v, v) of its visit.  Two more waves
// follow it flip by flip through flags in LDS and form the new columns of C and D (row l in
// lane l), and a fourth fetches the next block's visit records, so that a block ends when its
// last decision does.
constexpr int SB_V = 32;    // visits per block: g is SB_V x SB_V
constexpr int SB_A = 16;    // accepted flips per block
constexpr int SB_K = CHAIN_BLOCK_KMAX;   // accepted flips per round (delayed-update depth)
constexpr int SB_T = 512;   // threads: 8 waves, two MFMA streams per SIMD
constexpr int SB_W = SB_T / 64;
constexpr int SB_M = (SB_K + 15) / 16;   // 16-wide tiles of C and D
constexpr int SB_PS = SB_V + 1;          // row pitch of the tables indexed by the block's sites
constexpr int SB_PL = SB_K + 1;          // row pitch of C and D
static_assert(2 * SB_K <= CHAIN_CD_LD, "C beside D in a square of CHAIN_CD_LD");
static_assert((SB_K & (SB_K - 1)) == 0, "indexes into C and D by masks");
static_assert(SB_K == 16 * SB_M && SB_K <= 64, "whole tiles of C and D, row l in lane l of a wave");

typedef double v4d __attribute__((ext_vector_type(4)));

// z * 2^-e with |z| in [0.5, 1): an exact rescaling that keeps the running phase in range
__device__ __forceinline__ cplx renorm_pow2(cplx z) {
  const double mx = fmax(fabs(z.x), fabs(z.y));
  const int e = __builtin_amdgcn_frexp_exp(mx);
  return make_double2(ldexp(z.x, -e), ldexp(z.y, -e));
}

// the complex value of lane l (l uniform) in every lane
__device__ __forceinline__ cplx lane_c(cplx v, int l) {
  const long long re = __builtin_bit_cast(long long, v.x), im = __builtin_bit_cast(long long, v.y);
  const long long r = ((long long)(unsigned)__builtin_amdgcn_readlane((int)(re >> 32), l) << 32) |
                      (unsigned)__builtin_amdgcn_readlane((int)re, l);
  const long long i = ((long long)(unsigned)__builtin_amdgcn_readlane((int)(im >> 32), l) << 32) |
                      (unsigned)__builtin_amdgcn_readlane((int)im, l);
  return make_double2(__builtin_bit_cast(double, r), __builtin_bit_cast(double, i));
}

// lanes 0..31 of v in both halves of low, lanes 32..63 in both halves of high (register moves)
__device__ __forceinline__ void both_halves(double v, double& low, double& high) {
  const long long b = __double_as_longlong(v);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)(b & 0xffffffffLL), (unsigned)(b & 0xffffffffLL), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  low = __longlong_as_double(((long long)hi[0] << 32) | (long long)lo[0]);
  high = __longlong_as_double(((long long)hi[1] << 32) | (long long)lo[1]);
}

// A 16 x 16 complex tile in four real products.  (Three, with im = (ar + ai)(br + bi) - re parts,
// leave the imaginary parts the rounding of the real ones: the error of G over ten slices was
// 1.15 times as large.)
struct CTile {
  v4d r = {0, 0, 0, 0}, i = {0, 0, 0, 0}, t = {0, 0, 0, 0};
  __device__ __forceinline__ void mac(cplx a, cplx b) {
    r = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, r, 0, 0, 0);
    i = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.y, i, 0, 0, 0);
    t = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, t, 0, 0, 0);
    i = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, i, 0, 0, 0);
  }
  __device__ __forceinline__ cplx get(int q) const { return make_double2(r[q] - t[q], i[q]); }
};
// tile += sum over k0 <= k < kn (multiples of 4) of fa(k + lk) fb(k + lk), lk = lane / 16: the next
// step's operands are read while this step's products issue.  Register q of a lane holds the
// entry of fa's index 4 q + lane / 16 and fb's index lane % 16.
template <class FA, class FB>
__device__ __forceinline__ void tile_mac(CTile& c, int k0, int kn, int lk, FA fa, FB fb) {
  if (kn <= k0) return;
  cplx a = fa(k0 + lk), b = fb(k0 + lk);
  for (int k = k0 + 4; k < kn; k += 4) {
    const cplx an = fa(k + lk), bn = fb(k + lk);
    c.mac(a, b);
    a = an;
    b = bn;
  }
  c.mac(a, b);
}

// the value of v, which the compiler takes for a new one: address arithmetic made from it stays
// inside the loop that it is in, where it would otherwise be hoisted, held in registers over the
// whole loop and spilled
__device__ __forceinline__ int here(int v) {
  __asm__ volatile("" : "+v"(v));
  return v;
}

// What a wave hands to another through LDS: released before the flag is stored, acquired after it is
// read, so that the hand-over is ordered in the language and not by the LDS pipeline alone.  The
// fences name the LDS only: the deciding wave waits for its LDS writes, not for global memory.  One
// chain's sweep at 16 x 16 with them 61.4 ms, with a bare compiler barrier in their place 61.2.
__device__ __forceinline__ void lds_release() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local"); }
__device__ __forceinline__ void lds_acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local"); }

// Bound by two serial parts, for one chain of 16 x 16 24.7 us a launch (34.5 where one rank-1 update
// of X, Y and g was made per acceptance; its sweep 75.1 -> 61.4 ms with the flush), for 256 chains of
// 4 x 4 12.1 us (20.0).  The decisions: about 1240 clocks (0.52 us) from one acceptance to the next (LDS
// reads of the row and column, their dot product, the test, the ballot), 22 of them in a launch, so
// less than half of it.  The starts of its two to three blocks, most of the rest: the gathers of G at
// the block's sites, two phases of products with a short K and three barriers, overlapped by nothing.
// Rounds end at 32 flips because the tables do: at 48 they would take more than the LDS's 160 KB.
// No array of this kernel may leave the registers: one that the compiler moves to LDS by thread
// costs a read of the launch packet in host memory, 1.6 us and in a batch of 256 chains 8 us.
__global__ __launch_bounds__(SB_T, 2) void chain_block_kernel(ChainArgs a) {
  __shared__ cplx gs[SB_V][SB_PS];            // g(r, c) at [c][r]
  __shared__ cplx Tuw[SB_A][64];              // u_i(s), w_i(s) at [i][s], [i][32 + s]
  __shared__ cplx Cm[SB_K][SB_PL];            // C(l, j) at [j][l], l < SB_K, j < m
  __shared__ cplx Dm[SB_K][SB_PL];            // D(l, j) at [j][l]
  __shared__ cplx Xa[SB_K][SB_PS];            // G(S_s, A_l) at [l][s], then T1(s, l)
  __shared__ cplx Yh[SB_K][SB_PS];            // Yhat(S_s, l) at [l][s], then T2(l, s)
  __shared__ cplx Xb[SB_K][SB_PS];            // X(S_s, j) at [j][s]
  __shared__ cplx Yb[SB_K][SB_PS];            // Y(S_s, j) at [j][s]
  __shared__ BVisit vr[2][SB_V];
  __shared__ cplx s_x[SB_A];
  __shared__ int s_aP[SB_K];
  __shared__ int s_mb, s_k, s_stopped;
  // entry j: 1 + the index of flip j's site once flip j is in LDS, SB_FIN after the block's last
  __shared__ int s_pub[SB_A + 1];
  constexpr int SB_FIN = 0x100;

  auto publish = [&](int j, int what) {
    lds_release();
    __hip_atomic_store(&s_pub[j], what, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int n = a.n;
  a.G = chain_ptr(a.G, a.cs);
  a.X = chain_ptr(a.X, a.cs);
  a.Y = chain_ptr(a.Y, a.cs);
  a.f = chain_ptr(a.f, a.cs);
  a.rec = chain_ptr(a.rec, a.cs);
  a.st = chain_ptr(a.st, a.cs);
  a.CD = chain_ptr(a.CD, a.cs);
  a.amap = chain_ptr(a.amap, a.cs);
  ChainState* st = a.st;
  if (a.lz && a.slice >= a.lz[blockIdx.z]) {
    // a slice beyond this chain's Ltrot: no visits, no random numbers, nothing to flush
    if (tid == 0) st->m = 0;
    return;
  }
  // one lane reads the chain's state for the workgroup, with what it will need at the end
  __shared__ int s_pos0;
  __shared__ cplx s_phase;
  ChainState st0;
  if (tid == 0) {
    st0.nc = st->nc;
    st0.acc = st->acc;
    st0.rng_pos = st->rng_pos;
    st0.max_slice_acc = st->max_slice_acc;
    st0.slice_acc = a.first_round ? 0 : st->slice_acc;
    s_pos0 = a.first_round ? 0 : st->pos;
    s_phase = st->phase;
  }
  __syncthreads();
  if (s_pos0 >= a.n_op) {
    // the slice ended in an earlier round
    if (tid == 0) st->m = 0;
    return;
  }
  int pos = s_pos0, m = 0;
  cplx z = s_phase;           // the phase up to a positive factor (wave 0)
  long long nvisits = 0, naccepts = 0;
  const int kmax = a.Kmax < SB_K ? a.Kmax : SB_K;
  bool stopped = false;

  // ---- the records of visits v0 .. v0 + SB_V - 1, one per lane of one wave ----
  auto records = [&](int v0, int buf) {
    const int lane = here(tid & 63);
    BVisit w;
    w.ca = make_double2(1.0, 0.0); w.cb = make_double2(0.0, 0.0); w.delta = make_double2(0.0, 0.0);
    w.thr = 2.0; w.P = 0; w.fnew = VISIT_NONE;
    if (lane < SB_V && v0 + lane < a.n_op) w = a.rec[v0 + lane];
    w.loc = (short)lane;
    if (a.multi) {
      for (int t = 0; t < SB_V; ++t) {
        const int Pt = __builtin_amdgcn_readlane(w.P, t);
        if (t < w.loc && Pt == w.P) w.loc = (short)t;
      }
    }
    if (lane < SB_V) vr[buf][lane] = w;
  };

  // ---- G at the sites of a block and of the round's flips, in registers until the tables of
  // the block before are free ----
  constexpr int NE = (SB_V * SB_K + SB_T - 1) / SB_T;
  auto gather = [&](const BVisit* v, int nb, cplx (&gss)[4], cplx (&gsa)[NE], cplx (&gas)[NE]) {
    const int ln = here(lane), lr = ln & 15, lk = ln >> 4, td = here(tid);
    if (wave < 4) {
      // tile wave of G[S, S] in the layout of its product: rows lane % 16, columns 4 q + lane / 16
      const int r = 16 * (wave & 1) + lr;
      const long long Pr = v[r < nb ? r : 0].P;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = 16 * (wave >> 1) + 4 * q + lk;
        gss[q] = a.G[Pr + (long long)v[c < nb ? c : 0].P * n];
      }
    }
    const int s = td & (SB_V - 1), Ps = v[s < nb ? s : 0].P;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int l = (td >> 5) + (SB_T / SB_V) * e;
      if (l < m) {
        const int Pl = s_aP[l];
        // (by components: as a copy of the element the array would leave the registers)
        const cplx *const psa = a.G + Ps + (long long)Pl * n, *const pas = a.G + Pl + (long long)Ps * n;
        gsa[e] = make_double2(psa->x, psa->y);
        gas[e] = make_double2(pas->x, pas->y);
      }
    }
  };
  int cur = 1;
  bool cut = true;            // the records at vr[cur ^ 1] are not those of the visits from pos on
  while (true) {
    // ---- the next block: its sites' rows and columns of G are on their way ----
    const bool more = !stopped && pos < a.n_op && (m < kmax || a.final_round);
    cplx gss[4], gsa[NE], gas[NE];
    if (more) {
      if (cut) {
        if (wave == SB_W - 1) records(pos, cur ^ 1);
        __syncthreads();
      }
      cur ^= 1;
      gather(vr[cur], a.n_op - pos < SB_V ? a.n_op - pos : SB_V, gss, gsa, gas);
    }
    if (!more) break;
    if (m >= kmax) {
      // last round of the slice and the round is full: G += X Y^T in place
      for (int r = tid; r < n; r += SB_T) {
        for (int j = 0; j < m; ++j) {
          cplx x = make_double2(0.0, 0.0), y = make_double2(0.0, 0.0);
          for (int l = 0; l <= j; ++l) {
            const int P = s_aP[l];
            const cplx g = a.G[P + (long long)r * n];
            x = cfma(a.G[r + (long long)P * n], Cm[j][l], x);
            y = cfma(make_double2((r == P ? 1.0 : 0.0) - g.x, -g.y), Dm[j][l], y);
          }
          a.X[r + (long long)j * n] = x;
          a.Y[r + (long long)j * n] = y;
        }
      }
      __syncthreads();
      for (int r = tid; r < n; r += SB_T) {
        for (int c = 0; c < n; ++c) {
          cplx acc = a.G[r + (long long)c * n];
          for (int j = 0; j < m; ++j) acc = cfma(a.X[r + (long long)j * n], a.Y[c + (long long)j * n], acc);
          a.G[r + (long long)c * n] = acc;
        }
      }
      m = 0;
      __syncthreads();
      gather(vr[cur], a.n_op - pos < SB_V ? a.n_op - pos : SB_V, gss, gsa, gas);
    }
    const int nb = a.n_op - pos < SB_V ? a.n_op - pos : SB_V;
    const int m4 = (m + 3) & ~3, mt = (m + 15) >> 4;
    const BVisit* const vc = vr[cur];
    for (int e = here(tid); e < SB_A * 64; e += SB_T) (&Tuw[0][0])[e] = make_double2(0.0, 0.0);
    if (tid <= SB_A) s_pub[tid] = 0;
    if (m > 0) {
      // ---- G[S, A] and Yhat[S, A] ----
      const int ln = here(lane), lr = ln & 15, lk = ln >> 4, td = here(tid);
      const int s = td & (SB_V - 1), Ps = vc[s < nb ? s : 0].P;
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int l = (td >> 5) + (SB_T / SB_V) * e;
        if (l < m) {
          Xa[l][s] = make_double2(gsa[e].x, gsa[e].y);
          Yh[l][s] = make_double2((Ps == s_aP[l] ? 1.0 : 0.0) - gas[e].x, -gas[e].y);
        } else if (l < m4) {
          Xa[l][s] = make_double2(0.0, 0.0);
          Yh[l][s] = make_double2(0.0, 0.0);
        }
      }
      __syncthreads();
      // ---- X[S] = G[S, A] C (waves 0 .. 3) and Y[S] = Yhat[S, A] D (4 .. 7): tile t covers sites
      //      16 (t % 2) and columns 16 (t / 2) of C or D, which are zero below the diagonal ----
      for (int t = wave & 3; t < 2 * mt; t += 4) {
        const int sc = 16 * (t & 1) + lr, j0 = 16 * (t >> 1), kn = m4 < j0 + 16 ? m4 : j0 + 16;
        CTile c;
        if (wave < 4)
          tile_mac(c, 0, kn, lk, [&](int k) { return Cm[j0 + lr][k]; }, [&](int k) { return Xa[k][sc]; });
        else
          tile_mac(c, 0, kn, lk, [&](int k) { return Dm[j0 + lr][k]; }, [&](int k) { return Yh[k][sc]; });
        cplx(*const out)[SB_PS] = wave < 4 ? Xb : Yb;
#pragma unroll
        for (int r = 0; r < 4; ++r) out[j0 + 4 * r + lk][sc] = c.get(r);
      }
      __syncthreads();
    }
    // ---- g = G[S, S] + X[S] Y[S]^T (waves 0 .. 3); T1 = X[S] D^T and T2 = C Y[S]^T (4 .. 7) ----
    if (wave < 4) {
      const int ln = here(lane), lr = ln & 15, lk = ln >> 4;
      const int r = 16 * (wave & 1) + lr, c0 = 16 * (wave >> 1);
      CTile c;
      tile_mac(c, 0, m4, lk, [&](int k) { return Yb[k][c0 + lr]; }, [&](int k) { return Xb[k][r]; });
#pragma unroll
      for (int q = 0; q < 4; ++q) gs[c0 + 4 * q + lk][r] = cadd(gss[q], c.get(q));
    } else {
      const int ln = here(lane), lr = ln & 15, lk = ln >> 4;
      for (int t = wave & 3; t < 4 * mt; t += 4) {
        // rows l0 .. l0 + 15 of C and D begin at column l0
        const int sc = 16 * (t & 1) + lr, l0 = 16 * (t >> 2);
        const bool t1 = (t & 2) == 0;
        CTile c;
        if (t1)
          tile_mac(c, l0, m4, lk, [&](int k) { return Dm[k][l0 + lr]; }, [&](int k) { return Xb[k][sc]; });
        else
          tile_mac(c, l0, m4, lk, [&](int k) { return Cm[k][l0 + lr]; }, [&](int k) { return Yb[k][sc]; });
        cplx(*const out)[SB_PS] = t1 ? Xa : Yh;
#pragma unroll
        for (int r = 0; r < 4; ++r) out[l0 + 4 * r + lk][sc] = c.get(r);
      }
    }
    __syncthreads();

    // ---- the visits ----
    // A rejected proposal leaves g and the phase unchanged, so the decisions of all visits up to
    // the next acceptance follow from the same g: lane v (and v + 32) tests visit v, and the first
    // passing visit at or after k is the next acceptance.  Each lane also forms what its visit
    // would make of the phase and x = Delta / (1 + v_P Delta), v_P = 1 - G_cur(P,P), beside the test.
    if (wave == 0) {
      const int lane = here(tid), v = lane & (SB_V - 1);
      const bool high = lane >= SB_V;
      const BVisit rec = vc[v < nb ? v : nb - 1];
      const int loc = rec.loc;
      const unsigned have = (unsigned)__ballot(v < nb && rec.fnew != VISIT_NONE);
      const int nvis = ~have == 0u ? SB_V : __builtin_ctz(~have);
      // element p of this lane's row or column of g, and of the other half's u_i, w_i
      const cplx* const g_lane = high ? &gs[v][0] : &gs[0][v];
      const int g_step = high ? 1 : SB_PS;
      const cplx* const t_lane = high ? &Tuw[0][0] : &Tuw[0][32];
      cplx d = gs[v][v];
      int k = nvis, mb = 0, js_of = 0;     // js_of: the visit of the block's flip number `lane`
      unsigned live = nvis >= 32 ? ~0u : (1u << nvis) - 1u;
      auto decide = [&](auto NS2) {
        while (true) {
          const cplx ratio = make_double2(fma(-rec.cb.x, d.x, fma(rec.cb.y, d.y, rec.ca.x)),
                                          fma(-rec.cb.x, d.y, fma(-rec.cb.y, d.x, rec.ca.y)));
          cplx rt = ratio;
          if constexpr (decltype(NS2)::value) rt = cmul(ratio, ratio);
          else for (int s = 1; s < a.n_sun; ++s) rt = cmul(rt, ratio);
          const cplx zn = cmul(z, rt);
          const bool pass = fabs(zn.x) > rec.thr * fabs(z.x);
          const cplx delta = rec.delta;
          const cplx den = make_double2(1.0 + (1.0 - d.x) * delta.x + d.y * delta.y,
                                        (1.0 - d.x) * delta.y - d.y * delta.x);
          const double c2 = cabs2(den);
          double rden = __builtin_amdgcn_rcp(c2);          // two Newton steps: full precision
          rden = fma(fma(-c2, rden, 1.0), rden, rden);
          rden = fma(fma(-c2, rden, 1.0), rden, rden);
          const cplx xl = cscale(cmul(delta, cconj(den)), rden);
          // keep these beside the test, where its latency leaves room, instead of after the ballot
          __asm__ volatile("" ::"v"(xl.x), "v"(xl.y), "v"(zn.x), "v"(zn.y));
          const unsigned lo = (unsigned)__ballot(pass) & live;   // lanes 0..31: visits 0..31 of the block
          if (lo == 0) return;
          const int js = __builtin_amdgcn_readfirstlane(__builtin_ctz(lo));
          const int p = __builtin_amdgcn_readlane(loc, js);
          live &= ~1u << js;
          // column p (low lanes) and row p (high lanes) of the current g
          cplx col = g_lane[p * g_step], sum = make_double2(0.0, 0.0);
          const cplx* const oth = t_lane + p;
          // this lane's u_{mb} (low) = -x col, w_{mb} (high) = delta - col, as f0 + f1 col
          cplx f1;
          double f0;
          auto dot = [&](auto C) {
            constexpr int IN = decltype(C)::value;
            cplx mine[IN], their[IN];
#pragma unroll
            for (int i = 0; i < IN; ++i) {
              mine[i] = Tuw[i][lane];
              their[i] = oth[64 * i];
            }
            __builtin_amdgcn_sched_barrier(0);
            // in the shadow of the reads
            const cplx x = lane_c(xl, js);
            f0 = high && loc == p ? 1.0 : 0.0;
            f1 = high ? make_double2(-1.0, 0.0) : make_double2(-x.x, -x.y);
            z = lane_c(renorm_pow2(zn), js);
            js_of = lane == mb ? js : js_of;
#pragma unroll
            for (int i = 0; i < IN; i += 2) {
              col = cfma(mine[i], their[i], col);
              sum = cfma(mine[i + 1], their[i + 1], sum);
            }
          };
          // (u_i, w_i are zero for the flips not yet made)
          if (mb <= 4) dot(std::integral_constant<int, 4>{});
          else if (mb <= 8) dot(std::integral_constant<int, 8>{});
          else {
            dot(std::integral_constant<int, 8>{});
            for (int i0 = 8; i0 < mb; i0 += 4) {
              cplx mine[4], their[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                mine[i] = Tuw[i0 + i][lane];
                their[i] = oth[64 * (i0 + i)];
              }
#pragma unroll
              for (int i = 0; i < 4; i += 2) {
                col = cfma(mine[i], their[i], col);
                sum = cfma(mine[i + 1], their[i + 1], sum);
              }
            }
          }
          col = cadd(col, sum);
          const cplx res = make_double2(fma(f1.x, col.x, fma(-f1.y, col.y, f0)), fma(f1.x, col.y, f1.y * col.x));
          Tuw[mb][lane] = res;
          // g(v, v) += u(v) w(v)
          double ux, uy, wx, wy;
          both_halves(res.x, ux, wx);
          both_halves(res.y, uy, wy);
          d = cfma(make_double2(ux, uy), make_double2(wx, wy), d);
          if (lane == js) {
            s_x[mb] = xl;
            publish(mb, p + 1);
          }
          mb = __builtin_amdgcn_readfirstlane(mb + 1);
          if (m + mb >= kmax || mb >= SB_A) {
            k = js + 1;
            return;
          }
        }
      };
      if (a.n_sun == 2) decide(std::true_type{});
      else decide(std::false_type{});
      if (lane < mb) {
        const BVisit& w = vc[js_of];
        a.f[(long long)a.slice * a.n_op + (a.dir > 0 ? pos + js_of : a.n_op - 1 - pos - js_of)] = (int8_t)w.fnew;
        s_aP[m + lane] = w.P;
      }
      if (lane == 0) {
        s_mb = mb;
        s_k = k;
        s_stopped = k == nvis && nvis < nb;   // the random stream ends here
        publish(mb, SB_FIN);
      }
    } else if (wave <= 2) {
      // ---- the new columns of C (wave 1) and D (wave 2), row l in lane l ----
      const bool isc = wave == 1;
      const int l = here(lane), lc = l < SB_K ? l : SB_K - 1;
      const cplx* const T = isc ? &Yh[lc][0] : &Xa[lc][0];   // T2(l, :) / T1(:, l)
      const cplx* const N = &Tuw[0][isc ? 32 : 0];           // w_i(p) / u_i(p)
      cplx* const out = isc ? &Cm[m][0] : &Dm[m][0];
      int j = 0;
      while (true) {
        const int pub = __hip_atomic_load(&s_pub[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        lds_acquire();
        if (pub == 0) {
          __builtin_amdgcn_s_sleep(1);
          continue;
        }
        if (pub == SB_FIN) break;             // the deciding wave always ends with SB_FIN
        const int p = pub - 1;
        const cplx x = s_x[j];
        cplx acc = l < m ? T[p] : make_double2(0.0, 0.0), acc1 = make_double2(0.0, 0.0);
        for (int i0 = 0; i0 < j; i0 += 4) {
          cplx mine[4], their[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int ii = i0 + i < j ? i0 + i : 0;
            mine[i] = l < SB_K ? out[ii * SB_PL + l] : make_double2(0.0, 0.0);
            their[i] = i0 + i < j ? N[64 * ii + p] : make_double2(0.0, 0.0);
          }
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            acc = cfma(mine[i], their[i], acc);
            acc1 = cfma(mine[i + 1], their[i + 1], acc1);
          }
        }
        acc = cadd(acc, acc1);
        const double dl = l == m + j ? 1.0 : 0.0;
        const cplx r = isc ? cmul(make_double2(-x.x, -x.y), make_double2(dl + acc.x, acc.y))
                           : make_double2(dl - acc.x, -acc.y);
        if (l < SB_K) out[j * SB_PL + l] = r;
        ++j;
      }
      // zero up to a whole k-step of the products
      for (; (m + j) & 3; ++j)
        if (l < SB_K) out[j * SB_PL + l] = make_double2(0.0, 0.0);
    } else if (wave == SB_W - 1) {
      // the records of the block after this one, if this one is not cut short
      records(pos + nb, cur ^ 1);
    }
    __syncthreads();
    const int mb = s_mb;
    const int k = s_k;
    stopped = s_stopped != 0;
    m += mb;
    nvisits += k;
    naccepts += mb;
    cut = k < nb;                            // the next block does not start where the records do
    pos += k;
  }
  // ---- the round's flush operands: C, D and the site list ----
  for (int e = tid; e < SB_K * m; e += SB_T) {
    const int l = e & (SB_K - 1), j = e / SB_K;
    a.CD[l + CHAIN_CD_LD * j] = Cm[j][l];
    a.CD[l + CHAIN_CD_LD * (CHAIN_BLOCK_KMAX + j)] = Dm[j][l];
  }
  if (tid < CHAIN_KMAX) a.amap[tid] = tid < m ? s_aP[tid] : 0;
  if (tid == 0) {
    st->phase = cscale(z, 1.0 / sqrt(cabs2(z)));
    st->nc = st0.nc + nvisits;
    st->acc = st0.acc + naccepts;
    st->m = m;
    const int sl = st0.slice_acc + (int)naccepts;
    st->slice_acc = sl;
    if (stopped) {
      st->status = 1;
      st->rng_pos = st0.rng_pos + (unsigned long long)a.uoff[pos];
    }
    if (stopped || pos >= a.n_op) {
      // the slice is done (a stopped one is not revisited) and the stream behind it
      if (!stopped) st->rng_pos = st0.rng_pos + (unsigned long long)a.per;
      if (sl > st0.max_slice_acc) st->max_slice_acc = sl;
      pos = a.n_op;
    }
    st->pos = pos;
  }
}

// Diagonal exponentials of slices [s0, s0 + ns): for each site i,
//   d(i) = prod_{ops at i} E_exp(op, f),  dinv(i) = prod E_exp(op, -f),  dconj(i) = conj(d(i)).
__global__ void dvec_kernel(const int8_t* __restrict__ f, int n_op, int s0, int ns, int n,
                            const int* __restrict__ site_ptr, const int* __restrict__ site_ops,
                            const cplx* __restrict__ eexp, cplx* __restrict__ d, cplx* __restrict__ dinv,
                            cplx* __restrict__ dconj, long long cs) {
  f = chain_ptr(f, cs);
  eexp = chain_ptr(eexp, cs);
  d = chain_ptr(d, cs);
  dinv = chain_ptr(dinv, cs);
  dconj = chain_ptr(dconj, cs);
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * ns) return;
  const int i = idx % n, s = idx / n;
  const int slice = s0 + s;
  cplx p = make_double2(1.0, 0.0), q = make_double2(1.0, 0.0);
  for (int t = site_ptr[i]; t < site_ptr[i + 1]; ++t) {
    const int op = site_ops[t];
    const int sp = f[(long long)slice * n_op + op];
    p = cmul(p, eexp[op * 5 + (sp + 2)]);
    q = cmul(q, eexp[op * 5 + (2 - sp)]);
  }
  d[idx] = p;
  dinv[idx] = q;
  dconj[idx] = cconj(p);
}

// Op_phase: prod over (op, slice) of exp(i Im(g alpha phi(f))) as a block product.  A thread
// takes operators op = tid, tid + 256, ... over all count / n_op slices, as four partial
// products over the slices (so the factor loads run ahead of the multiplications), combined
// in a fixed order.
__global__ void opphase_kernel(const int8_t* __restrict__ f, long long count, int n_op,
                               const cplx* __restrict__ phasefac, cplx* __restrict__ out, long long cs) {
  __shared__ cplx sh[256];
  f = chain_ptr(f, cs);
  phasefac = chain_ptr(phasefac, cs);
  out = chain_ptr(out, cs);
  const long long nsl = count / n_op;
  cplx p = make_double2(1.0, 0.0);
  for (int op = threadIdx.x; op < n_op; op += blockDim.x) {
    const cplx* pf = phasefac + op * 5 + 2;
    cplx q[4] = {make_double2(1.0, 0.0), make_double2(1.0, 0.0), make_double2(1.0, 0.0), make_double2(1.0, 0.0)};
    long long sl = 0;
    for (; sl + 4 <= nsl; sl += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) q[u] = cmul(q[u], pf[f[(sl + u) * n_op + op]]);
    }
    for (; sl < nsl; ++sl) q[0] = cmul(q[0], pf[f[sl * n_op + op]]);
    p = cmul(p, cmul(cmul(q[0], q[1]), cmul(q[2], q[3])));
  }
  sh[threadIdx.x] = p;
  __syncthreads();
  for (int s = blockDim.x >> 1; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] = cmul(sh[threadIdx.x], sh[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = sh[0];
}

}  // namespace

int launch_philox_fill(double* u, ChainState* st, long long count, int nchain, long long cs, hipStream_t s) {
  if (count <= 0) return ST_NONE;
  hipLaunchKernelGGL(philox_fill_kernel, dim3((unsigned)((count + 255) / 256), 1, nchain), dim3(256), 0, s, u, st,
                     count, cs);
  HIP_OK(hipGetLastError());
  return ST_NONE;
}

int launch_visits(const VisitArgs& a, hipStream_t s) {
  const long long count = (long long)a.n_op * a.ns;
  if (count <= 0) return ST_NONE;
  hipLaunchKernelGGL(visit_kernel, dim3((unsigned)((count + 255) / 256), 1, a.nchain), dim3(256), 0, s, a);
  HIP_OK(hipGetLastError());
  return ST_NONE;
}

int chain_max_delay(int n) {
  (void)n;
  return SB_K;
}

int launch_chain(const ChainArgs& a, hipStream_t s, KTimer* t) {
  if (a.Kmax < 1 || a.Kmax > CHAIN_KMAX) {
    alfq_set_error("launch_chain: K outside [1, CHAIN_KMAX]");
    return ST_GENERIC;
  }
  if (a.Kmax <= SB_K && a.rec) {
    if (t && t->on) {
      if (t->used == t->ev.size()) {
        hipEvent_t e0, e1;
        // no system-scope release when the timing events are recorded: they bracket one
        // kernel on the device and nothing on the host reads its results in between
        HIP_OK(hipEventCreateWithFlags(&e0, hipEventDisableSystemFence));
        HIP_OK(hipEventCreateWithFlags(&e1, hipEventDisableSystemFence));
        t->ev.emplace_back(e0, e1);
      }
      auto& pr = t->ev[t->used++];
      hipExtLaunchKernelGGL(chain_block_kernel, dim3(1, 1, a.nchain), dim3(SB_T), 0, s, pr.first, pr.second, 0, a);
    } else {
      hipLaunchKernelGGL(chain_block_kernel, dim3(1, 1, a.nchain), dim3(SB_T), 0, s, a);
    }
    HIP_OK(hipGetLastError());
    return ST_NONE;
  }
  if (a.nchain > 1) {
    alfq_set_error("launch_chain: delays beyond the block kernel's depth are supported for single chains only");
    return ST_GENERIC;
  }
  hipLaunchKernelGGL(chain_kernel, dim3(1), dim3(256), 0, s, a);
  HIP_OK(hipGetLastError());
  return ST_NONE;
}

int launch_dvec(const int8_t* f, int n_op, int s0, int ns, int n, const int* site_ptr, const int* site_ops,
                const cplx* eexp, cplx* d, cplx* dinv, cplx* dconj, int nchain, long long cs, hipStream_t s) {
  const int total = n * ns;
  hipLaunchKernelGGL(dvec_kernel, dim3((total + 255) / 256, 1, nchain), dim3(256), 0, s, f, n_op, s0, ns, n,
                     site_ptr, site_ops, eexp, d, dinv, dconj, cs);
  HIP_OK(hipGetLastError());
  return ST_NONE;
}

int launch_opphase(const int8_t* f, long long count, int n_op, const cplx* phasefac, cplx* out, int nchain,
                   long long cs, hipStream_t s) {
  hipLaunchKernelGGL(opphase_kernel, dim3(1, 1, nchain), dim3(256), 0, s, f, count, n_op, phasefac, out, cs);
  HIP_OK(hipGetLastError());
  return ST_NONE;
}
