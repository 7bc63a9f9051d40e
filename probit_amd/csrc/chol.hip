// Blocked right-looking Cholesky A = L L^T (lower), replacing B.cholesky
// (probit/implicit/Laplace.py:24, probit/implicit/VB.py:10,25) and the LU
// solve of the Newton system (probit/implicit/solvers.py:24), whose matrix
// -(I + W K) is factored here in the symmetric form B = I + W^1/2 K W^1/2.
//
// Schedule for every batch member at once (c0 = 64k), with the block
// columns grouped into super-steps of G columns:
//   U_k  : left-looking update A_ik -= sum_c L_ic L_kc^T of column k (i >= k)
//          by the earlier columns c of k's super-step, 64x64 MFMA tiles;
//   F_k  : factor and invert diagonal block k (one workgroup per member);
//   P_k  : panel  L_ik = A_ik L_kk^-T for all row blocks i > k, as an MFMA
//          product with the stored inverse of L_kk;
//   O    : after the super-step's last column, the outer update of every
//          lower tile right of it with rank 64 G (FP64 / FP32 operands, or
//          BF16 operands with FP32 accumulation); part of it may run in the
//          next super-step's launch (k_superstep).
// A diagonal block is factored by one workgroup in FP64 together with its
// inverse (four columns at a time, the updates on FP64 MFMA); the FP64
// inverses (DINV) serve the panel products and the triangular solves.
#include <math.h>
#include <stdlib.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "chol_schedule.hpp"
#include "mfma.hpp"
#include "pgp_internal.hpp"

namespace pgp {

__device__ __forceinline__ void lower_tile_c(int t, int& ti, int& tj) {
  int i = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((i + 1) * (i + 2) / 2 <= t) ++i;
  while (i * (i + 1) / 2 > t) --i;
  ti = i;
  tj = t - i * (i + 1) / 2;
}

struct FactorOut {
  void* L;          // factor storage (T), ld
  int64_t ld;
  double* dinv;     // 64x64 FP64 inverse of this block, column-major
  double* logdiag;  // 64 entries for this block (may be null)
  double* diagval;  // 64 entries (may be null)
  int32_t* info;
};

// 1 / sqrt(p) in FP64: hardware estimate and one third-order step
// r <- r (1 + e / 2 + 3 e^2 / 8), e = 1 - p r^2.
__device__ __forceinline__ double rsqrt_f64(double p) {
  const double r = __builtin_amdgcn_rsq(p);
  const double e = fma(-p * r, r, 1.0);
  return fma(r * e, fma(e, 0.375, 0.5), r);
}

// LDS of the diagonal-block factor: the block A ([64][65] doubles) and the
// exchange area of its waves: the finished 16x16 blocks of three row blocks
// and the next diagonal sub-block, as register images.
constexpr int FX_BLOCK = 4 * 64;
constexpr int FX_DOUBLES = 7 * FX_BLOCK;  // two panels' blocks, one sub-block
constexpr int FACTOR_LDS = (TILE * (TILE + 1) + FX_DOUBLES) * 8;

// 1 / d in FP64: hardware estimate and one third-order step
// r <- r (1 + e + e^2), e = 1 - d r (three dependent operations, where two
// Newton steps take four).
__device__ __forceinline__ double rcp_f64(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  const double e = fma(-d, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// v[k]
__device__ __forceinline__ double pick4(const double (&v)[4], int k) {
  const double a = (k & 1) ? v[1] : v[0], b = (k & 1) ? v[3] : v[2];
  return (k & 2) ? b : a;
}

// Factor + inverse of a 64x64 SPD block held in LDS (`A`, [row][65], lower
// triangle read), blocked by 16 columns and, inside, by 4.
//
// The 64 rows of L and the 64 rows of Y = L^-T = I L^-T go through the same
// elimination, 16 rows per wave: in panel s (columns 16 s ..), wave w > s
// finishes block L_ws and wave w <= s finishes block Y_ws, so every panel
// gives each of the four waves one 16x16 block, and the inverse comes along
// with the factor.  A wave's row block stays in registers (R[c]: its block
// column c) in the transposed MFMA D layout, whose register r holds, at lane
// l, row l & 15 and column 4 r + (l >> 4): for the symmetric diagonal
// sub-block that is both D's layout and the layout of a four-column MFMA
// operand, so a rank-4 update needs no data movement.  Every wave eliminates
// the panel's diagonal sub-block S itself (redundantly: the pivots never
// cross waves), four columns at a time: the 4x4 pivot block is read through
// readlane and eliminated as L4 D L4^T in every lane (one reciprocal per
// pivot on the chain; square roots after it), an MFMA each applies L4^-T to
// the four columns of S and of the wave's block, and one each updates the
// rest.  After a panel the waves
// swap their finished blocks through LDS and update the next panel's columns;
// the later columns' update runs inside the next panel, beside its chain.
//
// Bound: the serial chain of 64 pivots in one workgroup.  A 16-column panel
// by one wave with the pivots and column values through readlane (about 125
// ns per pivot), then the inverse after the factor, took 14.1-14.6 us per
// block; this form takes 8.9 us, 8.2 to the inverse's stores (one workgroup
// alone; a four-column step is about 0.32 us).
//
// L (lower) goes to global storage as T, the inverse to o.dinv (FP64).  In
// LDS, L takes A's strict lower triangle and Y its strict upper one (the
// diagonals are dval and rinv).  `published(...)` runs (all threads) once
// the inverse's stores are issued, before L's: a caller that hands DINV to
// other workgroups publishes there.
struct NoPublish {
  __device__ void operator()() const {}
};
template <typename T, typename Pub = NoPublish>
__device__ __forceinline__ void factor_block_blocked(double (*A)[TILE + 1], double* fx, int64_t r0,
                                     const FactorOut& o, Pub published = Pub()) {
  __shared__ double dval[TILE], rinv[TILE];
  const int t = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const unsigned ul = t & 63;
  const int l = (int)ul;
  const int row = l & 15, kq = l >> 4;
  double* sbuf = fx + 6 * FX_BLOCK;
  __builtin_amdgcn_s_setprio(3);
  // entries above the diagonal of S reach only its finished rows and columns
  doublex4 R[4], S;
#pragma unroll
  for (int r = 0; r < 4; ++r) S[r] = A[row][4 * r + kq];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) R[c][r] = c <= w ? A[16 * w + row][16 * c + 4 * r + kq] : 0.0;
  double e[4];  // column kq of the 4x4 identity
#pragma unroll
  for (int q = 0; q < 4; ++q) e[q] = q == kq ? 1.0 : 0.0;
  __syncthreads();  // A is in registers: L and Y take its place
  double lp[4], fp[4][4];  // the previous panel's block and L blocks
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int o16 = 16 * s;
    double* fs = fx + 3 * FX_BLOCK * (s & 1);
    if (s > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) S[r] = sbuf[64 * r + l];
    }
    doublex4 B = R[s];
    if (w == s) {
#pragma unroll
      for (int r = 0; r < 4; ++r) B[r] = row == 4 * r + kq ? 1.0 : 0.0;
    }
    // the wave's finished block and the diagonal one, operand layout; 1 / sqrt(d)
    double lb[4], ls[4], rs[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int p0 = 4 * r;
      // the 4x4 pivot block (lane 16 b + p0 + a: row p0 + a, column p0 + b)
      auto piv = [&](int a, int b) { return bcast(S[r], 16 * b + p0 + a); };
      const double s10 = piv(1, 0), s20 = piv(2, 0), s30 = piv(3, 0);
      double s21 = piv(2, 1), s31 = piv(3, 1), s32 = piv(3, 2);
      double d[4] = {piv(0, 0), piv(1, 1), piv(2, 2), piv(3, 3)};
      // the previous panel's update of the columns after the next panel runs
      // beside the pivots' chain
#pragma unroll
      for (int c = s + 1; c < 4; ++c)
        if (s > 0) R[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(fp[c][r], lp[r], R[c], 0, 0, 0);
      // (the quotients l first, never a product of two entries, whose range is
      // the square of theirs)
      const double r0 = rcp_f64(d[0]);
      const double l10 = s10 * r0, l20 = s20 * r0, l30 = s30 * r0;
      d[1] = fma(-l10, s10, d[1]);
      d[2] = fma(-l20, s20, d[2]);
      d[3] = fma(-l30, s30, d[3]);
      s21 = fma(-l20, s10, s21);
      s31 = fma(-l30, s10, s31);
      s32 = fma(-l30, s20, s32);
      const double r1 = rcp_f64(d[1]);
      const double l21 = s21 * r1, l31 = s31 * r1;
      d[2] = fma(-l21, s21, d[2]);
      d[3] = fma(-l31, s31, d[3]);
      s32 = fma(-l31, s21, s32);
      const double r2 = rcp_f64(d[2]);
      const double l32 = s32 * r2;
      d[3] = fma(-l32, s32, d[3]);
      // X = (the four columns) L4^-T = L D, as X^T = L4^-1 (columns)^T: one
      // 4x4x4 MFMA for the four blocks of four rows, whose result is in the
      // operand layout again.  Lane l brings L4^-1(l & 3, l >> 4).
      double y[4];
      y[0] = e[0];
      y[1] = fma(-l10, e[0], e[1]);
      y[2] = fma(-l21, y[1], fma(-l20, e[0], e[2]));
      y[3] = fma(-l32, y[2], fma(-l31, y[1], fma(-l30, e[0], e[3])));
      const double inv4 = pick4(y, l & 3);
      const double xs = __builtin_amdgcn_mfma_f64_4x4x4f64(inv4, S[r], 0.0, 0, 0, 0);
      const double xb = __builtin_amdgcn_mfma_f64_4x4x4f64(inv4, B[r], 0.0, 0, 0, 0);
      rs[r] = rsqrt_f64(pick4(d, kq));
      ls[r] = xs * rs[r];
      lb[r] = xb * rs[r];
      if (r < 3) {
        S = __builtin_amdgcn_mfma_f64_16x16x4f64(-ls[r], ls[r], S, 0, 0, 0);
        B = __builtin_amdgcn_mfma_f64_16x16x4f64(-ls[r], lb[r], B, 0, 0, 0);
        // both in flight before the next step: B's would otherwise be
        // scheduled late and hold up that step's MFMAs
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (w > s) {
#pragma unroll
      for (int r = 0; r < 4; ++r) fs[(w - 1) * FX_BLOCK + 64 * r + l] = -lb[r];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int cl = 4 * r + kq;  // column inside the panel
      if (w != s) {
        A[16 * w + row][o16 + cl] = lb[r];
      } else {
        A[o16 + row][o16 + cl] = cl > row ? lb[r] : ls[r];
        if (row == cl) {
          dval[o16 + row] = ls[r];
          rinv[o16 + row] = rs[r];
        }
      }
    }
    __syncthreads();
    if (s == 3) break;
    // the wave's later block columns, R_wc -= (its block) L_cs^T: the next
    // panel's at once, the others beside that panel (in rows of L only
    // columns up to the wave's own exist; L_cs = 0 keeps the others zero)
#pragma unroll
    for (int c = s + 1; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        fp[c][r] = (w <= s || c <= w) ? fs[(c - 1) * FX_BLOCK + 64 * r + l] : 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      lp[r] = lb[r];
      R[s + 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(fp[s + 1][r], lb[r], R[s + 1], 0, 0, 0);
    }
    if (w == s + 1) {
#pragma unroll
      for (int r = 0; r < 4; ++r) sbuf[64 * r + l] = R[s + 1][r];
    }
    __syncthreads();
  }
  // a pivot that was not positive left no positive sqrt(d) (NaN)
  if (t < TILE && !(dval[t] > 0.0) && o.info) atomicOr(o.info, PGP_INFO_NOT_PD);
  __builtin_amdgcn_s_setprio(0);
  // columns w + 4q, one row per lane: whole columns per store
  {
    double v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = A[w + 4 * q][l];
    const double dg = rinv[l];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int c = w + 4 * q;
      // coherent: the column kernels hand DINV to other workgroups
      __hip_atomic_store(gbl(o.dinv) + c * TILE + ul, c < l ? v[q] : c == l ? dg : 0.0,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  published();
  if (t < TILE) {
    if (o.logdiag) o.logdiag[t] = log(dval[t]);
    if (o.diagval) o.diagval[t] = dval[t];
  }
  const auto L = gbl((T*)o.L) + r0 + r0 * o.ld;
  double v[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) v[q] = A[l][w + 4 * q];
  const double dg = dval[l];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int c = w + 4 * q;
    if (c <= l) (L + c * o.ld)[ul] = (T)(c == l ? dg : v[q]);
  }
}

// ---- F: first diagonal block -------------------------------------------------
template <typename T>
__device__ void factor_first(const T* A, int64_t ld, const FactorOut& o) {
  __shared__ double blk[TILE][TILE + 1];
  __shared__ double xd[FX_DOUBLES];
  const int m = threadIdx.x & 63, kb = threadIdx.x >> 6;
  for (int q = 0; q < 16; ++q) {
    const int c = kb + 4 * q;
    blk[m][c] = (double)A[(size_t)m + (size_t)c * ld];
  }
  __syncthreads();
  factor_block_blocked<T>(blk, xd, 0, o);
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_factor_first(Prob* const* probs) {
  const Prob& P = *probs[blockIdx.y];
  FactorOut o{P.L, P.Np, P.dinv, P.logdiag, P.diagval, P.info};
  factor_first<T>((const T*)P.L, P.Np, o);
}

// ---- P_k: panel rows below block k --------------------------------------------
// L_ik = A_ik DINV_k^T in the storage type: FP64 MFMA for an FP64 factor,
// FP32 MFMA (the FP64 inverse rounded to FP32) for an FP32 one, whose
// trailing updates carry FP32 rounding anyway.
template <typename T>
__device__ void panel_rows(T* A, int64_t ld, const double* dinv_k, int64_t c0, int64_t r0) {
  constexpr int PP = KP<T>::value;
  __shared__ T As[TILE * PP];
  __shared__ T Bs[TILE * PP];
  // As[p][m] = A(r0 + m, c0 + p); Bs[p][n] = DINV_k(n, p)
  load_block_kmajor<T, T>(As, PP, A, ld, r0, c0);
  {
    const int n = threadIdx.x & 63, pb = threadIdx.x >> 6;
    for (int q = 0; q < 16; ++q) {
      const int p = pb + 4 * q;
      Bs[p * PP + n] = (T)dinv_k[n + p * TILE];
    }
  }
  __syncthreads();
  typename Acc<T>::type acc[2][2];
  zero_acc<T>(acc);
  mma64_kmajor<T>(As, PP, Bs, PP, acc);
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        A[(size_t)(r0 + acc_row<T>(bm, r)) + (size_t)(c0 + acc_col(bn)) * ld] = (T)acc[bm][bn][r];
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_panel(Prob* const* probs, Sched sc, int k) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int64_t c0 = (int64_t)k * TILE;
  const int64_t r0 = c0 + (int64_t)TILE * (bx + 1);
  if (r0 >= P.Np) return;
  panel_rows<T>((T*)P.L, P.Np, P.dinv + (size_t)k * TILE * TILE, c0, r0);
}

// ---- S_k: trailing update; tile (k+1, k+1) then factors its block ----------
template <typename T, int BF16, int FUSE>
__device__ void syrk_tile(T* A, int64_t ld, int64_t c0, int64_t ri, int64_t rj, bool factor,
                          const FactorOut& o) {
  // one LDS arena: MMA operands, then (fused mode, tile (k+1, k+1) only) the
  // two FP64 blocks of the diagonal factorisation
  constexpr int PP = KP<T>::value;
  constexpr int OPER = BF16 ? 2 * TILE * 72 * 2 : 2 * TILE * PP * (int)sizeof(T);
  constexpr int BLK = FUSE ? FACTOR_LDS : 0;
  __shared__ __attribute__((aligned(16))) char arena[OPER > BLK ? OPER : BLK];
  typedef typename Acc<T>::type acc_t;
  acc_t acc[2][2];
  zero_acc<T>(acc);
  // the C tile is loaded first, so its latency overlaps the product
  T cpre[2][2][4];
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        cpre[bm][bn][r] = A[(size_t)(ri + acc_row<T>(bm, r)) + (size_t)(rj + acc_col(bn)) * ld];
  if constexpr (BF16) {
    unsigned short* si = (unsigned short*)arena;
    unsigned short* sj = si + TILE * 72;
    load_block_bf16_mmajor<T>(si, 72, A, ld, ri, c0);
    load_block_bf16_mmajor<T>(sj, 72, A, ld, rj, c0);
    __syncthreads();
    mma64_bf16(si, 72, sj, 72, acc);
  } else {
    T* si = (T*)arena;
    T* sj = si + TILE * PP;
    load_block_kmajor<T, T>(si, PP, A, ld, ri, c0);
    load_block_kmajor<T, T>(sj, PP, A, ld, rj, c0);
    __syncthreads();
    mma64_kmajor<T>(si, PP, sj, PP, acc);
  }
  if constexpr (!FUSE) factor = false;
  double (*blk)[TILE + 1] = (double (*)[TILE + 1])arena;
  if (factor) __syncthreads();  // operands are dead; the arena becomes the block
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn) {
      const int col = acc_col(bn);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = acc_row<T>(bm, r);
        const T v = cpre[bm][bn][r] - acc[bm][bn][r];
        if (factor)
          blk[row][col] = (double)v;
        else
          A[(size_t)(ri + row) + (size_t)(rj + col) * ld] = v;
      }
    }
  if constexpr (FUSE) {
    if (factor) {
      __syncthreads();
      factor_block_blocked<T>(blk, (double*)(blk + TILE), ri, o);
    }
  }
}

// The trailing updates of FP32 factors (outer update, column update, column
// kernel) stage their operands m-major for mma64_f32_mmajor; FP64 factors
// stay k-major and BF16 operands are m-major bf16.  All three kernels use
// the same form, so a tile's update is bitwise the same in each.
template <typename T, int BF16>
struct MmajorF32 {
  static constexpr bool value = std::is_same<T, float>::value && !BF16;
};

// k index of the q-th of the 16 operand values a thread (row m, group kb)
// fetches per 64-column chunk: 16 consecutive k for the m-major FP32 form,
// every fourth k otherwise.  Either way one fetch instruction reads one
// column's 64 consecutive rows.
template <bool MM>
__device__ __forceinline__ int operand_k(int kb, int q) {
  return MM ? 16 * kb + q : kb + 4 * q;
}

// d[m * pitch + 16 kb + q] = v[q], q = 0..15, as four 16-byte stores
// (pitch a multiple of 4).
template <typename T>
__device__ __forceinline__ void stash_f32_mmajor(T* d, int pitch, const T (&v)[16], int m, int kb) {
  static_assert(std::is_same<T, float>::value, "m-major FP32 operands only");
#pragma unroll
  for (int j = 0; j < 4; ++j)
    *(floatx4*)&d[m * pitch + 16 * kb + 4 * j] =
        floatx4{v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]};
}

// d[m * pitch + 16 kb + q] = bf16(v[q]), q = 0..15, as two 16-byte stores
// (pitch a multiple of 8): the same LDS image as one 2-byte store per value.
template <typename T>
__device__ __forceinline__ void stash_bf16_mmajor(unsigned short* d, int pitch, const T (&v)[16],
                                                  int m, int kb) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    u16x8 w;
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = f2bf((float)v[8 * j + e]);
    *(u16x8*)&d[m * pitch + 16 * kb + 8 * j] = w;
  }
}

// Workgroups of one launch are dealt to the 8 XCDs round-robin (workgroup g
// runs on XCD g % 8).  Renumber them so that each XCD gets one contiguous
// run of tiles: neighbouring tiles share panel rows, which then stay in that
// XCD's L2.
__device__ __forceinline__ int xcd_contiguous(int g, int total) {
  const int x = g & 7, q = total >> 3, r = total & 7;
  return x * q + (x < r ? x : r) + (g >> 3);
}

// C(ri.., rj..) -= sum over block columns c in [kc0, kc1) of
// A(ri.., 64c..) A(rj.., 64c..)^T for one 64x64 tile: the rank-64(kc1-kc0)
// update of a super-step, with the next 64-wide chunk of both panels loaded
// into registers while the current one is multiplied from LDS.  C is read
// and written once however long the K range.
// FUSE: the workgroup given factor = true (the tile that becomes the next
// diagonal block) keeps its updated tile in LDS and factors it at once.
// Requires kc1 > kc0 (both callers update by at least one block column).
// SH (BF16 factors, the outer update): the operand chunks come as BF16 from
// the super-step's panel copy (P.panel16, row r at (r - p16_row0) * pitch),
// the same values the stash would convert, so no conversion and half the
// operand bytes.
template <typename T, int BF16, int FUSE, bool SH = false>
__device__ __forceinline__ void syrk_tile_multi(T* A_, int ld_, int kc0, int kc1, int ri_, int rj_,
                                bool factor, const FactorOut& o,
                                const unsigned short* p16 = nullptr, int64_t p16_row0 = 0,
                                int p16_pitch = 0) {
  static_assert(!SH || BF16, "the panel copy holds BF16 operands");
  const auto A = gbl(uniform(A_));
  const int64_t ld = uniform(ld_), ri = uniform(ri_), rj = uniform(rj_);
  constexpr bool MM = MmajorF32<T, BF16>::value;
  constexpr int PITCH = BF16 ? 72 : MM ? 68 : KP<T>::value;
  typedef typename std::conditional<BF16 != 0, unsigned short, T>::type LT;
  constexpr int OPER = 2 * TILE * PITCH * (int)sizeof(LT);
  constexpr int BLK = FUSE ? FACTOR_LDS : 0;
  __shared__ __attribute__((aligned(16))) char arena[OPER > BLK ? OPER : BLK];
  LT* sa = (LT*)arena;
  LT* sb = sa + TILE * PITCH;
  typedef typename Acc<T>::type acc_t;
  const unsigned m = threadIdx.x & 63;
  const int kb = uniform((int)(threadIdx.x >> 6));
  T ra[16], rb[16];
  acc_t acc[2][2];
  zero_acc<T>(acc);
  // the m-major FP32 and BF16 stagings take 16 consecutive k per thread
  constexpr bool CK = MM || BF16;
  constexpr int KS = CK ? 1 : 4;
  u16x8 ua[2], ub[2];  // SH: a thread's 16 BF16 operand values of each row
  auto fetch = [&](int c) {
    if constexpr (SH) {
      const size_t kofs = (size_t)(c - kc0) * TILE + 16 * kb;
      const unsigned short* pa = p16 + (size_t)(ri + m - p16_row0) * p16_pitch + kofs;
      const unsigned short* pb = p16 + (size_t)(rj + m - p16_row0) * p16_pitch + kofs;
      ua[0] = *(const u16x8*)pa;
      ua[1] = *(const u16x8*)(pa + 8);
      ub[0] = *(const u16x8*)pb;
      ub[1] = *(const u16x8*)(pb + 8);
    } else {
      auto pa = A + (ri + ((int64_t)c * TILE + operand_k<CK>(kb, 0)) * ld);
      auto pb = A + (rj + ((int64_t)c * TILE + operand_k<CK>(kb, 0)) * ld);
#pragma unroll
      for (int q = 0; q < 16; ++q, pa += KS * ld, pb += KS * ld) {
        ra[q] = pa[m];
        rb[q] = pb[m];
      }
    }
  };
  fetch(kc0);
  auto stash = [&](LT* da, LT* db) {
    if constexpr (SH) {
      *(u16x8*)&da[m * PITCH + 16 * kb] = ua[0];
      *(u16x8*)&da[m * PITCH + 16 * kb + 8] = ua[1];
      *(u16x8*)&db[m * PITCH + 16 * kb] = ub[0];
      *(u16x8*)&db[m * PITCH + 16 * kb + 8] = ub[1];
    } else if constexpr (MM) {
      stash_f32_mmajor(da, PITCH, ra, m, kb);
      stash_f32_mmajor(db, PITCH, rb, m, kb);
    } else if constexpr (BF16) {
      stash_bf16_mmajor(da, PITCH, ra, m, kb);
      stash_bf16_mmajor(db, PITCH, rb, m, kb);
    } else {
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int k = kb + 4 * q;
        da[k * PITCH + m] = ra[q];
        db[k * PITCH + m] = rb[q];
      }
    }
  };
  auto mma = [&](const LT* da, const LT* db) {
    if constexpr (BF16)
      mma64_bf16(da, PITCH, db, PITCH, acc);
    else if constexpr (MM)
      mma64_f32_mmajor(da, PITCH, db, PITCH, acc);
    else
      mma64_kmajor<T>(da, PITCH, db, PITCH, acc);
  };
  for (int c = kc0; c < kc1 - 1; ++c) {
    if (c > kc0) __syncthreads();  // the previous chunk's products are done with LDS
    stash(sa, sb);
    __syncthreads();
    fetch(c + 1);
    mma(sa, sb);
  }
  if (kc1 - 1 > kc0) __syncthreads();
  stash(sa, sb);
  __syncthreads();
  // the C tile is loaded during the last chunk's product (the fetch
  // registers are free then), so its latency overlaps the product
  T cpre[2][2][4];
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        cpre[bm][bn][r] = A[(size_t)(ri + acc_row<T>(bm, r)) + (size_t)(rj + acc_col(bn)) * ld];
  mma(sa, sb);
  if constexpr (!FUSE) factor = false;
  double (*blk)[TILE + 1] = (double (*)[TILE + 1])arena;
  if (factor) __syncthreads();  // operands are dead; the arena becomes the block
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn) {
      const int col = acc_col(bn);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = acc_row<T>(bm, r);
        const T v = cpre[bm][bn][r] - (T)acc[bm][bn][r];
        if (factor)
          blk[row][col] = (double)v;
        else
          A[(size_t)(ri + row) + (size_t)(rj + col) * ld] = v;
      }
    }
  if constexpr (FUSE) {
    if (factor) {
      __syncthreads();
      factor_block_blocked<T>(blk, (double*)(blk + TILE), ri, o);
    }
  }
}

// Left-looking update of block column j inside its super-step [s0, ...):
// tiles (i, j), i >= j, receive A_ij -= sum_{c in [s0, j)} L_ic L_jc^T in one
// product (the same arithmetic as the column kernel's update), just before
// block j is factored and its panel formed.  FUSE: the workgroup of tile
// (j, j) factors that block at once.
template <typename T, int BF16, int FUSE>
__global__ __launch_bounds__(NTHREADS) void k_col_update(Prob* const* probs, Sched sc, int j,
                                                         int s0) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int nb = P.Np / TILE;
  const int i = j + bx;
  if (i >= nb) return;
  const int c1 = j * TILE;
  const FactorOut o{P.L, P.Np, P.dinv + (size_t)j * TILE * TILE,
                    P.logdiag ? P.logdiag + c1 : nullptr, P.diagval ? P.diagval + c1 : nullptr,
                    P.info};
  syrk_tile_multi<T, BF16, FUSE>((T*)P.L, P.Np, s0, j, i * TILE, j * TILE,
                                 FUSE && i == j, o);
}

// Tile t of a Tk x Tk lower triangle in blocked order: super-tiles of 8 x 8
// tiles, super-rows in order, the super-tiles of a super-row left to right
// (the diagonal one as a lower triangle), row-major inside.  Consecutive
// tiles (those one XCD runs together) then share a few 64-row panels, which
// stay in that XCD's L2.  Super-rows before I hold 32 I^2 + 4 I tiles.
__device__ __forceinline__ void blocked_tile(int t, int Tk, int& ti, int& tj) {
  int I = (int)((sqrt(16.0 + 128.0 * (double)t) - 4.0) / 64.0);
  while (32 * (I + 1) * (I + 1) + 4 * (I + 1) <= t) ++I;
  while (32 * I * I + 4 * I > t) --I;
  const int u = t - (32 * I * I + 4 * I);
  const int rI = min(8, Tk - 8 * I);
  const int off = rI * 8 * I;
  if (u < off) {
    const int J = u / (rI * 8), v = u - J * rI * 8;
    ti = 8 * I + (v >> 3);
    tj = 8 * J + (v & 7);
  } else {
    int a, c;
    lower_tile_c(u - off, a, c);
    ti = 8 * I + a;
    tj = 8 * I + c;
  }
}

// Tile t of the first w tile columns of a lower triangle: its top w x w
// triangle, then whole rows.
__device__ __forceinline__ void column_tile(int t, int w, int& ti, int& tj) {
  const int v = t - w * (w + 1) / 2;
  if (v < 0) {
    lower_tile_c(t, ti, tj);
  } else {
    ti = w + v / w;
    tj = v % w;
  }
}

// Outer update closing a super-step [s0, s_end): every lower tile (i, j),
// s_end <= j <= i, j < s_end + wd, gets A_ij -= sum_{c in [s0, s_end)} L_ic
// L_jc^T.
template <typename T, int BF16, int FUSE>
__global__ __launch_bounds__(NTHREADS) void k_syrk_outer(Prob* const* probs, Sched sc, int s0,
                                                         int s_end, int wd) {
  int bx;
  const int g = xcd_contiguous(blockIdx.x, gridDim.x);
  const Prob& P = *probs[sched_member(sc, g, bx)];
  const int Tk = uniform(P.Np) / TILE - s_end;
  if (Tk <= 0 || bx >= outer_tiles64(Tk, wd)) return;
  int ti, tj;
  if (wd >= Tk)
    blocked_tile(bx, Tk, ti, tj);
  else
    column_tile(bx, wd, ti, tj);
  ti = uniform(ti);  // (the square root's)
  tj = uniform(tj);
  const int c1 = s_end * TILE;
  const FactorOut o{P.L, P.Np, P.dinv + (size_t)s_end * TILE * TILE,
                    P.logdiag ? P.logdiag + c1 : nullptr, P.diagval ? P.diagval + c1 : nullptr,
                    P.info};
  // BF16 factors read the operands from the panel copy (k_panel_bf16)
  syrk_tile_multi<T, BF16, FUSE, BF16 != 0>(
      (T*)P.L, P.Np, s0, s_end, (s_end + ti) * TILE, (s_end + tj) * TILE,
      FUSE && ti == 0 && tj == 0, o, P.panel16, (int64_t)s_end * TILE, P.panel16_pitch);
}

// The outer update in tiles of 128 x 128, a wave 64 x 64 of it: half the
// operand bytes per flop of the 64-tiles.  The operands come in chunks of KC
// columns through two LDS buffers (one barrier per chunk), a chunk fetched
// into registers during the product before its own.  The k order inside and
// across the MFMA steps is the 64-tile's, so both give the same bits.  Bound
// by the MFMAs and then C's bytes (of N = 12288's 755 us a launch of 3496
// tiles, K = 384, 704 remain without the loop's fetches and LDS stores: 560 of
// MFMAs, and C's 180 partly under them); BF16 by C's bytes.  Per launch, 64-
// against 128-tiles: FP64, 184 block rows, K = 512: 1570 -> 1188 us (60
// TFLOP/s); FP32, 244, K = 768: 1946 -> 1569 (121); BF16, 248, K = 512: 622 ->
// 323.  A third of FP32's gain is the addresses: tile indices from a square
// root and descriptor fields arrive in vector registers, and 80 64-bit vector
// additions per chunk then hold up the MFMAs (hence uniform()).
template <typename T, int BF16>
struct Outer128;
template <>
struct Outer128<double, 0> {
  static constexpr int KC = 16, P = 144;  // k-major, rows of 128
  typedef double LT;
  static constexpr int OP = KC * P;  // elements of one operand chunk
};
template <>
struct Outer128<float, 0> {
  static constexpr int KC = 32, P = 36;  // m-major; 16-byte reads, 4 = P mod 32
  typedef float LT;
  static constexpr int OP = 128 * P;
};
template <>
struct Outer128<float, 1> {
  static constexpr int KC = 64, P = 72;  // m-major
  typedef unsigned short LT;
  static constexpr int OP = 128 * P;
};

template <typename T, int BF16>
constexpr OuterOp outer_op() {
  return std::is_same<T, double>::value ? OUTER_FP64 : BF16 ? OUTER_BF16 : OUTER_FP32;
}

// Tile bx (blocked_tile's order) of the lower triangle from block row and
// column `base` on, or (wd > 0) bx of its first wd block columns (even):
// A -= the product of the panel columns [s0, s1), s1 <= base.  lds: 4 OP
// elements.  All threads call it.
template <typename T, int BF16>
__device__ __forceinline__ void outer128_tile(const Prob& P, int bx, int s0, int s1, int base,
                                              int wd, typename Outer128<T, BF16>::LT* lds) {
  typedef Outer128<T, BF16> O;
  typedef typename O::LT LT;
  constexpr bool F64 = std::is_same<T, double>::value;
  const int Tb = uniform(P.Np) / TILE - base, Tk = (Tb + 1) / 2;
  int ti, tj;
  if (wd == 0)
    blocked_tile(bx, Tk, ti, tj);
  else
    column_tile(bx, wd / 2, ti, tj);
  ti = uniform(ti);  // (the square root's)
  tj = uniform(tj);
  const int64_t ld = uniform(P.Np);
  const int64_t ri = (int64_t)base * TILE + 128 * ti, rj = (int64_t)base * TILE + 128 * tj;
  // an odd last block row: the upper 64 rows of its tile stand in for the
  // missing ones, and the waves they belong to have nothing to do
  const bool fulli = 2 * ti + 1 < Tb, fullj = 2 * tj + 1 < Tb;
  const int t = threadIdx.x, l = t & 63, w = uniform(t >> 6);
  const int wr = 64 * (w >> 1), wc = 64 * (w & 1);
  const bool active = (wr == 0 || fulli) && (wc == 0 || fullj) && (ti != tj || wr >= wc);
  const int lr = l & 15, lk = l >> 4;
  typedef typename Acc<T>::type acc_t;
  acc_t acc[4][4];  // [row block][column block]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = (T)0;
  const auto A = gbl(uniform((T*)P.L));
  const int nc = (s1 - s0) * (TILE / O::KC);

  // ---- a chunk of both operands: registers, LDS, MFMA steps ----
  typedef double d2 __attribute__((ext_vector_type(2)));
  typedef typename std::conditional<
      F64, d2, typename std::conditional<BF16 != 0, u16x8, floatx4>::type>::type chunk_t;
  typedef typename std::conditional<F64, double, chunk_t>::type frag_t;
  chunk_t ra[4], rb[4];
  const int mt = F64 ? 2 * l : BF16 ? t >> 1 : t & 127;  // the thread's row of the tile
  const unsigned ma = fulli ? mt : mt & 63, mb = fullj ? mt : mt & 63;
  const unsigned pitch = uniform(P.panel16_pitch);  // (BF16: row s1 TILE is the first)
  const auto p16 = gbl(uniform((const unsigned short*)P.panel16)) +
                   (int64_t)(base - s1) * TILE * pitch;
  // Parts 0..3 of chunk c into registers, and from there into LDS buffer u.
  auto fetch = [&](int c, int q) {
    if constexpr (F64) {
      typedef const __attribute__((address_space(1))) d2* gd2;
      const auto p = A + ((int64_t)s0 * TILE + c * O::KC + w + 4 * q) * ld;
      ra[q] = *(gd2)(p + ri + ma);
      rb[q] = *(gd2)(p + rj + mb);
    } else if constexpr (BF16 != 0) {
      typedef const __attribute__((address_space(1))) u16x8* gu8;
      const unsigned h = 32 * (t & 1) + 8 * q;
      ra[q] = *(gu8)(p16 + (128 * ti * (int64_t)pitch + c * O::KC) + (ma * pitch + h));
      rb[q] = *(gu8)(p16 + (128 * tj * (int64_t)pitch + c * O::KC) + (mb * pitch + h));
    } else {
      // LDS column e holds k = 16 (e / 8) + 8 (chunk & 1) + e % 8 of a block of
      // 64: the k of eight of its sixteen MFMA steps (mma64_f32_mmajor's order)
      auto p = A + ((int64_t)s0 * TILE + (c >> 1) * TILE + 32 * (w >> 1) + 8 * (c & 1) +
                    16 * (q >> 1) + 4 * (q & 1)) * ld;
#pragma unroll
      for (int e = 0; e < 4; ++e, p += ld) {
        ra[q][e] = (p + ri)[ma];
        rb[q][e] = (p + rj)[mb];
      }
    }
  };
  auto stash = [&](int u, int q) {
    LT* da = lds + 2 * u * O::OP;
    LT* db = da + O::OP;
    const int o = F64 ? (w + 4 * q) * O::P + 2 * l
                      : mt * O::P + (BF16 ? 32 * (t & 1) + 8 * q : 16 * (w >> 1) + 4 * q);
    *(chunk_t*)&da[o] = ra[q];
    *(chunk_t*)&db[o] = rb[q];
  };
  // Operands of MFMA group s (F64: one step of four k; FP32: four steps; BF16:
  // one of 32 k).
  auto read = [&](const LT* da, int s, frag_t (&a)[4], frag_t (&b)[4]) {
    const LT* db = da + O::OP;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int oa = F64 ? (4 * s + lk) * O::P + wr + 16 * i + lr
                         : (wr + 16 * i + lr) * O::P + 8 * lk + (BF16 ? 32 : 4) * s;
      const int ob = F64 ? (4 * s + lk) * O::P + wc + 16 * i + lr
                         : (wc + 16 * i + lr) * O::P + 8 * lk + (BF16 ? 32 : 4) * s;
      a[i] = *(const frag_t*)&da[oa];
      b[i] = *(const frag_t*)&db[ob];
    }
  };
  constexpr int NG = F64 ? 4 : 2;  // MFMA groups of a chunk
  auto mfmas = [&](frag_t (&a)[4], frag_t (&b)[4], auto part) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < (F64 || BF16 ? 1 : 4); ++e) {
      if constexpr (!F64 && !BF16) {
        part(e);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // (FP64 transposed: rows of D are the tile's columns, so that 16
          // lanes hold consecutive rows of C, whole 128-byte lines)
          if constexpr (F64)
            acc[i][j] = mfma16(b[j], a[i], acc[i][j]);
          else if constexpr (BF16 != 0)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, a[i]), __builtin_bit_cast(bf16x8, b[j]), acc[i][j], 0,
                0, 0);
          else
            acc[i][j] = mfma16(a[i][e], b[j][e], acc[i][j]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Chunk c is multiplied from one buffer while chunk c + 1 goes from the
  // registers into the other and chunk c + 2 is fetched, a part at a time
  // between the MFMA groups.
  auto chunk = [&](int c, auto st, auto ft) {
    __syncthreads();  // chunk c is in its buffer; the other one is read
    const LT* da = lds + 2 * (c & 1) * O::OP;
    auto part = [&](int q) {
      if constexpr (st.value) stash((c & 1) ^ 1, q);
      if constexpr (ft.value) fetch(c + 2, q);
    };
    if (active) {
      frag_t a[2][4], b[2][4];
      read(da, 0, a[0], b[0]);
#pragma unroll
      for (int s = 0; s < NG; ++s) {
        if (s + 1 < NG) read(da, s + 1, a[(s & 1) ^ 1], b[(s & 1) ^ 1]);
        if constexpr (F64) part(s);
        if constexpr (BF16 != 0) {
          part(2 * s);
          part(2 * s + 1);
        }
        mfmas(a[s & 1], b[s & 1], [&](int e) {
          if ((e & 1) == 0) part(2 * s + e / 2);
        });
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) part(q);
    }
  };
#pragma unroll
  for (int q = 0; q < 4; ++q) fetch(0, q);
#pragma unroll
  for (int q = 0; q < 4; ++q) stash(0, q);
  if (nc > 1)
#pragma unroll
    for (int q = 0; q < 4; ++q) fetch(1, q);
  // (FP32: C arrives during the last chunk's product)
  typedef __attribute__((address_space(1))) floatx4* gf4;
  const auto C = A + (ri + wr + (rj + wc) * ld);
  floatx4 cv[F64 ? 1 : 4][4];
  int c = 0;
  for (; c + 2 < nc; ++c) chunk(c, std::true_type{}, std::true_type{});
  if (c + 1 < nc) chunk(c++, std::true_type{}, std::false_type{});
  if constexpr (!F64) {
    if (active) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          cv[i][j] = *(gf4)(C + (16 * i + 16 * j * ld) + (4 * lk + lr * (unsigned)ld));
    }
  }
  chunk(c, std::false_type{}, std::false_type{});
  if (!active) return;
  // ---- C -= acc ----
  if constexpr (F64) {
    const unsigned o = lr + lk * (unsigned)ld;
    double v[2][16];
    auto load = [&](int j) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[j & 1][4 * i + r] = (C + (16 * i + (16 * j + 4 * r) * ld))[o];
    };
    load(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < 3) load(j + 1);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          (C + (16 * i + (16 * j + 4 * r) * ld))[o] = v[j & 1][4 * i + r] - acc[i][j][r];
    }
  } else {
    const unsigned o = 4 * lk + lr * (unsigned)ld;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) *(gf4)(C + (16 * i + 16 * j * ld) + o) = cv[i][j] - acc[i][j];
  }
}

// The outer update closing a super-step [s0, s_end) in outer_tiles128's tiles.
template <typename T, int BF16>
__global__ __launch_bounds__(NTHREADS, 2) void k_syrk_outer128(Prob* const* probs, Sched sc,
                                                               int s0, int s_end, int wd) {
  __shared__ __attribute__((aligned(16))) typename Outer128<T, BF16>::LT
      lds[4 * Outer128<T, BF16>::OP];
  int bx;
  const int g = xcd_contiguous(blockIdx.x, gridDim.x);
  const Prob& P = *probs[sched_member(sc, g, bx)];
  int base = s_end;
  if (wd > 0) {
    const int tb = uniform(P.Np) / TILE - s_end, n = tiles128(tb) - tiles128(tb - wd);
    if (bx >= n) {
      bx -= n;
      base += wd;
      wd = 0;
    }
  }
  outer128_tile<T, BF16>(P, bx, s0, s_end, base, wd, lds);
}

// BF16 copy of the panel columns [s0, s_end) of the rows below the
// super-step, for its outer update: one workgroup per 64-row block, each
// thread converting 16 consecutive columns of one row per block column.
// The conversion is the one the update's stash applies (f2bf).
__global__ __launch_bounds__(NTHREADS) void k_panel_bf16(Prob* const* probs, Sched sc, int s0,
                                                         int s_end) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int nb = P.Np / TILE;
  if (bx >= nb - s_end) return;
  const int m = threadIdx.x & 63, kb = threadIdx.x >> 6;
  const int64_t r = (int64_t)(s_end + bx) * TILE + m;
  const auto A = gbl((const float*)P.L);
  unsigned short* dst = P.panel16 + (size_t)(r - (int64_t)s_end * TILE) * P.panel16_pitch;
  for (int c = s0; c < s_end; ++c) {
    float v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q)
      v[q] = A[(size_t)r + (size_t)((int64_t)c * TILE + 16 * kb + q) * P.Np];
    stash_bf16_mmajor(dst + (size_t)(c - s0) * TILE, 0, v, 0, kb);
  }
}

// ---- one launch per block column ---------------------------------------------
// C = A(ri.., rj..) - sum_{c in [kc0, kc1)} A(ri.., 64c..) A(rj.., 64c..)^T,
// computed as the trailing updates are (T / BF16 operands on MFMA, result
// rounded to T), then held in LDS as FP64: out[r][c] (kmajor = false) or
// out[c][r] (kmajor = true).  `arena` holds the operands first.
// SAME: the diagonal tile (ri == rj), whose two operand rows are the same:
// fetched and staged once.
template <typename T, int BF16, typename OT, bool SAME = false>
__device__ __forceinline__ void update_tile_to_lds(const T* A_, int64_t ld, int kc0, int kc1,
                                                   int64_t ri, int64_t rj, char* arena, OT* out,
                                                   int opitch, bool kmajor) {
  auto A = gbl(A_);
  constexpr bool MM = MmajorF32<T, BF16>::value;
  constexpr int PITCH = BF16 ? 72 : MM ? 68 : KP<T>::value;
  typedef typename std::conditional<BF16 != 0, unsigned short, T>::type LT;
  typedef typename Acc<T>::type acc_t;
  LT* sa = (LT*)arena;
  LT* sb = SAME ? sa : sa + TILE * PITCH;
  const int m = threadIdx.x & 63, kb = threadIdx.x >> 6;
  acc_t acc[2][2];
  zero_acc<T>(acc);
  if (kc1 > kc0) {
    T ra[16], rb[16];
    auto fetch = [&](int c) {
      const int64_t c0 = (int64_t)c * TILE;
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int k = operand_k<MM>(kb, q);
        ra[q] = A[(size_t)(ri + m) + (size_t)(c0 + k) * ld];
        if constexpr (!SAME) rb[q] = A[(size_t)(rj + m) + (size_t)(c0 + k) * ld];
      }
    };
    fetch(kc0);
    for (int c = kc0; c < kc1; ++c) {
      if (c > kc0) __syncthreads();
      if constexpr (MM) {
        stash_f32_mmajor(sa, PITCH, ra, m, kb);
        if constexpr (!SAME) stash_f32_mmajor(sb, PITCH, rb, m, kb);
      } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int k = kb + 4 * q;
          if constexpr (BF16) {
            sa[m * PITCH + k] = f2bf((float)ra[q]);
            if constexpr (!SAME) sb[m * PITCH + k] = f2bf((float)rb[q]);
          } else {
            sa[k * PITCH + m] = ra[q];
            if constexpr (!SAME) sb[k * PITCH + m] = rb[q];
          }
        }
      }
      __syncthreads();
      if (c + 1 < kc1) fetch(c + 1);
      if constexpr (BF16)
        mma64_bf16(sa, PITCH, sb, PITCH, acc);
      else if constexpr (MM)
        mma64_f32_mmajor(sa, PITCH, sb, PITCH, acc);
      else
        mma64_kmajor<T>(sa, PITCH, sb, PITCH, acc);
    }
    __syncthreads();  // operands are dead: `out` may overlay them
  }
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn) {
      const int col = acc_col(bn);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = acc_row<T>(bm, r);
        const T v = A[(size_t)(ri + row) + (size_t)(rj + col) * ld] - (T)acc[bm][bn][r];
        if (kmajor)
          out[col * opitch + row] = (OT)v;
        else
          out[row * opitch + col] = (OT)v;
      }
    }
  __syncthreads();
}

// LDS of the column kernels, used in turn by a tile update's operands, its
// FP64 result with the diagonal factor's inverse blocks (FACTOR_LDS), or a
// row tile's panel-product operands.
template <typename T, int BF16>
constexpr int col_arena_bytes() {
  constexpr int PP = KP<T>::value;
  constexpr int PITCH = BF16 ? 72 : MmajorF32<T, BF16>::value ? 68 : PP;
  constexpr int oper = 2 * TILE * PITCH * (BF16 ? 2 : (int)sizeof(T));
  constexpr int prod = 2 * TILE * PP * (int)sizeof(T);
  constexpr int a = oper > prod ? oper : prod;
  return a > FACTOR_LDS ? a : FACTOR_LDS;
}

// Column j of every member in one launch.  Tickets [0, nd) are the diagonal
// workgroups of members 0..nd-1 (members are sorted by size, so these are
// the members with more than j block columns); the rest are row workgroups
// listed by `rows`.  Within the super-step [s0, ...), column j has not yet
// received the updates of columns s0..j-1; each workgroup applies them to
// its own tile (left-looking, rank 64 (j - s0)).  The diagonal workgroup
// then factors and inverts block j and publishes; a row workgroup waits for
// its member's publication and forms L_ij = C_ij DINV_j^T (FP64 MFMA).
template <typename T, int BF16>
__global__ __launch_bounds__(NTHREADS) void k_column(Prob* const* probs, Sched rows, int nd,
                                                     uint32_t* ticket, uint32_t epoch, int j,
                                                     int s0) {
  __shared__ __attribute__((aligned(16))) char arena_b[col_arena_bytes<T, BF16>()];
  double (*arena)[TILE + 1] = (double (*)[TILE + 1])arena_b;
  double* xd = (double*)arena_b + TILE * (TILE + 1);
  __shared__ int s_val;
  const int t = take_ticket(ticket, &s_val);
  if ((unsigned)t >= gridDim.x) {  // counter not zero at launch: nothing to take
    flag_members_stalled(probs, nd);  // the diagonal workgroups' members: every member
    return;
  }
  const int64_t c0 = (int64_t)j * TILE;
  if (t < nd) {
    const Prob& P = *probs[t];
    update_tile_to_lds<T, BF16, double, true>((const T*)P.L, P.Np, s0, j, c0, c0, (char*)arena,
                                        &arena[0][0], TILE + 1, false);
    FactorOut o{P.L, P.Np, P.dinv + (size_t)j * TILE * TILE,
                P.logdiag ? P.logdiag + c0 : nullptr, P.diagval ? P.diagval + c0 : nullptr,
                P.info};
    factor_block_blocked<T>(arena, xd, c0, o);
    // every wave's DINV stores complete, then publish
    publish_wait();
    __syncthreads();
    if (threadIdx.x == 0)
      __hip_atomic_store(P.progress, ((uint64_t)epoch << 32) | 1u, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  int local;
  const Prob& P = *probs[sched_member(rows, t - nd, local)];
  const int64_t ri = c0 + (int64_t)TILE * (local + 1);
  // the panel product runs in the storage type (as panel_rows)
  constexpr int PP = KP<T>::value;
  T* ck = (T*)&arena[0][0];
  T* bk = ck + TILE * PP;
  update_tile_to_lds<T, BF16, T>((const T*)P.L, P.Np, s0, j, ri, c0, (char*)arena, ck, PP, true);
  if (threadIdx.x == 0) wait_progress(P.progress, epoch, 1, P.info);
  __syncthreads();
  // B[p][n] = DINV_j(n, p), published in this launch: coherent loads
  const double* Dj = P.dinv + (size_t)j * TILE * TILE;
  {
    const int n = threadIdx.x & 63, pb = threadIdx.x >> 6;
    for (int q = 0; q < 16; ++q) {
      const int pp = pb + 4 * q;
      bk[pp * PP + n] = (T)ld_coherent(&Dj[n + pp * TILE]);
    }
  }
  __syncthreads();
  typename Acc<T>::type acc[2][2];
  zero_acc<T>(acc);
  mma64_kmajor<T>(ck, PP, bk, PP, acc);
  T* L = (T*)P.L;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        L[(size_t)(ri + acc_row<T>(bm, r)) + (size_t)(c0 + acc_col(bn)) * P.Np] = acc[bm][bn][r];
}

// ---- column-form super-step in one launch ------------------------------------
// The tiles (i, j), j <= i < rlim, of the super-step's columns [s0, s1) in one
// launch: one workgroup per row block i of every member, which forms its
// tiles (i, s0), (i, s0 + 1), ... from left to right and, for a row block of
// the super-step itself, then factors and inverts its diagonal block.  For a
// tile it accumulates sum_{c in [s0, j)} L_ic L_jc^T from its own earlier
// tiles and row block j's (published in this launch: coherent loads once
// their flags show them final), waits for block j's inverse and multiplies:
// L_ij = C_ij DINV_j^T.  A row block of the super-step also accumulates its
// diagonal tile's update on the way, so the chain from one block column to
// the next is DINV_{i-1} -> L_{i,i-1} (in LDS) -> update of tile (i, i) ->
// factor -> DINV_i: one hand-off between workgroups per column.  With the
// super-step's rows s0..s1-1 cut off by rlim = s1 the rows below are left to
// k_panel_rows.  Same operations in the same order on every tile as
// k_column: the factor is bitwise the same.
//
// Bound: that chain.  With a workgroup per tile a block column took two
// hand-offs through memory and 33 us (FP64) / 29 us (FP32) of a lone N = 512
// factor; with one per row block 14.3 us (FP32) and 18 us (FP64, to 29 us in
// the last columns of 8, where the left-looking products are the longer
// side): 287 -> 164 us and 217 -> 114 us for the eight columns.  Super-steps of
// six, the zeros of the panel product and half the diagonal update left out:
// 15.8 us a column of an FP64 factor at N = 1537.
//
// Member sync words (Prob::csync, zeroed when the descriptor is written with
// reset): flag (i, c) at csync[(c - s0) MAXG + i - s0] holds the launch's
// epoch once tile (i, c), i < s1, is final (c = i: DINV_i); csync[16 nb]
// counts the member's finished workgroups.  The member's last workgroup
// resets the count and clears the flags, so no flag outlives its launch (a
// replayed graph of the launch, whose epoch is the captured one, starts from
// cleared flags).
constexpr int MAXG = 16;
// Tickets: the row blocks s0, s0 + 1, ... of the super-step, each for every
// member that has it, then the rows below, member after member; a workgroup
// waits only for row blocks of its member above its own, on lower tickets.
//
// Outer tiles: with the previous super-step's outer update done only for this
// one's columns, the rest of it (128-tiles from column s1 on) goes into this
// launch, where it fills the CUs that the column chain leaves idle.
// A factor of N = 4096 in FP64: super-steps of 100 us and outer updates of 82
// on average; with the tiles 124 to 101, and 39 to 24 for the columns before.
// Evidence and gradient 18.6 -> 16.4 ms; prior draw N = 12288 14.4 -> 13.7;
// FP32 posterior N = 8192 38.4 -> 35.1 (with tiles handed out by ticket, not
// in runs per XCD, only 37.6: a tile then took 80 us, not 60).
struct StepSched {
  int32_t count;             // members (sorted by size, descending)
  int32_t s0, s1;            // columns [s0, s1)
  int32_t rlim;              // row blocks [s0, min(nb, rlim))
  int32_t gbase[MAXG + 1];   // first ticket of row block s0 + g; [s1 - s0]: the end
  int32_t pre[MAXB + 1];     // rows below (i >= s1) of the members before m
  // the previous super-step's outer update from block column s1 on
  int32_t p0;                // its columns [p0, s0)
  int32_t ofirst;            // outer tiles before the rows below
  int32_t rest;              // at most so many of each member, its last ones
  int32_t opre[LOOKB + 1];   // outer tiles of the members before m (opre[count] = 0: none)
};

__device__ __forceinline__ uint32_t* tile_flag(uint32_t* csync, int s0, int i, int c) {
  return csync + (c - s0) * MAXG + (i - s0);
}

// Wave 0 waits (bounded, one flag per lane) until the flags of tiles (j, c),
// c in [ca, cb), equal `epoch`; then the workgroup proceeds.  All threads
// call it.
__device__ __forceinline__ void wait_tiles(uint32_t* csync, int32_t* info, int s0, int j, int ca,
                                           int cb, uint32_t epoch) {
  if (threadIdx.x < 64) {
    const int l = threadIdx.x;
    const uint32_t* f = l < cb - ca ? tile_flag(csync, s0, j, ca + l) : nullptr;
    for (int spins = 0;; ++spins) {
      const bool ok =
          !f || __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch;
      if (__builtin_amdgcn_ballot_w64(!ok) == 0) break;
      if (spins >= SPIN_LIMIT) {
        if (l == 0) atomicOr(info, PGP_INFO_STALLED);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
  __syncthreads();
}

// The thread's 16 operand values v (row m, the k indices operand_k<CK>(kb, q))
// into an operand buffer of the trailing updates' form.
template <typename T, int BF16, typename LT>
__device__ __forceinline__ void stash_operand(LT* d, const T (&v)[16], int m, int kb) {
  constexpr bool MM = MmajorF32<T, BF16>::value;
  if constexpr (BF16) {
    stash_bf16_mmajor(d, 72, v, m, kb);
  } else if constexpr (MM) {
    stash_f32_mmajor(d, 68, v, m, kb);
  } else {
#pragma unroll
    for (int q = 0; q < 16; ++q) d[(kb + 4 * q) * KP<T>::value + m] = v[q];
  }
}
template <typename T, int BF16, typename LT>
__device__ __forceinline__ void mma_operands(const LT* a, const LT* b,
                                             typename Acc<T>::type (&acc)[2][2]) {
  if constexpr (BF16)
    mma64_bf16(a, 72, b, 72, acc);
  else if constexpr (MmajorF32<T, BF16>::value)
    mma64_f32_mmajor(a, 68, b, 68, acc);
  else
    mma64_kmajor<T>(a, KP<T>::value, b, KP<T>::value, acc);
}

// The ten 16 x 16 blocks on and below the diagonal of a 64 x 64 product A A^T
// (k-major operand), at most three to a wave: block b of wave w.
__device__ __forceinline__ void lower_block(int w, int b, int& i, int& j) {
  // w = 0: (3,0) (3,1) (0,0); 1: (3,2) (3,3) (1,0); 2: (2,0) (2,1) (1,1); 3: (2,2)
  i = (0xa9a7cf >> (6 * w + 2 * b)) & 3;
  j = (0xa94384 >> (6 * w + 2 * b)) & 3;
}
template <typename T>
__device__ __forceinline__ void mma64_lower(const T* As, int p, typename Acc<T>::type (&acc)[3]) {
  const int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const T *a[3], *c[3];
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    int i, j;
    lower_block(w, b, i, j);
    a[b] = As + (l >> 4) * p + 16 * i + (l & 15);
    c[b] = As + (l >> 4) * p + 16 * j + (l & 15);
  }
  T av[2][3], cv[2][3];
  auto read = [&](int s) {
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      av[s & 1][b] = a[b][4 * s * p];
      cv[s & 1][b] = c[b][4 * s * p];
    }
  };
  read(0);
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    if (s < 15) read(s + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < 3; ++b) acc[b] = mfma16(av[s & 1][b], cv[s & 1][b], acc[b]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// LDS of the super-step kernel: the panel product's two operands and the
// updates' two, or the diagonal factor's block.
template <typename T, int BF16>
struct StepArena {
  static constexpr int OPER = TILE * (BF16 ? 72 : MmajorF32<T, BF16>::value ? 68 : KP<T>::value);
  static constexpr int all = 2 * TILE * KP<T>::value * (int)sizeof(T) +
                             2 * OPER * (BF16 ? 2 : (int)sizeof(T));
  static constexpr int outer = 4 * Outer128<T, BF16>::OP * (BF16 ? 2 : (int)sizeof(T));
  static constexpr int step = all > FACTOR_LDS ? all : FACTOR_LDS;
  static constexpr int bytes = step > outer ? step : outer;
};

template <typename T, int BF16>
__global__ __launch_bounds__(NTHREADS, sizeof(T) == 8 ? 1 : 2) void k_superstep(
    Prob* const* probs, StepSched ss, uint32_t* ticket, uint32_t epoch) {
  __shared__ __attribute__((aligned(16))) char arena[StepArena<T, BF16>::bytes];
  __shared__ int s_val;
  // the outer tiles wait for nothing: no ticket, and a run of tiles per XCD
  const int s0 = ss.s0, s1 = ss.s1;
  const int chain = ss.gbase[s1 - s0], rows = chain + ss.pre[ss.count];
  const int u = (int)blockIdx.x - chain;
  if (u >= 0 && (u < ss.ofirst || u >= ss.ofirst + rows - chain)) {
    int o = xcd_contiguous(u < ss.ofirst ? u : u - (rows - chain), gridDim.x - rows);
    int mo = 0;
    while (o >= ss.opre[mo + 1]) ++mo;
    const Prob& P = *uniform(probs[mo]);
    o += max(0, tiles128(uniform(P.Np) / TILE - s1) - ss.rest) - ss.opre[mo];
    outer128_tile<T, BF16>(P, o, ss.p0, s0, s1, 0, (typename Outer128<T, BF16>::LT*)arena);
    return;
  }
  const int t = take_ticket(ticket, &s_val, rows);
  if ((unsigned)t >= (unsigned)rows) {  // counter not zero at launch: nothing to take
    flag_members_stalled(probs, ss.count);
    return;
  }
  // ticket -> (member mi, row block i)
  int mi, i;
  if (t < chain) {
    int g = 0;
    while (t >= ss.gbase[g + 1]) ++g;
    mi = t - ss.gbase[g];
    i = s0 + g;
  } else {
    const int b = t - chain;
    int lo = 0, hi = ss.count;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (ss.pre[mid] <= b)
        lo = mid;
      else
        hi = mid;
    }
    mi = lo;
    i = s1 + b - ss.pre[lo];
  }
  const Prob& P = *uniform(probs[mi]);
  const int nb = uniform(P.Np) / TILE;
  int64_t ld = (int64_t)nb * TILE;
  const int64_t ri = (int64_t)i * TILE;
  T* const Lp = (T*)uniform((char*)P.L);
  double* const dinv = uniform(P.dinv);
  double* const logdiag = uniform(P.logdiag);
  double* const diagval = uniform(P.diagval);
  uint32_t* const csync = uniform(P.csync);
  int32_t* const info = uniform(P.info);
  const bool diag = i < s1;  // this row block factors its diagonal block
  constexpr bool CK = MmajorF32<T, BF16>::value || BF16;
  typedef typename std::conditional<BF16 != 0, unsigned short, T>::type LT;
  typedef typename Acc<T>::type acc_t;
  constexpr int PP = KP<T>::value;
  T* ck = (T*)arena;  // panel product operands: C_ij and DINV_j
  T* bk = ck + TILE * PP;
  LT* sa = (LT*)(bk + TILE * PP);  // update operands
  LT* sb = sa + StepArena<T, BF16>::OPER;
  // the wave index as a scalar: column addresses stay in scalar registers
  const unsigned m = threadIdx.x & 63;
  const int kb = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const auto A = gbl(Lp);
  // the wave's 16 columns of the tile at (r0, c0): every fourth one, or
  // (operands) its columns operand_k<CK>
  auto col4 = [&](int64_t r0, int64_t c0) { return A + (r0 + (c0 + kb) * ld); };
  auto colk = [&](int64_t r0, int64_t c0) { return A + (r0 + (c0 + operand_k<CK>(kb, 0)) * ld); };
  constexpr int KS = CK ? 1 : 4;
  // acc: update of the current (then the next) tile; accd: of the diagonal tile
  constexpr bool F64 = std::is_same<T, double>::value;
  acc_t acc[2][2], accd[2][2], accl[3], prod[4];
  zero_acc<T>(acc);
  zero_acc<T>(accd);
#pragma unroll
  for (int b = 0; b < 3; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) accl[b][r] = (T)0;
  T av[16], ra[2][16], rb[2][16];
  auto load_a = [&](int64_t c0) {
    auto p = col4(ri, c0);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += 4 * ld) av[q] = p[m];
  };
  // row block j's tile (j, c), published in this launch
  auto load_rb = [&](T (&v)[16], int j, int c) {
    auto p = colk((int64_t)j * TILE, (int64_t)c * TILE);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += KS * ld) v[q] = ld_coh(p + m);
  };
  // k-major LDS image of a D-layout tile
  auto to_lds = [&](T* d, const acc_t (&v)[2][2]) {
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
      for (int bn = 0; bn < 2; ++bn)
#pragma unroll
        for (int r = 0; r < 4; ++r) d[acc_col(bn) * PP + acc_row<T>(bm, r)] = (T)v[bm][bn][r];
  };
  const int jend = min(i, s1);
  load_a((int64_t)(jend > s0 ? s0 : i) * TILE);
  for (int j = s0; j < jend; ++j) {
    asm volatile("" : "+s"(ld));  // column addresses are formed where they are used
    const int64_t c0 = (int64_t)j * TILE;
    const bool next = j + 1 < jend;
    // C_ij = A_ij - acc
    if (j > s0) {
      to_lds(ck, acc);
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      T* p = &ck[(kb + 4 * q) * PP + m];
      *p = j > s0 ? av[q] - *p : av[q];
    }
    // while block j is factored: the next tile's update by the columns
    // before j (own tiles: complete, see below), two columns ahead in flight
    zero_acc<T>(acc);
    if (next && j > s0) {
      wait_tiles(csync, info, s0, j + 1, s0, j, epoch);
      auto fetch = [&](int c, T (&a)[16], T (&b)[16]) {
        auto p = colk(ri, (int64_t)c * TILE);
#pragma unroll
        for (int q = 0; q < 16; ++q, p += KS * ld) a[q] = p[m];
        load_rb(b, j + 1, c);
      };
      auto chunk = [&](int c, T (&a)[16], T (&b)[16]) {
        __syncthreads();  // the previous products are done with LDS
        stash_operand<T, BF16>(sa, a, m, kb);
        stash_operand<T, BF16>(sb, b, m, kb);
        __syncthreads();
        if (c + 2 < j) fetch(c + 2, a, b);
        mma_operands<T, BF16>(sa, sb, acc);
      };
      fetch(s0, ra[0], rb[0]);
      if (s0 + 1 < j) fetch(s0 + 1, ra[1], rb[1]);
      for (int c = s0; c < j; c += 2) {
        chunk(c, ra[0], rb[0]);
        if (c + 1 < j) chunk(c + 1, ra[1], rb[1]);
      }
    }
    wait_tiles(csync, info, s0, j, j, j + 1, epoch);  // block j factored, DINV_j published
    {
      const auto Dj = gbl((const double*)dinv + (size_t)j * TILE * TILE);
      double dv[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) dv[q] = ld_coh(Dj + (kb + 4 * q) * TILE + m);
      __builtin_amdgcn_sched_barrier(0);  // every load issued before the first is used
#pragma unroll
      for (int q = 0; q < 16; ++q) bk[(kb + 4 * q) * PP + m] = (T)dv[q];
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) prod[b][r] = (T)0;
    mma64_tri<T, false, false>(bk, PP, ck, PP, prod);
    __syncthreads();
    // L_ij through LDS: whole columns per store, and the operand of the
    // following updates
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        ck[(16 * b + (m & 15)) * PP + 16 * kb + acc_row<T>(0, r) - 32 * (kb >> 1)] = prod[b][r];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; ++q) ra[0][q] = ck[operand_k<CK>(kb, q) * PP + m];
    {
      auto p = colk(ri, c0);
      if (diag) {
#pragma unroll
        for (int q = 0; q < 16; ++q, p += KS * ld)
          __hip_atomic_store(p + m, ra[0][q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
#pragma unroll
        for (int q = 0; q < 16; ++q, p += KS * ld) p[m] = ra[0][q];
      }
    }
    if (next || diag) {
      load_a(c0 + TILE);  // the next tile (the diagonal one after the last)
      stash_operand<T, BF16>(sa, ra[0], m, kb);
      __syncthreads();
      if (diag) {
        if constexpr (F64)
          mma64_lower<T>(sa, PP, accl);
        else
          mma_operands<T, BF16>(sa, sa, accd);
      }
    }
    // every wave's stores complete: publish the tile (and read it back as an
    // operand of the next columns)
    publish_wait();
    __syncthreads();
    if (diag && threadIdx.x == 0)
      __hip_atomic_store(tile_flag(csync, s0, i, j), epoch, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    if (next) {
      // column j's part of the next tile's update
      wait_tiles(csync, info, s0, j + 1, j, j + 1, epoch);
      load_rb(rb[0], j + 1, j);
      stash_operand<T, BF16>(sb, rb[0], m, kb);
      __syncthreads();
      mma_operands<T, BF16>(sa, sb, acc);
    }
  }
  if (diag) {
    __syncthreads();
    double (*blk)[TILE + 1] = (double (*)[TILE + 1])arena;
    if constexpr (F64) {
      // (the blocks above the diagonal ones are not read by the factor)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        if (kb == 3 && b > 0) break;
        int bi, bj;
        lower_block(kb, b, bi, bj);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          blk[16 * bi + acc_row<T>(0, r) - 32 * (kb >> 1)][16 * bj + (m & 15)] = accl[b][r];
      }
    } else {
#pragma unroll
      for (int bm = 0; bm < 2; ++bm)
#pragma unroll
        for (int bn = 0; bn < 2; ++bn)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            blk[acc_row<T>(bm, r)][acc_col(bn)] = (double)(T)accd[bm][bn][r];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      double* p = &blk[m][kb + 4 * q];
      *p = (double)(av[q] - (T)*p);
    }
    __syncthreads();
    FactorOut o{Lp, ld, dinv + (size_t)i * TILE * TILE, logdiag ? logdiag + ri : nullptr,
                diagval ? diagval + ri : nullptr, info};
    // the rows below wait only for DINV_i: publish before L_ii is stored
    factor_block_blocked<T>(blk, (double*)(blk + TILE), ri, o, [&]() {
      publish_wait();
      __syncthreads();
      if (threadIdx.x == 0)
        __hip_atomic_store(tile_flag(csync, s0, i, i), epoch, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    });
  }
  // the member's last workgroup in this launch clears its sync words
  if (threadIdx.x == 0) {
    const uint32_t total = (uint32_t)(min(nb, ss.rlim) - s0);
    s_val = (atomicAdd(csync + (size_t)16 * nb, 1u) + 1u == total) ? 1 : 0;
  }
  __syncthreads();
  if (s_val) {
    const int e = min(s1, nb) - s0;
    for (int w = threadIdx.x; w < e * MAXG; w += NTHREADS)
      if (w % MAXG < e) __hip_atomic_store(csync + w, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x == 0)
      __hip_atomic_store(csync + (size_t)16 * nb, 0u, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Diagonal block k (k >= 1) after the trailing update of step k - 1 (separate
// mode): one workgroup per member.
template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_factor_diag(Prob* const* probs, Sched sc, int k) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int64_t c0 = (int64_t)k * TILE;
  if (c0 >= P.Np) return;
  __shared__ double blk[TILE][TILE + 1];
  __shared__ double xd[FX_DOUBLES];
  const T* A = (const T*)P.L;
  const int m = threadIdx.x & 63, kb = threadIdx.x >> 6;
  for (int q = 0; q < 16; ++q) {
    const int c = kb + 4 * q;
    blk[m][c] = (double)A[(size_t)(c0 + m) + (size_t)(c0 + c) * P.Np];
  }
  __syncthreads();
  FactorOut o{P.L, P.Np, P.dinv + (size_t)k * TILE * TILE, P.logdiag ? P.logdiag + c0 : nullptr,
              P.diagval ? P.diagval + c0 : nullptr, P.info};
  factor_block_blocked<T>(blk, xd, c0, o);
}

// ---- raw (kernel-level ABI) variants ----------------------------------------
template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_factor_first_raw(T* A, int64_t ld, double* dinv,
                                                               double* logdiag, int32_t* info) {
  FactorOut o{A, ld, dinv, logdiag, nullptr, info};
  factor_first<T>(A, ld, o);
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_panel_raw(T* A, int64_t N, int64_t ld,
                                                        const double* dinv, int k) {
  const int64_t c0 = (int64_t)k * TILE;
  const int64_t r0 = c0 + (int64_t)TILE * (blockIdx.x + 1);
  panel_rows<T>(A, ld, dinv + (size_t)k * TILE * TILE, c0, r0);
}

template <typename T, int BF16>
__global__ __launch_bounds__(NTHREADS) void k_syrk_raw(T* A, int64_t N, int64_t ld, int k,
                                                       double* dinv, double* logdiag,
                                                       int32_t* info) {
  const int64_t c0 = (int64_t)k * TILE, c1 = c0 + TILE;
  int ti, tj;
  lower_tile_c(blockIdx.x, ti, tj);
  const bool factor = (ti == 0 && tj == 0);
  FactorOut o{A, ld, dinv + (size_t)(k + 1) * TILE * TILE, logdiag ? logdiag + c1 : nullptr,
              nullptr, info};
  syrk_tile<T, BF16, 1>(A, ld, c0, c1 + (int64_t)TILE * ti, c1 + (int64_t)TILE * tj, factor, o);
}

// ---- inverse of every 64x64 diagonal block of a given factor (FP64) --------
// Used when a caller hands in a factor (kernel-level solves).  Lane i of each
// wave holds x_i of one column of inv(L_kk) during forward substitution.
template <typename T>
__device__ void invert_diag_block(const T* A, int64_t ld, int64_t c0, double* out) {
  __shared__ double Ls[TILE][TILE + 1];  // Ls[col][row]
  const int m = threadIdx.x & 63, kb = threadIdx.x >> 6;
  for (int q = 0; q < 16; ++q) {
    const int col = kb + 4 * q;
    Ls[col][m] = (m >= col) ? (double)A[(size_t)(c0 + m) + (size_t)(c0 + col) * ld] : 0.0;
  }
  __syncthreads();
  const int wv = threadIdx.x >> 6;
  const int i = threadIdx.x & 63;
  for (int cq = 0; cq < 16; ++cq) {
    const int c = wv * 16 + cq;
    double x = 0.0;
    double rhs = (i == c) ? 1.0 : 0.0;
    for (int j = c; j < 64; ++j) {
      if (i == j) x = rhs / Ls[j][j];
      const double xj = __shfl(x, j);
      if (i > j) rhs -= Ls[j][i] * xj;
    }
    out[(size_t)i + (size_t)c * TILE] = (i >= c) ? x : 0.0;
  }
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_dinv_raw(const T* A, int64_t ld, double* dinv) {
  invert_diag_block<T>(A, ld, (int64_t)blockIdx.x * TILE, dinv + (size_t)blockIdx.x * TILE * TILE);
}

// ---------------------------------------------------------------------------
// Schedule table (the autotuner's): per precision and size class, the
// super-step width G (rank-64G outer updates), COLUMN_MAX (super-steps whose
// first column has at most this many workgroups run in the column kernel;
// 0 disables), FUSE_MAX (update launches of at most this many tiles factor
// the next diagonal block inside the launch; 0 disables) and COLUMN_MERGE
// (how such a super-step is launched: 0 one k_column launch per column;
// 1 the diagonal block of tiles in one k_superstep launch, then the rows
// below in one k_panel_rows launch; 2 every tile in one k_superstep
// launch).
// Size class 0 holds the members with padded N <= TUNE_CLASS_NP, class 1 the
// larger ones; a batch is factored class by class, so a member's schedule --
// and with G its rounding -- depends only on its own size (a result is the
// same alone and in any mix, in the batcher or the single-problem path).
// COLUMN_MAX, FUSE_MAX and COLUMN_MERGE change only the launches, never the
// arithmetic.
// Initial values: PGP_SUPERSTEP / PGP_COLUMN_MAX / PGP_FUSE_MAX /
// PGP_COLUMN_MERGE from the environment, else 8 / 512 / 512 / 2.  Read at every factorisation, written
// rarely (pgp_tune_set): a mutex guards it.
// ---------------------------------------------------------------------------
constexpr int TUNE_CLASSES = 2;
constexpr int TUNE_CLASS_NP = 1024;

static int env_int(const char* name, int dflt) {
  const char* e = getenv(name);
  return e ? atoi(e) : dflt;
}

struct TuneTable {
  std::mutex mu;
  pgp_tune_entry_t e[3][TUNE_CLASSES];
  TuneTable() {
    const int cm = env_int("PGP_COLUMN_MAX", 512), fm = env_int("PGP_FUSE_MAX", 512);
    const int mg = std::min(2, std::max(0, env_int("PGP_COLUMN_MERGE", 2)));
    for (int p = 0; p < 3; ++p)
      for (int c = 0; c < TUNE_CLASSES; ++c) {
        // FP64 above the size class: the shorter column chain of six (N = 1537
        // 6.56 -> 6.07 ms a posterior, N = 4096 19.7 -> 18.6 the evidence and
        // gradient, N = 12288 14.55 -> 14.66 a prior draw)
        const int g = env_int("PGP_SUPERSTEP", p == PGP_PREC_FP64 && c == 1 ? 6 : 8);
        e[p][c] = pgp_tune_entry_t{std::min(16, std::max(1, g)), cm, fm, mg};
      }
  }
};
static TuneTable& tune_table() {
  static TuneTable t;
  return t;
}

int tune_class_of(int np) { return np > TUNE_CLASS_NP ? 1 : 0; }

pgp_tune_entry_t tune_get(int prec, int cls) {
  TuneTable& t = tune_table();
  std::lock_guard<std::mutex> lock(t.mu);
  return t.e[prec][cls];
}

void tune_set(int prec, int cls, const pgp_tune_entry_t& v) {
  TuneTable& t = tune_table();
  std::lock_guard<std::mutex> lock(t.mu);
  t.e[prec][cls] = v;
}

static bool sorted_desc(const Batch& b) {
  for (int m = 1; m < b.count; ++m)
    if (b.np(m) > b.np(m - 1)) return false;
  return true;
}

template <typename T, int BF16>
static void column_launch(const Batch& b, int j, int s0, bool tpa, hipStream_t s) {
  constexpr double F3 = TILE * TILE * TILE / 3.0;
  constexpr double G64 = 2.0 * TILE * TILE * TILE;
  for (int off = 0; off < b.count; off += MAXB) {
    const int n = std::min(MAXB, b.count - off);
    Sched sc;
    sc.count = n;
    int tot = 0, nd = 0;
    double fl = 0.0;
    for (int m = 0; m < n; ++m) {
      const int nbm = b.np(off + m) / TILE;
      sc.pre[m] = tot;
      if (nbm > j) {
        ++nd;
        tot += nbm - j - 1;
        fl += F3 + (double)(nbm - j) * G64 * (j - s0) + (double)(nbm - j - 1) * G64;
      }
    }
    sc.pre[n] = tot;
    if (nd == 0) continue;
    const uint32_t ep = next_epoch();
    if (tpa) timer_begin(TC_PANEL, s);
    hipLaunchKernelGGL((k_column<T, BF16>), dim3(nd + tot), dim3(NTHREADS), 0, s, b.dprobs + off,
                       sc, nd, b.ticket, ep, j, s0);
    if (tpa) timer_end(TC_PANEL, s, fl, 0.0);
  }
}

// Phase B: row block i = s1 + local of a member with more than s1 block
// columns, columns [s0, s1): L_ij = (A_ij - sum_{c in [s0, j)} L_ic L_jc^T)
// DINV_j^T, j in order.  L_jc and DINV_j come from phase A (the previous
// launch), L_ic from this workgroup's earlier iterations.
template <typename T, int BF16>
struct RowsArena {
  static constexpr int PP = KP<T>::value;
  static constexpr int OPND = BF16 ? 72 * 2 : (MmajorF32<T, BF16>::value ? 68 * 4 : PP * (int)sizeof(T));
  static constexpr int A = 2 * TILE * OPND;                   // update operands
  static constexpr int B = 2 * TILE * PP * (int)sizeof(T);  // C_ij and DINV_j
  static constexpr int bytes = A > B ? A : B;
};

template <typename T, int BF16>
__global__ __launch_bounds__(NTHREADS) void k_panel_rows(Prob* const* probs, Sched sc, int s0,
                                                         int s1) {
  constexpr int PP = KP<T>::value;
  __shared__ __attribute__((aligned(16))) char arena[RowsArena<T, BF16>::bytes];
  int local;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, local)];
  const int i = s1 + local;
  if (i >= P.Np / TILE) return;
  const int64_t ri = (int64_t)i * TILE;
  T* ck = (T*)arena;
  T* bk = ck + TILE * PP;
  T* L = (T*)P.L;
  const int n = threadIdx.x & 63, pb = threadIdx.x >> 6;
  for (int j = s0; j < s1; ++j) {
    const int64_t c0 = (int64_t)j * TILE;
    update_tile_to_lds<T, BF16, T>((const T*)P.L, P.Np, s0, j, ri, c0, arena, ck, PP, true);
    const double* Dj = P.dinv + (size_t)j * TILE * TILE;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int pp = pb + 4 * q;
      bk[pp * PP + n] = (T)Dj[n + pp * TILE];
    }
    __syncthreads();
    typename Acc<T>::type acc[2][2];
    zero_acc<T>(acc);
    mma64_kmajor<T>(ck, PP, bk, PP, acc);
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
      for (int bn = 0; bn < 2; ++bn)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          L[(size_t)(ri + acc_row<T>(bm, r)) + (size_t)(c0 + acc_col(bn)) * P.Np] =
              acc[bm][bn][r];
    // the tile is an operand of this row's next columns; LDS is free again
    publish_wait();
    __syncthreads();
  }
}

template <typename T, int BF16>
static void rows_launch(const Batch& b, int s0, int s1, bool tpa, hipStream_t s) {
  constexpr double G64 = 2.0 * TILE * TILE * TILE;
  sched_launch(
      b, [&](int m) { return std::max(0, b.np(m) / TILE - s1); },
      [&](Prob* const* dp, const Sched& sc, int n) {
        if (tpa) timer_begin(TC_PANEL, s);
        hipLaunchKernelGGL((k_panel_rows<T, BF16>), dim3(n), dim3(NTHREADS), 0, s, dp, sc, s0, s1);
        if (tpa) {
          const int off = (int)(dp - b.dprobs);
          double fl = 0.0;
          const double per_row = G64 * (double)(s1 - s0) * (s1 - s0 + 1) / 2.0;
          for (int m = off; m < off + sc.count; ++m)
            fl += std::max(0, b.np(m) / TILE - s1) * per_row;
          timer_end(TC_PANEL, s, fl, 0.0);
        }
      });
}

template <typename T, int BF16>
static void superstep_launch(const Batch& b, int s0, int s1, int rlim, int p0, int rest, bool tpa,
                             hipStream_t s) {
  constexpr double F3 = TILE * TILE * TILE / 3.0;
  constexpr double G64 = 2.0 * TILE * TILE * TILE;
  for (int off = 0; off < b.count; off += MAXB) {
    const int n = std::min(MAXB, b.count - off);
    StepSched ss;
    ss.count = n;
    ss.s0 = s0;
    ss.s1 = s1;
    ss.rlim = rlim;
    double fl = 0.0;
    ss.pre[0] = 0;
    for (int m = 0; m < n; ++m) {
      const int nbm = b.np(off + m) / TILE, nbr = std::min(nbm, rlim);
      ss.pre[m + 1] = ss.pre[m] + std::max(0, nbr - s1);
      for (int j = s0; j < std::min(s1, nbm); ++j)
        fl += F3 + (double)(nbr - j) * G64 * (j - s0) + (double)(nbr - j - 1) * G64;
    }
    const int ncols = s1 - s0;
    ss.gbase[0] = 0;
    for (int g = 0; g < ncols; ++g) {
      int nd = 0;
      for (int m = 0; m < n; ++m)
        if (b.np(off + m) / TILE > s0 + g) ++nd;
      ss.gbase[g + 1] = ss.gbase[g] + nd;
    }
    ss.p0 = p0;
    ss.rest = rest;
    ss.opre[0] = 0;
    if (p0 >= 0) {
      for (int m = 0; m < n; ++m) {
        const int t = std::min(rest, tiles128(b.np(off + m) / TILE - s1));
        ss.opre[m + 1] = ss.opre[m] + t;
        fl += 4.0 * t * G64 * (s0 - p0);
      }
    } else {
      ss.opre[std::min(n, LOOKB)] = 0;
    }
    const int nouter = ss.opre[std::min(n, LOOKB)];
    look_tiles(outer_op<T, BF16>(), ss.gbase[ncols], ss.pre[n], ss.ofirst);
    ss.ofirst = std::min(ss.ofirst, nouter);
    // with outer tiles one workgroup a CU: a second one would slow the chain's
    const int lds = nouter > 0 && sizeof(T) == 4 ? 8192 : 0;
    const int tot = ss.gbase[ncols] + ss.pre[n] + nouter;
    if (tot == 0) continue;
    const uint32_t ep = next_epoch();
    const bool tsu = timer_on(TC_SUPER);
    double by = 0.0;
    if (tsu) {
      // algorithmic bytes: every tile of the launch read and written once in
      // the storage type, and each diagonal block's FP64 inverse written once
      constexpr double TB = (double)TILE * TILE;
      for (int m = 0; m < n; ++m) {
        const int nbm = b.np(off + m) / TILE, nbr = std::min(nbm, rlim);
        for (int j = s0; j < std::min(s1, nbm); ++j)
          by += (double)(nbr - j) * 2.0 * TB * sizeof(T) + TB * 8.0;
        if (p0 >= 0)
          by += std::min(rest, tiles128(nbm - s1)) * 8.0 * TB * sizeof(T) +
                std::max(0, nbm - s1) * TB * (s0 - p0) * (BF16 ? 2.0 : sizeof(T));
      }
      timer_begin(TC_SUPER, s);
    }
    hipLaunchKernelGGL((k_superstep<T, BF16>), dim3(tot), dim3(NTHREADS), lds, s, b.dprobs + off,
                       ss, b.ticket, ep);
    if (tsu) timer_end(TC_SUPER, s, fl, by);
  }
}

// ---------------------------------------------------------------------------
// Per block column k (every member at once), in super-steps of G columns:
//   separate kernels: U_k left-looking update of column k by the super-step's
//     earlier panels; F_k factor of block k (inside U_k when that launch is
//     small); P_k panel; at the super-step's last column O, the outer update
//     of everything right of it (factoring its first block when small);
//   column kernel: one k_column launch per column (the same update, factor
//     and panel), then O at the super-step's end.
// Both forms apply the same operations in the same order to every tile, so a
// member's factor does not depend on which form its batch used.
template <typename T, int BF16>
static void potrf_steps(const Batch& b, hipStream_t s, const pgp_tune_entry_t& te) {
  const int nb = b.maxNp / TILE;
  const int G = te.superstep;
  const int column_max = te.column_max, fuse_max = te.fuse_max;
  const bool tsy = timer_on(TC_SYRK), tpa = timer_on(TC_PANEL);
  constexpr double F3 = TILE * TILE * TILE / 3.0;  // factor of one 64x64 block
  constexpr double G64 = 2.0 * TILE * TILE * TILE;  // one 64x64x64 product
  // algorithmic flops of the members [off, off + n) of a launch
  auto flops = [&](const Sched& sc, Prob* const* dp, auto per_member) {
    const int off = (int)(dp - b.dprobs);
    double f = 0.0;
    for (int m = off; m < off + sc.count; ++m) f += per_member(b.np(m) / TILE);
    return f;
  };
  const bool colok = column_max > 0 && b.ticket && sorted_desc(b);
  // workgroups of the column launch at the first column of a super-step;
  // non-increasing in s0, so once a super-step uses the column kernel all
  // later ones do
  auto col_style = [&](int s0) {
    if (!colok) return false;
    long long w = 0;
    for (int m = 0; m < b.count; ++m) w += std::max(0, b.np(m) / TILE - s0);
    return w <= column_max;
  };
  auto nb_of = [&](int m) { return b.np(m) / TILE; };
  // rest >= 0: all but the last `rest` 128-tiles of each member's triangle from
  // the next super-step's end on, which go into that super-step's launch
  auto outer_launch = [&](int s0, int s_end, bool fuse, int rest) {
    if constexpr (BF16 != 0) {
      // the BF16 copy of the panel rows below the super-step, which the
      // outer update reads instead of converting at every stash
      sched_launch(
          b, [&](int m) { return std::max(0, b.np(m) / TILE - s_end); },
          [&](Prob* const* dp, const Sched& sc, int n) {
            hipLaunchKernelGGL(k_panel_bf16, dim3(n), dim3(NTHREADS), 0, s, dp, sc, s0, s_end);
          });
    }
    const int wd = rest < 0 ? 0 : G;  // its columns, if it has to be split
    auto tiles128_of = [&](int m) { return outer_tiles128(b.np(m) / TILE - s_end, wd, rest); };
    auto tiles64_of = [&](int m) {
      return outer_tiles64(std::max(0, b.np(m) / TILE - s_end), wd > 0 ? wd : nb);
    };
    const bool wide =
        !fuse && outer_takes_wide(outer_op<T, BF16>(), b.count, nb_of, s_end, wd, rest);
    auto tiles = [&](int m) { return wide ? tiles128_of(m) : tiles64_of(m); };
    sched_launch(b, tiles, [&](Prob* const* dp, const Sched& sc, int n) {
      if (tsy) timer_begin(TC_SYRK, s);
      if (fuse)
        hipLaunchKernelGGL((k_syrk_outer<T, BF16, 1>), dim3(n), dim3(NTHREADS), 0, s, dp, sc, s0,
                           s_end, nb);
      else if (wide)
        hipLaunchKernelGGL((k_syrk_outer128<T, BF16>), dim3(n), dim3(NTHREADS), 0, s, dp, sc, s0,
                           s_end, wd);
      else
        hipLaunchKernelGGL((k_syrk_outer<T, BF16, 0>), dim3(n), dim3(NTHREADS), 0, s, dp, sc, s0,
                           s_end, wd > 0 ? wd : nb);
      if (tsy) {
        // outer update: an n x n lower triangle (n = 64 T) with rank K = 64 G
        // counts n (n + 1) K flops (a part of it, its tiles' products); bytes:
        // every tile read and written once, each trailing row block's G panel
        // blocks read once
        const double es = sizeof(T);
        auto part = [&](int nbm) {  // 64-tiles of a split update
          return wide ? 4.0 * outer_tiles128(nbm - s_end, wd, rest)
                      : (double)outer_tiles64(std::max(0, nbm - s_end), wd);
        };
        timer_end(TC_SYRK, s, flops(sc, dp,
                                    [&](int nbm) {
                                      const double nn = (double)std::max(0, nbm - s_end) * TILE;
                                      return wd > 0 ? part(nbm) * G64 * G
                                                    : nn * (nn + 1) * (double)(TILE * G);
                                    }),
                  flops(sc, dp, [&](int nbm) {
                    // (BF16 factors read the panel from its BF16 copy)
                    const double t = std::max(0, nbm - s_end);
                    return (wd > 0 ? 2.0 * part(nbm) : t * (t + 1)) * TILE * TILE * es +
                           t * TILE * TILE * G * (BF16 ? 2.0 : es);
                  }));
      }
    });
  };
  auto total_units = [&](auto units) {
    int t = 0;
    for (int m = 0; m < b.count; ++m) t += units(m);
    return t;
  };
  if (!col_style(0)) {
    if (tpa) timer_begin(TC_PANEL, s);
    hipLaunchKernelGGL(k_factor_first<T>, dim3(1, b.count), dim3(NTHREADS), 0, s, b.dprobs);
    if (tpa) timer_end(TC_PANEL, s, b.count * F3, 0.0);
  }
  int ahead = -1;  // tiles of the last outer update left to the next super-step (-1: none)
  for (int k = 0; k < nb; ++k) {
    const int s0 = k / G * G, s_end = s0 + G;
    const bool outer = (k + 1 == s_end);
    if (col_style(s0)) {
      if (te.column_merge == 2) {
        // every row block of the super-step's columns in the one launch, with
        // the rest of the previous super-step's outer update
        if (k == s0)
          superstep_launch<T, BF16>(b, s0, std::min(s_end, nb), nb, ahead < 0 ? -1 : s0 - G,
                                    ahead, tpa, s);
      } else if (te.column_merge == 1) {
        if (k == s0) {
          superstep_launch<T, BF16>(b, s0, std::min(s_end, nb), s_end, -1, 0, tpa, s);
          if (s_end < nb) rows_launch<T, BF16>(b, s0, s_end, tpa, s);
        }
      } else {
        column_launch<T, BF16>(b, k, s0, tpa, s);
      }
      if (outer && s_end < nb) {
        ahead = te.column_merge == 2
                    ? outer_ahead(outer_op<T, BF16>(), b.count, nb_of, s_end, G)
                    : -1;
        outer_launch(s0, s_end, false, ahead);
      }
      continue;
    }
    // U_k (k > s0): left-looking update of column k, factoring block k inside
    // the launch when it is small, else F_k after it.  Block s0 of a
    // super-step was factored at the end of the previous one (or by F_0).
    if (k > s0) {
      auto tiles = [&](int m) { return std::max(0, b.np(m) / TILE - k); };
      const bool fused = total_units(tiles) <= fuse_max;
      sched_launch(b, tiles, [&](Prob* const* dp, const Sched& sc, int n) {
        if (tpa) timer_begin(TC_PANEL, s);
        if (fused)
          hipLaunchKernelGGL((k_col_update<T, BF16, 1>), dim3(n), dim3(NTHREADS), 0, s, dp, sc, k,
                             s0);
        else
          hipLaunchKernelGGL((k_col_update<T, BF16, 0>), dim3(n), dim3(NTHREADS), 0, s, dp, sc, k,
                             s0);
        if (tpa)
          timer_end(TC_PANEL, s,
                    flops(sc, dp, [&](int nbm) {
                      return nbm > k ? (double)(nbm - k) * G64 * (k - s0) + (fused ? F3 : 0.0)
                                     : 0.0;
                    }),
                    0.0);
      });
      if (!fused)
        sched_launch(
            b, [&](int m) { return b.np(m) / TILE > k ? 1 : 0; },
            [&](Prob* const* dp, const Sched& sc, int n) {
              if (tpa) timer_begin(TC_PANEL, s);
              hipLaunchKernelGGL(k_factor_diag<T>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, k);
              if (tpa) timer_end(TC_PANEL, s, n * F3, 0.0);
            });
    }
    if (k + 1 >= nb) break;
    sched_launch(
        b, [&](int m) { return std::max(0, b.np(m) / TILE - k - 1); },
        [&](Prob* const* dp, const Sched& sc, int n) {
          if (tpa) timer_begin(TC_PANEL, s);
          hipLaunchKernelGGL(k_panel<T>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, k);
          if (tpa)
            timer_end(TC_PANEL, s,
                      flops(sc, dp, [&](int nbm) { return std::max(0, nbm - k - 1) * G64; }), 0.0);
        });
    if (outer) {
      // O closes the super-step; block s_end is factored inside it when the
      // launch is small, else by F_s_end -- unless the next super-step uses
      // the column kernel, which factors it itself
      const bool next_col = col_style(s_end);
      const bool fused = !next_col && total_units([&](int m) {
                                        const int t = std::max(0, b.np(m) / TILE - s_end);
                                        return t * (t + 1) / 2;
                                      }) <= fuse_max;
      outer_launch(s0, s_end, fused, -1);
      if (!fused && !next_col)
        sched_launch(
            b, [&](int m) { return b.np(m) / TILE > s_end ? 1 : 0; },
            [&](Prob* const* dp, const Sched& sc, int n) {
              if (tpa) timer_begin(TC_PANEL, s);
              hipLaunchKernelGGL(k_factor_diag<T>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, s_end);
              if (tpa) timer_end(TC_PANEL, s, n * F3, 0.0);
            });
    }
  }
}

static void potrf_class(const Batch& b, int prec, hipStream_t s) {
  if (b.count <= 0) return;
  const pgp_tune_entry_t te = tune_get(prec, tune_class_of(b.maxNp));
  if (prec == PGP_PREC_FP64)
    potrf_steps<double, 0>(b, s, te);
  else if (prec == PGP_PREC_FP32)
    potrf_steps<float, 0>(b, s, te);
  else
    potrf_steps<float, 1>(b, s, te);
}

// The members of a batch are sorted by size (largest first), so the large
// size class is a prefix: each class is factored with its own schedule.
void launch_potrf(const Batch& b, int prec, hipStream_t s) {
  int k = 0;
  while (k < b.count && tune_class_of(b.np(k)) == 1) ++k;
  if (k == 0 || k == b.count) {
    potrf_class(b, prec, s);
    return;
  }
  Batch big = b, small = b;
  big.count = k;
  small.dprobs = b.dprobs + k;
  small.count = b.count - k;
  small.maxNp = b.np(k);
  if (b.hnp) small.hnp = b.hnp + k;
  if (b.hm) small.hm = b.hm + k;
  potrf_class(big, prec, s);
  potrf_class(small, prec, s);
}

template <typename T, int BF16>
static void potrf_raw_steps(T* A, int64_t N, int64_t ld, double* dinv, double* logdiag,
                            int32_t* info, hipStream_t s) {
  const int nb = (int)(N / TILE);
  hipLaunchKernelGGL(k_factor_first_raw<T>, dim3(1), dim3(NTHREADS), 0, s, A, ld, dinv, logdiag,
                     info);
  for (int k = 0; k + 1 < nb; ++k) {
    const int below = nb - k - 1;
    hipLaunchKernelGGL(k_panel_raw<T>, dim3(below), dim3(NTHREADS), 0, s, A, N, ld,
                       (const double*)dinv, k);
    hipLaunchKernelGGL((k_syrk_raw<T, BF16>), dim3(below * (below + 1) / 2), dim3(NTHREADS), 0, s,
                       A, N, ld, k, dinv, logdiag, info);
  }
}

int launch_potrf_raw(int prec, void* A, int64_t N, int64_t ld, double* dinv, double* logdiag,
                     int32_t* info, hipStream_t s) {
  if (prec == PGP_PREC_FP64)
    potrf_raw_steps<double, 0>((double*)A, N, ld, dinv, logdiag, info, s);
  else if (prec == PGP_PREC_FP32)
    potrf_raw_steps<float, 0>((float*)A, N, ld, dinv, logdiag, info, s);
  else
    potrf_raw_steps<float, 1>((float*)A, N, ld, dinv, logdiag, info, s);
  return 0;
}

int launch_dinv_raw(int prec, const void* A, int64_t N, int64_t ld, double* dinv, hipStream_t s) {
  if (prec == PGP_PREC_FP64)
    hipLaunchKernelGGL(k_dinv_raw<double>, dim3((unsigned)(N / TILE)), dim3(NTHREADS), 0, s,
                       (const double*)A, ld, dinv);
  else
    hipLaunchKernelGGL(k_dinv_raw<float>, dim3((unsigned)(N / TILE)), dim3(NTHREADS), 0, s,
                       (const float*)A, ld, dinv);
  return 0;
}

}  // namespace pgp
