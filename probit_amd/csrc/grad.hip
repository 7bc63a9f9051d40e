// Adjoint of the Laplace evidence and the VB traces.
//
// The reference differentiates objective_LA (probit/implicit/Laplace.py:12-30)
// with jax.value_and_grad through the implicit fixed-point layer
// (probit/implicit/solvers.py:28-64, probit/approximators.py:132-134).  At the
// fixed point that derivative has the closed form (Rasmussen & Williams
// Alg. 5.1, extended to likelihood parameters):
//   C = W^1/2 B^-1 W^1/2,  Sigma_ii = K_ii - (K C K)_ii,  s2 = -1/2 Sigma_ii d3_i,
//   shat = (I - C K) s2,
//   d/dtheta_K = sum_ij dK_ij/dtheta G_ij,  G = C/2 - a a^T/2 + (shat a^T + a shat^T)/2,
//   d/dtheta_l = sum_i [-L_p - Sigma_ii L_ffp / 2 + (K shat)_i L_fp].
// This file holds the O(N^3) pieces reused from the resident factor:
//   * k_inv_merge: Linv = L^-1 by doubling;
//   * k_sym_from_inv: C = S (Linv^T Linv) S (or Linv^T Linv for VB), lower;
//   * k_grad_trace: tiles of sum_ij dK_ij/dtheta G_ij with dK recomputed from
//     X in registers, lower tiles only (off-diagonal tiles count twice),
//     per-tile partials reduced in a fixed order by k_sum_partials;
//   * k_vb_trace: tr(C) and sum_ij K_ij C_ij of objective_VB
//     (probit/implicit/VB.py:28-30).
#include <math.h>

#include <algorithm>

#include "mfma.hpp"
#include "pgp_internal.hpp"

namespace pgp {

constexpr int GMAXD = 16;  // input dimensions supported by the gradient kernel
constexpr int NPAR = 1 + 2 * GMAXD;

__device__ __forceinline__ void lower_tile_g(int t, int& ti, int& tj) {
  int i = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((i + 1) * (i + 2) / 2 <= t) ++i;
  while (i * (i + 1) / 2 > t) --i;
  ti = i;
  tj = t - i * (i + 1) / 2;
}

// ---- X = L^-1 ------------------------------------------------------------------
// The explicit inverse of the resident factor (lower triangular, in P.S) by
// doubling: its diagonal tiles are DINV; two neighbouring inverted diagonal
// blocks of h tiles give the inverse of their 2h-tile block,
//   X_21 = -X_22 (L_21 X_11),
// two launches per doubling, every tile of every pair its own workgroup.  The
// product L_21 X_11 waits in the unused upper tiles (tile (i, j) of it at
// (j, i)).  Bound: FP64 MFMA once the blocks are large (N^3 / 3 flops in
// all), the launches before.  A forward substitution of the identity has
// the factor's block rows as a serial chain instead: 3.1 ms at N = 4096
// (FP64), 16 x 22 us at N = 512, where this takes 0.87 ms and 6 x 10 us.
template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_inv_diag(Prob* const* probs) {
  const Prob& P = *probs[blockIdx.y];
  const int i = blockIdx.x;
  if (i >= P.Np / TILE) return;
  const auto D = gbl(P.dinv + (size_t)i * TILE * TILE);
  const auto X = gbl((T*)P.S) + (size_t)i * TILE * (P.Np + 1);
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int e = threadIdx.x + NTHREADS * q;
    X[(size_t)(e >> 6) * P.Np + (e & 63)] = (T)D[e];
  }
}

template <typename T, bool SECOND>
__global__ __launch_bounds__(NTHREADS) void k_inv_merge(Prob* const* probs, int h) {
  const Prob& P = *probs[blockIdx.z];
  const int nb = uniform(P.Np) / TILE;
  const int a = 2 * h * blockIdx.y, mid = a + h;
  // the longest sums first: first product k from j, second k up to i
  const int j = uniform(a + (int)blockIdx.x % h);
  const int i = uniform(SECOND ? min(nb, mid + h) - 1 - (int)blockIdx.x / h
                               : mid + (int)blockIdx.x / h);
  if (i >= nb || i < mid) return;
  const int64_t ld = uniform(P.Np);
  const unsigned m = threadIdx.x & 63;
  const int kb = uniform((int)(threadIdx.x >> 6));
  const auto L = gbl(uniform((const T*)P.L));
  const auto X = gbl(uniform((T*)P.S));
  __shared__ GemmLds<T> lds;
  typename Acc<T>::type acc[2][2];
  zero_acc<T>(acc);
  auto tile = [&](auto base, int r, int c, T (&v)[16]) {
    auto p = base + ((int64_t)r * TILE + ((int64_t)c * TILE + kb) * ld);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += 4 * ld) v[q] = p[m];
  };
  if constexpr (!SECOND)
    gemm_tiles<T, false>(
        j, mid, [&](int k, T (&v)[16]) { tile(L, i, k, v); },
        [&](int k, T (&v)[16]) { tile(X, k, j, v); }, lds, acc);
  else
    gemm_tiles<T, false>(
        mid, i + 1, [&](int k, T (&v)[16]) { tile(X, i, k, v); },
        [&](int k, T (&v)[16]) { tile(X, j, k, v); }, lds, acc);
  const int r0 = SECOND ? i : j, c0 = SECOND ? j : i;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        X[(size_t)(r0 * TILE + acc_row<T>(bm, r)) + (size_t)(c0 * TILE + acc_col(bn)) * ld] =
            (T)(SECOND ? -acc[bm][bn][r] : acc[bm][bn][r]);
}

template <typename T>
static void tri_inverse(const Batch& b, hipStream_t s) {
  const int nb = b.maxNp / TILE;
  hipLaunchKernelGGL(k_inv_diag<T>, dim3(nb, b.count), dim3(NTHREADS), 0, s, b.dprobs);
  for (int h = 1; h < nb; h *= 2) {
    const dim3 g(h * std::min(h, nb - h), (nb - h + 2 * h - 1) / (2 * h), b.count);
    hipLaunchKernelGGL((k_inv_merge<T, false>), g, dim3(NTHREADS), 0, s, b.dprobs, h);
    hipLaunchKernelGGL((k_inv_merge<T, true>), g, dim3(NTHREADS), 0, s, b.dprobs, h);
  }
}

void launch_tri_inverse(const Batch& b, int prec, hipStream_t s) {
  if (prec == PGP_PREC_FP64)
    tri_inverse<double>(b, s);
  else
    tri_inverse<float>(b, s);
}

// C(i0.., j0..) = scale_i * sum_k X(k, i) X(k, j) * scale_j, X = L^-1, so the
// k range starts at i0 >= j0: the lower tiles of C (its readers take the
// lower triangle only), those with the longest sums first.
template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_sym_from_inv(Prob* const* probs, int use_scale) {
  const Prob& P = *probs[blockIdx.y];
  const int nb = uniform(P.Np) / TILE;
  if ((int)blockIdx.x >= nb * (nb + 1) / 2) return;
  int ti, tj;
  lower_tile_g(blockIdx.x, ti, tj);
  ti = uniform(ti);
  tj = uniform(tj);
  const int64_t ld = uniform(P.Np);
  const auto X = gbl(uniform((const T*)P.S));
  __shared__ GemmLds<T> lds;
  typename Acc<T>::type acc[2][2];
  zero_acc<T>(acc);
  const unsigned m = threadIdx.x & 63;
  const int kb = uniform((int)(threadIdx.x >> 6));
  auto rows = [&](int k, int t, T (&v)[16]) {
    auto p = X + ((int64_t)k * TILE + ((int64_t)t * TILE + kb) * ld);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += 4 * ld) v[q] = p[m];
  };
  gemm_tiles<T, true>(
      ti, nb, [&](int k, T (&v)[16]) { rows(k, ti, v); },
      [&](int k, T (&v)[16]) { rows(k, tj, v); }, lds, acc);
  const auto S = gbl(vslot(P, V_S));
  const auto C = gbl(P.C);
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int i = ti * TILE + acc_row<T>(bm, rr);
        const int j = tj * TILE + acc_col(bn);
        double v = (double)acc[bm][bn][rr];
        if (use_scale) v *= S[i] * S[j];
        if (i >= P.N || j >= P.N) v = 0.0;
        C[(size_t)i + (size_t)j * ld] = v;
      }
}

void launch_sym_from_inv(const Batch& b, int prec, int use_scale, hipStream_t s) {
  const int nb = b.maxNp / TILE;
  dim3 g(nb * (nb + 1) / 2, b.count);
  if (prec == PGP_PREC_FP64)
    hipLaunchKernelGGL(k_sym_from_inv<double>, g, dim3(NTHREADS), 0, s, b.dprobs, use_scale);
  else
    hipLaunchKernelGGL(k_sym_from_inv<float>, g, dim3(NTHREADS), 0, s, b.dprobs, use_scale);
}

// Where W_i is not positive, (K C)_ii = W_i Sigma_ii says nothing about
// Sigma_ii: there it is K_ii - ||V_:,i||^2, V = L^-1 S K.  A workgroup per row
// block I and column block J of V, the longest sums first: if one of J's
// columns has such a W, their norms over I's rows take the place of their row
// sums of K o C in slot I of J (k_symv_reduce then adds squares).  N^3 flops at
// worst, as the solve it stands for; none of it where all W > 0.  A gradient at
// N = 4096 takes 1.8 ms, 2.0 with 40 such W and 3.7 with 3686; with the
// quadratic form of C by one workgroup per such W 10.2 and 29.3.
__global__ __launch_bounds__(NTHREADS) void k_sigma_squares(Prob* const* probs) {
  const Prob& P = *probs[blockIdx.z];
  const int nb = uniform(P.Np) / TILE, J = blockIdx.y;
  const int I = nb - 1 - (int)blockIdx.x;
  if (I < 0 || J >= nb) return;
  const unsigned m = threadIdx.x & 63;
  const int kb = uniform((int)(threadIdx.x >> 6));
  const int64_t ld = uniform(P.Np);
  const auto W = gbl(vslot(P, V_W)) + J * TILE;
  const bool mine = J * TILE + (int)m < P.N && !(W[m] > 0.0);
  const uint64_t which = __builtin_amdgcn_ballot_w64(mine);  // the same in every wave
  if (which == 0) return;
  const auto X = gbl(uniform((const double*)P.S));  // L^-1
  const auto K = gbl(uniform(P.K));
  const auto S = gbl(vslot(P, V_S));
  __shared__ GemmLds<double> lds;
  doublex4 acc[2][2];
  zero_acc<double>(acc);
  gemm_tiles<double, false>(
      0, I + 1,
      [&](int k, double (&v)[16]) {
        auto p = X + ((int64_t)I * TILE + ((int64_t)k * TILE + kb) * ld);
#pragma unroll
        for (int q = 0; q < 16; ++q, p += 4 * ld) v[q] = p[m];
      },
      [&](int k, double (&v)[16]) {
        const double sk = S[(int64_t)k * TILE + m];
        auto p = K + ((int64_t)k * TILE + ((int64_t)J * TILE + kb) * ld);
#pragma unroll
        for (int q = 0; q < 16; ++q, p += 4 * ld) v[q] = sk * p[m];
      },
      lds, acc);
  constexpr int PB = GemmLds<double>::PB;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double v = acc[bm][bn][r];
        lds.b[acc_row<double>(bm, r) * PB + acc_col(bn)] = v * v;
      }
  __syncthreads();
  if (kb == 0 && mine) {
    double a = 0.0;
    for (int r = 0; r < TILE; ++r) a += lds.b[r * PB + m];
    P.symv[((size_t)J * nb + I) * TILE + m] = a;
  }
}

// Right-hand side S_i K_ij of V = L^-1 S K (factors stored in FP32).
__global__ __launch_bounds__(NTHREADS) void k_fill_rhs(Prob* const* probs) {
  const Prob& P = *probs[blockIdx.y];
  const int64_t e = (int64_t)blockIdx.x * NTHREADS + threadIdx.x;
  if (e >= (int64_t)P.Np * P.Np) return;
  ((float*)P.S)[e] = (float)(vslot(P, V_S)[e % P.Np] * P.K[e]);
}

// Sigma_jj = K_jj - ||V_:,j||^2 into X1 (one wave per column).
__global__ __launch_bounds__(NTHREADS) void k_sigma_norms(Prob* const* probs) {
  const Prob& P = *probs[blockIdx.y];
  const int j = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (j >= P.Np) return;
  const int lane = threadIdx.x & 63;
  const float* V = (const float*)P.S + (size_t)j * P.Np;
  double q = 0.0;
  for (int i = lane; i < P.Np; i += 64) {
    const double v = (double)V[i];
    q += v * v;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) q += __shfl_xor(q, off);
  if (lane == 0) vslot(P, V_X1)[j] = (j < P.N) ? P.K[(size_t)j * P.Np + j] - q : 0.0;
}

// diag Sigma into X1, Sigma = (K^-1 + W)^-1 = K - K C K.  FP64 factors: from C
// and K.  Sigma W = K C, so Sigma_ii = (sum_j K_ij C_ij) / W_i, two N^2 passes
// where the column norms of L^-1 S K take a solve with N right-hand sides (N^3
// flops: 3.2 ms at N = 4096, now 0.05), except where W_i <= 0
// (k_sigma_squares).  The sum cancels as K W grows, like the norms': an entry's
// error is up to nine times theirs (N = 400, Gaussian noise 1e-3: 9e-8 and 9e-9
// relative, both with the condition of B), but the gradient, which adds the
// entries up, is as accurate (noise 1e-3: 6.6e-10 and 5.7e-10; 0.03: 3.6e-13
// and 2.4e-13; probit noise 0.1, N = 400: 2.9e-12 and 3.3e-12).
// Factors stored in FP32 keep the column norms: C then carries the factor's
// FP32 error, which the norms damp (noise gradient of a Gaussian fit at N =
// 2000: 7e-5 relative error from the norms, 1e-3 from C).
void launch_sigma_diag(const Batch& b, int prec, hipStream_t s) {
  if (prec == PGP_PREC_FP64) {
    const int nb = b.maxNp / TILE;
    launch_hadamard_tiles(b, s);
    hipLaunchKernelGGL(k_sigma_squares, dim3(nb, nb, b.count), dim3(NTHREADS), 0, s, b.dprobs);
    launch_symv_reduce(b, V_X1, V_X1, 4, s);
    return;
  }
  const int64_t n2 = (int64_t)b.maxNp * b.maxNp;
  hipLaunchKernelGGL(k_fill_rhs, dim3((unsigned)((n2 + NTHREADS - 1) / NTHREADS), b.count),
                     dim3(NTHREADS), 0, s, b.dprobs);
  launch_trsm(b, prec, b.maxNp, s);
  hipLaunchKernelGGL(k_sigma_norms, dim3((b.maxNp + 3) / 4, b.count), dim3(NTHREADS), 0, s,
                     b.dprobs);
}

// Parameter p of (variance, lengthscale[GMAXD], period[GMAXD]) is one of the
// kernel's.
__device__ __forceinline__ bool grad_par_used(int p, int D, int periodic) {
  return p <= D || (periodic && p > GMAXD && p <= GMAXD + D);
}

// Fused trace: partials[tile][p] = w_tile * sum_{(i,j) in tile} dK_ij/dtheta_p G_ij
// with theta = (variance, lengthscale[D], period[D]) and G built from
// C (P.C), a (V_Z) and shat (V_X3).
__global__ __launch_bounds__(NTHREADS) void k_grad_trace(Prob* const* probs, double* partials) {
  const Prob& P = *probs[blockIdx.y];
  const int T = P.Np / TILE;
  const int ntiles = T * (T + 1) / 2;
  if ((int)blockIdx.x >= ntiles) return;
  int ti, tj;
  lower_tile_g(blockIdx.x, ti, tj);
  const int D = P.D;
  __shared__ double xs[TILE * GMAXD];
  __shared__ double zs[TILE * GMAXD];
  for (int e = threadIdx.x; e < TILE * D; e += NTHREADS) {
    const int r = e / D, d = e - r * D;
    const int gi = ti * TILE + r, gj = tj * TILE + r;
    xs[r * D + d] = gi < P.N ? P.X[(size_t)gi * D + d] : 0.0;
    zs[r * D + d] = gj < P.N ? P.X[(size_t)gj * D + d] : 0.0;
  }
  __syncthreads();
  const int il = threadIdx.x & 63, jg = threadIdx.x >> 6;
  const int i = ti * TILE + il;
  const double* a = vslot(P, V_Z);
  const double* sh = vslot(P, V_X3);
  const double ai = a[i], shi = sh[i];
  double acc[NPAR];
#pragma unroll
  for (int p = 0; p < NPAR; ++p) acc[p] = 0.0;
  const double wt = (ti == tj) ? 1.0 : 2.0;
  const bool eq = P.kern_kind == PGP_KERNEL_EQ;
  for (int c = 0; c < 16; ++c) {
    const int jl = jg * 16 + c;
    const int j = tj * TILE + jl;
    if (i >= P.N || j >= P.N) continue;
    const double G = wt * (0.5 * P.C[(size_t)i + (size_t)j * P.Np] - 0.5 * ai * a[j] +
                           0.5 * (shi * a[j] + ai * sh[j]));
    double q[GMAXD];
    double r2 = 0.0;
#pragma unroll
    for (int d = 0; d < GMAXD; ++d) {
      q[d] = 0.0;
      if (d < D) {
        const double df = xs[il * D + d] - zs[jl * D + d];
        if (P.periodic) {
          const double sn = sin(P.pi_over_per[d] * df);
          q[d] = 4.0 * sn * sn;
        } else {
          q[d] = df * df;
        }
        r2 += q[d] * P.inv_ls2[d];
      }
    }
    double kap, dk_dr2;
    if (eq) {
      kap = exp(-0.5 * r2);
      dk_dr2 = -0.5 * P.variance * kap;
    } else {
      const double r = sqrt(r2);
      kap = exp(-r);
      dk_dr2 = (r > 0.0) ? -P.variance * kap / (2.0 * r) : 0.0;
    }
    acc[0] += G * kap;
    const double gd = G * dk_dr2;
#pragma unroll
    for (int d = 0; d < GMAXD; ++d) {
      if (d < D) {
        const double l = P.ls[d];
        acc[1 + d] += gd * (-2.0 * q[d] * P.inv_ls2[d] / l);
        if (P.periodic) {
          const double df = xs[il * D + d] - zs[jl * D + d];
          const double per = P.per[d];
          const double dq = -4.0 * sin(2.0 * P.pi_over_per[d] * df) * M_PI * df / (per * per);
          acc[1 + GMAXD + d] += gd * dq * P.inv_ls2[d];
        }
      }
    }
  }
  // fixed-order block reduction of the accumulators in use
  __shared__ double red[NPAR][4];
#pragma unroll
  for (int p = 0; p < NPAR; ++p) {
    if (!grad_par_used(p, D, P.periodic)) continue;
    double v = acc[p];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if ((threadIdx.x & 63) == 0) red[p][threadIdx.x >> 6] = v;
  }
  __syncthreads();
  const int p = threadIdx.x;
  if (p < NPAR && grad_par_used(p, D, P.periodic))
    partials[((size_t)blockIdx.y * ntiles + blockIdx.x) * NPAR + p] =
        (red[p][0] + red[p][1]) + (red[p][2] + red[p][3]);
}

// out[b * NPAR + p] = sum over tiles (fixed order), one workgroup per p
__global__ __launch_bounds__(NTHREADS) void k_sum_partials(Prob* const* probs,
                                                           const double* partials, double* out) {
  const Prob& P = *probs[blockIdx.y];
  const int T = P.Np / TILE;
  const int ntiles = T * (T + 1) / 2;
  const int p = blockIdx.x;
  __shared__ double red[NTHREADS];
  double v = 0.0;
  if (grad_par_used(p, P.D, P.periodic))
    for (int t = threadIdx.x; t < ntiles; t += NTHREADS)
      v += partials[((size_t)blockIdx.y * ntiles + t) * NPAR + p];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int st = NTHREADS / 2; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[(size_t)blockIdx.y * NPAR + p] = red[0];
}

int grad_npar() { return NPAR; }
int grad_maxd() { return GMAXD; }

void launch_grad_trace(const Batch& b, double* partials, double* out, hipStream_t s) {
  const int T = b.maxNp / TILE;
  dim3 g(T * (T + 1) / 2, b.count);
  hipLaunchKernelGGL(k_grad_trace, g, dim3(NTHREADS), 0, s, b.dprobs, partials);
  hipLaunchKernelGGL(k_sum_partials, dim3(NPAR, b.count), dim3(NTHREADS), 0, s, b.dprobs, partials, out);
}

// VB traces: out[0] = tr(C), out[1] = sum_ij K_ij C_ij over the N x N block
// (the row sums of K o C, in X1).
__global__ __launch_bounds__(NTHREADS) void k_vb_trace(Prob* const* probs, double* out) {
  const Prob& P = *probs[blockIdx.x];
  const double* rows = vslot(P, V_X1);
  double tr = 0.0, kc = 0.0;
  for (int i = threadIdx.x; i < P.N; i += NTHREADS) {
    kc += rows[i];
    tr += P.C[(size_t)i + (size_t)i * P.Np];
  }
  __shared__ double r1[NTHREADS], r2[NTHREADS];
  r1[threadIdx.x] = tr;
  r2[threadIdx.x] = kc;
  __syncthreads();
  for (int st = NTHREADS / 2; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) {
      r1[threadIdx.x] += r1[threadIdx.x + st];
      r2[threadIdx.x] += r2[threadIdx.x + st];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[2 * blockIdx.x] = r1[0];
    out[2 * blockIdx.x + 1] = r2[0];
  }
}

void launch_vb_trace(const Batch& b, double* out, hipStream_t s) {
  launch_hadamard_tiles(b, s);
  launch_symv_reduce(b, V_X1, V_X1, 0, s);
  hipLaunchKernelGGL(k_vb_trace, dim3(b.count), dim3(NTHREADS), 0, s, b.dprobs, out);
}

// The VB adjoint's noise-std terms besides the likelihood partials:
// out[0] = tr(C), out[1] = v . (d1 - 2 sigma a) with v in X4.
__global__ __launch_bounds__(NTHREADS) void k_vb_sigma_terms(Prob* const* probs, double* out) {
  const Prob& P = *probs[blockIdx.x];
  const double* v = vslot(P, V_X4);
  const double* a = vslot(P, V_Z);
  const double* g = vslot(P, V_G);
  double tr = 0.0, dv = 0.0;
  for (int i = threadIdx.x; i < P.N; i += NTHREADS) {
    tr += P.C[(size_t)i + (size_t)i * P.Np];
    dv += v[i] * (g[i] - 2.0 * P.noise_std * a[i]);
  }
  __shared__ double r1[NTHREADS], r2[NTHREADS];
  r1[threadIdx.x] = tr;
  r2[threadIdx.x] = dv;
  __syncthreads();
  for (int st = NTHREADS / 2; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) {
      r1[threadIdx.x] += r1[threadIdx.x + st];
      r2[threadIdx.x] += r2[threadIdx.x + st];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[2 * blockIdx.x] = r1[0];
    out[2 * blockIdx.x + 1] = r2[0];
  }
}

void launch_vb_sigma_terms(const Batch& b, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_vb_sigma_terms, dim3(b.count), dim3(NTHREADS), 0, s, b.dprobs, out);
}

}  // namespace pgp
