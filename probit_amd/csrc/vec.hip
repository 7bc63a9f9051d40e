// FP64 vector work of the Newton / fixed-point loops and the predict epilogue.
//
//  * symmetric GEMV y = K x: each lower 64x64 tile of K is read once (row
//    and column sums into per-tile slots, then a fixed-order reduction with
//    a fused epilogue: f = K a, S .* K r, refinement residuals), so HBM
//    reads half of K per product.
//    Replaces `K @ weight` (probit/implicit/Laplace.py:8,22,
//    probit/approximators.py:273,338) and the matvecs inside the reference's
//    dense Jacobian (probit/implicit/solvers.py:24).
//  * elementwise Newton updates and fixed-order per-problem reductions
//    (step norm for the jaxopt stopping rule, sum log p, f.a, log|B|).
//  * predict epilogue: mean_j = sum of per-tile partials, var_j = Kss -
//    ||V_:,j||^2 (probit/approximators.py:176-179).
#include "pgp_internal.hpp"

namespace pgp {

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// mode 0: out = Kx
// mode 1: out = SF .* Kx              (SF: the W^1/2 of the factored B)
// mode 2: out = R - DL - S^2 .* Kx     (Laplace residual of (I + W K) d = r, x = DL)
// mode 3: out = X1 - sigma^2 x - Kx    (VB residual of (sigma^2 I + K) w = rhs, rhs in X1)
// mode 4: out = Kx / W within [0, K_ii], or K_ii - Kx where W <= 0: diag of
//         (K^-1 + W)^-1 from the row sums of K o C, or the squares of
//         k_sigma_squares
// (modes >= 10: the same with the matrix C in place of K)
__device__ __forceinline__ void gemv_epilogue(const Prob& P, int i, const double* x, int os,
                                              int mode, double sum) {
  double v;
  switch (mode) {
    case 0:
      v = sum;
      break;
    case 1:
      v = vslot(P, V_SF)[i] * sum;
      break;
    case 2: {
      const double si = vslot(P, V_S)[i];
      v = vslot(P, V_R)[i] - x[i] - si * si * sum;
      break;
    }
    case 4: {
      const double W = vslot(P, V_W)[i], kii = P.variance;
      v = W > 0.0 ? sum / W : kii - sum;
      if (W > 0.0) v = v < 0.0 ? 0.0 : v > kii ? kii : v;  // (a NaN stays one)
      if (i >= P.N) v = 0.0;
      break;
    }
    default: {
      const double s2 = (i < P.N) ? P.noise_std * P.noise_std : 1.0;
      v = vslot(P, V_X1)[i] - s2 * x[i] - sum;
      break;
    }
  }
  vslot(P, os)[i] = v;
}

// Symmetric product y = K x reading each lower 64x64 tile of K once: the
// tile (I, J) gives its row sums K_IJ x_J (towards y_I) and, off the
// diagonal, its column sums K_IJ^T x_I (towards y_J), each written to its
// own slot part[I][J] / part[J][I] (64 doubles).  k_symv_reduce then adds
// the nb slots of every row block in a fixed order, so the result does not
// depend on scheduling, and applies the epilogue.
__device__ __forceinline__ void lower_tile_v(int t, int& ti, int& tj) {
  int i = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while ((i + 1) * (i + 2) / 2 <= t) ++i;
  while (i * (i + 1) / 2 > t) --i;
  ti = i;
  tj = t - i * (i + 1) / 2;
}

// MAT: the matrix is K, C, or (with x = 1: row sums) K o C.
enum SymvMat { SYMV_K = 0, SYMV_C = 1, SYMV_HADAMARD = 2 };
template <int MAT>
__global__ __launch_bounds__(NTHREADS) void k_symv_tiles(Prob* const* probs, Sched sc, int xs) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int nb = uniform(P.Np) / TILE;
  if (bx >= nb * (nb + 1) / 2) return;
  int ti, tj;
  lower_tile_v(bx, ti, tj);
  ti = uniform(ti);
  tj = uniform(tj);
  __shared__ double rpart[4][TILE];
  const int64_t ld = uniform(P.Np);
  const unsigned r = threadIdx.x & 63;
  const int w = uniform((int)(threadIdx.x >> 6));
  const double* xp = uniform(P.vec) + xs * ld;
  const auto x = gbl(xp);
  const auto xj = scalar(xp) + (tj * TILE + w);
  const int64_t tile = ti * TILE + (tj * TILE + w) * ld;
  const auto Kt = gbl(uniform(MAT == SYMV_C ? P.C : P.K)) + tile;
  // lane r holds row r of the wave's 16 columns c = w + 4q (coalesced down
  // each column); the tile never goes through LDS
  double k[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) k[q] = (Kt + 4 * q * ld)[r];
  if constexpr (MAT == SYMV_HADAMARD) {
    const auto Ct = gbl(uniform(P.C)) + tile;
    double c[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) c[q] = (Ct + 4 * q * ld)[r];
#pragma unroll
    for (int q = 0; q < 16; ++q) k[q] *= c[q];
  }
  const double xi = MAT == SYMV_HADAMARD ? 1.0 : x[ti * TILE + r];
  double rs = 0.0;
#pragma unroll
  for (int q = 0; q < 16; ++q)
    rs += MAT == SYMV_HADAMARD ? k[q] : k[q] * xj[4 * q];
  rpart[w][r] = rs;
  const auto part = gbl(uniform(P.symv));
  if (ti != tj) {
    // column sums K_IJ^T x_I of the wave's 16 columns: lane l ends with column
    // q = (l >> 2) & 15
    double v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = k[q] * xi;
    const double cs = column_sums(v);
    if ((r & 3) == 0)
      part[((size_t)tj * nb + ti) * TILE + w + 4 * ((r >> 2) & 15)] = cs;
  }
  __syncthreads();
  if (w == 0)
    part[((size_t)ti * nb + tj) * TILE + r] = (rpart[0][r] + rpart[1][r]) + (rpart[2][r] + rpart[3][r]);
}

// One workgroup per row block, its waves every fourth slot: with a thread a row
// a workgroup read 256 rows' slots one after another (N = 4096: 11.3 us, 5.2
// with four times the workgroups and loads in flight).
__global__ __launch_bounds__(NTHREADS) void k_symv_reduce(Prob* const* probs, Sched sc, int xs,
                                                          int os, int mode) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int nb = uniform(P.Np) / TILE;
  if (bx >= nb) return;
  const unsigned r = threadIdx.x & 63;
  const int w = uniform((int)(threadIdx.x >> 6));
  const auto part = gbl(uniform(P.symv)) + (size_t)bx * nb * TILE;
  double a0 = 0.0, a1 = 0.0;
  int J = w;
#pragma unroll 4
  for (; J + 4 < nb; J += 8) {
    a0 += (part + (size_t)J * TILE)[r];
    a1 += (part + (size_t)(J + 4) * TILE)[r];
  }
  if (J < nb) a0 += (part + (size_t)J * TILE)[r];
  __shared__ double sum[4][TILE];
  sum[w][r] = a0 + a1;
  __syncthreads();
  if (w == 0)
    gemv_epilogue(P, bx * TILE + r, vslot(P, xs), os, mode,
                  (sum[0][r] + sum[1][r]) + (sum[2][r] + sum[3][r]));
}

template <int MAT>
static void symv_tiles(const Batch& b, int x_slot, hipStream_t s) {
  sched_launch(
      b,
      [&](int m) {
        const int t = b.np(m) / TILE;
        return t * (t + 1) / 2;
      },
      [&](Prob* const* dp, const Sched& sc, int n) {
        hipLaunchKernelGGL(k_symv_tiles<MAT>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, x_slot);
      });
}

void launch_gemv_sym(const Batch& b, int x_slot, int out_slot, int mode, hipStream_t s) {
  if (mode >= 10)
    symv_tiles<SYMV_C>(b, x_slot, s);
  else
    symv_tiles<SYMV_K>(b, x_slot, s);
  launch_symv_reduce(b, x_slot, out_slot, mode % 10, s);
}

void launch_symv_tiles(const Batch& b, int x_slot, hipStream_t s) {
  symv_tiles<SYMV_K>(b, x_slot, s);
}

void launch_hadamard_tiles(const Batch& b, hipStream_t s) {
  symv_tiles<SYMV_HADAMARD>(b, V_X1, s);
}

void launch_symv_reduce(const Batch& b, int x_slot, int out_slot, int mode, hipStream_t s) {
  sched_launch(
      b, [&](int m) { return b.np(m) / TILE; },
      [&](Prob* const* dp, const Sched& sc, int n) {
        hipLaunchKernelGGL(k_symv_reduce, dim3(n), dim3(NTHREADS), 0, s, dp, sc, x_slot, out_slot,
                           mode);
      });
}



__global__ __launch_bounds__(NTHREADS) void k_vec(Prob* const* probs, Sched sc, int op) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int i = bx * NTHREADS + threadIdx.x;
  if (i >= P.Np) return;
  switch (op) {
    case OP_STEP:
      vslot(P, V_DL)[i] = vslot(P, V_R)[i] - vslot(P, V_SF)[i] * vslot(P, V_U)[i];
      break;
    case OP_IRCORR:
      vslot(P, V_DL)[i] += vslot(P, V_Q)[i] - vslot(P, V_SF)[i] * vslot(P, V_U)[i];
      break;
    case OP_SNAP:
      vslot(P, V_SF)[i] = vslot(P, V_S)[i];
      break;
    case OP_ZERO_Z:  // the zero weight and its latent f = K 0
      vslot(P, V_Z)[i] = 0.0;
      vslot(P, V_F)[i] = 0.0;
      break;
    case OP_OUT:
      if (i < P.N) {
        if (P.out_weight) P.out_weight[i] = vslot(P, V_Z)[i];
        if (P.out_prec) P.out_prec[i] = vslot(P, V_W)[i];
        if (P.out_latent) P.out_latent[i] = vslot(P, V_F)[i];
      }
      break;
    case OP_VB_RHS:
      vslot(P, V_X1)[i] = vslot(P, V_F)[i] + P.noise_std * vslot(P, V_G)[i];
      break;
    case OP_VB_STEP:
      vslot(P, V_DL)[i] = vslot(P, V_U)[i] - vslot(P, V_Z)[i];
      break;
    case OP_VB_IRCORR:
      vslot(P, V_U)[i] += vslot(P, V_X4)[i];
      break;
    case OP_GRAD_S2:
      vslot(P, V_X2)[i] = -0.5 * vslot(P, V_X1)[i] * vslot(P, V_D3)[i];
      break;
    case OP_GRAD_SHAT:
      vslot(P, V_X3)[i] = vslot(P, V_X2)[i] - vslot(P, V_T)[i];
      break;
    case OP_VBG_R:
      vslot(P, V_X1)[i] = vslot(P, V_Z)[i] - vslot(P, V_G)[i];
      break;
    case OP_VBG_T:
      vslot(P, V_T)[i] = vslot(P, V_S)[i] * vslot(P, V_X2)[i];
      break;
    case OP_VBG_Z:
      vslot(P, V_X4)[i] = vslot(P, V_S)[i] * vslot(P, V_U)[i];
      break;
    case OP_VBG_V:
      vslot(P, V_X4)[i] =
          (vslot(P, V_X2)[i] - vslot(P, V_X3)[i]) / (P.noise_std * P.noise_std);
      break;
    case OP_VBG_SHAT: {
      const double v = vslot(P, V_X4)[i];
      vslot(P, V_X3)[i] = vslot(P, V_Z)[i] - vslot(P, V_G)[i] - P.noise_std * vslot(P, V_W)[i] * v;
      vslot(P, V_X1)[i] = 0.0;
      vslot(P, V_X2)[i] = P.noise_std * v;
      break;
    }
    case OP_VB_PREC: {
      const double w = (i < P.N) ? 1.0 / (P.noise_std * P.noise_std) : 0.0;
      vslot(P, V_W)[i] = w;
      vslot(P, V_S)[i] = sqrt(w);
      break;
    }
    default:
      break;
  }
}

void launch_vec_op(const Batch& b, int op, hipStream_t s) {
  sched_launch(
      b, [&](int m) { return (b.np(m) + NTHREADS - 1) / NTHREADS; },
      [&](Prob* const* dp, const Sched& sc, int n) {
        hipLaunchKernelGGL(k_vec, dim3(n), dim3(NTHREADS), 0, s, dp, sc, op);
      });
}

__global__ __launch_bounds__(NTHREADS) void k_load_state(Prob* const* probs, Sched sc,
                                                         const double* weight, const double* W) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int i = bx * NTHREADS + threadIdx.x;
  if (i >= P.Np) return;
  if (weight) vslot(P, V_Z)[i] = (i < P.N) ? weight[i] : 0.0;
  if (W) {
    const double w = (i < P.N) ? W[i] : 0.0;
    vslot(P, V_W)[i] = w;
    vslot(P, V_S)[i] = sqrt(fmax(w, 0.0));
  }
}

void launch_load_state(const Batch& b, const double* weight, const double* W, hipStream_t s) {
  sched_launch(
      b, [&](int m) { return (b.np(m) + NTHREADS - 1) / NTHREADS; },
      [&](Prob* const* dp, const Sched& sc, int n) {
        hipLaunchKernelGGL(k_load_state, dim3(n), dim3(NTHREADS), 0, s, dp, sc, weight, W);
      });
}

// Copy a vector slot between problems' slots (same problem): dst = src.
__global__ __launch_bounds__(NTHREADS) void k_copy_slot(Prob* const* probs, Sched sc, int src,
                                                        int dst) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int i = bx * NTHREADS + threadIdx.x;
  if (i >= P.Np) return;
  vslot(P, dst)[i] = vslot(P, src)[i];
}

void launch_copy_slot(const Batch& b, int src, int dst, hipStream_t s) {
  sched_launch(
      b, [&](int m) { return (b.np(m) + NTHREADS - 1) / NTHREADS; },
      [&](Prob* const* dp, const Sched& sc, int n) {
        hipLaunchKernelGGL(k_copy_slot, dim3(n), dim3(NTHREADS), 0, s, dp, sc, src, dst);
      });
}

// ---- fixed-order block reduction ----
__device__ double block_sum(double v) {
  __shared__ double ws[NTHREADS / 64];
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
  __syncthreads();
  return (ws[0] + ws[1]) + (ws[2] + ws[3]);
}



// One workgroup per member: at N = 16384 a thread has 64 elements, some 10 us;
// a launch each for the step, the update and the norm cost a small fit as much
// (N = 20, with the status and the norm read back in one copy: 359 -> 308 us a
// fit and its predict).
__global__ __launch_bounds__(NTHREADS) void k_newton_step(Prob* const* probs, int op,
                                                          double* gather) {
  const Prob& P = *probs[blockIdx.x];
  const int np = uniform(P.Np);
  const double* vec = uniform(P.vec);
  const auto slot = [&](int v) { return gbl((double*)vec + (size_t)v * np); };
  const auto DL = slot(V_DL), Z = slot(V_Z);
  const auto U = slot(V_U), R = slot(op == OP_IRCORR ? V_Q : V_R), SF = slot(V_SF);
  const bool take = !(P.info[0] & PGP_INFO_NOT_PD);  // no step from a failed factor
  double a = 0.0;
#pragma unroll 4
  for (int i = threadIdx.x; i < np; i += NTHREADS) {
    const double z = Z[i];
    double d = op == OP_VB_STEP ? U[i] - z : R[i] - SF[i] * U[i];
    if (op == OP_IRCORR) d += DL[i];
    DL[i] = d;
    if (take) Z[i] = z + d;
    a += d * d;
  }
  const double s = block_sum(a);
  if (threadIdx.x == 0) {
    P.red[R_STEP2] = s;
    if (gather) gather[blockIdx.x] = s;
  }
}

void launch_newton_step(const Batch& b, int op, double* gather, hipStream_t s) {
  hipLaunchKernelGGL(k_newton_step, dim3(b.count), dim3(NTHREADS), 0, s, b.dprobs, op, gather);
}

__global__ __launch_bounds__(NTHREADS) void k_reduce(Prob* const* probs, int what,
                                                     double* gather) {
  const Prob& P = *probs[blockIdx.x];
  const double* ll = vslot(P, V_LL);
  const double* f = vslot(P, V_F);
  const double* z = vslot(P, V_Z);
  const double* w = vslot(P, V_W);
  double a = 0.0, b = 0.0, c = 0.0, n = 0.0;
  for (int i = threadIdx.x; i < P.Np; i += NTHREADS) {
    a += ll[i];
    b += f[i] * z[i];
    c += P.logdiag[i];
    n += (i < P.N && w[i] < 0.0) ? 1.0 : 0.0;
    if (what == RED_FINAL_OUT && i < P.N) {  // OP_OUT
      if (P.out_weight) P.out_weight[i] = z[i];
      if (P.out_prec) P.out_prec[i] = w[i];
      if (P.out_latent) P.out_latent[i] = f[i];
    }
  }
  const double sa = block_sum(a);
  const double sb = block_sum(b);
  const double sc = block_sum(c);
  const double sn = block_sum(n);
  if (threadIdx.x == 0) {
    P.red[R_SUMLL] = sa;
    P.red[R_FA] = sb;
    P.red[R_LOGDET] = sc;
    P.red[R_NEGW] = sn;
    if (gather) {
      gather[8 * blockIdx.x + 0] = sa;
      gather[8 * blockIdx.x + 1] = sb;
      gather[8 * blockIdx.x + 2] = sc;
      gather[8 * blockIdx.x + 3] = sn;
      gather[8 * blockIdx.x + 4] = (double)P.info[0];
    }
  }
}
void launch_reduce(const Batch& b, int what, double* gather, hipStream_t s) {
  hipLaunchKernelGGL(k_reduce, dim3(b.count), dim3(NTHREADS), 0, s, b.dprobs, what, gather);
}

// ---- predict epilogue: one wave per test point ----
template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_predict_final(Prob* const* probs, Sched sc) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int j = bx * 4 + (threadIdx.x >> 6);
  if (j >= P.M) return;
  const int lane = threadIdx.x & 63;
  const int nrt = P.Np / TILE;
  double q;
  if (P.qpart) {  // the FP64-corrected quadratic forms, summed over row tiles
    double qa = 0.0;
    for (int rt = lane; rt < nrt; rt += 64) qa += P.qpart[(size_t)rt * P.Mp + j];
    q = wave_sum(qa);
  } else {
    const T* S = (const T*)P.S + (size_t)j * P.Np;
    double q0 = 0.0, q1 = 0.0;
    int i = lane;
    for (; i + 64 < P.Np; i += 128) {
      const double v0 = (double)S[i], v1 = (double)S[i + 64];
      q0 += v0 * v0;
      q1 += v1 * v1;
    }
    for (; i < P.Np; i += 64) {
      const double v = (double)S[i];
      q0 += v * v;
    }
    q = wave_sum(q0 + q1);
  }
  double mu = 0.0;
  for (int rt = lane; rt < nrt; rt += 64) mu += P.mupart[(size_t)rt * P.Mp + j];
  mu = wave_sum(mu);
  if (lane == 0) {
    P.pmean[j] = mu;
    P.pvar[j] = P.variance - q;
  }
}

void launch_predict_final(const Batch& b, int prec, int maxM, hipStream_t s) {
  sched_launch(
      b, [&](int m) { return (b.mcount(m, maxM) + 3) / 4; },
      [&](Prob* const* dp, const Sched& sc, int n) {
        if (prec == PGP_PREC_FP64)
          hipLaunchKernelGGL(k_predict_final<double>, dim3(n), dim3(NTHREADS), 0, s, dp, sc);
        else
          hipLaunchKernelGGL(k_predict_final<float>, dim3(n), dim3(NTHREADS), 0, s, dp, sc);
      });
}

}  // namespace pgp
