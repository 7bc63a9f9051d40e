// GP prior sampling: f = L_K z with L_K the Cholesky factor of K + jitter I
// (probit's data generators: examples/regression.py:52-58,
// examples/classification.py:227-234).  The Gram matrix and the factor come
// from the library's FP64 kernels; this file holds the two pieces around
// them: the jitter / padding of K and the lower-triangular product L z.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mfma.hpp"
#include "pgp_internal.hpp"

namespace pgp {

// The factor's descriptor, status word, ticket and sync words (one workgroup).
struct PriorPage {
  Prob prob;
  Prob* self;
  int32_t info[4];
  uint64_t progress;
  uint32_t ticket;
};
static_assert(sizeof(PriorPage) <= 4096, "the page fits its workspace");

__global__ __launch_bounds__(NTHREADS) void k_prior_page(PriorPage* page, Prob val) {
  const uint64_t* src = reinterpret_cast<const uint64_t*>(&val);
  uint64_t* d = reinterpret_cast<uint64_t*>(&page->prob);
  for (int i = threadIdx.x; i < (int)(sizeof(Prob) / 8); i += NTHREADS) d[i] = src[i];
  if (threadIdx.x == 0) {
    page->self = &page->prob;
    page->progress = 0;
    page->ticket = 0;
  }
  if (threadIdx.x < 4) page->info[threadIdx.x] = 0;
  for (int64_t w = threadIdx.x; w < csync_words(val.Np); w += NTHREADS) val.csync[w] = 0;
}

// K (Np x Np, column-major, ld) after the Gram kernel wrote its N x N block:
// jitter on the diagonal, identity in the padding (rows / columns N..Np-1,
// so the padded factor is the identity there).  One workgroup per column.
__global__ __launch_bounds__(NTHREADS) void k_prior_prepare(double* A, int64_t ld, int N, int Np,
                                                           double jitter) {
  const int j = blockIdx.x;
  double* col = A + (size_t)j * ld;
  if (j < N) {
    if (threadIdx.x == 0) col[j] += jitter;
    for (int i = N + threadIdx.x; i < Np; i += NTHREADS) col[i] = 0.0;
  } else {
    for (int i = threadIdx.x; i < Np; i += NTHREADS) col[i] = (i == j) ? 1.0 : 0.0;
  }
}

// f(64 I.., 64 c..) = sum_{J <= I} L(64 I.., 64 J..) z(64 J.., 64 c..) on
// FP64 MFMA, one workgroup per 64 x 64 output tile (the longest sums first).
// The diagonal block's upper triangle is masked (the factor storage holds
// only the lower triangle); rows of z past N and columns past S read as zero.
__global__ __launch_bounds__(NTHREADS) void k_trmm_lower(const double* L, int64_t ld, int N,
                                                        const double* z, int64_t ldz, int S,
                                                        double* f, int64_t ldf) {
  __shared__ GemmLds<double> lds;
  const int I = gridDim.x - 1 - blockIdx.x, c = blockIdx.y;
  const unsigned m = threadIdx.x & 63;
  const int kb = uniform((int)(threadIdx.x >> 6));
  const int64_t r0 = (int64_t)I * TILE, n0 = (int64_t)c * TILE;
  doublex4 acc[2][2];
  zero_acc<double>(acc);
  gemm_tiles<double, false>(
      0, I + 1,
      [&](int J, double (&v)[16]) {
        auto p = gbl(L) + (r0 + ((int64_t)J * TILE + kb) * ld);
#pragma unroll
        for (int q = 0; q < 16; ++q, p += 4 * ld) {
          v[q] = p[m];
          if (J == I && kb + 4 * q > (int)m) v[q] = 0.0;
        }
      },
      [&](int J, double (&v)[16]) {
        const int64_t k = (int64_t)J * TILE + m;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int64_t n = n0 + kb + 4 * q;
          v[q] = k < N && n < S ? gbl(z)[(size_t)k + (size_t)n * ldz] : 0.0;
        }
      },
      lds, acc);
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t i = r0 + acc_row<double>(bm, r), j = n0 + acc_col(bn);
        if (i < N && j < S) f[(size_t)i + (size_t)j * ldf] = acc[bm][bn][r];
      }
}

// The same for at most TRMV_S columns, where the MFMA form would multiply
// padding and walk the tiles of a block row one after the other: a workgroup
// takes `per` tiles of block row I and the sums of its 64 rows wait in part
// [chunk][I][column][row]; k_trmv_sum adds the chunks in order.  Bound: one
// read of L's lower triangle (0.15 ms at N = 12288, S = 1, 4.0 TB/s; the MFMA
// form took 1.73 ms).
constexpr int TRMV_S = 8;

__global__ __launch_bounds__(NTHREADS) void k_trmv_part(const double* L, int64_t ld, int N,
                                                       const double* z, int64_t ldz, int S,
                                                       int per, double* part) {
  const int I = gridDim.x - 1 - blockIdx.x, chunk = blockIdx.y;
  const int J0 = chunk * per, J1 = min(I + 1, J0 + per);
  if (J0 > I) return;
  __shared__ double zs[TRMV_S][TILE];
  __shared__ double red[4][TRMV_S][TILE];
  const unsigned m = threadIdx.x & 63;
  const int w = uniform((int)(threadIdx.x >> 6));
  double acc[TRMV_S];
#pragma unroll
  for (int c = 0; c < TRMV_S; ++c) acc[c] = 0.0;
  for (int J = J0; J < J1; ++J) {
    double k[16];
    auto p = gbl(L) + ((int64_t)I * TILE + ((int64_t)J * TILE + 16 * w) * ld);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += ld) k[q] = p[m];
    if (J == I) {
#pragma unroll
      for (int q = 0; q < 16; ++q)
        if (16 * w + q > (int)m) k[q] = 0.0;
    }
    __syncthreads();  // the previous tile's z is read
    for (int e = threadIdx.x; e < S * TILE; e += NTHREADS) {
      const int64_t r = (int64_t)J * TILE + (e & 63);
      zs[e >> 6][e & 63] = r < N ? z[(size_t)r + (size_t)(e >> 6) * ldz] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < TRMV_S; ++c) {
      if (c >= S) break;
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[c] = fma(k[q], zs[c][16 * w + q], acc[c]);
    }
  }
#pragma unroll
  for (int c = 0; c < TRMV_S; ++c)
    if (c < S) red[w][c][m] = acc[c];
  __syncthreads();
  double* out = part + ((size_t)chunk * gridDim.x + I) * S * TILE;
  for (int e = threadIdx.x; e < S * TILE; e += NTHREADS) {
    const int c = e >> 6, r = e & 63;
    out[e] = (red[0][c][r] + red[1][c][r]) + (red[2][c][r] + red[3][c][r]);
  }
}

__global__ __launch_bounds__(NTHREADS) void k_trmv_sum(const double* part, int nb, int N, int S,
                                                      int per, double* f, int64_t ldf) {
  const int I = blockIdx.x;
  for (int e = threadIdx.x; e < S * TILE; e += NTHREADS) {
    const int64_t r = (int64_t)I * TILE + (e & 63);
    double v = 0.0;
    for (int c = 0; c * per <= I; ++c) v += part[((size_t)c * nb + I) * S * TILE + e];
    if (r < N) f[(size_t)r + (size_t)(e >> 6) * ldf] = v;
  }
}

int launch_prior_sample(const pgp_kernel_t* kernel, const double* X, int64_t N, double jitter,
                        const double* z, int64_t S, int64_t ldz, double* f, int64_t ldf,
                        char* ws, hipStream_t s) {
  const int64_t Np = (N + TILE - 1) / TILE * TILE;
  double* A = (double*)ws;
  double* dinv = (double*)(ws + prior_ws_offset_dinv(Np));
  PriorPage* page = (PriorPage*)(ws + prior_ws_offset_page(Np));
  launch_gram_raw(kernel, 0, X, N, X, N, A, Np, s);
  hipLaunchKernelGGL(k_prior_prepare, dim3((unsigned)Np), dim3(NTHREADS), 0, s, A, Np, (int)N,
                     (int)Np, jitter);
  // the fits' blocked factorisation (super-steps) on this matrix
  Prob p = {};
  p.N = (int32_t)N;
  p.Np = (int32_t)Np;
  p.prec = PGP_PREC_FP64;
  p.L = A;
  p.dinv = dinv;
  p.info = page->info;
  p.progress = &page->progress;
  p.csync = (uint32_t*)(ws + prior_ws_offset_csync(Np));
  hipLaunchKernelGGL(k_prior_page, dim3(1), dim3(NTHREADS), 0, s, page, p);
  Batch b;
  b.dprobs = &page->self;
  b.count = 1;
  b.maxNp = (int)Np;
  b.ticket = &page->ticket;
  launch_potrf(b, PGP_PREC_FP64, s);
  const int nb = (int)(Np / TILE);
  if (S <= TRMV_S) {
    // the chunks' sums take the place of the diagonal inverses (dead after
    // the factor): chunks x nb x S x 64 doubles of nb x 64 x 64
    const int chunks = std::min(nb, TILE / (int)S), per = (nb + chunks - 1) / chunks;
    hipLaunchKernelGGL(k_trmv_part, dim3((unsigned)nb, (unsigned)((nb + per - 1) / per)),
                       dim3(NTHREADS), 0, s, (const double*)A, Np, (int)N, z, ldz, (int)S, per,
                       dinv);
    hipLaunchKernelGGL(k_trmv_sum, dim3((unsigned)nb), dim3(NTHREADS), 0, s, (const double*)dinv,
                       nb, (int)N, (int)S, per, f, ldf);
    return 0;
  }
  hipLaunchKernelGGL(k_trmm_lower, dim3((unsigned)nb, (unsigned)((S + TILE - 1) / TILE)),
                     dim3(NTHREADS), 0, s, (const double*)A, Np, (int)N, z, ldz, (int)S, f, ldf);
  return 0;
}

}  // namespace pgp
