// Triangular solves with the resident Cholesky factor.
//
// TRSV (one right-hand side per problem) serves the Newton step
// (I + W K)^-1 r = r - W^1/2 B^-1 W^1/2 K r (the reference's dense LU solve,
// probit/implicit/solvers.py:24) and B.cholesky_solve (probit/implicit/VB.py:11).
// TRSM (many right-hand sides) serves predict's solve against Kfs
// (probit/approximators.py:177) and the explicit inverses of
// probit/implicit/VB.py:26-27.
//
// Both are blocked by 64 and run as one wavefront launch (k_trsv_seg,
// k_trsm_rows), or without a ticket counter as a launch per block step.  The
// diagonal block is applied as a product with its precomputed FP64 inverse
// (DINV), so no step has a serial substitution chain; the off-diagonal update
// is a GEMV / MFMA GEMM.  Vectors are FP64 throughout; TRSM runs in the
// factor's storage type.
#include <stdlib.h>

#include <algorithm>
#include <atomic>

#include "mfma.hpp"
#include "pgp_internal.hpp"
#include "solve_schedule.hpp"

namespace pgp {

// x = DINV_k b_k (trans = 0) or DINV_k^T b_k (trans = 1), 64 outputs in xs.
__device__ __forceinline__ void apply_dinv(const double* Dk, const double* bk_lds, double* xs,
                                           int trans) {
  __shared__ double part[4][TILE];
  const int i = threadIdx.x & 63, q = threadIdx.x >> 6;
  double acc = 0.0;
#pragma unroll 4
  for (int p = 16 * q; p < 16 * q + 16; ++p) {
    const double d = trans ? Dk[p + i * TILE] : Dk[i + p * TILE];
    acc += d * bk_lds[p];
  }
  part[q][i] = acc;
  __syncthreads();
  if (threadIdx.x < TILE) xs[i] = (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]);
  __syncthreads();
}

template <typename T>
__device__ void trsv_fwd_step(const T* L, int64_t ld, int64_t Np, const double* dinv, int k,
                              double* b, double* x, int w) {
  __shared__ double bk[TILE], xk[TILE];
  __shared__ double part[4][TILE];
  const int64_t c0 = (int64_t)k * TILE;
  if (threadIdx.x < TILE) bk[threadIdx.x] = b[c0 + threadIdx.x];
  __syncthreads();
  apply_dinv(dinv + (size_t)k * TILE * TILE, bk, xk, 0);
  const int i = threadIdx.x & 63, q = threadIdx.x >> 6;
  if (w == 0) {
    if (threadIdx.x < TILE) x[c0 + i] = xk[i];
    return;
  }
  const int64_t R = c0 + (int64_t)TILE * w + i;
  double acc = 0.0;
#pragma unroll 4
  for (int p = 16 * q; p < 16 * q + 16; ++p)
    acc += (double)L[(size_t)R + (size_t)(c0 + p) * ld] * xk[p];
  part[q][i] = acc;
  __syncthreads();
  if (threadIdx.x < TILE) b[R] -= (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]);
}

template <typename T>
__device__ void trsv_bwd_step(const T* L, int64_t ld, const double* dinv, int k, double* b,
                              double* x, int w) {
  __shared__ double bk[TILE], xk[TILE];
  const int64_t c0 = (int64_t)k * TILE;
  if (threadIdx.x < TILE) bk[threadIdx.x] = b[c0 + threadIdx.x];
  __syncthreads();
  apply_dinv(dinv + (size_t)k * TILE * TILE, bk, xk, 1);
  const int i = threadIdx.x & 63, q = threadIdx.x >> 6;
  if (w == 0) {
    if (threadIdx.x < TILE) x[c0 + i] = xk[i];
    return;
  }
  // columns m in [64 (w-1), 64 w): b_m -= sum_i L[c0 + i][m] x_i
  const double xi = xk[i];
  for (int cq = 0; cq < 16; ++cq) {
    const int64_t m = (int64_t)TILE * (w - 1) + 16 * q + cq;
    double v = (double)L[(size_t)(c0 + i) + (size_t)m * ld] * xi;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if (i == 0) b[m] -= v;
  }
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_trsv(Prob* const* probs, Sched sc, int k, int trans,
                                                   int in, int out) {
  int w;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, w)];
  const int nb = P.Np / TILE;
  if (k >= nb) return;
  double* b = vslot(P, in);
  double* x = vslot(P, out);
  if (!trans) {
    if (w >= nb - k) return;
    trsv_fwd_step<T>((const T*)P.L, P.Np, P.Np, P.dinv, k, b, x, w);
  } else {
    if (w > k) return;
    trsv_bwd_step<T>((const T*)P.L, P.Np, P.dinv, k, b, x, w);
  }
}

// ---- single-launch TRSV in segments ------------------------------------------
// x = L^-1 b (or L^-T b) for every member in one launch: one workgroup of 16
// waves per segment of SEG block rows, in sweep order (forward: from the
// first block row; transposed: from the last one up).  Wave (rb, cg) takes 16
// columns (cg) of block row rb of the segment: it streams the tiles of that
// block row left (transposed: below) of the segment as their x becomes
// known, two tiles ahead in registers.  Then the segment's own blocks follow in turn, x_r =
// DINV_r v_r by the four waves of block row r, handed to the later block
// rows through LDS.
//
// x travels between workgroups as tagged words: value halves in two 64-bit
// words, each with the launch's epoch in its upper half, so a reader polls
// the data itself and no separate flag has to follow the data's completion.
// Both sweeps of a solve write the same buffer (Prob::xpub) in full under
// different epochs, so a replayed graph of a solve, whose epochs are the
// captured ones, never finds its own epoch left from the last replay.  One
// wave of a workgroup polls (one block ahead) and shares x through LDS.
//
// Bound: the chain of blocks.  One workgroup per block row with a progress
// word cost a hand-off through memory per block, 4.7-4.8 us; here the
// hand-off falls on every SEG-th block, and a sweep over N = 1537 takes 48-52
// us (FP64) / 33-34 us (FP32) where it took 119.  SEG = 4: the tiles a
// workgroup streams per block (SEG x 32 KB in FP64) then take about the time
// its chain needs for one.
//
// Workgroups take their segment from a ticket counter in start order, segment
// major, so a workgroup only waits for running ones, and every wait is
// bounded (SPIN_LIMIT polls): the member is then flagged PGP_INFO_STALLED and
// the sweep runs on, so every workgroup exits.
constexpr int SEG = 4;
constexpr int SEG_THREADS = 256 * SEG;

template <typename T, bool TR>
__global__ __launch_bounds__(SEG_THREADS) void k_trsv_seg(Prob* const* probs, Sched segs,
                                                          uint32_t* ticket, uint32_t epoch,
                                                          int in, int out) {
  __shared__ double xs[2][TILE];      // x of the block being streamed
  __shared__ double part[sizeof(T) == 8 ? 8 : 16][TILE];  // sums of block row r
  __shared__ double vs[4][TILE];      // v_r, one copy per wave
  __shared__ double xq[2][TILE];      // x of the segment's blocks
  constexpr bool DL = sizeof(T) == 8;
  __shared__ double dl[DL ? SEG : 1][DL ? TILE : 1][TILE + 1];  // FP64: DINV of the blocks
  __shared__ int s_val;
  const int tk = take_ticket(ticket, &s_val);
  if ((unsigned)tk >= gridDim.x) {  // counter not zero at launch: no segment to take
    flag_members_stalled(probs, segs.pre[1] - segs.pre[0]);  // segment 0 lists every member
    return;
  }
  int mi;
  const int seg = sched_member(segs, tk, mi);
  const Prob& P = *uniform(probs[mi]);
  const int nb = uniform(P.Np) / TILE;
  int64_t ld = (int64_t)nb * TILE;
  const auto L = gbl((const T*)uniform((char*)P.L));
  const auto dinv = gbl((const double*)uniform(P.dinv));
  double* const vec = uniform(P.vec);
  const auto bv = gbl((const double*)vec + (size_t)in * ld);
  const auto xv = gbl(vec + (size_t)out * ld);
  uint64_t* const pub = uniform(P.xpub);
  int32_t* const info = uniform(P.info);
  const unsigned l = threadIdx.x & 63;
  const int w = uniform((int)(threadIdx.x >> 6));
  const int rb = w >> 2, cg = w & 3;
  const int b0 = SEG * seg, nblk = min(SEG, nb - b0);
  auto block = [&](int s) { return TR ? nb - 1 - s : s; };  // sweep position -> block
  const bool act = rb < nblk;
  const int i = block(act ? b0 + rb : b0);
  const int ntile = act ? b0 + rb : 0;  // tiles of this wave's block row
  // a lane's part of the wave's 64 x 16 strip of a tile: VEC rows from
  // VEC lr (one 16-byte load) in each of NC columns from NC lg
  constexpr int VEC = 16 / (int)sizeof(T), RL = TILE / VEC, CG = 64 / RL, NC = 16 / CG;
  typedef T vec_t __attribute__((ext_vector_type(VEC)));
  const unsigned lr = l % RL, lg = l / RL;
  constexpr int DEPTH = 2;
  vec_t st[DEPTH][NC];
  auto load = [&](vec_t (&v)[NC], int s) {
    const int64_t j = block(s);
    auto p = TR ? L + (j * TILE + ((int64_t)i * TILE + 16 * cg) * ld)
                : L + ((int64_t)i * TILE + (j * TILE + 16 * cg) * ld);
    p += lg * NC * ld;
#pragma unroll
    for (int c = 0; c < NC; ++c, p += ld)
      v[c] = *(const __attribute__((address_space(1))) vec_t*)(p + VEC * lr);
  };
#pragma unroll
  for (int u = 0; u < DEPTH; ++u)
    if (u < ntile) load(st[u], u);
  // forward: sums of the lane's VEC rows; transposed: of its NC columns
  constexpr int NA = TR ? NC : VEC;
  double acc[NA];
#pragma unroll
  for (int c = 0; c < NA; ++c) acc[c] = 0.0;
  auto consume = [&](const vec_t (&v)[NC], const double* x) {
    if constexpr (TR) {
      double xe[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) xe[e] = x[VEC * lr + e];
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[c] = fma((double)v[c][e], xe[e], acc[c]);
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const double xc = x[16 * cg + NC * lg + c];
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] = fma((double)v[c][e], xc, acc[e]);
      }
    }
  };
  // x_r = DINV_r v_r (transposed: DINV_r^T): wave cg of block row r forms rows
  // 16 cg + (l & 15), a lane 16 of the 64 terms (from 16 (l >> 4)).  DINV_r is
  // fetched ahead of the stream: into registers, or (FP64, whose tiles take
  // them) into LDS
  const unsigned xr = 16 * cg + (l & 15), kq = 16 * (l >> 4);
  double dv[DL ? 1 : 16];
  if (act) {
    const auto D = dinv + (size_t)i * TILE * TILE;
    if constexpr (DL) {
      double t[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) t[k] = D[(16 * cg + k) * TILE + l];
#pragma unroll
      for (int k = 0; k < 16; ++k) dl[rb][16 * cg + k][l] = t[k];
    } else {
#pragma unroll
      for (int k = 0; k < 16; ++k) dv[k] = TR ? D[TILE * xr + kq + k] : D[(kq + k) * TILE + xr];
    }
  }
  // DINV_r(xr, kq + k), transposed DINV_r(kq + k, xr)
  auto dval = [&](int k) {
    if constexpr (DL)
      return TR ? dl[rb][xr][kq + k] : dl[rb][kq + k][xr];
    else
      return dv[k];
  };
  const double b = bv[(size_t)i * TILE + l];
  uint64_t wa = 0, wb = 0;  // the polling wave's next words
  auto peek = [&](int s) {
    const uint64_t* p = pub + 2 * ((size_t)block(s) * TILE + l);
    wa = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    wb = __hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (w == 0 && b0 > 0) peek(0);
  auto stream = [&](int s, vec_t (&v)[NC]) {
    asm volatile("" : "+s"(ld));  // column addresses are formed where they are used
    if (w == 0) {
      for (int spins = 0;; ++spins) {
        const bool ok = (uint32_t)(wa >> 32) == epoch && (uint32_t)(wb >> 32) == epoch;
        if (__builtin_amdgcn_ballot_w64(!ok) == 0) break;
        if (spins >= SPIN_LIMIT) {
          if (l == 0) atomicOr(info, PGP_INFO_STALLED);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
        peek(s);
      }
      xs[s & 1][l] = __longlong_as_double((long long)((wb << 32) | (wa & 0xffffffffu)));
      if (s + 1 < b0) peek(s + 1);
    }
    __syncthreads();
    if (act) {
      consume(v, xs[s & 1]);
      if (s + DEPTH < ntile) load(v, s + DEPTH);
    }
  };
  for (int s = 0; s < b0; s += DEPTH) {  // b0 is a multiple of DEPTH
    stream(s, st[0]);
    stream(s + 1, st[1]);
  }
#pragma unroll
  for (int r = 0; r < SEG; ++r) {
    if (r >= nblk) break;
    if (rb == r) {
      if constexpr (TR) {
        // column sums over the lane's row lanes by a transposing butterfly:
        // row lane lr ends with column (lr / (RL / NC)) of the NC
        double v[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) v[c] = acc[c];
#pragma unroll
        for (int h = NC / 2, bit = RL / 2; h >= 1; h >>= 1, bit >>= 1) {
          const bool up = (l & bit) != 0;
#pragma unroll
          for (int q = 0; q < h; ++q) {
            const double give = up ? v[q] : v[q + h];
            const double keep = up ? v[q + h] : v[q];
            v[q] = keep + __shfl_xor(give, bit);
          }
        }
        double cs = v[0];
#pragma unroll
        for (int bit = RL / NC / 2; bit >= 1; bit >>= 1) cs += __shfl_xor(cs, bit);
        if (lr % (RL / NC) == 0) part[0][16 * cg + NC * lg + lr / (RL / NC)] = cs;
      } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) part[CG * cg + lg][VEC * lr + e] = acc[e];
      }
    }
    __syncthreads();
    if (rb == r) {
      double sum = 0.0;
      if constexpr (TR) {
        sum = part[0][l];
      } else {
#pragma unroll
        for (int g = 0; g < 4 * CG; ++g) sum += part[g][l];
      }
      vs[cg][l] = b - sum;  // read back by this wave only
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      double a0 = 0.0, a1 = 0.0;
#pragma unroll
      for (int k = 0; k < 16; k += 2) {
        a0 = fma(dval(k), vs[cg][kq + k], a0);
        a1 = fma(dval(k + 1), vs[cg][kq + k + 1], a1);
      }
      double x = a0 + a1;
      x += __shfl_xor(x, 16);
      x += __shfl_xor(x, 32);
      if (l < 16) {
        xq[r & 1][xr] = x;
        const uint64_t u = (uint64_t)__double_as_longlong(x), tag = (uint64_t)epoch << 32;
        uint64_t* p = pub + 2 * ((size_t)i * TILE + xr);
        __hip_atomic_store(p, tag | (u & 0xffffffffu), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(p + 1, tag | (u >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        xv[(size_t)i * TILE + xr] = x;
      }
    }
    if (r + 1 >= nblk) break;
    __syncthreads();
    if (act && rb > r) {
      consume(st[r % DEPTH], xq[r & 1]);
      if (r + DEPTH < rb) load(st[r % DEPTH], b0 + r + DEPTH);
    }
  }
}

static bool wavefront_trsv() {
  static const bool v = [] {
    const char* e = getenv("PGP_TRSV_WAVEFRONT");
    return !(e && e[0] == '0');
  }();
  return v;
}

uint32_t next_epoch() {
  static std::atomic<uint32_t> g{0};
  uint32_t e = ++g;
  if (e == 0) e = ++g;
  return e;
}

void launch_trsv(const Batch& bt, int prec, int trans, int in, int out, hipStream_t s) {
  const int nseg = (bt.maxNp / TILE + SEG - 1) / SEG;
  if (bt.ticket && wavefront_trsv() && nseg <= MAXB) {
    // segment-major schedule: segment t holds the members with more than t
    // segments (a prefix: members are sorted by size), one workgroup each
    Sched rows;
    rows.count = nseg;
    int tot = 0;
    for (int st = 0; st < nseg; ++st) {
      rows.pre[st] = tot;
      for (int m = 0; m < bt.count; ++m)
        if (bt.np(m) / TILE > SEG * st) ++tot;
    }
    rows.pre[nseg] = tot;
    if (tot == 0) return;
    const bool on = timer_on(TC_TRSV);
    const double esz = prec == PGP_PREC_FP64 ? 8.0 : 4.0;
    // algorithmic work: Np^2 flops; bytes: the lower triangle of L and the
    // diagonal-block inverses, read once
    double fl = 0.0, by = 0.0;
    if (on) {
      for (int m = 0; m < bt.count; ++m) {
        const double np = bt.np(m);
        fl += np * np;
        by += 0.5 * np * (np + TILE) * esz + np * TILE * 8.0;
      }
      timer_begin(TC_TRSV, s);
    }
    const uint32_t ep = next_epoch();
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(tot), dim3(SEG_THREADS), 0, s, bt.dprobs, rows, bt.ticket,
                         ep, in, out);
    };
    if (prec == PGP_PREC_FP64)
      trans ? go(k_trsv_seg<double, true>) : go(k_trsv_seg<double, false>);
    else
      trans ? go(k_trsv_seg<float, true>) : go(k_trsv_seg<float, false>);
    if (on) timer_end(TC_TRSV, s, fl, by);
    return;
  }
  const int nb = bt.maxNp / TILE;
  for (int step = 0; step < nb; ++step) {
    const int k = trans ? nb - 1 - step : step;
    sched_launch(
        bt,
        [&](int m) {
          const int nbm = bt.np(m) / TILE;
          return k < nbm ? (trans ? k + 1 : nbm - k) : 0;
        },
        [&](Prob* const* dp, const Sched& sc, int n) {
          if (prec == PGP_PREC_FP64)
            hipLaunchKernelGGL(k_trsv<double>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, k, trans, in,
                               out);
          else
            hipLaunchKernelGGL(k_trsv<float>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, k, trans, in,
                               out);
        });
  }
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_trsv_raw(const T* L, int64_t N, int64_t ld,
                                                       const double* dinv, int k, int trans,
                                                       double* b, double* x) {
  if (!trans)
    trsv_fwd_step<T>(L, ld, N, dinv, k, b, x, blockIdx.x);
  else
    trsv_bwd_step<T>(L, ld, dinv, k, b, x, blockIdx.x);
}

int launch_trsv_raw_dinv(int prec, const void* L, int64_t N, int64_t ld, const double* dinv,
                         double* b, double* x, int trans, hipStream_t s) {
  const int nb = (int)(N / TILE);
  for (int step = 0; step < nb; ++step) {
    const int k = trans ? nb - 1 - step : step;
    dim3 g(trans ? k + 1 : nb - k);
    if (prec == PGP_PREC_FP64)
      hipLaunchKernelGGL(k_trsv_raw<double>, g, dim3(NTHREADS), 0, s, (const double*)L, N, ld,
                         dinv, k, trans, b, x);
    else
      hipLaunchKernelGGL(k_trsv_raw<float>, g, dim3(NTHREADS), 0, s, (const float*)L, N, ld, dinv,
                         k, trans, b, x);
  }
  return 0;
}

// ---- TRSM: S <- L^-1 S, S is Np x Mp (ld lds) ----
// With a ticket counter and up to ROWS_MAX block rows a solve is one wavefront
// launch (k_trsm_rows, below) with the roundings of the schedule its width would
// take without: a launch per block row (up to TRSM_WIDE column tiles) or per
// super-step of G block rows, which subtract each block row's (super-step's)
// product from S.
//
// Per block row (lagged).
// Lagged schedule.  Launch k, workgroup (w, ct), row block i = k + w:
//   S_i[:, ct] -= L_{i,k-1} X_{k-1}[:, ct]   (k >= 1; X_{k-1} = S_{k-1}, final
//                                            since launch k - 1)
//   w == 0 then finishes block k: S_k[:, ct] = DINV_k S_k[:, ct].
// Every workgroup writes only its own rows and reads only rows finished in
// earlier launches, so workgroups of one launch never race, whatever order
// they run in.  Launch 0 holds only the w == 0 workgroups.
template <typename T>
__device__ __forceinline__ void trsm_step(const T* L, int64_t ld, const double* dinv, int k, T* S, int64_t lds,
                          int w, int ct) {
  constexpr int PP = KP<T>::value;  // A operand: conflict-free MFMA reads
  constexpr int PB = TILE + 1;       // B operand: written transposed, conflict-free stores
  __shared__ T As[TILE * PP];
  __shared__ T Bs[TILE * PB];
  typedef typename Acc<T>::type acc_t;
  const int64_t r0 = (int64_t)(k + w) * TILE;
  const int64_t n0 = (int64_t)ct * TILE;
  acc_t acc[2][2];
  zero_acc<T>(acc);
  if (k > 0) {
    const int64_t cp = (int64_t)(k - 1) * TILE;
    // A = L(r0.., cp..) (k-major), B[kk][n] = S(cp + kk, n0 + n)
    load_block_kmajor<T, T>(As, PP, L, ld, r0, cp);
    {
      const int r = threadIdx.x & 63, cb = threadIdx.x >> 6;
#pragma unroll 4
      for (int q = 0; q < 16; ++q) {
        const int c = cb + 4 * q;
        Bs[r * PB + c] = S[(size_t)(cp + r) + (size_t)(n0 + c) * lds];
      }
    }
    __syncthreads();
    mma64_kmajor<T>(As, PP, Bs, PB, acc);
    __syncthreads();
  }
  if (w > 0) {
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
      for (int bn = 0; bn < 2; ++bn)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          T* p = &S[(size_t)(r0 + acc_row<T>(bm, r)) + (size_t)(n0 + acc_col(bn)) * lds];
          *p = *p - acc[bm][bn][r];
        }
    return;
  }
  // block k: S_k - update (rounded to T) as the k-major B operand, DINV_k as A
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = acc_row<T>(bm, r), col = acc_col(bn);
        Bs[row * PB + col] =
            S[(size_t)(r0 + row) + (size_t)(n0 + col) * lds] - acc[bm][bn][r];
      }
  load_block_kmajor<double, T>(As, PP, dinv + (size_t)k * TILE * TILE, TILE, 0, 0);
  __syncthreads();
  zero_acc<T>(acc);
  mma64_kmajor<T>(As, PP, Bs, PB, acc);
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[(size_t)(r0 + acc_row<T>(bm, r)) + (size_t)(n0 + acc_col(bn)) * lds] = acc[bm][bn][r];
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_trsm_lagged(Prob* const* probs, Sched sc, int k) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int nb = P.Np / TILE;
  if (k >= nb) return;
  const int rows = k == 0 ? 1 : nb - k;  // row blocks of this launch
  const int w = bx % rows, ct = bx / rows;
  if (ct >= P.Mp / TILE) return;
  trsm_step<T>(uniform((const T*)P.L), uniform(P.Np), uniform(P.dinv), k, uniform((T*)P.S),
               uniform(P.Np), uniform(w), uniform(ct));
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_trsm_lagged_raw(const T* L, int64_t ld,
                                                              const double* dinv, int k, T* S,
                                                              int64_t lds) {
  trsm_step<T>(L, ld, dinv, k, S, lds, blockIdx.x, blockIdx.y);
}

// Workgroup tk of a wide solve's launch: block row (in sweep order), member,
// column tile of the launch.
__device__ __forceinline__ void solve_unit(const SolveSched& ss, int tk, int& row, int& m,
                                           int& ct) {
  auto find = [](const int32_t* pre, int n, int v) {  // the last i < n with pre[i] <= v
    int lo = 0, hi = n;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (pre[mid] <= v)
        lo = mid;
      else
        hi = mid;
    }
    return lo;
  };
  const int r = find(ss.rows, ss.count, tk), local = tk - ss.rows[r];
  row = ss.row0 + r;
  if (ss.nct > 0) {
    m = uniform(local / ss.nct);
    ct = local - m * ss.nct;
  } else {
    m = find(ss.tiles, ss.members, local);
    ct = local - ss.tiles[m];
  }
}

// The launches of a wide solve (at most maxMp / 64 column tiles a member):
// per PROGRESS_CT column tiles, per schedule's members and block rows, each
// member with its own column tiles (256 requests of 700 to 1024 points, one
// with 5000 test points and the others with 64, a step of a stream: 14.3 ms in
// FP32 and 11.9 in FP64 with the widest member's tiles listed for every member,
// now 8.1 and 9.0).
// go(dprobs, schedule, first column tile, workgroups, epoch).
template <class Go>
static void solve_launches(const Batch& bt, int maxMp, hipStream_t s, Go go) {
  auto mt_of = [&](int m) { return bt.hm ? (bt.hm[m] + TILE - 1) / TILE : maxMp / TILE; };
  const bool on = timer_on(TC_TRSM);
  for (int ct0 = 0; ct0 < maxMp / TILE; ct0 += PROGRESS_CT) {
    for (int m0 = 0, n = 0; m0 < bt.count; m0 += n) {
      auto nct_of = [&](int m) {
        return std::min(PROGRESS_CT, std::max(0, mt_of(m0 + m) - ct0));
      };
      auto nb_of = [&](int m) { return bt.np(m0 + m) / TILE; };
      SolveSched ss;
      n = fill_tiles(ss, bt.count - m0, nct_of);
      double fl = 0.0;
      if (on) {
        for (int m = 0; m < n; ++m) {
          const double np = bt.np(m0 + m);
          fl += np * np * TILE * nct_of(m);
        }
        timer_begin(TC_TRSM, s);
      }
      for (int row0 = 0; row0 < nb_of(0); row0 += ROWS_MAX) {
        const int tot = fill_rows(ss, row0, nb_of);
        if (tot > 0) go(bt.dprobs + m0, ss, ct0, tot, next_epoch());
      }
      if (on) timer_end(TC_TRSM, s, fl, 0.0);
    }
  }
}

// Wavefront TRSM for the column tiles [ct0, ct0 + nct) (nct <= PROGRESS_CT),
// all members in one launch: one workgroup per (block row i, member, column
// tile ct), numbered row-major so that the wave front moves through every
// member and column tile at once.  Workgroup (i, ct) accumulates L_ij X_j[:,
// ct] for every block j < i as soon as (j, ct) publishes, then forms X_i =
// DINV_i (S_i - acc) and publishes it: X_i through agent-scope stores, a wait
// for their completion, then the member's progress word of column tile ct.
// S is read and written once.  Start-order tickets and bounded waits as in
// k_trsv_seg.
//
// Bound by the tile products once a row's work (nct products per earlier
// block, over 256 CUs) exceeds the chain's step (the last product, DINV's and
// the hand-off, ~9 us); FP64 at N = 3000, M = 5000: 2400 us as 12 super-step
// launches, whose solving workgroups run 30 tile products in a row; 1712 in
// one wavefront launch; 1207 (38 TFLOP/s) with the operands fetched a product
// ahead; 1110 (41) with DINV's zeros left out and X_i stored by whole columns
// (256 test points, FP32, a stream of fits: 68.5 -> 65.8 ms); 1061 (43) with
// the sums taken off in groups and so S_i fetched first.  N = 1537, M = 501: 590
// -> 269 -> 181 us.  Transposed, FP32 at N = 8192, M = 4096: 20.3 ms in 16
// launches of 4 column tiles, 2.8 ms (98 TFLOP/s) in one.
//
// GRP: the sum is taken off S_i, in its type, after every 1 << lg blocks but
// the last whole group before i's own: the roundings of the schedules of one
// launch per block row (lg = 0) or super-step of TRSM_G (lg = 2), which solves
// of more than WAVE_NCT column tiles follow without a ticket counter.  A row's
// whole sum taken off at once is less accurate (FP64, N = 3000, M = 5000:
// 2.6e-13 from 64-bit references, grouped 1.1e-13).
// lg goes by the member's own column tiles (up to WAVE_NCT: no group is ever
// whole), so that its results do not depend on the rest of the batch.
constexpr int WAVE_NCT = 4;
// Right-hand sides of at least this many column tiles take the super-step
// schedule.
constexpr int TRSM_WIDE = 16;

template <typename T, bool GRP>
__global__ __launch_bounds__(NTHREADS, sizeof(T) == 8 ? 2 : 3) void k_trsm_rows(
    Prob* const* probs, SolveSched ss, int ct0, uint32_t* ticket, uint32_t epoch) {
  constexpr int PP = KP<T>::value;  // A operand: conflict-free MFMA reads
  constexpr int PB = TILE + 1;       // B operand: written transposed, conflict-free stores
  __shared__ T As[TILE * PP];
  __shared__ T Bs[TILE * PB];
  __shared__ int s_val;
  typedef typename Acc<T>::type acc_t;
  const int tk = take_ticket(ticket, &s_val);
  if ((unsigned)tk >= gridDim.x) {  // counter not zero at launch: no block to take
    flag_members_stalled(probs, ss.members);
    return;
  }
  int i, m, lct;
  solve_unit(ss, uniform(tk), i, m, lct);
  const int ct = ct0 + lct;
  const Prob& P = *probs[m];
  const int mt = uniform(P.Mp) / TILE;
  if (ct >= mt || i >= P.Np / TILE) return;
  const int lg = mt <= WAVE_NCT ? 30 : mt < TRSM_WIDE ? 0 : 2;
  uint64_t* prog = P.progress_ct + lct;
  const auto L = gbl(uniform((const T*)P.L));
  const auto S = gbl(uniform((T*)P.S));
  const int64_t ld = uniform(P.Np);
  const int64_t ri = (int64_t)i * TILE, n0 = (int64_t)ct * TILE;
  const unsigned r = threadIdx.x & 63;
  const int cb = uniform((int)(threadIdx.x >> 6));
  // la: the next A operand (L_ij, at last DINV_i), fetched during the
  // product before its own; xb: the next X_j, fetched as early when it is
  // known to be published, and (sv) during the last product S_i.
  T la[16], xb[16], si[GRP ? 16 : 1];
  T(&sv)[16] = [&]() -> T(&)[16] {
    if constexpr (GRP)
      return si;
    else
      return xb;
  }();
  auto fetch_l = [&](int k) {
    auto p = L + (ri + ((int64_t)k * TILE + cb) * ld);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += 4 * ld) la[q] = p[r];
  };
  auto fetch_d = [&]() {
    const auto D = gbl(uniform(P.dinv)) + ((size_t)i * TILE * TILE + (size_t)cb * TILE);
#pragma unroll
    for (int q = 0; q < 16; ++q) la[q] = (T)D[r + (size_t)(4 * q) * TILE];
  };
  auto fetch_s = [&](T (&v)[16]) {  // accumulator layout
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
      for (int bn = 0; bn < 2; ++bn)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[8 * bm + 4 * bn + q] =
              S[(size_t)(ri + acc_row<T>(bm, q)) + (size_t)(n0 + acc_col(bn)) * ld];
  };
  auto fetch_x = [&](int k) {  // published in this launch: coherent loads
    auto p = S + ((int64_t)k * TILE + (n0 + cb) * ld);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += 4 * ld)
      xb[q] = __hip_atomic_load(p + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if constexpr (GRP) fetch_s(sv);
  if (i > 0) {
    fetch_l(0);
  } else {
    fetch_d();
    if constexpr (!GRP) fetch_s(sv);
  }
  acc_t acc[2][2];
  zero_acc<T>(acc);
  int done = 0, ready = 0;
  while (done < i) {
    if (done >= ready) {
      __syncthreads();  // everyone has read the previous s_val
      if (threadIdx.x == 0) s_val = wait_progress(prog, epoch, done + 1, P.info);
      __syncthreads();
      ready = min(__builtin_amdgcn_readfirstlane(s_val), i);
      fetch_x(done);
    }
    __syncthreads();  // the previous product is done with LDS
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      As[(cb + 4 * q) * PP + r] = la[q];
      Bs[r * PB + cb + 4 * q] = xb[q];  // B(k, n) = X_j(k, n)
    }
    ++done;
    if (done < i) {
      fetch_l(done);
      if (done < ready) fetch_x(done);
    } else {
      fetch_d();
      if constexpr (!GRP) fetch_s(sv);
    }
    __syncthreads();
    mma64_kmajor<T>(As, PP, Bs, PB, acc);
    if constexpr (GRP) {
      if ((done & ((1 << lg) - 1)) == 0 && (done >> lg) < (i >> lg)) {
#pragma unroll
        for (int bm = 0; bm < 2; ++bm)
#pragma unroll
          for (int bn = 0; bn < 2; ++bn)
#pragma unroll
            for (int q = 0; q < 4; ++q) sv[8 * bm + 4 * bn + q] -= acc[bm][bn][q];
        zero_acc<T>(acc);
      }
    }
  }
  // X_i = DINV_i (S_i - acc)
  __syncthreads();
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = acc_row<T>(bm, q), col = acc_col(bn);
        Bs[row * PB + col] = sv[8 * bm + 4 * bn + q] - acc[bm][bn][q];
      }
#pragma unroll
  for (int q = 0; q < 16; ++q) As[(cb + 4 * q) * PP + r] = la[q];
  __syncthreads();
  acc_t prod[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int q = 0; q < 4; ++q) prod[b][q] = (T)0;
  mma64_tri<T, true, false>(As, PP, Bs, PB, prod);
  __syncthreads();
  // X_i through LDS: whole columns per store
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      Bs[(16 * cb + (r & 15)) * PB + 16 * b + acc_row<T>(0, q) - 32 * (cb >> 1)] = prod[b][q];
  __syncthreads();
  {
    auto p = S + (ri + (n0 + cb) * ld);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += 4 * ld)
      __hip_atomic_store(p + r, Bs[(cb + 4 * q) * PB + r], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  publish_wait();  // every wave's X_i stores complete ...
  __syncthreads();
  if (threadIdx.x == 0)  // ... before (i + 1, ct) may read them
    __hip_atomic_store(prog, ((uint64_t)epoch << 32) | (uint64_t)(i + 1), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// Transposed wavefront TRSM: X <- L^-T X in place on the predict buffer S,
// for the column tiles [ct0, ct0 + nct) (nct <= PROGRESS_CT), all members in
// one launch.  Step t of a member is its block row i = nb - 1 - t (the sweep
// runs from the last block row up): workgroup (t, member, ct) accumulates
// L_ji^T X_j[:, ct] for every j > i as soon as step nb - 1 - j publishes,
// then forms X_i = DINV_i^T (X_i - acc) and publishes step t.  Operands as in
// k_trsm_rows with both L_ji and DINV_i transposed on their way into LDS
// (rows of the stored tile are the k index, read coalesced along k).
template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_trsm_rows_t(Prob* const* probs, SolveSched ss,
                                                          int ct0, uint32_t* ticket,
                                                          uint32_t epoch) {
  constexpr int PA = TILE + 1;  // A operand, written row by row
  constexpr int PB = TILE + 1;  // B operand, written transposed
  __shared__ T As[TILE * PA];
  __shared__ T Bs[TILE * PB];
  __shared__ int s_val;
  typedef typename Acc<T>::type acc_t;
  const int tk = take_ticket(ticket, &s_val);
  if ((unsigned)tk >= gridDim.x) {  // counter not zero at launch: no block to take
    flag_members_stalled(probs, ss.members);
    return;
  }
  int t, m, lct;
  solve_unit(ss, uniform(tk), t, m, lct);
  const Prob& P = *probs[m];
  const int nb = uniform(P.Np) / TILE, ct = ct0 + lct;
  if (ct >= P.Mp / TILE || t >= nb) return;
  const int i = nb - 1 - t;
  uint64_t* prog = P.progress_ct + lct;
  const auto L = gbl(uniform((const T*)P.L));
  const auto S = gbl(uniform((T*)P.S));
  const int64_t ld = uniform(P.Np);
  const int64_t ri = (int64_t)i * TILE, n0 = (int64_t)ct * TILE;
  const unsigned r = threadIdx.x & 63;
  const int cb = uniform((int)(threadIdx.x >> 6));
  // la: the next A operand (L_ji, at last DINV_i), fetched during the
  // product before its own; xb: the next X_j, fetched as early when it is
  // known to be published, and during the last product S_i.
  T la[16], xb[16];
  // fetch_l(k): la[q] = L_ji(r, cb + 4q), j = nb - 1 - k: A(m, k) = L_ji(k, m)
  auto fetch_l = [&](int k) {
    auto p = L + ((int64_t)(nb - 1 - k) * TILE + (ri + cb) * ld);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += 4 * ld) la[q] = p[r];
  };
  auto fetch_d = [&]() {
    const auto D = gbl(uniform(P.dinv)) + ((size_t)i * TILE * TILE + (size_t)cb * TILE);
#pragma unroll
    for (int q = 0; q < 16; ++q) la[q] = (T)D[r + (size_t)(4 * q) * TILE];
  };
  auto fetch_s = [&]() {  // accumulator layout
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
      for (int bn = 0; bn < 2; ++bn)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          xb[8 * bm + 4 * bn + q] =
              S[(size_t)(ri + acc_row<T>(bm, q)) + (size_t)(n0 + acc_col(bn)) * ld];
  };
  auto fetch_x = [&](int k) {  // published in this launch: coherent loads
    auto p = S + ((int64_t)(nb - 1 - k) * TILE + (n0 + cb) * ld);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += 4 * ld)
      xb[q] = __hip_atomic_load(p + r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (t > 0) {
    fetch_l(0);
  } else {
    fetch_d();
    fetch_s();
  }
  acc_t acc[2][2];
  zero_acc<T>(acc);
  int done = 0, ready = min(ss.row0, t);  // steps known to be published
  if (ready > 0) fetch_x(0);
  while (done < t) {
    if (done >= ready) {
      __syncthreads();  // everyone has read the previous s_val
      if (threadIdx.x == 0) s_val = wait_progress(prog, epoch, done + 1, P.info);
      __syncthreads();
      ready = min(__builtin_amdgcn_readfirstlane(s_val), t);
      fetch_x(done);
    }
    __syncthreads();  // the previous product is done with LDS
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      As[r * PA + cb + 4 * q] = la[q];
      Bs[r * PB + cb + 4 * q] = xb[q];  // B(k, n) = X_j(k, n)
    }
    ++done;
    if (done < t) {
      fetch_l(done);
      if (done < ready) fetch_x(done);
    } else {
      fetch_d();
      fetch_s();
    }
    __syncthreads();
    mma64_kmajor<T>(As, PA, Bs, PB, acc);
  }
  // X_i = DINV_i^T (X_i - acc)
  __syncthreads();
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = acc_row<T>(bm, q), col = acc_col(bn);
        Bs[row * PB + col] = xb[8 * bm + 4 * bn + q] - acc[bm][bn][q];
      }
#pragma unroll
  for (int q = 0; q < 16; ++q) As[r * PA + cb + 4 * q] = la[q];  // A(m, k) = DINV_i(k, m)
  __syncthreads();
  acc_t prod[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int q = 0; q < 4; ++q) prod[b][q] = (T)0;
  mma64_tri<T, true, true>(As, PA, Bs, PB, prod);
  __syncthreads();
  // X_i through LDS: whole columns per store
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      Bs[(16 * cb + (r & 15)) * PB + 16 * b + acc_row<T>(0, q) - 32 * (cb >> 1)] = prod[b][q];
  __syncthreads();
  {
    auto p = S + (ri + (n0 + cb) * ld);
#pragma unroll
    for (int q = 0; q < 16; ++q, p += 4 * ld)
      __hip_atomic_store(p + r, Bs[(cb + 4 * q) * PB + r], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  publish_wait();  // every wave's X_i stores complete ...
  __syncthreads();
  if (threadIdx.x == 0)  // ... before step t + 1 may read them
    __hip_atomic_store(prog, ((uint64_t)epoch << 32) | (uint64_t)(t + 1), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// S <- L^-T S for every member's Mp right-hand sides (Mp <= maxMp).
void launch_trsm_t(const Batch& bt, int prec, int maxMp, hipStream_t s) {
  solve_launches(bt, maxMp, s, [&](Prob* const* dp, const SolveSched& ss, int ct0, int tot,
                                   uint32_t ep) {
    if (prec == PGP_PREC_FP64)
      hipLaunchKernelGGL(k_trsm_rows_t<double>, dim3(tot), dim3(NTHREADS), 0, s, dp, ss, ct0,
                         bt.ticket, ep);
    else
      hipLaunchKernelGGL(k_trsm_rows_t<float>, dim3(tot), dim3(NTHREADS), 0, s, dp, ss, ct0,
                         bt.ticket, ep);
  });
}

static bool wavefront_trsm() {
  static const bool v = [] {
    const char* e = getenv("PGP_TRSM_WAVEFRONT");
    return !(e && e[0] == '0');
  }();
  return v;
}

// Super-steps of G block rows.
// One launch per super-step q of block rows SS_q = [Gq, Gq + G), with
// P = SS_{q-1} the super-step finished by the previous launch:
//   solve workgroup (column tile ct), for k in SS_q in order:
//     X_k = DINV_k (S_k - sum_{c in [G(q-1), k)} L_kc X_c)   (left-looking)
//   update workgroups (row block i >= G(q+1), column tile ct):
//     S_i -= sum_{c in P} L_ic X_c                          (rank 64 G)
// so every later row block receives each finished super-step in one
// rank-64G product: S is read and written once per super-step, not once per
// block row.  A workgroup writes only its own rows and reads rows finished
// in earlier launches (or by itself), so workgroups of one launch never
// race.
constexpr int TRSM_G = 4;

// acc += sum_{c in [c0, c1)} L(r0.., 64c..) S(64c.., n0..): MFMA tile
// products with the next chunk fetched into registers during the current.
// Rows of S from block c_fresh on were written by this workgroup in this
// launch: they are read with coherent loads (past the CU's L1, which may
// still hold the values they replaced).
template <typename T>
__device__ __forceinline__ void trsm_acc(const T* L, int64_t ld, const T* S, int64_t lds, int64_t r0, int64_t n0,
                         int c0, int c1, int c_fresh, T* As, T* Bs,
                         typename Acc<T>::type (&acc)[2][2]) {
  constexpr int PP = KP<T>::value;  // A operand: conflict-free MFMA reads
  constexpr int PB = TILE + 1;       // B operand: written transposed, conflict-free stores
  if (c0 >= c1) return;
  const unsigned m = threadIdx.x & 63;
  const int kb = uniform((int)(threadIdx.x >> 6));
  T ra[16], rb[16];
  auto fetch = [&](int c) {
    const int64_t cc = (int64_t)c * TILE;
    auto pa = gbl(L) + (r0 + (cc + kb) * ld);  // A(m, k)
    auto pb = gbl(S) + (cc + (n0 + kb) * lds);  // B(m, k): row m, column k
#pragma unroll
    for (int q = 0; q < 16; ++q, pa += 4 * ld) ra[q] = pa[m];
    if (c >= c_fresh) {
#pragma unroll
      for (int q = 0; q < 16; ++q, pb += 4 * lds)
        rb[q] = __hip_atomic_load(pb + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
#pragma unroll
      for (int q = 0; q < 16; ++q, pb += 4 * lds) rb[q] = pb[m];
    }
  };
  fetch(c0);
  for (int c = c0; c < c1; ++c) {
    if (c > c0) __syncthreads();  // the previous chunk's products are done with LDS
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int k = kb + 4 * q;
      As[k * PP + m] = ra[q];
      Bs[m * PB + k] = rb[q];
    }
    __syncthreads();
    if (c + 1 < c1) fetch(c + 1);
    mma64_kmajor<T>(As, PP, Bs, PB, acc);
  }
  __syncthreads();  // LDS free for the caller
}

// Workgroup `u` of launch q for one right-hand side of nct column tiles:
// u < nct solves SS_q for column tile u; the others update one row block.
template <typename T>
__device__ __forceinline__ void trsm_ss(const T* L, int64_t ld, const double* dinv, int nb, int q, T* S,
                        int64_t lds, int nct, int u) {
  constexpr int PP = KP<T>::value;
  constexpr int PB = TILE + 1;
  __shared__ T As[TILE * PP];
  __shared__ T Bs[TILE * PB];
  typedef typename Acc<T>::type acc_t;
  constexpr int G = TRSM_G;
  u = uniform(u);
  const int p0 = q > 0 ? G * (q - 1) : 0;  // first column of P (or of SS_0)
  acc_t acc[2][2];
  if (u < nct) {
    const int ct = u;
    const int64_t n0 = (int64_t)ct * TILE;
    const int kend = min(G * q + G, nb);
    for (int k = G * q; k < kend; ++k) {
      const int64_t r0 = (int64_t)k * TILE;
      zero_acc<T>(acc);
      trsm_acc<T>(L, ld, S, lds, r0, n0, p0, k, G * q, As, Bs, acc);
      // B = S_k - acc (rounded to T), A = DINV_k
#pragma unroll
      for (int bm = 0; bm < 2; ++bm)
#pragma unroll
        for (int bn = 0; bn < 2; ++bn)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = acc_row<T>(bm, r), col = acc_col(bn);
            Bs[row * PB + col] =
                S[(size_t)(r0 + row) + (size_t)(n0 + col) * lds] - acc[bm][bn][r];
          }
      load_block_kmajor<double, T>(As, PP, dinv + (size_t)k * TILE * TILE, TILE, 0, 0);
      __syncthreads();
      zero_acc<T>(acc);
      mma64_kmajor<T>(As, PP, Bs, PB, acc);
#pragma unroll
      for (int bm = 0; bm < 2; ++bm)
#pragma unroll
        for (int bn = 0; bn < 2; ++bn)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            S[(size_t)(r0 + acc_row<T>(bm, r)) + (size_t)(n0 + acc_col(bn)) * lds] =
                acc[bm][bn][r];
      publish_wait();   // X_k reaches L2 ...
      __syncthreads();  // ... before the next row of this super-step reads it back
    }
    return;
  }
  // update of row block i >= G(q+1) by P = [G(q-1), Gq)
  const int v = u - nct;
  const int ct = uniform(v % nct);
  const int i = uniform(G * (q + 1) + v / nct);
  if (q == 0 || i >= nb) return;
  const int64_t r0 = (int64_t)i * TILE, n0 = (int64_t)ct * TILE;
  zero_acc<T>(acc);
  trsm_acc<T>(L, ld, S, lds, r0, n0, p0, G * q, G * q, As, Bs, acc);
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        T* p = &S[(size_t)(r0 + acc_row<T>(bm, r)) + (size_t)(n0 + acc_col(bn)) * lds];
        *p = *p - acc[bm][bn][r];
      }
}

// workgroups of launch q: nct solvers plus nct per row block below SS_q
static inline int trsm_units(int nb, int q, int nct) {
  const int rows = q > 0 ? std::max(0, nb - TRSM_G * (q + 1)) : 0;
  return nb > TRSM_G * q ? nct * (1 + rows) : 0;
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_trsm(Prob* const* probs, Sched sc, int q) {
  int bx;
  const Prob& P = *probs[sched_member(sc, blockIdx.x, bx)];
  const int np = uniform(P.Np);
  trsm_ss<T>(uniform((const T*)P.L), np, uniform(P.dinv), np / TILE, q, uniform((T*)P.S), np,
             uniform(P.Mp) / TILE, bx);
}

static void launch_trsm_lagged(const Batch& bt, int prec, int maxMp, hipStream_t s) {
  const int nb = bt.maxNp / TILE;
  const bool on = timer_on(TC_TRSM);
  for (int k = 0; k < nb; ++k) {
    auto nct_of = [&](int m) {
      const int mp = bt.hm ? (bt.hm[m] + TILE - 1) / TILE * TILE : maxMp;
      return mp / TILE;
    };
    sched_launch(
        bt,
        [&](int m) {
          const int nbm = bt.np(m) / TILE;
          return k < nbm ? (k == 0 ? 1 : nbm - k) * nct_of(m) : 0;
        },
        [&](Prob* const* dp, const Sched& sc, int n) {
          if (on) timer_begin(TC_TRSM, s);
          if (prec == PGP_PREC_FP64)
            hipLaunchKernelGGL(k_trsm_lagged<double>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, k);
          else
            hipLaunchKernelGGL(k_trsm_lagged<float>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, k);
          if (on) {
            // step k of an N^2 M-flop solve: the update of rows k.. by block
            // k - 1 (2 * 64 per entry) and the 64-row triangle (64^2 per column)
            double fl = 0.0;
            const int off = (int)(dp - bt.dprobs);
            for (int m = off; m < off + sc.count; ++m) {
              const int nbm = bt.np(m) / TILE;
              if (k >= nbm) continue;
              const double cols = (double)nct_of(m) * TILE;
              fl += cols * (TILE * TILE + (k > 0 ? 2.0 * TILE * TILE * (nbm - k) : 0.0));
            }
            timer_end(TC_TRSM, s, fl, 0.0);
          }
        });
  }
}

void launch_trsm(const Batch& bt, int prec, int maxMp, hipStream_t s) {
  if (bt.ticket && bt.maxNp / TILE <= ROWS_MAX && wavefront_trsm()) {
    const bool narrow = maxMp / TILE <= WAVE_NCT;
    solve_launches(bt, maxMp, s, [&](Prob* const* dp, const SolveSched& ss, int ct0, int tot,
                                     uint32_t ep) {
      const auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(tot), dim3(NTHREADS), 0, s, dp, ss, ct0, bt.ticket, ep);
      };
      if (prec == PGP_PREC_FP64)
        narrow ? go(k_trsm_rows<double, false>) : go(k_trsm_rows<double, true>);
      else
        narrow ? go(k_trsm_rows<float, false>) : go(k_trsm_rows<float, true>);
    });
    return;
  }
  if (maxMp / TILE < TRSM_WIDE) {
    launch_trsm_lagged(bt, prec, maxMp, s);
    return;
  }
  const int nb = bt.maxNp / TILE;
  const int nq = (nb + TRSM_G - 1) / TRSM_G;
  const bool on = timer_on(TC_TRSM);
  auto nct_of = [&](int m) {
    const int mp = bt.hm ? (bt.hm[m] + TILE - 1) / TILE * TILE : maxMp;
    return mp / TILE;
  };
  for (int q = 0; q < nq; ++q) {
    sched_launch(
        bt, [&](int m) { return trsm_units(bt.np(m) / TILE, q, nct_of(m)); },
        [&](Prob* const* dp, const Sched& sc, int n) {
          if (on) timer_begin(TC_TRSM, s);
          if (prec == PGP_PREC_FP64)
            hipLaunchKernelGGL(k_trsm<double>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, q);
          else
            hipLaunchKernelGGL(k_trsm<float>, dim3(n), dim3(NTHREADS), 0, s, dp, sc, q);
          if (on) {
            // super-step q of an N^2 M-flop solve: its rows' left-looking
            // products and triangles, and the rank-64G update of the rows
            // below by the previous super-step (full right-hand side)
            constexpr double T3 = 2.0 * TILE * TILE * TILE;
            double fl = 0.0;
            const int off = (int)(dp - bt.dprobs);
            for (int m = off; m < off + sc.count; ++m) {
              const int nbm = bt.np(m) / TILE, nct = nct_of(m);
              if (nbm <= TRSM_G * q) continue;
              const int p0 = q > 0 ? TRSM_G * (q - 1) : 0;
              for (int k = TRSM_G * q; k < std::min(nbm, TRSM_G * q + TRSM_G); ++k)
                fl += nct * (T3 * (k - p0) + T3 / 2);
              if (q > 0)
                fl += (double)nct * std::max(0, nbm - TRSM_G * (q + 1)) * T3 * TRSM_G;
            }
            timer_end(TC_TRSM, s, fl, 0.0);
          }
        });
  }
}

template <typename T>
__global__ __launch_bounds__(NTHREADS) void k_trsm_raw(const T* L, int64_t ld, const double* dinv,
                                                       int nb, int q, T* S, int64_t lds, int nct) {
  trsm_ss<T>(L, ld, dinv, nb, q, S, lds, nct, blockIdx.x);
}

int launch_trsm_raw_dinv(int prec, const void* L, int64_t N, int64_t ld, const double* dinv,
                         void* S, int64_t M, int64_t lds, hipStream_t s) {
  const int nb = (int)(N / TILE), nct = (int)(M / TILE);
  if (nct < TRSM_WIDE) {
    for (int k = 0; k < nb; ++k) {
      dim3 g(k == 0 ? 1 : nb - k, (unsigned)nct);
      if (prec == PGP_PREC_FP64)
        hipLaunchKernelGGL(k_trsm_lagged_raw<double>, g, dim3(NTHREADS), 0, s, (const double*)L,
                           ld, dinv, k, (double*)S, lds);
      else
        hipLaunchKernelGGL(k_trsm_lagged_raw<float>, g, dim3(NTHREADS), 0, s, (const float*)L, ld,
                           dinv, k, (float*)S, lds);
    }
    return 0;
  }
  const int nq = (nb + TRSM_G - 1) / TRSM_G;
  for (int q = 0; q < nq; ++q) {
    const dim3 g((unsigned)trsm_units(nb, q, nct));
    if (prec == PGP_PREC_FP64)
      hipLaunchKernelGGL(k_trsm_raw<double>, g, dim3(NTHREADS), 0, s, (const double*)L, ld, dinv,
                         nb, q, (double*)S, lds, nct);
    else
      hipLaunchKernelGGL(k_trsm_raw<float>, g, dim3(NTHREADS), 0, s, (const float*)L, ld, dinv,
                         nb, q, (float*)S, lds, nct);
  }
  return 0;
}

}  // namespace pgp
