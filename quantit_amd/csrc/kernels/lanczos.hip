// Kernels of the k-step Lanczos eigensolver of the two-site update (FP64).
//
// The Krylov vectors of one update share one flat layout (the blocks of the
// two-site state, back to back), so they are the rows of one matrix V
// (row pitch ld): the full reorthogonalisation is a pair of skinny
// products c = V w and w -= V^T c, and the Ritz vector is V^T y.  All
// reductions run in a fixed order (no atomics), so results do not depend on
// what else runs on the device.
#include "../kernels.hpp"

namespace qtt {
namespace kern {

namespace {

constexpr int kThreads = 256;

__device__ double block_reduce(double v, double* sh) {
  const int tid = threadIdx.x;
  sh[tid] = v;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (tid < w) sh[tid] += sh[tid + w];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

}  // namespace

// partial[i * G + b] = sum over chunk b of V[i][e] * w[e]; the thread keeps
// its kKrylovPerThread elements of w in registers across the m rows.
__global__ __launch_bounds__(kThreads) void k_krylov_dot_partial(double* __restrict__ base, int64_t v_off, int64_t ld,
                                                                 int m, int64_t w_off, int64_t n,
                                                                 int64_t partial_off) {
  __shared__ double sh[kThreads];
  const int G = gridDim.x;
  const int64_t e0 = int64_t(blockIdx.x) * kKrylovChunk + threadIdx.x;
  const double* w = base + w_off;
  double wr[kKrylovPerThread];
#pragma unroll
  for (int q = 0; q < kKrylovPerThread; ++q) {
    const int64_t e = e0 + int64_t(q) * kThreads;
    wr[q] = e < n ? w[e] : 0.0;
  }
  for (int i = 0; i < m; ++i) {
    const double* v = base + v_off + int64_t(i) * ld;
    double acc = 0.0;
#pragma unroll
    for (int q = 0; q < kKrylovPerThread; ++q) {
      const int64_t e = e0 + int64_t(q) * kThreads;
      if (e < n) acc += v[e] * wr[q];
    }
    const double r = block_reduce(acc, sh);
    if (threadIdx.x == 0) base[partial_off + int64_t(i) * G + blockIdx.x] = r;
  }
}

// out[i] = sum_b partial[i * G + b], b ascending.
__global__ void k_krylov_dot_final(double* __restrict__ base, int64_t partial_off, int G, int m, int64_t out_off) {
  for (int i = threadIdx.x; i < m; i += blockDim.x) {
    double acc = 0.0;
    const double* p = base + partial_off + int64_t(i) * G;
    for (int b = 0; b < G; ++b) acc += p[b];
    base[out_off + i] = acc;
  }
}

void krylov_dot(hipStream_t s, double* base, int64_t v_off, int64_t ld, int m, int64_t w_off, int64_t n,
                int64_t partial_off, int64_t out_off) {
  if (m <= 0) return;
  const int G = int((n + kKrylovChunk - 1) / kKrylovChunk);
  if (G > 0)
    hipLaunchKernelGGL(k_krylov_dot_partial, dim3(G), dim3(kThreads), 0, s, base, v_off, ld, m, w_off, n,
                       partial_off);
  hipLaunchKernelGGL(k_krylov_dot_final, dim3(1), dim3(64), 0, s, base, partial_off, G, m, out_off);
}

// dst[e] = src[e] + sign * sum_i coef[i] V[i][e] (src_off < 0: no src term;
// scale_off >= 0: the result is divided by sqrt(base[scale_off])).
__global__ __launch_bounds__(kThreads) void k_krylov_axpy(double* __restrict__ base, int64_t v_off, int64_t ld, int m,
                                                          int64_t coef_off, double sign, int64_t src_off,
                                                          int64_t dst_off, int64_t n, int64_t scale_off) {
  const int64_t e = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (e >= n) return;
  double acc = 0.0;
  for (int i = 0; i < m; ++i) acc += base[coef_off + i] * base[v_off + int64_t(i) * ld + e];
  double r = (src_off >= 0 ? base[src_off + e] : 0.0) + sign * acc;
  if (scale_off >= 0) r = r / sqrt(base[scale_off]);
  base[dst_off + e] = r;
}

void krylov_axpy(hipStream_t s, double* base, int64_t v_off, int64_t ld, int m, int64_t coef_off, double sign,
                 int64_t src_off, int64_t dst_off, int64_t n, int64_t scale_off) {
  if (n <= 0) return;
  const int64_t G = (n + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(k_krylov_axpy, dim3(unsigned(G)), dim3(kThreads), 0, s, base, v_off, ld, m, coef_off, sign,
                     src_off, dst_off, n, scale_off);
}

namespace {

__device__ __forceinline__ double fast_rcp(double x) {  // estimate (2^-24) and one third-order step
  const double z = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, z, 1.0);
  return fma(z, fma(e, e, e), z);
}

struct TridiagLds {
  double alpha[kMaxKrylov], beta[kMaxKrylov], b2[kMaxKrylov], y[kMaxKrylov], l[kMaxKrylov], rd[kMaxKrylov];
  double bracket[2];
};

// Number of eigenvalues of the symmetric tridiagonal T (alpha, beta) below
// x: the negative pivots of the LDL^T factorisation of T - x I (Sturm).
__device__ int sturm_count(const TridiagLds& S, int m, double x, double tiny) {
  int cnt = 0;
  double q = S.alpha[0] - x;
  if (fabs(q) < tiny) q = -tiny;
  cnt += q < 0.0;
  for (int i = 1; i < m; ++i) {
    q = S.alpha[i] - x - S.b2[i - 1] * fast_rcp(q);
    if (fabs(q) < tiny) q = -tiny;
    cnt += q < 0.0;
  }
  return cnt;
}

// LDS written by lanes of this wave is seen by all of them.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Three inverse iterations with L D L^T = T - sigma I (l, 1 / D = rd) from the
// vector of ones, normalised with y[0] >= 0.
template <int M>
__device__ __forceinline__ void inverse_iterate(int m, const double (&l)[M], const double (&rd)[M], double (&y)[M]) {
#pragma unroll
  for (int i = 0; i < M; ++i) y[i] = 1.0;
  for (int it = 0; it < 3; ++it) {
#pragma unroll
    for (int i = 1; i < M; ++i)
      if (i < m) y[i] -= l[i - 1] * y[i - 1];  // L z = y
#pragma unroll
    for (int i = 0; i < M; ++i) y[i] *= rd[i];  // D
#pragma unroll
    for (int i = M - 2; i >= 0; --i)
      if (i + 1 < m) y[i] -= l[i] * y[i + 1];  // L^T
    double nrm = 0.0;
#pragma unroll
    for (int i = 0; i < M; ++i)
      if (i < m) nrm += y[i] * y[i];
    const double f = (y[0] < 0.0 ? -1.0 : 1.0) / sqrt(nrm);
#pragma unroll
    for (int i = 0; i < M; ++i) y[i] *= f;
  }
}

// The lowest eigenpair of the leading m x m tridiagonal in S (alpha, beta);
// one wave calls this:
// * eigenvalue by multisection: 64 lanes evaluate Sturm counts at 64 interior
//   points of the bracket, which shrinks 65-fold per round, from the
//   Gershgorin interval down to a few ulps;
// * eigenvector by three inverse iterations with T - sigma I, sigma just below
//   the eigenvalue (positive definite: its LDL^T pivots stay positive),
//   normalised with y[0] >= 0.
// out: [0] eigenvalue, [1] residual norm beta[m-1] |y[m-1]|, [2] beta[m-1],
// [3 ..] y.  host (pinned memory): the first three and [3] = 1 where a NaN
// appeared, 0 otherwise; stored there directly, a copy would be one more
// dispatch before the host's wait.
__device__ void tridiag_lowest(TridiagLds& S, int m, double* __restrict__ out, double* __restrict__ host) {
  const int tid = threadIdx.x;
  if (tid < m) S.b2[tid] = S.beta[tid] * S.beta[tid];
  if (tid == 0) {
    double lo = S.alpha[0], hi = S.alpha[0];
    for (int i = 0; i < m; ++i) {
      const double r = (i > 0 ? fabs(S.beta[i - 1]) : 0.0) + (i + 1 < m ? fabs(S.beta[i]) : 0.0);
      lo = fmin(lo, S.alpha[i] - r);
      hi = fmax(hi, S.alpha[i] + r);
    }
    const double pad = 2.2e-16 * (fmax(fabs(lo), fabs(hi)) + 1e-300);
    S.bracket[0] = lo - pad;
    S.bracket[1] = hi + pad;
  }
  wave_sync();
  const double scale = fmax(fabs(S.bracket[0]), fabs(S.bracket[1]));
  const double tiny = 1e-300 + 2.2e-16 * 1e-30 * scale;
  // invariant: count(bracket[0]) == 0, count(bracket[1]) >= 1
  for (int round = 0; round < 12; ++round) {
    const double lo = S.bracket[0], hi = S.bracket[1];
    if (!(hi - lo > 4.4e-16 * fmax(fabs(lo), fabs(hi)))) break;
    const double x = lo + (hi - lo) * double(tid + 1) / 65.0;
    const unsigned long long ge = __ballot(sturm_count(S, m, x, tiny) >= 1);
    if (tid == 0) {
      if (ge == 0ull) {
        S.bracket[0] = lo + (hi - lo) * 64.0 / 65.0;
      } else {
        const int f = __ffsll(static_cast<long long>(ge)) - 1;  // first lane whose point holds an eigenvalue below
        S.bracket[1] = lo + (hi - lo) * double(f + 1) / 65.0;
        if (f > 0) S.bracket[0] = lo + (hi - lo) * double(f) / 65.0;
      }
    }
    wave_sync();
  }
  if (tid != 0) return;
  const double lam = 0.5 * (S.bracket[0] + S.bracket[1]);
  // sigma below lam: T - sigma I positive definite (pivots > 0)
  const double sigma = lam - fmax(8.0 * (S.bracket[1] - S.bracket[0]), 4.4e-16 * fmax(scale, 1e-300));
  S.rd[0] = 1.0 / (S.alpha[0] - sigma);
  for (int i = 1; i < m; ++i) {
    S.l[i - 1] = S.beta[i - 1] * S.rd[i - 1];
    double d = S.alpha[i] - sigma - S.l[i - 1] * S.beta[i - 1];
    if (!(d > 0.0)) d = 1e-300 + 2.2e-16 * scale;
    S.rd[i] = 1.0 / d;
  }
  if (m <= 8) {  // in registers: one lane waits for every LDS access
    double l[8], rd[8], y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      l[i] = i + 1 < m ? S.l[i] : 0.0;
      rd[i] = i < m ? S.rd[i] : 0.0;
    }
    inverse_iterate(m, l, rd, y);
#pragma unroll
    for (int i = 0; i < 8; ++i) S.y[i] = y[i];
  } else {
    for (int i = 0; i < m; ++i) S.y[i] = 1.0;
    for (int it = 0; it < 3; ++it) {
      for (int i = 1; i < m; ++i) S.y[i] -= S.l[i - 1] * S.y[i - 1];   // L z = y
      for (int i = 0; i < m; ++i) S.y[i] *= S.rd[i];                    // D
      for (int i = m - 2; i >= 0; --i) S.y[i] -= S.l[i] * S.y[i + 1];  // L^T
      double nrm = 0.0;
      for (int i = 0; i < m; ++i) nrm += S.y[i] * S.y[i];
      const double f = (S.y[0] < 0.0 ? -1.0 : 1.0) / sqrt(nrm);
      for (int i = 0; i < m; ++i) S.y[i] *= f;
    }
  }
  const double bj = S.beta[m - 1];
  const double res = fabs(bj * S.y[m - 1]);
  out[0] = lam;
  out[1] = res;
  out[2] = bj;
  bool bad = isnan(lam) || isnan(res);
  for (int i = 0; i < m; ++i) {
    out[3 + i] = S.y[i];
    bad |= isnan(S.y[i]);
  }
  host[0] = lam;
  host[1] = res;
  host[2] = bj;
  host[3] = bad ? 1.0 : 0.0;
}

}  // namespace

// Stores alpha[j] = c1[j] + c2[j] and beta[j] = sqrt(nrm2) into T (alpha at
// T[0..K), beta at T[K..2K)), then the lowest eigenpair of the leading (j+1) x
// (j+1) tridiagonal.
__global__ __launch_bounds__(64) void k_lanczos_tridiag(double* __restrict__ base, int64_t t_off, int K, int j,
                                                        int64_t c1_off, int64_t c2_off, int64_t nrm2_off,
                                                        int64_t out_off, double* __restrict__ host) {
  __shared__ TridiagLds S;
  const int m = j + 1;
  if (threadIdx.x == 0) {
    base[t_off + j] = base[c1_off + j] + base[c2_off + j];
    base[t_off + K + j] = sqrt(base[nrm2_off]);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < m; i += 64) {
    S.alpha[i] = base[t_off + i];
    S.beta[i] = base[t_off + K + i];
  }
  __syncthreads();
  tridiag_lowest(S, m, base + out_off, host);
}

void lanczos_tridiag(hipStream_t s, double* base, int64_t t_off, int K, int j, int64_t c1_off, int64_t c2_off,
                     int64_t nrm2_off, int64_t out_off, double* host) {
  hipLaunchKernelGGL(k_lanczos_tridiag, dim3(1), dim3(64), 0, s, base, t_off, K, j, c1_off, c2_off, nrm2_off,
                     out_off, host);
}

// A whole Lanczos step after the matvec for short vectors, by one work-group:
// two Gram-Schmidt passes of w against v_0 .. v_j, |w|^2, the tridiagonal
// eigensolve, and v_{j+1} = w / |w| when V has the row.  In launches of their
// own these are ten, each shorter than the launch of the next.  w stays in
// registers, V is read up to four times from the caches, by one CU: up to 8192
// elements that is no slower for any m (n = 1000, m = 4: 12.8 us against 34.1;
// m = 16: 46 against 87; n = 8000, m = 4: 21 against 40; m = 64: 336 against 339).
constexpr int kStepThreads = 512;
static_assert(kKrylovStepMaxN == 16 * kStepThreads, "the widest variant holds 16 elements per thread");
template <int Q>  // elements of a vector per thread
__global__ __launch_bounds__(kStepThreads) void k_krylov_step(double* __restrict__ base, int64_t v_off, int64_t ld,
                                                              int j, int K, int64_t w_off, int n, int64_t t_off,
                                                              int64_t nrm2_off, int64_t out_off,
                                                              double* __restrict__ host) {
  __shared__ TridiagLds S;
  __shared__ double part[kMaxKrylov + 3][kStepThreads / 64], cs[kMaxKrylov + 3], alpha_j;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = j + 1;
  const double* V = base + v_off;
  double w[Q], v[4][Q];
  auto load = [&](const double* x, double (&r)[Q]) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int e = tid + q * kStepThreads;
      r[q] = x[min(e, n - 1)];
      if (e >= n) r[q] = 0.0;
    }
  };
  auto rows = [&](int i0) {  // four rows at a time (past the last: it again)
#pragma unroll
    for (int u = 0; u < 4; ++u) load(V + int64_t(min(i0 + u, m - 1)) * ld, v[u]);
  };
  auto wave_sum = [&](double x) {
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    return x;
  };
  load(base + w_off, w);
  if (tid == 0) alpha_j = 0.0;
  for (int pass = 0; pass < 2; ++pass) {
    for (int i0 = 0; i0 < m; i0 += 4) {
      rows(i0);
      double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[u] = fma(v[u][q], w[q], acc[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] = wave_sum(acc[u]);
      if (lane == 0)
#pragma unroll
        for (int u = 0; u < 4; ++u) part[i0 + u][wave] = acc[u];
    }
    __syncthreads();
    if (tid < (m + 3) / 4 * 4) {
      double c = 0.0;
#pragma unroll
      for (int u = 0; u < kStepThreads / 64; ++u) c += part[tid][u];
      cs[tid] = tid < m ? c : 0.0;
      if (tid == j) alpha_j += c;
    }
    __syncthreads();
    for (int i0 = 0; i0 < m; i0 += 4) {
      if (m > 4) rows(i0);  // else still there
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double c = cs[i0 + u];
#pragma unroll
        for (int q = 0; q < Q; ++q) w[q] = fma(-c, v[u][q], w[q]);
      }
    }
  }
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < Q; ++q) acc = fma(w[q], w[q], acc);
  acc = wave_sum(acc);
  if (lane == 0) part[0][wave] = acc;
  __syncthreads();
  double nrm2 = 0.0;
#pragma unroll
  for (int u = 0; u < kStepThreads / 64; ++u) nrm2 += part[0][u];
  const double nrm = sqrt(nrm2);
  if (m < K) {
    double* next = base + v_off + int64_t(m) * ld;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int e = tid + q * kStepThreads;
      if (e < n) next[e] = w[q] / nrm;
    }
  }
  if (tid == 0) {
    base[nrm2_off] = nrm2;
    base[t_off + j] = alpha_j;
    base[t_off + K + j] = nrm;
  }
  if (tid < m) {
    S.alpha[tid] = tid == j ? alpha_j : base[t_off + tid];
    S.beta[tid] = tid == j ? nrm : base[t_off + K + tid];
  }
  __syncthreads();
  if (wave == 0) tridiag_lowest(S, m, base + out_off, host);
}

void krylov_step(hipStream_t s, double* base, int64_t v_off, int64_t ld, int j, int K, int64_t w_off, int64_t n,
                 int64_t t_off, int64_t nrm2_off, int64_t out_off, double* host) {
  auto* k = n <= 2 * kStepThreads   ? k_krylov_step<2>
            : n <= 4 * kStepThreads ? k_krylov_step<4>
            : n <= 8 * kStepThreads ? k_krylov_step<8>
                                    : k_krylov_step<16>;
  hipLaunchKernelGGL(k, dim3(1), dim3(kStepThreads), 0, s, base, v_off, ld, j, K, w_off, int(n), t_off, nrm2_off,
                     out_off, host);
}

}  // namespace kern
}  // namespace qtt
