// Gram-matrix eigenvectors for sectors wider than one work-group's LDS holds
// (k > kGramEigMaxK).  G = Y^T Y (k x k, column-major, leading dimension k)
// lives in device memory; the steps mirror the LDS solver of svd_jacobi.hip:
//
//   k_gram_check    orthogonality test of the columns behind G (relative, or
//                   absolute with respect to the largest singular value),
//   k_pchol_panel   one panel of nb columns of the pivoted Cholesky
//                   P^T G P = R^T R (left-looking inside the panel; the
//                   trailing matrix is updated by a GEMM G -= Lp Lp^T after
//                   each panel).  L = R^T is kept with its rows in the
//                   original order, so L L^T = G and the Jacobi rounds on the
//                   columns of L (gram_rounds.hip) yield G's eigenvectors
//                   as the normalised columns,
//   k_gram_vectors  normalises the columns of the rotated L into W and
//                   completes zero columns from the unit vector with the
//                   largest residual (two projection passes).
#include <algorithm>
#include <cfloat>
#include <climits>
#include <stdexcept>

#include "../kernels.hpp"

namespace qtt {
namespace kern {

namespace {

__device__ double block_max(double v, double* sh) {
  const int tid = threadIdx.x;
  sh[tid] = v;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if (tid < w) sh[tid] = fmax(sh[tid], sh[tid + w]);
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

__device__ double block_sum(double v, double* sh) {
  const int tid = threadIdx.x;
  sh[tid] = v;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if (tid < w) sh[tid] += sh[tid + w];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

// 1/sqrt(x) by the hardware estimate (2^-24) and one third-order step.
__device__ __forceinline__ double fast_rsqrt_pc(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

}  // namespace

constexpr int kLargeThreads = 1024;

template <class L>
__global__ void k_gram_check_zero(double*, L l, int n, int* __restrict__ flags) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const SmallJacobi J = l.template list<SmallJacobi>()[i];
    if (J.flag_idx >= 0) flags[J.flag_idx] = 0;
    if (J.aux_idx >= 0) flags[J.aux_idx] = 0;
  }
}

// flags[flag_idx] += pairs failing both tests, flags[aux_idx] += pairs passing
// only the absolute one (same tests as k_gram_eig, on squares), both zeroed
// beforehand.  Work-group y of a sector takes the columns c = y (mod
// gridDim.y); the diagonal sits in LDS (dynamic, k doubles); wave w scans the
// upper part of its w-th, (w + 16)-th, ... column with coalesced reads.
template <class L>
__global__ __launch_bounds__(kLargeThreads) void k_gram_check(double* __restrict__ base, L l, int* __restrict__ flags,
                                                              double tol) {
  extern __shared__ double dg[];
  __shared__ double sh[kLargeThreads];
  __shared__ int nv, na;
  const SmallJacobi J = l.template list<SmallJacobi>()[blockIdx.x];
  const int k = J.k;
  const double* G = base + J.y_off;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwave = blockDim.x >> 6;
  const int ny = gridDim.y, y = blockIdx.y;
  if (tid == 0) nv = na = 0;
  double dm = 0.0;
  for (int i = tid; i < k; i += blockDim.x) {
    dg[i] = G[int64_t(i) * J.ldy + i];
    dm = fmax(dm, dg[i]);
  }
  const double g2max = block_max(dm, sh);  // also orders the dg writes before the reads
  const double t2 = tol * tol;
  int my = 0, mya = 0;
  for (int c = y + ny * wave; c < k; c += ny * nwave) {
    const double gjj = dg[c];
    const double* col = G + int64_t(c) * J.ldy;
#pragma unroll 4
    for (int r = lane; r < c; r += 64) {
      const double gii = dg[r], g = col[r];
      const double g2 = g * g;
      if (gii > 0.0 && gjj > 0.0 && g2 > t2 * gii * gjj) {
        if (g2 > t2 * fmax(gii, gjj) * g2max)
          ++my;
        else
          ++mya;
      }
    }
  }
  if (my) atomicAdd(&nv, my);
  if (mya) atomicAdd(&na, mya);
  __syncthreads();
  if (tid == 0) {
    if (J.flag_idx >= 0 && nv) atomicAdd(&flags[J.flag_idx], nv);
    if (J.aux_idx >= 0 && na) atomicAdd(&flags[J.aux_idx], na);
  }
}

void gram_check(hipStream_t st, double* base, const Lists& descs, int n, int* flags, double tol, int kmax) {
  if (n <= 0) return;
  static const size_t limit = [] {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) v = 65536;
    const size_t l = size_t(v) - kLargeThreads * sizeof(double) - 64;
    for (const void* f : {reinterpret_cast<const void*>(&k_gram_check<DevLists>),
                          reinterpret_cast<const void*>(&k_gram_check<ArgLists>)})
      (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, int(l));
    return l;
  }();
  const size_t lds = size_t(kmax) * sizeof(double);
  if (lds > limit) throw std::runtime_error("gram check: sector wider than the LDS holds");
  const int ny = std::max(1, std::min(8, kmax / 64));  // about 64 columns per work-group
  launch_lists(k_gram_check_zero<DevLists>, k_gram_check_zero<ArgLists>, descs, dim3(1), dim3(256), 0, st, base, n, flags);
  launch_lists(k_gram_check<DevLists>, k_gram_check<ArgLists>, descs, dim3(n, ny), dim3(kLargeThreads), lds, st, base, flags, tol);
}

// One panel [j0, j0 + nb) of the pivoted Cholesky of G (already updated by
// the previous panels).  state[0] = rank found so far (k while running),
// state[1 + i] = 1 once original index i has been pivoted.  L is k x ldl
// (column-major, leading dimension k), rows in the original order.  The
// panel's columns are also written to Lp (k x nb, column-major) for the
// trailing update.  LDS: the nb panel columns, the running diagonal dg
// (G_ii less this panel's columns so far) and the pivoted flags, k each.
// The pivot is the largest remaining diagonal up to 2^-7 of it, the smallest
// index on ties: the key is the value's upper word with the inverted index in
// its low 13 bits (k <= 8192); non-positive values never beat positive ones.
//
// A step is bound by its chain (the waves' candidates, the pivot's column of G,
// one barrier) and by LDS reads, which cost the same for one address as for 64
// (a candidate per lane, not all by every thread).  ONE: one row to a thread (k
// <= 1024), whose panel entries, diagonal and flag stay in registers; only the
// pivot's row comes from LDS.  k = 544: 44 us a panel of 32, against 58 for
// 64-bit keys and rows read from LDS.
constexpr int kPanelMax = 32;
template <bool ONE>
__global__ __launch_bounds__(kLargeThreads) void k_pchol_panel(double* __restrict__ base,
                                                               const CholPanel* __restrict__ ps, int j0, int nb) {
  extern __shared__ double lds[];
  __shared__ int wkey[2][kLargeThreads / 64];  // the waves' candidates, by step parity
  __shared__ double wval[2][kLargeThreads / 64];
  const CholPanel P = ps[blockIdx.x];
  const int k = P.k;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const double* G = base + P.g_off;
  double* L = base + P.l_off;
  double* Lp = base + P.lp_off;
  int* state = reinterpret_cast<int*>(base + P.state_off);
  double* col = lds;       // nb columns of length k
  double* dg = col + int64_t(nb) * k;
  int* used = reinterpret_cast<int*>(dg + k);
  if (state[0] < k || j0 >= k) {  // already rank-deficient or finished: zero panel
    for (int64_t e = tid; e < int64_t(k) * nb; e += blockDim.x) Lp[e] = 0.0;
    return;
  }
  const int nwv = min(int(blockDim.x) >> 6, (k + 63) >> 6);  // waves that hold rows
  auto key_of = [&](double d, int i) { return (int(__double_as_longlong(d) >> 32) & ~0x1FFF) | (8191 - i); };
  // the wave's best row, from each lane's best (key, diagonal)
  auto publish = [&](int key, double d, int slot) {
    int top = max(key, __builtin_amdgcn_mov_dpp(key, 0xB1, 0xF, 0xF, false));
    top = max(top, __builtin_amdgcn_mov_dpp(top, 0x4E, 0xF, 0xF, false));
    top = max(top, __builtin_amdgcn_mov_dpp(top, 0x141, 0xF, 0xF, false));
    top = max(top, __builtin_amdgcn_mov_dpp(top, 0x140, 0xF, 0xF, false));
    top = max(top, __builtin_amdgcn_ds_swizzle(top, 0x401F));
    top = max(top, __shfl_xor(top, 32));
    if (key == top) {  // one lane, or all of a wave without a row left
      wkey[slot][wave] = top;
      wval[slot][wave] = d;
    }
  };
  double lr[ONE ? kPanelMax : 1], mydg = -1.0;
  bool out = true;  // ONE: no row, or a pivoted one
#pragma unroll
  for (int t = 0; t < (ONE ? kPanelMax : 1); ++t) lr[t] = 0.0;
  if (wave < nwv) {
    int key = INT_MIN;
    double d = -1.0;
    for (int i = tid; i < k; i += blockDim.x) {
      const double di = G[int64_t(i) * k + i];
      const int u = state[1 + i];
      const int ki = u ? INT_MIN : key_of(di, i);
      if (ki > key) {
        key = ki;
        d = di;
      }
      if constexpr (ONE) {
        mydg = di;
        out = u != 0;
      } else {
        dg[i] = di;
        used[i] = u;
      }
    }
    publish(key, d, 0);
  }
  __syncthreads();
  // One barrier per step: a thread forms the next step's key from its own
  // diagonal entries right after updating them, and the candidates go to the
  // other parity's slots (last read before the previous barrier).
  int rank = k;
  for (int jj = 0; jj < nb; ++jj) {
    const int j = j0 + jj;
    if (j >= k) {
      for (int i = tid; i < k; i += blockDim.x) col[jj * k + i] = 0.0;
      continue;
    }
    // lane w < nwv looks at wave w's candidate
    const int cand = lane < nwv ? wkey[jj & 1][lane] : INT_MIN;
    const double cval = lane < nwv ? wval[jj & 1][lane] : -1.0;
    int top = max(cand, __builtin_amdgcn_mov_dpp(cand, 0xB1, 0xF, 0xF, false));
    top = max(top, __builtin_amdgcn_mov_dpp(top, 0x4E, 0xF, 0xF, false));
    top = max(top, __builtin_amdgcn_mov_dpp(top, 0x141, 0xF, 0xF, false));
    top = max(top, __builtin_amdgcn_mov_dpp(top, 0x140, 0xF, 0xF, false));
    top = __builtin_amdgcn_readfirstlane(top);
    const int who = __ffsll((unsigned long long)__ballot(cand == top)) - 1;
    const long long cb = __double_as_longlong(cval);
    const int plo = __builtin_amdgcn_readlane(int(cb & 0xffffffffLL), who);
    const int phi = __builtin_amdgcn_readlane(int(cb >> 32), who);
    const double pv = __longlong_as_double((long long)(unsigned)plo | ((long long)phi << 32));
    const int p = 8191 - (top & 0x1FFF);
    if (top == INT_MIN || !(pv > 0.0)) {  // uniform: the rest is zero or negative noise
      for (int t = jj; t < nb; ++t)
        for (int i = tid; i < k; i += blockDim.x) col[t * k + i] = 0.0;
      rank = j;
      break;
    }
    if (wave < nwv) {
      const double isq = fast_rsqrt_pc(pv), ljj = pv * isq;
      int key = INT_MIN;
      double d = -1.0;
      if constexpr (ONE) {
        // the load of G's column p does not depend on the sum over the panel's
        // earlier columns, so its latency overlaps that
        const double gpi = out ? 0.0 : G[int64_t(p) * k + tid];
        double acc[2] = {0.0, 0.0};
#pragma unroll
        for (int t0 = 0; t0 < kPanelMax; t0 += 8)
          if (t0 < jj) {  // entries past jj meet zeros of lr
            double lp[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) lp[u] = col[min(t0 + u, jj - 1) * k + p];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc[u & 1] = fma(lr[t0 + u], lp[u], acc[u & 1]);
          }
        const bool here = tid == p;
        const double v = here ? ljj : out ? 0.0 : (gpi - (acc[0] + acc[1])) * isq;
        mydg = here ? -1.0 : fma(-v, v, mydg);
        out = out || here;
        if (tid < k) col[jj * k + tid] = v;
#pragma unroll
        for (int t0 = 0; t0 < kPanelMax; t0 += 8)
          if (t0 == (jj & ~7))
#pragma unroll
            for (int u = 0; u < 8; ++u) lr[t0 + u] = u == (jj & 7) ? v : lr[t0 + u];
        key = out ? INT_MIN : key_of(mydg, tid);
        d = mydg;
      } else {
        for (int i = tid; i < k; i += blockDim.x) {
          double v = 0.0;
          if (i == p) {
            v = ljj;
            used[p] = 1;
          } else if (!used[i]) {
            const double gpi = G[int64_t(p) * k + i];
            double acc = 0.0;
#pragma unroll 8
            for (int t = 0; t < jj; ++t) acc = fma(col[t * k + i], col[t * k + p], acc);
            v = (gpi - acc) * isq;
            dg[i] -= v * v;
          }
          col[jj * k + i] = v;
          const int ki = used[i] ? INT_MIN : key_of(dg[i], i);
          if (ki > key) {
            key = ki;
            d = dg[i];
          }
        }
      }
      publish(key, d, (jj + 1) & 1);
    }
    __syncthreads();
  }
  if constexpr (ONE)
    if (tid < k) used[tid] = out;
  __syncthreads();  // the copies below read other threads' column entries
  for (int i = tid; i < k; i += blockDim.x) state[1 + i] = used[i];
  if (tid == 0 && rank < k) state[0] = rank;
  for (int t = wave; t < nb; t += int(blockDim.x) >> 6)
    for (int i = lane; i < k; i += 64) {
      const double v = col[t * k + i];
      Lp[int64_t(t) * k + i] = v;
      if (j0 + t < k) L[int64_t(j0 + t) * k + i] = v;
    }
  if (rank > 0 && rank < k) {
    // the factor of G + delta^2 I on the rows without a pivot, as in k_gram_eig
    __syncthreads();  // the zero columns copied above are overwritten
    const double* first = j0 == 0 ? col : L;
    const double* end = rank > j0 ? col + (rank - 1 - j0) * k : L + int64_t(rank - 1) * k;
    double top = 0.0, last = 0.0;
    for (int i = lane; i < k; i += 64) {
      top = fmax(top, fabs(first[i]));
      last = fmax(last, fabs(end[i]));
    }
    for (int off = 32; off > 0; off >>= 1) {
      top = fmax(top, __shfl_xor(top, off));
      last = fmax(last, __shfl_xor(last, off));
    }
    top = fmin(top * 0x1p-27, last);
    for (int i = tid; i < k; i += blockDim.x) {
      if (used[i]) continue;
      int c = rank;
      for (int j = 0; j < i; ++j) c += used[j] ? 0 : 1;
      L[int64_t(c) * k + i] = top;
    }
  }
}

__global__ __launch_bounds__(256) void k_pchol_init(double* __restrict__ base, const CholPanel* __restrict__ ps) {
  const CholPanel P = ps[blockIdx.x];
  int* state = reinterpret_cast<int*>(base + P.state_off);
  for (int i = threadIdx.x; i <= P.k; i += blockDim.x) state[i] = i == 0 ? P.k : 0;
}

void pchol_init(hipStream_t st, double* base, const void* descs, int n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_pchol_init, dim3(n), dim3(256), 0, st, base, static_cast<const CholPanel*>(descs));
}

void pchol_panel(hipStream_t st, double* base, const void* descs, int n, int j0, int nb, int kmax) {
  if (n <= 0) return;
  if (nb > kPanelMax) throw std::runtime_error("Cholesky panel wider than 32 columns");
  const size_t lds = size_t(kmax) * (nb + kPcholExtra) * sizeof(double);
  const auto* ps = static_cast<const CholPanel*>(descs);
  if (kmax <= kLargeThreads)
    hipLaunchKernelGGL(k_pchol_panel<true>, dim3(n), dim3((kmax + 63) / 64 * 64), lds, st, base, ps, j0, nb);
  else
    hipLaunchKernelGGL(k_pchol_panel<false>, dim3(n), dim3(kLargeThreads), lds, st, base, ps, j0, nb);
}

size_t pchol_lds_limit() {
  static const size_t limit = [] {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) v = 65536;
    const size_t l = size_t(v) - 1024;  // static arrays of the kernel
    for (const void* f : {reinterpret_cast<const void*>(&k_pchol_panel<true>),
                          reinterpret_cast<const void*>(&k_pchol_panel<false>)})
      (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, int(l));
    return l;
  }();
  return limit;
}

// W = columns of X (k x k at x_off, leading dimension ldx) normalised, by
// k_gram_vec_norm over (sector, 64-column) work-groups (wave w takes four
// columns, rows in flight four at a time); then k_gram_vectors completes the
// zero columns from the unit vector with the largest residual (two
// projection passes), one work-group per sector, and returns at once when
// there are none.  W is written at w_off with leading dimension ldw;
// scratch_off: 3k doubles (norms, two work vectors).
template <class L>
__global__ __launch_bounds__(kLargeThreads) void k_gram_vec_norm(double* __restrict__ base,
                                                                 L l) {
  const GramVec J = l.template list<GramVec>()[blockIdx.x];
  const int k = J.k;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c0 = blockIdx.y * 64 + wave * 4;
  if (c0 >= k) return;
  const double* X = base + J.x_off;
  double* W = base + J.w_off;
  double* nrm = base + J.scratch_off;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const double* col[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) col[c] = X + int64_t(min(c0 + c, k - 1)) * J.ldx;
  for (int r0 = lane; r0 < k; r0 += 256) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = r0 + 64 * u;
      const int rr = r < k ? r : k - 1;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const double x = col[c][rr];
        acc[c] += r < k ? x * x : 0.0;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    double a = acc[c];
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off);
    acc[c] = sqrt(a);
    if (lane == 0 && c0 + c < k) nrm[c0 + c] = acc[c];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (c0 + c >= k) break;
    const double v = acc[c];
    double* w = W + int64_t(c0 + c) * J.ldw;
    for (int r = lane; r < k; r += 64) w[r] = v > 1e-300 ? col[c][r] / v : 0.0;
  }
}

template <class L>
__global__ __launch_bounds__(kLargeThreads) void k_gram_vectors(double* __restrict__ base,
                                                                L l) {
  __shared__ double sh[kLargeThreads];
  __shared__ int best, nzero;
  const GramVec J = l.template list<GramVec>()[blockIdx.x];
  const int k = J.k;
  const int tid = threadIdx.x;
  double* W = base + J.w_off;
  double* nrm = base + J.scratch_off;  // k
  double* vec = nrm + k;               // k
  double* hh = vec + k;                // k
  if (tid == 0) nzero = 0;
  __syncthreads();
  int z = 0;
  for (int c = tid; c < k; c += blockDim.x) z += nrm[c] > 1e-300 ? 0 : 1;
  if (z) atomicAdd(&nzero, z);
  __syncthreads();
  if (nzero == 0) return;  // uniform
  for (int c = 0; c < k; ++c) {
    if (nrm[c] > 1e-300) continue;  // uniform
    for (int r = tid; r < k; r += blockDim.x) {
      double q = 1.0;
      for (int j = 0; j < k; ++j) q -= W[int64_t(j) * J.ldw + r] * W[int64_t(j) * J.ldw + r];
      vec[r] = q;
    }
    __syncthreads();
    if (tid == 0) {
      int bi = 0;
      for (int r = 1; r < k; ++r)
        if (vec[r] > vec[bi]) bi = r;
      best = bi;
    }
    __syncthreads();
    const int e0 = best;
    for (int r = tid; r < k; r += blockDim.x) {
      double q = r == e0 ? 1.0 : 0.0;
      for (int j = 0; j < k; ++j) q -= W[int64_t(j) * J.ldw + r] * W[int64_t(j) * J.ldw + e0];
      vec[r] = q;
    }
    __syncthreads();
    for (int j = tid; j < k; j += blockDim.x) {
      double q = 0.0;
      for (int r = 0; r < k; ++r) q += W[int64_t(j) * J.ldw + r] * vec[r];
      hh[j] = q;
    }
    __syncthreads();
    for (int r = tid; r < k; r += blockDim.x) {
      double q = vec[r];
      for (int j = 0; j < k; ++j) q -= W[int64_t(j) * J.ldw + r] * hh[j];
      vec[r] = q;
    }
    __syncthreads();
    double a = 0.0;
    for (int r = tid; r < k; r += blockDim.x) a += vec[r] * vec[r];
    const double n = sqrt(block_sum(a, sh));
    for (int r = tid; r < k; r += blockDim.x) W[int64_t(c) * J.ldw + r] = vec[r] / n;
    if (tid == 0) nrm[c] = n;
    __syncthreads();
  }
}

void gram_vectors(hipStream_t st, double* base, const Lists& descs, int n, int kmax) {
  if (n <= 0 || kmax <= 0) return;
  launch_lists(k_gram_vec_norm<DevLists>, k_gram_vec_norm<ArgLists>, descs, dim3(n, (kmax + 63) / 64), dim3(kLargeThreads),
               0, st, base);
  launch_lists(k_gram_vectors<DevLists>, k_gram_vectors<ArgLists>, descs, dim3(n), dim3(kLargeThreads), 0, st, base);
}

}  // namespace kern
}  // namespace qtt
