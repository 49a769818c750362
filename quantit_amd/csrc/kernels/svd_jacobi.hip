// Batched FP64 block SVD for gfx950: block one-sided (Hestenes) Jacobi.
//
// Each sector matrix is held as Y (ell x kp, column-major) with
// ell = max(m,n) rows and kp >= min(m,n) columns (zero padded to a multiple of
// 2*kSvdBlock); W (kp x kp) accumulates the right rotations (Y W = Z with
// mutually orthogonal columns).  One launch = one round of the round-robin
// tournament over column blocks of kSvdBlock columns: every work-group takes
// a disjoint block pair (p, q) of one sector and
//   1. forms the 32x32 Gram matrix G = [Y_p Y_q]^T [Y_p Y_q] with
//      v_mfma_f64_16x16x4_f64 (Y staged through LDS in 64-row chunks),
//   2. returns if every column pair is orthogonal to the tolerance
//      (|G_ij| <= tol sqrt(G_ii G_jj)),
//   3. diagonalises G with a cyclic two-sided Jacobi in LDS (16 disjoint
//      rotations per step, circle ordering) accumulating Q,
//   4. applies Y_pq <- Y_pq Q and W_pq <- W_pq Q with MFMA.
// The singular values are the final column norms of Y (computed from the
// columns, so the small ones keep absolute accuracy eps*||A||), which matches
// the accuracy class of LAPACK gesdd used by the reference
// (sources/btensor_linalg.cpp:483).
#include <algorithm>
#include <cfloat>
#include <climits>
#include <stdexcept>

#include "../kernels.hpp"

namespace qtt {
namespace kern {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int NB2 = 2 * kSvdBlock;  // 32 columns per work-group
constexpr int YC = 128;             // rows of Y staged per chunk
constexpr int YP = YC + 2;          // LDS pitch of the staged Y chunk
constexpr int GP = NB2 + 1;         // LDS pitch of G and Q

// Y and its partner zero, W and its partner the identity, for every sector;
// gridDim.y work-groups share a sector.
template <class L>
__global__ __launch_bounds__(256) void k_svd_prepare(double* __restrict__ base, L l) {
  const SvdPrep s = l.template list<SvdPrep>()[blockIdx.x];
  const int t0 = blockIdx.y * blockDim.x + threadIdx.x, step = gridDim.y * blockDim.x;
  const int64_t ny = int64_t(s.ell) * s.kp;
  for (int64_t e = t0; e < ny; e += step) {
    base[s.y_off + e] = 0.0;
    if (s.y2_off >= 0) base[s.y2_off + e] = 0.0;
  }
  const uint32_t kp = s.kp, nw = kp * kp;  // k is far below 2^16
  for (uint32_t e = t0; e < nw; e += step) {
    const double v = e % (kp + 1) == 0 ? 1.0 : 0.0;
    base[s.w_off + e] = v;
    if (s.w2_off >= 0) base[s.w2_off + e] = v;
  }
}

void svd_prepare(hipStream_t st, double* base, const Lists& secs, int nsec, int64_t max_elems) {
  if (nsec <= 0) return;
  const int ny = int(std::min<int64_t>(std::max<int64_t>(max_elems / 2048, 4), 128));  // about 8 elements a thread
  launch_lists(k_svd_prepare<DevLists>, k_svd_prepare<ArgLists>, secs, dim3(nsec, ny), dim3(256), 0, st, base);
}

__device__ __forceinline__ int circle_block(int pos, int round, int nb) {
  return pos == 0 ? 0 : 1 + ((pos - 1 + round) % (nb - 1));
}

// Reciprocal square root and reciprocal: the hardware estimates (relative error
// up to 2^-24 measured) and one third-order step, 2^-72 before rounding and a
// shorter chain than two Newton steps; the division and square root the
// compiler expands to correctly rounded sequences take several times longer.
__device__ __forceinline__ double fast_rsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}
__device__ __forceinline__ double fast_rcp(double x) {
  const double z = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, z, 1.0);
  return fma(z, fma(e, e, e), z);
}

// Jacobi rotation (c, s) annihilating the off-diagonal h/2 of the symmetric
// 2x2 [[a, h/2], [h/2, b]] with |angle| <= pi/4, from d = b - a:
// t = sign(d) h / (|d| + sqrt(d^2 + h^2)), c = 1/sqrt(1 + t^2), s = c t.
__device__ __forceinline__ void jacobi_cs(double d, double h, double& c, double& sn) {
  const double q2 = d * d + h * h;
  const double r = q2 * fast_rsqrt(q2);
  const double t = (d >= 0.0 ? h : -h) * fast_rcp(fabs(d) + r);
  c = fast_rsqrt(1.0 + t * t);
  sn = c * t;
}

// lane i of each 16-lane row <- lane (i + 1) mod 16 (DPP row rotate right by
// 15), on a double as two 32-bit moves.
__device__ __forceinline__ double dpp_row_next(double v) {
  const long long b = __double_as_longlong(v);
  int lo = int(b & 0xffffffffLL), hi = int(b >> 32);
  lo = __builtin_amdgcn_mov_dpp(lo, 0x12F, 0xF, 0xF, false);
  hi = __builtin_amdgcn_mov_dpp(hi, 0x12F, 0xF, 0xF, false);
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}

// Apply the 32x32 rotation Q (LDS, pitch GP) to the 32 selected columns of a
// column-major matrix M (rows x ld) in place, YC rows at a time (each wave
// owns two 16-row MFMA tiles of a chunk).
__device__ void apply_rotation(double* __restrict__ M, int64_t ld, int rows, const int* cols,
                               double (*Ys)[YP], const double (*Q)[GP]) {
  constexpr int PER = YC / 8;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool act = tid < 256;  // the first four waves work, every thread meets the barriers
  const int c = act ? tid >> 3 : 0, lq = (tid & 7) * PER;
  const double* src = M + int64_t(cols[c]) * ld;
  double buf[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) buf[i] = (act && lq + i < rows) ? src[lq + i] : 0.0;
  for (int l0 = 0; l0 < rows; l0 += YC) {
    if (act) {
#pragma unroll
      for (int i = 0; i < PER; ++i) Ys[c][lq + i] = buf[i];
    }
    __syncthreads();
    if (act && l0 + YC < rows) {
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int l = l0 + YC + lq + i;
        buf[i] = (l < rows) ? src[l] : 0.0;
      }
    }
    v4d acc[2][2] = {{v4d{0.0, 0.0, 0.0, 0.0}, v4d{0.0, 0.0, 0.0, 0.0}},
                     {v4d{0.0, 0.0, 0.0, 0.0}, v4d{0.0, 0.0, 0.0, 0.0}}};
#pragma unroll
    for (int kk = 0; kk < NB2 && act; kk += 4) {
      const int kr = kk + (lane >> 4), cl = lane & 15;
      const double a0 = Ys[kr][wave * 32 + cl], a1 = Ys[kr][wave * 32 + 16 + cl];
      const double b0 = Q[kr][cl], b1 = Q[kr][16 + cl];
      acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
    __syncthreads();  // every wave has read its Ys rows before they are overwritten
    if (!act) continue;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = l0 + wave * 32 + rt * 16 + 4 * r + (lane >> 4);  // f64 MFMA output layout
          const int col = jt * 16 + (lane & 15);
          if (row < rows) M[int64_t(cols[col]) * ld + row] = acc[rt][jt][r];
        }
  }
}

// RESIDENT: the block pair's ell x 32 columns are loaded into dynamic LDS
// once (ell <= the LDS capacity), the Gram matrix and the rotated columns are
// computed from there and written back once; otherwise 128-row chunks are
// staged twice (Gram, then rotation).
template <bool RESIDENT>
__global__ __launch_bounds__(RESIDENT ? 1024 : 256) void k_svd_round(double* __restrict__ base,
                                                   const RoundWork* __restrict__ work, int round,
                                                   int* __restrict__ counters, const int* __restrict__ skip,
                                                   double tol, int inner_sweeps, int pitch, int cross_after0) {
  extern __shared__ double dyn[];
  __shared__ double G[1][NB2][GP];
  __shared__ double Q[1][NB2][GP];
  __shared__ int cols[NB2];
  __shared__ int flag, nrot;
  double (*Ys)[YP] = reinterpret_cast<double (*)[YP]>(dyn);  // chunk staging (aliases the resident block)

  const RoundWork s = work[blockIdx.x];
  const int pi = s.pair;
  const int nb = s.nb;
  if (round >= nb - 1) return;
  // a sector whose previous sweep rotated nothing has converged
  if (skip && skip[s.flag_idx] == 0) return;
  const int p = circle_block(pi, round, nb);
  const int q = circle_block(nb - 1 - pi, round, nb);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid < NB2) cols[tid] = tid < kSvdBlock ? p * kSvdBlock + tid : q * kSvdBlock + (tid - kSvdBlock);
  if (tid == 0) flag = 0;
  __syncthreads();

  double* Y = base + s.y_off;
  const int64_t ld = s.ell;
  const int ell = s.ell;
  // ---- 1. Gram matrix ------------------------------------------------------
  const int wi = wave >> 1, wj = wave & 1;
  v4d g = v4d{0.0, 0.0, 0.0, 0.0};
  if (RESIDENT) {
    // all 32 columns at once: 32 lanes per column take rows (tid & 31) + 32u,
    // up to 36 loads per thread in flight (one pass for the resident sizes)
    double* Yl = dyn;  // Yl[c * pitch + r]
    {
      constexpr int CH = 36;
      const int c = tid >> 5, part = tid & 31;
      const double* src = Y + int64_t(cols[c]) * ld;
      double* dst = Yl + c * pitch;
      for (int o = 0; o < ell; o += 32 * CH) {
        double v[CH];
        // 32-row slices wholly past ell are skipped (a uniform branch): their
        // clamped loads would only occupy the address units
#pragma unroll
        for (int u = 0; u < CH; ++u) {
          const int r = o + part + 32 * u;
          v[u] = 0.0;
          if (o + 32 * u < ell) v[u] = src[r < ell ? r : ell - 1];
        }
#pragma unroll
        for (int u = 0; u < CH; ++u) {
          const int r = o + part + 32 * u;
          if (r < ell) dst[r] = v[u];
        }
      }
    }
    __syncthreads();
    // G is symmetric: the three distinct 16x16 tiles (0,0), (0,1), (1,1),
    // five waves each on the 4-row slices 4 part + 20 t (two accumulation
    // chains); the fifths are summed into G in a fixed order below and the
    // (0,1) tile is mirrored into (1,0).  Wave 15 only meets the barriers.
    const int cl = lane & 15, kq = lane >> 4;
    constexpr int kParts = 5;
    const bool gw = wave < 3 * kParts;
    const int tile = gw ? wave % 3 : 0, part = gw ? wave / 3 : kParts;
    const int ti = tile == 2 ? 1 : 0, tj = tile == 0 ? 0 : 1;
    const double* ya = Yl + (ti * 16 + cl) * pitch + kq;
    const double* yb = Yl + (tj * 16 + cl) * pitch + kq;
    v4d g1 = v4d{0.0, 0.0, 0.0, 0.0};
    if (gw && ti == tj) {  // diagonal tile: both operands are the same columns
      int kk = 4 * part;
      for (; kk + 4 * kParts < ell; kk += 8 * kParts) {
        const bool in1 = kk + 4 * kParts + kq < ell;
        const double a0 = ya[kk];
        const double a1 = in1 ? ya[kk + 4 * kParts] : 0.0;
        g = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, a0, g, 0, 0, 0);
        g1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, a1, g1, 0, 0, 0);
      }
      for (; kk < ell; kk += 4 * kParts) {
        const double xa = kk + kq < ell ? ya[kk] : 0.0;
        g = __builtin_amdgcn_mfma_f64_16x16x4f64(xa, xa, g, 0, 0, 0);
      }
      g = g + g1;
    } else if (gw) {
      int kk = 4 * part;
      for (; kk + 4 * kParts < ell; kk += 8 * kParts) {
        const bool in1 = kk + 4 * kParts + kq < ell;
        const double a0 = ya[kk], b0 = yb[kk];
        const double a1 = ya[in1 ? kk + 4 * kParts : 0], b1 = yb[in1 ? kk + 4 * kParts : 0];
        g = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, g, 0, 0, 0);
        g1 = __builtin_amdgcn_mfma_f64_16x16x4f64(in1 ? a1 : 0.0, in1 ? b1 : 0.0, g1, 0, 0, 0);
      }
      for (; kk < ell; kk += 4 * kParts) {
        const bool in = kk + kq < ell;
        const double xa = ya[in ? kk : 0], xb = yb[in ? kk : 0];
        g = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? xa : 0.0, in ? xb : 0.0, g, 0, 0, 0);
      }
      g = g + g1;
    }
#pragma unroll
    for (int qq = 0; qq < kParts; ++qq) {
      if (part == qq) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int gi = ti * 16 + 4 * r + (lane >> 4), gj = tj * 16 + (lane & 15);
          double& dst = G[0][gi][gj];
          const double v = qq == 0 ? g[r] : dst + g[r];
          dst = v;
          if (tile == 1) G[0][gj][gi] = v;
        }
      }
      __syncthreads();
    }
  } else {
    // YC-row chunks staged through LDS; the next chunk's global loads are
    // issued before the MFMAs of the current one
    constexpr int PER = YC / 8;
    const int c = tid >> 3, lq = (tid & 7) * PER;
    const double* src = Y + int64_t(cols[c]) * ld;
    double buf[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) buf[i] = (lq + i < ell) ? src[lq + i] : 0.0;
    for (int l0 = 0; l0 < ell; l0 += YC) {
#pragma unroll
      for (int i = 0; i < PER; ++i) Ys[c][lq + i] = buf[i];
      __syncthreads();
      if (l0 + YC < ell) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const int l = l0 + YC + lq + i;
          buf[i] = (l < ell) ? src[l] : 0.0;
        }
      }
#pragma unroll
      for (int kk = 0; kk < YC; kk += 4) {
        const int kr = kk + (lane >> 4), cl = lane & 15;
        g = __builtin_amdgcn_mfma_f64_16x16x4f64(Ys[wi * 16 + cl][kr], Ys[wj * 16 + cl][kr], g, 0, 0, 0);
      }
      __syncthreads();
    }
  }
  if (!RESIDENT) {  // the resident path has summed its quarters into G already
#pragma unroll
    for (int r = 0; r < 4; ++r) G[0][wi * 16 + 4 * r + (lane >> 4)][wj * 16 + (lane & 15)] = g[r];
  }
  __syncthreads();
  // ---- 2. convergence test ---------------------------------------------------
  for (int e = tid; e < NB2 * NB2; e += blockDim.x) {
    const int i = e / NB2, j = e % NB2;
    if (i < j) {
      const double gii = G[0][i][i], gjj = G[0][j][j], gij = G[0][i][j];
      if (gii > 0.0 && gjj > 0.0 && gij * gij > (tol * gii) * (tol * gjj)) flag = 1;
    }
  }
  __syncthreads();
  if (flag == 0) return;
  if (tid == 0) atomicAdd(&counters[s.flag_idx], 1);
  // ---- 3. eigen-decomposition of G by cyclic two-sided Jacobi -----------------
  // Thread (P, R) owns the 2x2 block of G at the row pair P and column pair R
  // of the round (circle ordering, 16 disjoint pairs): it computes both
  // pairs' rotations from the diagonal blocks, then applies J_P^T (rows) and
  // J_R (columns) to its block and J_R to the same rows of Q, in place.  The
  // 256 blocks tile G and Q, so one round is two barriers and no other LDS
  // traffic.
  for (int e = tid; e < NB2 * NB2; e += blockDim.x) {
    const int i = e / NB2, j = e % NB2;
    Q[0][i][j] = (i == j) ? 1.0 : 0.0;
  }
  __syncthreads();
  {
    // Step r: the 16 threads tid < 16 compute the rotations of the 16 pairs
    // (one each) into rc/rs; after a barrier thread (P, R) applies J_P^T
    // (rows) and J_R (columns) to its 2x2 block of G and J_R to the same rows
    // of Q, in place.  The 256 blocks tile G and Q, so a step is two barriers
    // and no chain of dependent LDS accesses beyond the diagonal reads.
    // With cross_after0, rounds after the first of a sweep take only the 256
    // pairs across the two blocks (pairs (i, 16 + (i + r) mod 16), 16
    // steps): the first round of every sweep holds each block once and takes
    // all 496 pairs, so a sweep still meets every column pair.
    __shared__ double rc[NB2 / 2], rs[NB2 / 2];
    const bool blk = tid < NB2 * NB2 / 4;  // 256 threads own the 2x2 blocks; the rest meet the barriers
    const int P = blk ? tid >> 4 : 0, R = tid & 15;
    const bool cross = cross_after0 && round > 0;
    const int nsteps = cross ? NB2 / 2 : NB2 - 1;
    auto pair_of = [&](int i, int r, int& x, int& y) {
      if (cross) {
        x = i;
        y = NB2 / 2 + ((i + r) & (NB2 / 2 - 1));
      } else {
        const int x0 = circle_block(i, r, NB2), x1 = circle_block(NB2 - 1 - i, r, NB2);
        x = min(x0, x1);
        y = max(x0, x1);
      }
    };
    if (cross && inner_sweeps == 1) {
      // The same cross sweep with G and Q held in registers.  Thread (P, R)
      // keeps g00 = G[P][R], g01 = G[P][b2], g10 = G[a2][R], g11 = G[a2][b2]
      // and Q's (P, R), (P, b2), (P+16, R), (P+16, b2), where a2 = 16 +
      // (P + r) mod 16 and b2 = 16 + (R + r) mod 16 move with the step r:
      // the diagonal owner (P == R) holds pair P's 2x2 block and computes
      // its rotation; after the update the moving columns come from lane
      // R + 1 of the same 16-lane row (DPP row rotate) and the moving rows
      // from thread P + 1 through LDS (G's area, which is dead from here
      // on).  After 16 steps every value is back at its first position.
      double (*s10)[NB2 / 2 + 1] = reinterpret_cast<double (*)[NB2 / 2 + 1]>(&G[0][0][0]);
      double (*s11)[NB2 / 2 + 1] = s10 + NB2 / 2;
      double g00 = 0.0, g01 = 0.0, g10 = 0.0, g11 = 0.0, qa0 = 0.0, qa1 = 0.0, qb0 = 0.0, qb1 = 0.0;
      constexpr int H = NB2 / 2;
      if (blk) {
        g00 = G[0][P][R];
        g01 = G[0][P][H + R];
        g10 = G[0][H + P][R];
        g11 = G[0][H + P][H + R];
        qa0 = Q[0][P][R];
        qa1 = Q[0][P][H + R];
        qb0 = Q[0][H + P][R];
        qb1 = Q[0][H + P][H + R];
      }
      __syncthreads();  // every read of G precedes the exchange writes into its area
      for (int r = 0; r < H; ++r) {
        if (blk && P == R) {
          const double app = g00, aqq = g11, apq = g01;
          const bool rot = app > 0.0 && aqq > 0.0 && apq * apq > (DBL_EPSILON * app) * (DBL_EPSILON * aqq);
          double cc, ss;
          jacobi_cs(aqq - app, 2.0 * apq, cc, ss);
          rc[P] = rot ? cc : 1.0;
          rs[P] = rot ? ss : 0.0;
        }
        __syncthreads();  // rotations published
        if (blk) {
          const double cp = rc[P], sp = rs[P], cq = rc[R], sq = rs[R];
          const double h00 = cp * g00 - sp * g10, h01 = cp * g01 - sp * g11;
          const double h10 = cp * g10 + sp * g00, h11 = cp * g11 + sp * g01;
          g00 = cq * h00 - sq * h01;
          g01 = cq * h01 + sq * h00;
          g10 = cq * h10 - sq * h11;
          g11 = cq * h11 + sq * h10;
          const double na1 = cq * qa1 + sq * qa0, nb1 = cq * qb1 + sq * qb0;
          qa0 = cq * qa0 - sq * qa1;
          qb0 = cq * qb0 - sq * qb1;
          g01 = dpp_row_next(g01);
          g11 = dpp_row_next(g11);
          qa1 = dpp_row_next(na1);
          qb1 = dpp_row_next(nb1);
          s10[P][R] = g10;
          s11[P][R] = g11;
        }
        __syncthreads();  // moving rows published; the next step's rotations wait for these reads
        if (blk) {
          g10 = s10[(P + 1) & (H - 1)][R];
          g11 = s11[(P + 1) & (H - 1)][R];
        }
      }
      __syncthreads();
      if (blk) {
        Q[0][P][R] = qa0;
        Q[0][P][H + R] = qa1;
        Q[0][H + P][R] = qb0;
        Q[0][H + P][H + R] = qb1;
      }
      __syncthreads();
    } else
    for (int sweep = 0; sweep < inner_sweeps; ++sweep) {
      if (tid == 0) nrot = 0;
      __syncthreads();
      for (int r = 0; r < nsteps; ++r) {
        int a, a2, b, b2;
        pair_of(P, r, a, a2);
        pair_of(R, r, b, b2);
        // The block owners issue their reads first, so that their latency
        // runs under the rotations below (only the owners read: the other
        // waves would multiply the LDS traffic).
        double g00 = 0.0, g01 = 0.0, g10 = 0.0, g11 = 0.0, q00 = 0.0, q01 = 0.0, q10 = 0.0, q11 = 0.0;
        if (blk) {
          g00 = G[0][a][b];
          g01 = G[0][a][b2];
          g10 = G[0][a2][b];
          g11 = G[0][a2][b2];
          q00 = Q[0][a][b];
          q01 = Q[0][a][b2];
          q10 = Q[0][a2][b];
          q11 = Q[0][a2][b2];
        }
        if (tid < NB2 / 2) {
          int x, y;
          pair_of(tid, r, x, y);
          const double app = G[0][x][x], aqq = G[0][y][y], apq = G[0][x][y];
          // computed unconditionally and selected, so that the chain has no
          // branch (an unselected result may be NaN, e.g. for a zero column)
          const bool rot = app > 0.0 && aqq > 0.0 && apq * apq > (DBL_EPSILON * app) * (DBL_EPSILON * aqq);
          double cc, ss;
          jacobi_cs(aqq - app, 2.0 * apq, cc, ss);
          rc[tid] = rot ? cc : 1.0;
          rs[tid] = rot ? ss : 0.0;
          if (rot) nrot = 1;  // a flag: every writer stores the same value
        }
        __syncthreads();  // rotations published; every read of this step precedes the writes
        if (blk) {
          const double cp = rc[P], sp = rs[P], cq = rc[R], sq = rs[R];
          // rows a, a2 by J_P^T; columns b, b2 by J_R (row' a = c a - s a2, row' a2 = c a2 + s a)
          const double h00 = cp * g00 - sp * g10, h01 = cp * g01 - sp * g11;
          const double h10 = cp * g10 + sp * g00, h11 = cp * g11 + sp * g01;
          G[0][a][b] = cq * h00 - sq * h01;
          G[0][a][b2] = cq * h01 + sq * h00;
          G[0][a2][b] = cq * h10 - sq * h11;
          G[0][a2][b2] = cq * h11 + sq * h10;
          Q[0][a][b] = cq * q00 - sq * q01;
          Q[0][a][b2] = cq * q01 + sq * q00;
          Q[0][a2][b] = cq * q10 - sq * q11;
          Q[0][a2][b2] = cq * q11 + sq * q10;
        }
        __syncthreads();
      }
      if (nrot == 0) break;
      __syncthreads();
    }
  }
  const int cur = 0;
  // ---- 4. rotate the columns of Y and W ---------------------------------------
  if (RESIDENT) {
    // (Y Q)^T = Q^T Y^T tile by tile: the MFMA output then holds 16
    // consecutive rows of one column per 16 lanes, so the stores coalesce
    const double* Yl = dyn;
    const int nw = blockDim.x >> 6;
    for (int l0 = 0; l0 < ell; l0 += nw * 32) {
      v4d acc[2][2] = {{v4d{0.0, 0.0, 0.0, 0.0}, v4d{0.0, 0.0, 0.0, 0.0}},
                       {v4d{0.0, 0.0, 0.0, 0.0}, v4d{0.0, 0.0, 0.0, 0.0}}};
      const int cl = lane & 15;
      const int r0 = l0 + wave * 32 + cl, r1 = r0 + 16;
#pragma unroll
      for (int kk = 0; kk < NB2; kk += 4) {
        const int kr = kk + (lane >> 4);
        const double a0 = r0 < ell ? Yl[kr * pitch + r0] : 0.0;
        const double a1 = r1 < ell ? Yl[kr * pitch + r1] : 0.0;
        const double b0 = Q[cur][kr][cl], b1 = Q[cur][kr][16 + cl];
        acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(b0, a0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(b1, a0, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(b0, a1, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(b1, a1, acc[1][1], 0, 0, 0);
      }
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int jt = 0; jt < 2; ++jt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = (rt ? r1 : r0);
            const int col = jt * 16 + 4 * r + (lane >> 4);  // f64 MFMA output layout, transposed tile
            if (row < ell) Y[int64_t(cols[col]) * ld + row] = acc[rt][jt][r];
          }
    }
  } else {
    apply_rotation(Y, ld, ell, cols, Ys, Q[cur]);
  }
  __syncthreads();  // the staging area below aliases the resident block
  const int kp = nb * kSvdBlock;
  apply_rotation(base + s.w_off, kp, kp, cols, Ys, Q[cur]);
}

// Rows of a block pair that stay resident in LDS (dynamic size at most the
// device's per-block LDS less the static arrays).
// (Thread-safe static initialisation: concurrent solves on several host
// threads see the limit only after the attribute has been set.)
int svd_round_dyn_max() {
  static const int dyn_max = [] {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) v = 65536;
    const int m = v - int(2 * NB2 * GP * sizeof(double)) - 1024;
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_svd_round<true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, m);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_svd_round<false>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, m);
    return m;
  }();
  return dyn_max;
}

// LDS pitch (doubles) of a resident column: at least ell and 2 (mod 32), so
// that a 32-lane phase of the Gram's reads (16 columns x 2 rows) meets each
// of the 64 banks once.
int resident_pitch(int ell) { return (ell + 29) / 32 * 32 + 2; }

void svd_round(hipStream_t st, double* base, const RoundWork* work, int nwork, int round, int* counters,
               const int* skip, double tol, int inner_sweeps, int max_ell, int cross_after0) {
  if (nwork <= 0) return;
  const size_t staging = size_t(NB2) * YP * sizeof(double);
  const int pitch = resident_pitch(max_ell);
  if (int64_t(pitch) * NB2 * int64_t(sizeof(double)) <= svd_round_dyn_max()) {
    const size_t lds = std::max(size_t(NB2) * pitch * sizeof(double), staging);
    hipLaunchKernelGGL(k_svd_round<true>, dim3(nwork), dim3(1024), lds, st, base, work, round, counters, skip, tol,
                       inner_sweeps, pitch, cross_after0);
  } else {
    hipLaunchKernelGGL(k_svd_round<false>, dim3(nwork), dim3(256), staging, st, base, work, round, counters, skip,
                       tol, inner_sweeps, 0, cross_after0);
  }
}

// Block-wide reductions (fixed order, deterministic).
__device__ double wg_sum(double v, double* sh) {
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

// ---- eigenvectors of a Gram matrix by one-sided Jacobi without accumulation --
// One work-group per k x k Gram matrix G (k <= kGramEigMaxK) held in LDS.
//
// 1. Test: a pair (i, j) of the columns behind G is converged when
//    |g_ij| <= tol sqrt(g_ii g_jj) (relative orthogonality) or
//    |g_ij| <= tol sqrt(max(g_ii, g_jj)) sqrt(max_l g_ll) (its coupling moves
//    the larger column's share of the smaller one by at most tol times the
//    largest singular value: absolute accuracy, the class of LAPACK gesdd).
//    flags[flag_idx] = pairs failing both; flags[J.aux_idx] (when >= 0) = pairs
//    converged only in the absolute sense.  No failing pair: W = I exactly.
// 2. Preconditioning (precond != 0): pivoted Cholesky P^T G P = R^T R in
//    place (diagonal pivoting; from a non-positive pivot on, the factor of a
//    diagonal below G's rounding), X = R^T.  This
//    is the QR-with-pivoting preconditioner of Drmac and Veselic (SIAM J.
//    Matrix Anal. Appl. 29, 2008) applied through G: on graded spectra the
//    Jacobi below then needs a few sweeps instead of tens.  Without it X = G.
// 3. One-sided Jacobi drives X W to mutually orthogonal columns.  Since
//    X X^T = P^T G P (or G^2), the normalised columns of the result are the
//    eigenvectors of P^T G P and no rotation is accumulated.  Rotations are
//    made down to tol/16, so the columns end orthonormal well inside tol
//    whatever the accuracy of the small eigenpairs; zero columns are
//    completed from the unit vector with the largest residual (two
//    projection passes).
// 4. W is written with the rows un-permuted (W = P Q).
// Sum over aligned groups of g lanes (g a power of two <= 16) with DPP moves:
// xor 1 and xor 2 by quad permutes, then the 8- and 16-lane mirrors (after
// the previous steps every lane of a half holds the same partial sum, so the
// mirror partner holds the other half's).
__device__ __forceinline__ double dpp_bits(double v, int ctrl_id) {
  const long long b = __double_as_longlong(v);
  int lo = int(b & 0xffffffffLL), hi = int(b >> 32);
  switch (ctrl_id) {
    case 0:
      lo = __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xF, 0xF, false);
      hi = __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xF, 0xF, false);
      break;
    case 1:
      lo = __builtin_amdgcn_mov_dpp(lo, 0x4E, 0xF, 0xF, false);
      hi = __builtin_amdgcn_mov_dpp(hi, 0x4E, 0xF, 0xF, false);
      break;
    case 2:
      lo = __builtin_amdgcn_mov_dpp(lo, 0x141, 0xF, 0xF, false);
      hi = __builtin_amdgcn_mov_dpp(hi, 0x141, 0xF, 0xF, false);
      break;
    default:
      lo = __builtin_amdgcn_mov_dpp(lo, 0x140, 0xF, 0xF, false);
      hi = __builtin_amdgcn_mov_dpp(hi, 0x140, 0xF, 0xF, false);
      break;
  }
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}

__device__ __forceinline__ void group_sum3(double& a, double& b, double& c, int g) {
  if (g > 16) {
    for (int off = g >> 1; off > 0; off >>= 1) {
      a += __shfl_xor(a, off, g);
      b += __shfl_xor(b, off, g);
      c += __shfl_xor(c, off, g);
    }
    return;
  }
  for (int st = 0; (2 << st) <= g; ++st) {
    const double ta = dpp_bits(a, st), tb = dpp_bits(b, st), tc = dpp_bits(c, st);
    a += ta;
    b += tb;
    c += tc;
  }
}

// Lanes per column pair: enough for about 16 rows per lane, at most what the
// block holds for all pairs.
__host__ __device__ inline int gram_eig_gsz(int k, int threads) {
  const int npairs = (k + (k & 1)) / 2;
  int g = 1;
  while (g < 16 && g * 16 < k) g <<= 1;
  while (g > 1 && g * npairs > threads) g >>= 1;
  return g;
}


// ---- wave-local block Jacobi ---------------------------------------------------
// The columns of X form NB = 2*ceil(k/16) blocks of 8 (columns >= k are zero
// and never stored).  A work-group round pairs the blocks by the circle
// ordering, one block pair (P, Q) per wave.  Inside the wave, 8-lane group g
// keeps column g of P and column g of Q in registers (rows li + 8j), so the 64
// column pairs across P and Q take 8 steps with no barrier: between steps the
// Q columns move between groups by a lane xor (group offsets in Gray-code
// order 0,1,3,2,6,7,5,4, so every group meets every Q column once).  The first
// round of a sweep also takes the 28 pairs inside each block, by xor pairing
// of the groups (both groups of a pair compute the same rotation from the same
// sums and update their own column).  One barrier per round instead of one per
// column pair, and the columns cross LDS once per round.  Each lane keeps R
// rows of a column, R the smallest even count with 8 R >= k.
// Nine waves: one per block pair at k = 144 (18 blocks), and at most three
// waves per SIMD, so each keeps two 18-row columns and the shifted copy in
// registers without spilling.
constexpr int kGramEigThreads = 576;
static_assert(kGramEigMaxK <= 8 * 18, "the widest wave-local variant holds 18 rows per lane");

__device__ __forceinline__ double dpp_ror8(double v) {  // lane i <- lane i ^ 8 within 16-lane rows
  const long long b = __double_as_longlong(v);
  int lo = int(b & 0xffffffffLL), hi = int(b >> 32);
  lo = __builtin_amdgcn_mov_dpp(lo, 0x128, 0xF, 0xF, false);
  hi = __builtin_amdgcn_mov_dpp(hi, 0x128, 0xF, 0xF, false);
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}

// Lane permutations without index registers where the hardware allows: xor 8
// by a DPP row rotation, xor 16 by ds_swizzle (bit-mask mode), xor 32 by
// ds_bpermute.  The vector unit's row swaps (v_permlane16_swap and 32) take
// five instructions a word against one: the steps below are bound by issue.
__device__ __forceinline__ int xor16(int v) { return __builtin_amdgcn_ds_swizzle(v, 0x401F); }
__device__ __forceinline__ double xor16(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = xor16(int(b & 0xffffffffLL)), hi = xor16(int(b >> 32));
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}
__device__ __forceinline__ int xor32(int v) { return __shfl_xor(v, 32); }
__device__ __forceinline__ double xor32(double v) { return __shfl_xor(v, 32); }

__device__ __forceinline__ void sum8(double& a) {
#pragma unroll
  for (int st = 0; st < 3; ++st) a += dpp_bits(a, st);
}

// A column in registers: true column = d * v (rows li + 8j), n = its squared
// norm.  Short columns (R <= 8) keep d = 1 and rotate both by c and s, 4 R
// operations; longer ones rotate in the scaled form, two FMAs per row (x' = x -
// t r y with r a ratio of scales) with the cosine folded into d.  n follows the
// exact identities |x'|^2 = |x|^2 - t x.y, |y'|^2 = |y|^2 + t x.y and is
// recomputed from the rows when it falls below a quarter of its value
// (cancellation).  The scales start at 1 when a column is loaded, so with at
// most 15 rotations between a load and a store they stay above 0.7^15.
template <int R>
struct WlCol {
  static constexpr bool kScaled = R > 8;
  double v[R];
  double d, n;
};

template <int R>
__device__ __forceinline__ double wl_norm(const WlCol<R>& x) {
  double s = 0.0;
#pragma unroll
  for (int j = 0; j < R; ++j) s += x.v[j] * x.v[j];
  sum8(s);
  return WlCol<R>::kScaled ? s * x.d * x.d : s;
}

// Column c of X (pitch k) into rows li + 8j.  Rows past k read the next
// column (or, for the last one, the arrays that follow X in LDS) and are
// masked; columns past k are zero.  One base address per column keeps the
// loads on immediate offsets.
template <int R>
__device__ __forceinline__ void wl_load(const double* X, int k, int c, int li, WlCol<R>& x) {
  const bool cin = c < k;
  const double* col = X + (cin ? c * k : 0) + li;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const double v = col[8 * j];
    x.v[j] = (cin && li + 8 * j < k) ? v : 0.0;
  }
  x.d = 1.0;
  x.n = wl_norm<R>(x);
}

template <int R>
__device__ __forceinline__ void wl_store(double* X, int k, int c, int li, const WlCol<R>& x) {
  if (c >= k) return;
  double* col = X + c * k + li;
#pragma unroll
  for (int j = 0; j < R; ++j)
    if (li + 8 * j < k) col[8 * j] = WlCol<R>::kScaled ? x.v[j] * x.d : x.v[j];
}

// The rotation of a column pair (x, y) from its squared norms and product:
// x' = c (x - t y), y' = c (y + t x) with c = 1 / sqrt(1 + t^2).  It is
// orthogonal for any t, so t comes from the bare estimates (2^-23 of the
// coupling is left, well below tol_rot once couplings are small); c is exact.
// big: the rotation could leave couplings over tol_rot, see wl_sweeps (t^2
// (xx^2 + yy^2) / (xx yy) bounds the tangent times the ratio of the lengths).
constexpr double kWlSmall = 1e-9;
struct WlRot {
  double t, c;
  bool big;
};
__device__ __forceinline__ WlRot wl_rotation(double xx, double yy, double xx_yy, double xy, double xy2) {
  WlRot r;
  const double d = yy - xx, h = xy + xy;
  const double q2 = fma(d, d, 4.0 * xy2);
  const double den = fma(q2, __builtin_amdgcn_rsq(q2), fabs(d));
  r.t = h * copysign(__builtin_amdgcn_rcp(den), d);
  const double t2 = r.t * r.t, lim = (kWlSmall * kWlSmall) * xx_yy;
  r.c = fast_rsqrt(1.0 + t2);
  r.big = (xy2 > lim) | (t2 * fma(2.0, xx_yy, q2) > lim);
  return r;
}

template <int R>
__device__ __forceinline__ double wl_dot(const double* x, const double* y) {
  double r0 = 0.0, r1 = 0.0;
#pragma unroll
  for (int j = 0; j < R; j += 2) {
    r0 = fma(x[j], y[j], r0);
    r1 = fma(x[j + 1], y[j + 1], r1);
  }
  r0 += r1;
  sum8(r0);
  return r0;
}

// x from the lanes of group (own group) ^ m, m uniform.
template <int R>
__device__ __forceinline__ void wl_xor(WlCol<R>& x, int m) {
  if (m & 1) {
#pragma unroll
    for (int j = 0; j < R; ++j) x.v[j] = dpp_ror8(x.v[j]);
    if constexpr (WlCol<R>::kScaled) x.d = dpp_ror8(x.d);
    x.n = dpp_ror8(x.n);
  }
  if (m & 2) {
#pragma unroll
    for (int j = 0; j < R; ++j) x.v[j] = xor16(x.v[j]);
    if constexpr (WlCol<R>::kScaled) x.d = xor16(x.d);
    x.n = xor16(x.n);
  }
  if (m & 4) {
#pragma unroll
    for (int j = 0; j < R; ++j) x.v[j] = xor32(x.v[j]);
    if constexpr (WlCol<R>::kScaled) x.d = xor32(x.d);
    x.n = xor32(x.n);
  }
}

// Squared norms after a rotation (an, bn by the identities), recomputed from
// the rows on cancellation.
template <int R>
__device__ __forceinline__ void wl_norms(WlCol<R>& a, WlCol<R>& b, double an, double bn) {
  const bool lost = (an < 0.25 * a.n) | (bn < 0.25 * b.n);
  a.n = an;
  b.n = bn;
  if (lost) {  // uniform in the group
    a.n = wl_norm<R>(a);
    b.n = wl_norm<R>(b);
  }
}

// Pairs (g, g ^ m) inside one block: x is the lower group's column.  Both
// groups form the same sums (the products commute and the reduction order is
// the same), so they compute the same rotation and each updates its own
// column.  Without a branch, so that the chains of two blocks interleave.
template <int R>
__device__ __forceinline__ void wl_intra(WlCol<R>& x, int m, int grp, double tol2, int& big) {
  const bool lower = grp < (grp ^ m);
  WlCol<R> p = x;
  wl_xor<R>(p, m);
  double xy = wl_dot<R>(x.v, p.v), ratio = 1.0;
  if constexpr (WlCol<R>::kScaled) {
    ratio = p.d * fast_rcp(x.d);
    xy *= x.d * p.d;
  }
  const double xy2 = xy * xy, w = x.n * p.n;
  WlRot r = wl_rotation(lower ? x.n : p.n, lower ? p.n : x.n, w, xy, xy2);
  const bool rot = xy2 > tol2 * w;
  big |= int(rot & r.big);
  // lower: x' = x - t (d_y / d_x) y;  upper: y' = y + t (d_x / d_y) x
  const double t = rot ? (lower ? -r.t : r.t) : 0.0;
  const double c = rot ? r.c : 1.0;
  if constexpr (WlCol<R>::kScaled) {
#pragma unroll
    for (int j = 0; j < R; ++j) x.v[j] = fma(t * ratio, p.v[j], x.v[j]);
    x.d *= c;
  } else {
    const double sn = t * c;
#pragma unroll
    for (int j = 0; j < R; ++j) x.v[j] = fma(sn, p.v[j], c * x.v[j]);
  }
  const double n = fma(t, xy, x.n);
  const bool lost = n < 0.25 * x.n;
  x.n = n;
  if (lost) x.n = wl_norm<R>(x);
}

template <int R>
__device__ __forceinline__ void wl_cross(WlCol<R>& a, WlCol<R>& b, double tol2, int& big) {
  double ab = wl_dot<R>(a.v, b.v), ra, rb;
  if constexpr (WlCol<R>::kScaled) {
    ra = b.d * fast_rcp(a.d);
    rb = a.d * fast_rcp(b.d);
    ab *= a.d * b.d;
  }
  const double ab2 = ab * ab, w = a.n * b.n;
  if (ab2 > tol2 * w) {
    const WlRot r = wl_rotation(a.n, b.n, w, ab, ab2);
    big |= int(r.big);
    if constexpr (WlCol<R>::kScaled) {
      const double fa = -r.t * ra, fb = r.t * rb;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const double x = a.v[j], y = b.v[j];
        a.v[j] = fma(fa, y, x);
        b.v[j] = fma(fb, x, y);
      }
      a.d *= r.c;
      b.d *= r.c;
    } else {
      const double sn = r.t * r.c;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const double x = a.v[j], y = b.v[j];
        a.v[j] = fma(-sn, y, r.c * x);
        b.v[j] = fma(sn, x, r.c * y);
      }
    }
    wl_norms<R>(a, b, fma(-r.t, ab, a.n), fma(r.t, ab, b.n));
  }
}

// Sweeps until one has no big rotation (or max_sweeps); nrot[2] are shared
// counters, zero on entry.  Every thread of the block calls this.
//
// A rotation adds to a coupling that is already zeroed at most the product of
// its own size (the coupling, or for columns of about equal length the
// tangent, times the ratio of the lengths) and another coupling.  After a
// sweep in which both stayed below kWlSmall = 1e-9 every pair is below k 1e-18
// + 2^-23 1e-9, inside tol_rot: a sweep more would only confirm it.  For k =
// 24 .. 130 that is one of 3 .. 9 sweeps.
template <int R>
__device__ __forceinline__ void wl_sweeps(double* X, int k, double tol_rot, int max_sweeps, int* nrot) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, grp = lane >> 3, li = lane & 7;
  const int NB = 2 * ((k + 15) / 16);
  const bool active = wave < NB / 2;
  const double tol2 = tol_rot * tol_rot;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    // of this lane's group: the groups rotate or not independently (an integer,
    // in a vector register: lane masks cost more)
    int big = 0;
    for (int t = 0; t < NB - 1; ++t) {
      if (active) {
        const int P = circle_block(wave, t, NB), Q = circle_block(NB - 1 - wave, t, NB);
        WlCol<R> a, b;
        wl_load<R>(X, k, P * 8 + grp, li, a);
        if (t == 0) {  // round 0 holds every block once: pairs inside the blocks
          if constexpr (R <= 10) {
            wl_load<R>(X, k, Q * 8 + grp, li, b);
#pragma unroll 1
            for (int m = 1; m < 8; ++m) {
              wl_intra<R>(a, m, grp, tol2, big);
              wl_intra<R>(b, m, grp, tol2, big);
            }
          } else {  // one block at a time: two with their partners' copies would spill
#pragma unroll 1
            for (int m = 1; m < 8; ++m) wl_intra<R>(a, m, grp, tol2, big);
            wl_load<R>(X, k, Q * 8 + grp, li, b);
#pragma unroll 1
            for (int m = 1; m < 8; ++m) wl_intra<R>(b, m, grp, tol2, big);
          }
        } else {
          wl_load<R>(X, k, Q * 8 + grp, li, b);
        }
        // group g pairs its P column with the Q column of group g ^ gray(u);
        // a loop of two steps, as eight unrolled overflow the instruction cache
#pragma unroll 1
        for (int u = 0; u < 4; ++u) {
          wl_cross<R>(a, b, tol2, big);
          wl_xor<R>(b, 1);
          wl_cross<R>(a, b, tol2, big);
          wl_xor<R>(b, (u & 1) ? 4 : 2);
        }
        wl_store<R>(X, k, P * 8 + grp, li, a);
        wl_store<R>(X, k, Q * 8 + grp, li, b);  // the eight moves of b have come round
      }
      __syncthreads();
    }
    const bool any = __any(big != 0);
    if (lane == 0 && any) atomicAdd(&nrot[sweep & 1], 1);
    __syncthreads();
    const int n = nrot[sweep & 1];
    if (tid == 0) nrot[(sweep + 1) & 1] = 0;
    __syncthreads();
    if (n == 0) break;
  }
}

// Pivoted Cholesky of G (in X, k x k column-major, k <= 8 R <= 64): column j
// of X receives column j of L in the original row order (X X^T = G), pivoted[i]
// whether row i was a pivot; returns the rank, pv0 and pv1 the first and the
// last pivot.  Every thread of the block calls this.
//
// Left-looking, eight lanes to a row: a step forms the pivot's column only,
// G(:, p) minus the product of the columns of L so far, so its chain is one
// read of the pivot, one of the pivot's row of L (in X), an eight-lane sum and
// one barrier.  Lane li keeps the entries li, li + 8, ... of its row of G and
// of L.  The pivot is the largest remaining diagonal up to 2^-12 of it (the key
// has 20 bits of the value's mantissa less the row's eight), the smallest row
// on ties; wkey, wval: shared, the waves' candidates by step parity.  k = 12,
// 24, 40: 6, 14, 31 us against 9, 17, 43 for one wave that updates the trailing
// matrix in its registers.
template <int R>
__device__ __forceinline__ int chol_rows(double* X, int* pivoted, int k, int (*wkey)[16], double (*wval)[16],
                                         double& pv0, double& pv1) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = tid & 7;
  const int nwv = (k + 7) >> 3;  // waves that hold rows
  const bool has = (tid >> 3) < k;
  const int row = has ? tid >> 3 : 0;  // reads stay inside X
  double g[R], lr[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int c = li + 8 * q;
    g[q] = has && c < k ? X[c * k + row] : 0.0;
    lr[q] = 0.0;
  }
  double dg = X[row * k + row];
  bool out = !has;  // no row, or a pivoted one
  auto publish = [&](int slot) {
    const int hi = int(__double_as_longlong(dg) >> 32);
    const int key = out ? INT_MIN : (hi & ~0xFF) | (255 - row);
    int top = max(key, __builtin_amdgcn_mov_dpp(key, 0x128, 0xF, 0xF, false));
    top = max(top, xor16(top));
    top = max(top, xor32(top));
    if (key == top && li == 0) {
      wkey[slot][wave] = top;
      wval[slot][wave] = dg;
    }
  };
  if (wave < nwv) publish(0);
  __syncthreads();  // also: every read of G precedes the columns of L
  int rk = k;
  for (int j = 0; j < k; ++j) {
    // lane w < nwv looks at wave w's candidate
    const int cand = lane < nwv ? wkey[j & 1][lane] : INT_MIN;
    const double cval = lane < nwv ? wval[j & 1][lane] : -1.0;
    int top = max(cand, __builtin_amdgcn_mov_dpp(cand, 0xB1, 0xF, 0xF, false));
    top = max(top, __builtin_amdgcn_mov_dpp(top, 0x4E, 0xF, 0xF, false));
    top = max(top, __builtin_amdgcn_mov_dpp(top, 0x141, 0xF, 0xF, false));
    top = __builtin_amdgcn_readfirstlane(top);
    const int who = __ffsll((unsigned long long)__ballot(cand == top)) - 1;
    const long long cb = __double_as_longlong(cval);
    const int plo = __builtin_amdgcn_readlane(int(cb & 0xffffffffLL), who);
    const int phi = __builtin_amdgcn_readlane(int(cb >> 32), who);
    const double pv = __longlong_as_double((long long)(unsigned)plo | ((long long)phi << 32));
    const int p = 255 - (top & 0xFF);
    if (top == INT_MIN || !(pv > 0.0)) {  // uniform: the rest is zero or negative noise
      rk = j;
      break;
    }
    if (j == 0) pv0 = pv;
    pv1 = pv;
    if (wave < nwv) {
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (q == (p >> 3)) s = g[q];
      s = li == (p & 7) ? s : 0.0;
      // entries of L past the j that exist meet zeros of lr
#pragma unroll
      for (int q0 = 0; q0 < R; q0 += 2)
        if (8 * q0 < j) {
          const double l0 = X[min(li + 8 * q0, j - 1) * k + p], l1 = X[min(li + 8 * q0 + 8, j - 1) * k + p];
          s = fma(-lr[q0], l0, s);
          s = fma(-lr[q0 + 1], l1, s);
        }
      const double isq = fast_rsqrt(pv);
      sum8(s);
      const bool here = has && row == p;
      const double l = here ? pv * isq : (out ? 0.0 : s * isq);
      if (li == 0 && has) X[j * k + row] = l;
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (q == (j >> 3)) lr[q] = li == (j & 7) ? l : lr[q];
      dg = here ? -1.0 : dg - l * l;
      out = out || here;
      publish((j + 1) & 1);
    }
    __syncthreads();
  }
  if (li == 0 && has) pivoted[row] = out;
  return rk;
}

template <class L>
__global__ __launch_bounds__(kGramEigThreads) void k_gram_eig(double* __restrict__ base,
                                                            L l,
                                                            int* __restrict__ flags, double tol, int max_sweeps,
                                                            int precond) {
  extern __shared__ double lds[];
  __shared__ int nrot[2];
  __shared__ int nviol, nabs, best;
  const SmallJacobi J = l.template list<SmallJacobi>()[blockIdx.x];
  const int k = J.k;
  const int ke = k + (k & 1);
  const int tid = threadIdx.x;
  double* X = lds;                         // k x ke, column-major
  double* nrm = lds + int64_t(k) * ke;     // ke
  double* vec = nrm + ke;                  // ke
  double* hh = vec + ke;                   // ke
  int* perm = reinterpret_cast<int*>(hh + ke);  // ke
  double* Gg = base + J.y_off;
  double* Wg = base + J.w_off;
  const int npairs = ke / 2;
  const int gsz = gram_eig_gsz(k, int(blockDim.x));
  if (k <= 0) return;
  if (k > kGramEigMaxK) {  // never launched so by the host
    for (int64_t e = tid; e < int64_t(k) * k; e += blockDim.x)
      Wg[(e / k) * J.ldw + e % k] = (e / k == e % k) ? 1.0 : 0.0;
    if (tid == 0 && J.flag_idx >= 0) flags[J.flag_idx] = -1;
    return;
  }
  for (int e = tid; e < k * ke; e += blockDim.x) {
    const int r = e % k, c = e / k;
    X[e] = c < k ? Gg[int64_t(c) * J.ldy + r] : 0.0;
  }
  for (int e = tid; e < ke; e += blockDim.x) perm[e] = e;
  if (tid == 0) {
    nviol = 0;
    nabs = 0;
    nrot[0] = nrot[1] = 0;
  }
  __syncthreads();
  // ---- 0. shift of an eigh -----------------------------------------------------
  // The solver takes a positive definite matrix.  A density matrix is one up to
  // its rounding, and its factor is as graded as its spectrum, so the sweeps
  // are few; shifted by its norm all columns are about equally long and the
  // rounding of their products keeps the sweeps going to their limit (sectors up
  // to k = 68, twelve decades: 30 sweeps and 976 us, against 440).  So the shift is first the
  // rounding a Cholesky factorisation may meet, and the norm only where that
  // fails.
  const bool eig = J.shift_off >= 0;
  double shift = 0.0, fro = 0.0;
  bool by_norm = false;  // counted, not compared: the norm may be a NaN
  auto add_shift = [&] {
    if (tid < k) X[tid * k + tid] += shift;
    __syncthreads();
  };
  if (eig) {
    __shared__ double red[3][kGramEigThreads / 64];
    double ss = 0.0, lo = INFINITY, hi = 0.0;
    for (int e = tid; e < k * k; e += blockDim.x) ss = fma(X[e], X[e], ss);
    if (tid < k) {
      lo = X[tid * k + tid];
      hi = fmax(lo, 0.0);
    }
    for (int off = 32; off > 0; off >>= 1) {
      ss += __shfl_xor(ss, off);
      lo = fmin(lo, __shfl_xor(lo, off));
      hi = fmax(hi, __shfl_xor(hi, off));
    }
    if ((tid & 63) == 0) {
      red[0][tid >> 6] = ss;
      red[1][tid >> 6] = lo;
      red[2][tid >> 6] = hi;
    }
    __syncthreads();
    ss = 0.0;
    for (int w = 0; w < kGramEigThreads / 64; ++w) {
      ss += red[0][w];
      lo = fmin(lo, red[1][w]);
      hi = fmax(hi, red[2][w]);
    }
    fro = sqrt(ss);
    shift = 4.0 * k * DBL_EPSILON * hi;
    // without the factorisation nothing would tell that the shift is too small
    by_norm = !precond || !(lo + shift > 0.0);
    if (by_norm) shift = fro;
    add_shift();
  }
  // ---- 1. orthogonality test on G -------------------------------------------
  {
    double dm = 0.0;
    for (int i = tid; i < k; i += blockDim.x) dm = fmax(dm, X[i * k + i]);
    if (tid == 0) nrm[0] = 0.0;  // scratch for the maximum (nrm is free until the Jacobi ends)
    __syncthreads();
    for (int off = 32; off > 0; off >>= 1) dm = fmax(dm, __shfl_xor(dm, off));
    if ((tid & 63) == 0) atomicMax(reinterpret_cast<unsigned long long*>(nrm),
                                   static_cast<unsigned long long>(__double_as_longlong(dm)));
    __syncthreads();
    // the two tests on squares: g^2 > tol^2 g_ii g_jj (relative) and
    // g^2 > tol^2 max(g_ii, g_jj) max_l g_ll (absolute); wave w scans the
    // upper part of columns w, w + nwave, ...
    const double g2max = nrm[0], t2 = tol * tol;
    const int lane = tid & 63, nwave = blockDim.x >> 6;
    int my = 0, mya = 0;
    for (int c = tid >> 6; c < k; c += nwave) {
      const double gjj = X[c * k + c];
      for (int r = lane; r < c; r += 64) {
        const double gii = X[r * k + r], g = X[c * k + r], g2 = g * g;
        if (gii > 0.0 && gjj > 0.0 && g2 > t2 * gii * gjj) {
          if (g2 > t2 * fmax(gii, gjj) * g2max)
            ++my;
          else
            ++mya;
        }
      }
    }
    if (my) atomicAdd(&nviol, my);
    if (mya) atomicAdd(&nabs, mya);
  }
  __syncthreads();
  const bool ident = nviol == 0 || k < 2;
  if (!ident && precond) {
    // ---- 2. pivoted Cholesky --------------------------------------------------
    // Up to k = 64 by chol_rows.  Wider, thread t owns an 8 x 5 tile of G.
    // Step j picks the largest remaining diagonal p (smallest index on ties),
    // the owners of column p publish l = G(:, p) / sqrt(G(p, p)) (zero on rows
    // already pivoted), every tile takes the rank-one update and vec keeps the
    // remaining diagonal; column j of X receives l (k = 80: 102 us, 133 for
    // chol_rows, which reads all columns so far each step).  perm flags the
    // pivoted rows here and is reset to the identity afterwards.
    __shared__ int wkey[2][16];
    __shared__ double wval[2][16];
    int rk;
    double pv0 = 0.0, pv1 = 0.0;  // first and last pivot
    for (;;) {
      rk = k;
      if (k <= 64) {
        rk = k <= 16   ? chol_rows<2>(X, perm, k, wkey, wval, pv0, pv1)
             : k <= 32 ? chol_rows<4>(X, perm, k, wkey, wval, pv0, pv1)
             : k <= 48 ? chol_rows<6>(X, perm, k, wkey, wval, pv0, pv1)
                       : chol_rows<8>(X, perm, k, wkey, wval, pv0, pv1);
        __syncthreads();
      } else {
        constexpr int TR = 8, TC = 5;
        const int ntc = (k + TC - 1) / TC;
        const bool owner = tid < ((k + TR - 1) / TR) * ntc;
        const int tr = owner ? tid / ntc : 0, tc = owner ? tid % ntc : 0;
        double g[TR][TC];
  #pragma unroll
        for (int a = 0; a < TR; ++a)
  #pragma unroll
          for (int b = 0; b < TC; ++b) {
            const int i = tr * TR + a, l = tc * TC + b;
            g[a][b] = (owner && i < k && l < k) ? X[l * k + i] : 0.0;
          }
        // Pivot keys: the top 54 bits of the remaining diagonal and the inverted
        // index in the low 10 bits (k <= 1023), so the largest key is the largest
        // value, smallest index on ties; pivoted entries hold -1, and non-positive
        // values never win over positive ones under a signed compare.  Thread i <
        // k keeps row i; each wave holding rows reduces its keys and publishes the
        // maximum in tkey[parity of the step it serves], which every thread reads
        // after the step's second barrier.
        __shared__ long long tkey[2][kGramEigThreads / 64];
        const int nwv = (k + 63) >> 6;  // waves that hold rows
        auto publish = [&](int slot) {
          long long key = LLONG_MIN;
          if (tid < k) key = (__double_as_longlong(vec[tid]) & ~0x3FFLL) | (1023 - tid);
  #pragma unroll
          for (int st = 0; st < 4; ++st) {
            const long long o = __double_as_longlong(dpp_bits(__longlong_as_double(key), st));
            key = o > key ? o : key;
          }
          long long o = __double_as_longlong(xor16(__longlong_as_double(key)));
          key = o > key ? o : key;
          o = __double_as_longlong(xor32(__longlong_as_double(key)));
          key = o > key ? o : key;
          if ((tid & 63) == 0) tkey[slot][tid >> 6] = key;
        };
        if (tid < k) {
          vec[tid] = X[tid * k + tid];
          perm[tid] = 0;
        }
        if ((tid >> 6) < nwv) publish(0);
        __syncthreads();  // every read of G from X precedes the L columns written below
        // Each step: (1) every thread takes the pivot p from the wave maxima and
        // the owners of column p copy it to hh; (2) thread i forms l_i, writes it
        // to nrm and to column j of X, updates vec[i] and the waves publish the
        // next keys; (3) the tiles take the rank-one update.  Two barriers a step:
        // hh and nrm are written one phase after their last reads, behind a
        // barrier, and the wave maxima alternate between two slots.
        for (int j = 0; j < k; ++j) {
          long long top = tkey[j & 1][0];
          for (int w = 1; w < nwv; ++w) top = tkey[j & 1][w] > top ? tkey[j & 1][w] : top;
          const int p = top == LLONG_MIN ? -1 : 1023 - int(top & 0x3FF);
          const double pmx = p >= 0 ? vec[p] : 0.0;
          if (!(pmx > 0.0)) {  // uniform: the rest of the matrix is zero or negative noise
            rk = j;
            break;
          }
          if (j == 0) pv0 = pmx;
          pv1 = pmx;
          const double isq = fast_rsqrt(pmx), sq = pmx * isq;
          if (owner && tc == p / TC) {
            // column p - tc TC of the tile by 0/1 weights: a select on the index
            // would be folded into an indexed load and move the tile to scratch
            double m[TC];
  #pragma unroll
            for (int b = 0; b < TC; ++b) m[b] = (p - tc * TC == b) ? 1.0 : 0.0;
  #pragma unroll
            for (int a = 0; a < TR; ++a) {
              double v = 0.0;
  #pragma unroll
              for (int b = 0; b < TC; ++b) v += g[a][b] * m[b];
              if (tr * TR + a < k) hh[tr * TR + a] = v;
            }
          }
          __syncthreads();
          if (tid < k) {
            const int i = tid;
            const double l = i == p ? sq : (perm[i] ? 0.0 : hh[i] * isq);
            nrm[i] = l;
            X[j * k + i] = l;
            if (i == p) {
              vec[p] = -1.0;
              perm[p] = 1;
            } else {
              vec[i] -= l * l;  // pivoted rows hold -1 and l = 0
            }
          }
          if ((tid >> 6) < nwv) publish((j + 1) & 1);
          __syncthreads();
          if (owner) {
            double li[TR], lc[TC];
  #pragma unroll
            for (int a = 0; a < TR; ++a) li[a] = tr * TR + a < k ? nrm[tr * TR + a] : 0.0;
  #pragma unroll
            for (int b = 0; b < TC; ++b) lc[b] = tc * TC + b < k ? nrm[tc * TC + b] : 0.0;
  #pragma unroll
            for (int a = 0; a < TR; ++a)
  #pragma unroll
              for (int b = 0; b < TC; ++b) g[a][b] -= li[a] * lc[b];
          }
        }
      }
      if (!eig || rk == k || by_norm) break;
      __syncthreads();  // not definite: again under the norm
      for (int e = tid; e < k * k; e += blockDim.x) X[e] = Gg[int64_t(e / k) * J.ldy + e % k];
      __syncthreads();
      by_norm = true;
      shift = fro;
      add_shift();
    }
    // Columns from the rank on: small multiples of the unit vectors of the rows
    // without a pivot, the factor of G + delta^2 I there with delta^2 the last
    // pivot, 2^-54 of the largest diagonal at most: below the rounding of G,
    // which is that small for the short columns of a graded matrix.  The Jacobi
    // sweeps then make the null space's basis with all others (a numpy model
    // takes the same number of sweeps or one more); completing zero columns one
    // by one took 640 of 1780 us for two sectors of k = 98 with spectra over ten
    // decades.  (2^-54 of the largest diagonal throughout left couplings among
    // short columns when the spectrum fell below 1e-16, and the iteration ran to
    // its cap: 300 columns over 30 decades 61 ms and V^T V - I = 4e-13, now 38 ms
    // and 3e-15.)  G = 0 leaves zero columns.
    for (int e = rk * k + tid; e < k * k; e += blockDim.x) X[e] = 0.0;
    const double delta = sqrt(fmin(pv0 * 0x1p-54, pv1));
    __syncthreads();
    if (rk > 0 && tid < k && !perm[tid]) {
      int c = rk;
      for (int i = 0; i < tid; ++i) c += perm[i] ? 0 : 1;
      X[c * k + tid] = delta;
    }
    __syncthreads();
    for (int i = tid; i < ke; i += blockDim.x) perm[i] = i;
    __syncthreads();
  }
  // ---- 3. one-sided Jacobi on the columns of X ------------------------------
  // (under a shift by the norm, tol / 16 is below the products' rounding)
  const double tol_rot = tol * (by_norm ? 0.5 : 1.0 / 16.0);
  const int pi = tid / gsz, li = tid % gsz;
  if (!ident) {
    if (k <= 16)
      wl_sweeps<2>(X, k, tol_rot, max_sweeps, nrot);
    else if (k <= 32)
      wl_sweeps<4>(X, k, tol_rot, max_sweeps, nrot);
    else if (k <= 48)
      wl_sweeps<6>(X, k, tol_rot, max_sweeps, nrot);
    else if (k <= 64)
      wl_sweeps<8>(X, k, tol_rot, max_sweeps, nrot);
    else if (k <= 80)
      wl_sweeps<10>(X, k, tol_rot, max_sweeps, nrot);
    else if (k <= 96)
      wl_sweeps<12>(X, k, tol_rot, max_sweeps, nrot);
    else if (k <= 112)
      wl_sweeps<14>(X, k, tol_rot, max_sweeps, nrot);
    else if (k <= 128)
      wl_sweeps<16>(X, k, tol_rot, max_sweeps, nrot);
    else
      wl_sweeps<18>(X, k, tol_rot, max_sweeps, nrot);
  }
  if (!ident) {
    // ---- 4. normalise, complete zero columns --------------------------------
    // column norms: the pairs of round 0 cover every column once
    if (pi < npairs) {
      const int a = circle_block(pi, 0, ke), b = circle_block(ke - 1 - pi, 0, ke);
      double al = 0.0, be = 0.0;
      double zero = 0.0;
      for (int l = li; l < k; l += gsz) {
        al += X[a * k + l] * X[a * k + l];
        be += X[b * k + l] * X[b * k + l];
      }
      group_sum3(al, be, zero, gsz);
      if (li == 0) {
        nrm[a] = sqrt(al);
        nrm[b] = sqrt(be);
      }
    }
    __syncthreads();
    for (int e = tid; e < k * k; e += blockDim.x) {
      const double v = nrm[e / k];
      X[e] = v > 1e-300 ? X[e] / v : 0.0;
    }
    __syncthreads();
    for (int c = 0; c < k; ++c) {
      if (nrm[c] > 1e-300) continue;  // uniform: nrm is shared
      for (int r = tid; r < k; r += blockDim.x) {
        double q = 1.0;
        for (int j = 0; j < k; ++j) q -= X[j * k + r] * X[j * k + r];
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
        for (int j = 0; j < k; ++j) q -= X[j * k + r] * X[j * k + e0];
        vec[r] = q;
      }
      __syncthreads();
      for (int j = tid; j < k; j += blockDim.x) {
        double q = 0.0;
        for (int r = 0; r < k; ++r) q += X[j * k + r] * vec[r];
        hh[j] = q;
      }
      __syncthreads();
      for (int r = tid; r < k; r += blockDim.x) {
        double q = vec[r];
        for (int j = 0; j < k; ++j) q -= X[j * k + r] * hh[j];
        vec[r] = q;
      }
      __syncthreads();
      if (tid == 0) {
        double q = 0.0;
        for (int r = 0; r < k; ++r) q += vec[r] * vec[r];
        nrm[c] = sqrt(q);
      }
      __syncthreads();
      for (int r = tid; r < k; r += blockDim.x) X[c * k + r] = vec[r] / nrm[c];
      __syncthreads();
    }
  }
  // ---- 5. W = P Q ---------------------------------------------------------------
  for (int e = tid; e < k * k; e += blockDim.x) {
    const int r = e % k, c = e / k;
    if (ident)
      Wg[int64_t(c) * J.ldw + r] = (r == c) ? 1.0 : 0.0;
    else
      Wg[int64_t(c) * J.ldw + perm[r]] = X[e];
  }
  if (tid == 0 && eig) base[J.shift_off] = shift;
  if (tid == 0 && J.flag_idx >= 0) flags[J.flag_idx] = nviol;
  if (tid == 0 && J.aux_idx >= 0) flags[J.aux_idx] = nabs;
}

// First-order Gram-Schmidt step on columns whose Gram matrix is G (k x k,
// leading dimension ldy): T = I - M with M_ij = g_ij / g_ii when column i is
// longer than column j (ties: lower index), so Z T removes from every column
// its components along the longer ones.  T is written k x k at w_off
// (leading dimension ldw).
//
// Columns that the last pass takes for zero (norms up to ell eps times the
// largest) hold rounding only, and there are often many of them in few
// directions: they are freed of the others, not the others of them, which
// would add them up (300 columns of rank 10: null values of 9e-13 and U S V^T
// off by 1e-11, against 6e-16 and 2e-14).
template <class L>
__global__ __launch_bounds__(256) void k_gs_step(double* __restrict__ base, L l) {
  const SmallJacobi J = l.template list<SmallJacobi>()[blockIdx.x];
  const int k = J.k;
  const int j0 = blockIdx.y * 8;  // eight columns of T per work-group
  if (j0 >= k) return;
  const double* G = base + J.y_off;
  double* T = base + J.w_off;
  double top = 0.0;  // every wave for itself: no barrier before the loads below
  for (int i = threadIdx.x & 63; i < k; i += 64) top = fmax(top, G[int64_t(i) * J.ldy + i]);
  for (int off = 32; off > 0; off >>= 1) top = fmax(top, __shfl_xor(top, off));
  const double rel = double(J.ell) * DBL_EPSILON, null2 = rel * rel * top;
  double dj[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) dj[c] = j0 + c < k ? G[int64_t(j0 + c) * J.ldy + j0 + c] : 0.0;
  for (int i = threadIdx.x; i < k; i += blockDim.x) {
    const double di = G[int64_t(i) * J.ldy + i];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int j = j0 + c;
      if (j < k) {
        double v = i == j ? 1.0 : 0.0;
        if (i != j && di > null2 && (di > dj[c] || (di == dj[c] && i < j))) v = -G[int64_t(j) * J.ldy + i] / di;
        T[int64_t(j) * J.ldw + i] = v;
      }
    }
  }
}

void gs_step(hipStream_t st, double* base, const Lists& descs, int n, int kmax) {
  if (n <= 0 || kmax <= 0) return;
  launch_lists(k_gs_step<DevLists>, k_gs_step<ArgLists>, descs, dim3(n, (kmax + 7) / 8), dim3(256), 0, st, base);
}

void gram_eig(hipStream_t st, double* base, const Lists& descs, int n, int* flags, double tol, int max_sweeps,
              int precond, size_t lds_bytes) {
  if (n <= 0) return;
  launch_lists(k_gram_eig<DevLists>, k_gram_eig<ArgLists>, descs, dim3(n), dim3(kGramEigThreads), lds_bytes, st, base, flags,
               tol, max_sweeps, precond);
}

// X, nrm, vec, hh and perm, and 16 doubles beyond them: the wave-local loads
// of the last column read up to 8 R - k - 1 <= 15 rows past its end (masked).
size_t gram_eig_lds_bytes(int k) {
  const int64_t ke = k + (k & 1);
  return size_t(int64_t(k) * ke + 3 * ke + 16) * sizeof(double) + size_t(ke) * sizeof(int);
}

size_t gram_eig_lds_limit() {
  static const size_t limit = [] {
    int dev = 0;
    int v = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) v = 65536;
    for (const void* f : {reinterpret_cast<const void*>(&k_gram_eig<DevLists>),
                          reinterpret_cast<const void*>(&k_gram_eig<ArgLists>)})
      (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, v - 64);
    return size_t(v);
  }();
  return limit;
}

// ---- finalize ----------------------------------------------------------------
constexpr int kFinishMaxK = 64, kFinishMaxEll = 256, kFinishMaxTasks = 256;
// aux = base + w_off + kp*kp holds 2*kp + ell doubles: column norms, ranks and
// the completion vector.

// One work-group per sector: singular values (column norms of Y), their rank
// in descending order (ties broken by column index) and the sorted values.
// Column norms of Y: grid (sector, chunk of 16 columns); each wave sums
// four columns at once (four independent loads per row step).
template <class L>
__global__ __launch_bounds__(256) void k_svd_colnorms(double* __restrict__ base, L l) {
  const SvdSector s = l.template list<SvdSector>()[blockIdx.x];
  const int k = s.k, ell = s.ell, kp = s.nb * kSvdBlock;
  const int c0 = blockIdx.y * 16 + (threadIdx.x >> 6) * 4;
  if (c0 >= k) return;
  const double* Y = base + s.y_off;
  double* sig = base + s.w_off + int64_t(kp) * kp;
  const int lane = threadIdx.x & 63;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const double* col[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) col[c] = Y + int64_t(min(c0 + c, k - 1)) * ell;  // columns past k: masked below
  for (int l = lane; l < ell; l += 256) {  // 16 loads in flight per lane
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = l + 64 * u;
      const int rr = r < ell ? r : ell - 1;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const double x = col[c][rr];
        acc[c] += (r < ell && c0 + c < k) ? x * x : 0.0;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    double a = acc[c];
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off);
    if (lane == 0 && c0 + c < k) sig[c0 + c] = sqrt(a);
  }
}

// Rank of every singular value of a sector in descending order (ties broken
// by column index) and the sorted values.  Work-group (sector, y) is one wave
// that ranks values 64 y ... 64 y + 63 against all k, compared from LDS 1024
// at a time.
constexpr int kNormsWave = 64;
template <class L>
__global__ __launch_bounds__(kNormsWave) void k_svd_norms(double* __restrict__ base,
                                                           L l) {
  constexpr int kChunk = 1024;
  __shared__ double chunk[kChunk];
  const SvdSector s = l.template list<SvdSector>()[blockIdx.x];
  const int k = s.k, kp = s.nb * kSvdBlock;
  const int j0 = blockIdx.y * kNormsWave;
  if (j0 >= k) return;  // uniform
  double* aux = base + s.w_off + int64_t(kp) * kp;
  double* sig = aux;
  double* rnk = aux + kp;
  double* S = base + s.s_off;
  const int tid = threadIdx.x;
  const int j = j0 + tid;
  const double sj = j < k ? sig[j] : 0.0;
  int r = 0;
  for (int i0 = 0; i0 < k; i0 += kChunk) {
    const int n = min(kChunk, k - i0);
    __syncthreads();  // the previous chunk has been read
    for (int t = tid; t < n; t += blockDim.x) chunk[t] = sig[i0 + t];
    __syncthreads();
    for (int t = 0; t < n; ++t) {
      const double si = chunk[t];
      r += (si > sj) || (si == sj && i0 + t < j);
    }
  }
  if (j < k) {
    rnk[j] = double(r);
    if (s.eig_shift)
      S[k - 1 - r] = sj - base[s.shift_off];
    else
      S[r] = sj;
  }
}

// Scatter of one 64x64 tile of a column-major source (Y: ell x k, or W: k x k
// leading block of kp x kp) into the row-major output with permuted, scaled
// columns, transposed through LDS so both the reads and the writes are
// coalesced.  task = (sector, part, row0, col0); part 0: Y -> Z side
// (columns divided by their norm, zero when numerically null), part 1: W.
template <class L>
__global__ __launch_bounds__(256) void k_svd_write(double* __restrict__ base, L l, uint32_t tasks) {
  __shared__ double tile[64][65];
  __shared__ int perm[64];
  __shared__ double scl[64];
  const int4 t = l.template list<int4>(tasks)[blockIdx.x];
  const SvdSector s = l.template list<SvdSector>()[t.x];
  const int k = s.k, kp = s.nb * kSvdBlock;
  const double* aux = base + s.w_off + int64_t(kp) * kp;
  const double* sig = aux;
  const double* rnk = aux + kp;
  const bool zpart = t.y == 0;
  const int rows = zpart ? s.ell : k;
  const int64_t ld = zpart ? s.ell : kp;
  const double* src = base + (zpart ? s.y_off : s.w_off);
  double* dst;
  if (s.eig_shift)
    dst = base + s.u_off;
  else
    dst = base + ((zpart != (s.transposed != 0)) ? s.u_off : s.v_off);
  const int r0 = t.z, c0 = t.w;
  const int tid = threadIdx.x;
  const double smax = base[s.s_off + (s.eig_shift ? k - 1 : 0)];
  if (tid < 64) {
    const int c = c0 + tid;
    if (c < k) {
      const int r = int(rnk[c]);
      perm[tid] = s.eig_shift ? k - 1 - r : r;
      if (zpart) {
        const double sj = sig[c];
        const double thr = (s.eig_shift ? 0.0 : smax) * double(s.ell) * DBL_EPSILON;
        scl[tid] = (sj > thr && sj > 0.0) ? 1.0 / sj : 0.0;
      } else {
        scl[tid] = 1.0;
      }
    }
  }
  for (int i = 0; i < 16; ++i) {
    const int cl = (tid >> 6) + 4 * i;
    const int rl = tid & 63;
    const int r = r0 + rl, c = c0 + cl;
    tile[cl][rl] = (r < rows && c < k) ? src[int64_t(c) * ld + r] : 0.0;
  }
  __syncthreads();
  for (int i = 0; i < 16; ++i) {
    const int rl = (tid >> 6) + 4 * i;
    const int cl = tid & 63;
    const int r = r0 + rl, c = c0 + cl;
    if (r < rows && c < k) dst[int64_t(r) * k + perm[cl]] = tile[cl][rl] * scl[cl];
  }
}

// Norms, ranks and the scatter in one launch for calls whose sectors are all
// narrow (kFinishMaxK columns, kFinishMaxEll rows): every tile's work-group
// forms the norms and ranks it needs itself from Y, which it or a neighbour
// reads anyway, and the tile's own loads are in flight meanwhile.  The same
// bits in every work-group; the first tile of a sector stores its values.
// Bound by one chain of memory latencies instead of three with two launches
// between them: 7 sectors of 30 x 60 7.6 us against 12.1, 9 of 64 x 64 8.0
// against 15.3, of 64 x 256 9.8 against 15.7.  More tiles than work-groups
// run at once pay for the repeated norms (60 sectors of 64 x 256, 300 tiles:
// 16.3 against 17.7; 200, 1000 tiles: 34.6 against 27.7): kFinishMaxTasks.
template <class L>
__global__ __launch_bounds__(256) void k_svd_finish(double* __restrict__ base, L l, uint32_t tasks) {
  __shared__ double tile[64][65];
  __shared__ double sig[kFinishMaxK], scl[kFinishMaxK], smax;
  __shared__ int less[4][kFinishMaxK], perm[kFinishMaxK];
  const int4 t = l.template list<int4>(tasks)[blockIdx.x];
  const SvdSector s = l.template list<SvdSector>()[t.x];
  const int k = s.k, ell = s.ell, kp = s.nb * kSvdBlock;
  const bool zpart = t.y == 0;
  const int rows = zpart ? ell : k, ld = zpart ? ell : kp;
  const double* Y = base + s.y_off;
  const double* src = base + (zpart ? s.y_off : s.w_off);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r0 = t.z;
  double v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = src[min(wave + 4 * i, k - 1) * ld + min(r0 + lane, rows - 1)];
  // columns 16 wave .. + 15: lane sums, then a butterfly that halves the
  // columns a lane holds; column 16 wave + (lane >> 2) is left
  double acc[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) acc[c] = 0.0;
  if (16 * wave < k)
    for (int r = lane; r < ell; r += 64) {
      double x[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) x[c] = Y[min(16 * wave + c, k - 1) * ell + r];
#pragma unroll
      for (int c = 0; c < 16; ++c) acc[c] = fma(x[c], x[c], acc[c]);
    }
#pragma unroll
  for (int h = 8; h > 0; h >>= 1) {
    const bool up = lane & (4 * h);
#pragma unroll
    for (int c = 0; c < h; ++c) {
      const double keep = up ? acc[c + h] : acc[c], give = up ? acc[c] : acc[c + h];
      acc[c] = keep + __shfl_xor(give, 4 * h);
    }
  }
  acc[0] += __shfl_xor(acc[0], 2);
  acc[0] += __shfl_xor(acc[0], 1);
  if ((lane & 3) == 0) {
    const int c = 16 * wave + (lane >> 2);
    sig[c] = c < k ? sqrt(acc[0]) : -1.0;  // behind every norm
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) tile[wave + 4 * i][lane] = v[i];
  __syncthreads();
  const double sj = sig[lane];
  int r = 0;
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int i = 16 * wave + u;
    const double si = sig[i];
    r += int(si > sj) | (int(si == sj) & int(i < lane));
  }
  less[wave][lane] = r;
  __syncthreads();
  r = less[0][lane] + less[1][lane] + less[2][lane] + less[3][lane];
  if (wave == 0 && lane < k) {
    perm[lane] = s.eig_shift ? k - 1 - r : r;
    if (r == 0) smax = sj;
    if (r0 == 0 && (zpart || s.eig_shift)) base[s.s_off + perm[lane]] = s.eig_shift ? sj - base[s.shift_off] : sj;
  }
  __syncthreads();
  if (wave == 0 && lane < k) {
    const double thr = (s.eig_shift ? 0.0 : smax) * double(ell) * DBL_EPSILON;
    scl[lane] = !zpart ? 1.0 : sj > thr && sj > 0.0 ? 1.0 / sj : 0.0;
  }
  __syncthreads();
  double* dst = base + (s.eig_shift || zpart == (s.transposed == 0) ? s.u_off : s.v_off);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int q = r0 + wave + 4 * i;
    if (q < rows && lane < k) dst[int64_t(q) * k + perm[lane]] = tile[lane][wave + 4 * i] * scl[lane];
  }
}

// Orthonormal completion of the Z-side columns whose singular value is
// numerically zero, columns t < limit: starting from unit vectors, classical
// Gram-Schmidt twice against all earlier columns (the dot products of one
// pass in one step, thread per column; the update thread per row), keeping
// the first candidate whose residual norm exceeds 0.7 / sqrt(ell): the
// residuals' squares sum to the number of missing columns, so one of the ell
// candidates always does (1/2 was out of reach when few columns are missing:
// every candidate was tried and the columns stayed zero).  One work-group
// per sector.
template <class L>
__global__ __launch_bounds__(256) void k_svd_complete(double* __restrict__ base,
                                                      L l) {
  __shared__ double sh[256];
  __shared__ int first_sh;
  const CompleteTask T = l.template list<CompleteTask>()[blockIdx.x];
  const int k = T.k, ell = T.ell, lim = T.limit < k ? T.limit : k;
  if (lim <= 0) return;
  const double* S = base + T.s_off;
  double* v = base + T.v_off;
  double* p = base + T.p_off;
  double* Z = base + T.z_off;  // ell x k row-major
  const double null_thr = S[0] * double(ell) * DBL_EPSILON;
  const int tid = threadIdx.x;
  // the first numerically zero value below the limit (lim when none)
  if (tid == 0) first_sh = lim;
  __syncthreads();
  for (int t = tid; t < lim; t += blockDim.x)
    if (!(S[t] > null_thr && S[t] > 0.0)) atomicMin(&first_sh, t);
  __syncthreads();
  const int first_null = first_sh;
  for (int t = first_null; t < lim; ++t) {
    for (int cand = 0; cand < ell; ++cand) {
      const int e0 = (t + cand) % ell;
      for (int l = tid; l < ell; l += blockDim.x) v[l] = (l == e0) ? 1.0 : 0.0;
      __syncthreads();
      for (int pass = 0; pass < 2; ++pass) {
        for (int c = tid; c < t; c += blockDim.x) {
          double acc = 0.0;
          for (int l = 0; l < ell; ++l) acc = fma(Z[int64_t(l) * k + c], v[l], acc);
          p[c] = acc;
        }
        __syncthreads();
        for (int l = tid; l < ell; l += blockDim.x) {
          const double* zr = Z + int64_t(l) * k;
          double acc = 0.0;
          for (int c = 0; c < t; ++c) acc = fma(zr[c], p[c], acc);
          v[l] -= acc;
        }
        __syncthreads();
      }
      double acc = 0.0;
      for (int l = tid; l < ell; l += blockDim.x) acc += v[l] * v[l];
      const double nrm = sqrt(wg_sum(acc, sh));
      if (nrm * nrm * double(ell) > 0.49) {
        for (int l = tid; l < ell; l += blockDim.x) Z[int64_t(l) * k + t] = v[l] / nrm;
        __syncthreads();
        break;
      }
    }
  }
}

void svd_complete(hipStream_t st, double* base, const Lists& tasks, int n) {
  if (n <= 0) return;
  launch_lists(k_svd_complete<DevLists>, k_svd_complete<ArgLists>, tasks, dim3(n), dim3(256), 0, st, base);
}

void svd_finalize(hipStream_t st, double* base, const Lists& l, const SvdSector* host_secs, int nsec, int ntasks) {
  if (nsec <= 0) return;
  int kmax = 1, ellmax = 1;
  for (int i = 0; i < nsec; ++i) {
    kmax = std::max(kmax, host_secs[i].k);
    ellmax = std::max(ellmax, host_secs[i].ell);
  }
  if (kmax <= kFinishMaxK && ellmax <= kFinishMaxEll && ntasks <= kFinishMaxTasks) {
    if (ntasks > 0)
      launch_lists(k_svd_finish<DevLists>, k_svd_finish<ArgLists>, l, dim3(ntasks), dim3(256), 0, st, base, l.at[1]);
    return;
  }
  launch_lists(k_svd_colnorms<DevLists>, k_svd_colnorms<ArgLists>, l, dim3(nsec, (kmax + 15) / 16), dim3(256), 0, st, base);
  launch_lists(k_svd_norms<DevLists>, k_svd_norms<ArgLists>, l, dim3(nsec, (kmax + kNormsWave - 1) / kNormsWave),
               dim3(kNormsWave), 0, st, base);
  if (ntasks > 0)
    launch_lists(k_svd_write<DevLists>, k_svd_write<ArgLists>, l, dim3(ntasks), dim3(256), 0, st, base, l.at[1]);
}

template <class L>
__global__ __launch_bounds__(256) void k_svd_shift(double* __restrict__ base, L l, int norm) {
  __shared__ double sh[256];
  const SvdSector s = l.template list<SvdSector>()[blockIdx.x];
  double* Y = base + s.y_off;
  double c;
  if (norm) {
    const int64_t n = int64_t(s.ell) * s.k;
    double acc = 0.0;
    for (int64_t e = threadIdx.x; e < n; e += blockDim.x) acc += Y[e] * Y[e];
    c = sqrt(wg_sum(acc, sh));
  } else {
    c = base[s.shift_off];
  }
  for (int i = threadIdx.x; i < s.k; i += blockDim.x) Y[int64_t(i) * s.ell + i] += c;
  if (norm && threadIdx.x == 0) base[s.shift_off] = c;
}

void svd_shift(hipStream_t st, double* base, const Lists& secs, int nsec, bool norm) {
  if (nsec <= 0) return;
  launch_lists(k_svd_shift<DevLists>, k_svd_shift<ArgLists>, secs, dim3(nsec), dim3(256), 0, st, base, int(norm));
}

__global__ void k_fill_i32(int32_t* p, int n, int32_t v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void fill_i32(hipStream_t st, int32_t* p, int n, int32_t v) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_i32, dim3((n + 255) / 256), dim3(256), 0, st, p, n, v);
}

// ---- global truncation ------------------------------------------------------
// The values of all sectors are gathered, sorted descending (bitonic, in LDS
// when 2^ceil(log2 total) doubles fit, else in the scratch area) and the cut
// is found by the reference's sequential tail accumulation.
//
// Up to kRankSort values are put in order by counting, for each, the values
// before it: reads of LDS that do not wait for each other and two barriers,
// where the bitonic sort has a barrier of 16 waves at each of its steps (36 of
// them at 256 values): the whole kernel at the 150 values of a D = 48 update
// 12.7 -> 8.9 us.
constexpr int kRankSort = 512;
template <class L, bool IN_LDS>
__global__ __launch_bounds__(1024) void k_truncate(double* __restrict__ base, L l, uint32_t at_pos, uint32_t at_ks,
                                                   int nsec, int64_t scratch_off,
                                                   int64_t total, double tol, double pw, int64_t min_size,
                                                   int64_t max_size, double null_scale,
                                                   int32_t* __restrict__ kept, double* __restrict__ thr_out) {
  extern __shared__ double vl[];
  __shared__ double thr_sh;
  __shared__ int before[kRankSort], null_sh;
  const int64_t* s_offs = l.template list<int64_t>();
  const int64_t* s_pos = l.template list<int64_t>(at_pos);
  const int32_t* ks = l.template list<int32_t>(at_ks);
  double* v = IN_LDS ? vl : base + scratch_off;
  int64_t n2 = 1;
  while (n2 < total) n2 <<= 1;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  // gather (sector lists concatenated in order, s_pos[i] = start of sector i),
  // one wave per sector, pad with -inf
  for (int i = wave; i < nsec; i += nw) {
    const double* src = base + s_offs[i];
    const int64_t pos = s_pos[i];
    const int n = ks[i];
    for (int j = lane; j < n; j += 64) v[pos + j] = src[j];
  }
  for (int64_t j = total + tid; j < n2; j += blockDim.x) v[j] = -INFINITY;
  if (tid < kRankSort) before[tid] = 0;
  __syncthreads();
  const bool by_rank = IN_LDS && total <= kRankSort;
  if (by_rank) {  // value j by blockDim.x / n2 threads, each counting a part
    const int n = int(total), m = int(n2), parts = blockDim.x / m;
    const int j = tid & (m - 1), step = (n + parts - 1) / parts;
    const int i0 = tid / m * step, i1 = min(i0 + step, n);
    const double x = v[j];
    int r = 0;
#pragma unroll 8
    for (int i = i0; i < i1; ++i) r += int(v[i] > x) | (int(v[i] == x) & int(i < j));
    double* sorted = vl + m;
    if (tid < m) sorted[tid] = x;  // no hole where a NaN has no place
    if (j < n) atomicAdd(&before[j], r);
    __syncthreads();
    if (tid < n) sorted[before[tid]] = x;
    __syncthreads();
    v = sorted;
  }
  // bitonic sort, descending (n2 < 2^31; strides are powers of two, so the
  // pair index is formed with masks, not divisions)
  const int m2 = by_rank ? 0 : int(n2);
  for (int size = 2; size <= m2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = tid; i < m2 / 2; i += blockDim.x) {
        const int lo = ((i & ~(stride - 1)) << 1) | (i & (stride - 1));
        const int hi = lo + stride;
        const bool desc = ((lo & size) == 0);
        const double a = v[lo], b = v[hi];
        if (desc ? (a < b) : (a > b)) {
          v[lo] = b;
          v[hi] = a;
        }
      }
      __syncthreads();
    }
  }
  // compute_last_index (sources/LinearAlgebra.cpp:57-75), sequential as in the reference
  if (tid == 0) {
    // the same steps in the same order, the next eight values read ahead
    // (a dependent read per step would dominate the scan) and summed before
    // the first test (the kernel at the 1200 values of a D = 301 update 43 ->
    // 31 us, at the 150 of D = 48 8.9 -> 6.8); the square and
    // the general power are separate loops, so that the common pw = 2 scan
    // evaluates no pow()
    auto scan = [&](auto power) {
      const double toln = power(tol);
      int64_t last = total - 1;
      double trunc = power(fabs(v[last]));
      for (bool done = false; !done;) {
        double buf[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) buf[j] = last - 1 - j >= 0 ? v[last - 1 - j] : 0.0;
        // all eight steps at once where none of them can stop: the sum only
        // grows, so its value before the eighth decides (a NaN goes step by step)
        if (last - 7 >= min_size && last - 7 > 0) {
          double t[8];
          t[0] = trunc;
#pragma unroll
          for (int j = 1; j < 8; ++j) t[j] = t[j - 1] + power(fabs(buf[j - 1]));
          if (last - 7 >= max_size || t[7] <= toln) {
            last -= 8;
            trunc = t[7] + power(fabs(buf[7]));
            continue;
          }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (!(last >= min_size && last > 0) || (trunc > toln && last < max_size)) {
            done = true;
            break;
          }
          --last;
          trunc += power(fabs(buf[j]));
        }
      }
      return last;
    };
    const int64_t last = pw == 2.0 ? scan([](double x) { return x * x; })
                                   : scan([pw](double x) { return pow(x, pw); });
    const double sl = v[last];
    thr_sh = sl - 2.0 * sl * DBL_EPSILON;
    thr_out[0] = thr_sh;
    null_sh = 0;
  }
  __syncthreads();
  const double thr = thr_sh;
  // kept[i] = index of the first value of sector i that is not above thr
  // (its length when none), one wave per sector, 64 values per ballot; the
  // chunks are all read (no early exit) so that their loads overlap
  for (int i = wave; i < nsec; i += nw) {
    const double* src = base + s_offs[i];
    const int n = ks[i];
    int c = n;
#pragma unroll 4
    for (int j0 = 0; j0 < n; j0 += 64) {
      const int j = j0 + lane;
      const unsigned long long m = __ballot(j < n && !(src[j < n ? j : 0] > thr));
      if (m && c == n) c = j0 + __ffsll((long long)m) - 1;
    }
    if (lane == 0) {
      kept[i] = c;
      if (c > 0 && !(src[c - 1] > src[0] * null_scale)) null_sh = 1;
    }
  }
  __syncthreads();
  if (tid == 0) kept[nsec] = null_sh;
}

void truncate_select(hipStream_t st, double* base, const Lists& l, int nsec, int64_t scratch_off, int64_t total, double tol, double pw, int64_t min_size,
                     int64_t max_size, double null_scale, int32_t* kept, double* thr_out) {
  int64_t n2 = 1;
  while (n2 < total) n2 <<= 1;
  if (n2 > (int64_t(1) << 30)) throw std::runtime_error("truncation: more than 2^30 values");
  const size_t lds = size_t(n2) * sizeof(double) * (total <= kRankSort ? 2 : 1);
  static const size_t limit = [] {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) v = 65536;
    for (const void* f : {reinterpret_cast<const void*>(&k_truncate<DevLists, true>),
                          reinterpret_cast<const void*>(&k_truncate<ArgLists, true>)})
      (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, v - 256 - kRankSort * int(sizeof(int)));
    return size_t(v) - 256 - kRankSort * sizeof(int);
  }();
  if (lds <= limit)
    launch_lists(k_truncate<DevLists, true>, k_truncate<ArgLists, true>, l, dim3(1), dim3(1024), lds, st, base, l.at[1],
                 l.at[2], nsec, scratch_off, total, tol, pw, min_size, max_size, null_scale, kept, thr_out);
  else
    launch_lists(k_truncate<DevLists, false>, k_truncate<ArgLists, false>, l, dim3(1), dim3(1024), 0, st, base, l.at[1],
                 l.at[2], nsec, scratch_off, total, tol, pw, min_size, max_size, null_scale, kept, thr_out);
}

}  // namespace kern
}  // namespace qtt
