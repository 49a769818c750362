// Two-sided block Jacobi rounds for the Gram eigenproblem of wide sectors.
//
// X (k x kp, column-major, leading dimension k) is driven to orthogonal
// columns by sweeps over column blocks of 16 (nb of them, round-robin
// tournament, pairs of blocks as in k_svd_round).  A sweep starts from a
// fresh G = X^T X (kp x kp, one grouped GEMM) and carries G along under the
// rotations, so a round works on 32 x 32 blocks of G only and never touches
// the columns' full length on its critical path:
//
//   launch r   solve(r)       one work-group per block pair: its 32 x 32
//                             diagonal block of G after round r - 1, a Jacobi
//                             sweep on it, Q_r and the rotated block D_r;
//              apply(r - 1)   the remaining work-groups: G <- Q^T G Q tile by
//                             tile into the other of two buffers, X <- X Q.
//
// solve(r) does not wait for apply(r - 1): the 16 x 16 block that couples its
// two column blocks is Q_a^T G Q_b of the round before, two small products,
// and the diagonal 16 x 16 blocks are parts of D_{r-1}.  So one launch per
// round suffices and the applications, which fill the chip, run beside the
// solves, which are a chain of dependent steps.
//
// The two-sided update of G keeps the small entries of a graded positive
// matrix to relative accuracy (Demmel and Veselic, SIAM J. Matrix Anal. Appl.
// 13, 1992), and every sweep measures its convergence on a G formed anew.
#include <cfloat>
#include <climits>

#include "../kernels.hpp"

namespace qtt {
namespace kern {

typedef double v4d __attribute__((ext_vector_type(4)));

namespace {

constexpr int B = kSvdBlock;  // 16 columns per block
constexpr int B2 = 2 * B;     // 32 columns per pair
constexpr int PT = B2 + 2;    // LDS pitch of a 32 x 32 block

__device__ __forceinline__ int circle(int pos, int round, int nb) {
  return pos == 0 ? 0 : 1 + ((pos - 1 + round) % (nb - 1));
}
// pair and side (0: first block) that hold block p in a round
__device__ __forceinline__ void pair_side(int p, int round, int nb, int& pair, int& side) {
  const int m = nb - 1;
  const int pos = p == 0 ? 0 : 1 + ((p - 1 - round) % m + m) % m;
  side = pos >= nb / 2;
  pair = side ? nb - 1 - pos : pos;
}

// Rotations (c, s) of two symmetric 2 x 2 blocks [[a, q], [q, b]], their two
// chains of dependent operations side by side (stage by stage; left to itself
// the compiler puts one after the other, 1040 cycles a step against 990, and 840
// with the diagonal blocks written without a branch).  The
// tangent needs only a few digits (the next meeting of the pair removes what
// is left: a numpy model of the sweeps with tangents rounded to 24 bits takes
// the same number of sweeps), so it comes from the bare hardware estimates;
// the cosine is 1 / sqrt(1 + t^2) to the last bits (one cubic step from the
// estimate), so the rotation is orthogonal.
__device__ __forceinline__ void rotations(const double (&a)[2], const double (&b)[2], const double (&q)[2],
                                          double (&c)[2], double (&s)[2]) {
  double d[2], h[2], hh[2], ab[2], q2[2], y[2], t[2], e[2];
  auto sign_of = [](double x, double d) {  // x with its sign turned by d's
    return __longlong_as_double(__double_as_longlong(x) ^ (__double_as_longlong(d) & LLONG_MIN));
  };
#define QTT_STAGE(expr)                                  \
  _Pragma("unroll") for (int u = 0; u < 2; ++u) { expr; } \
  __builtin_amdgcn_sched_barrier(0)
  QTT_STAGE(d[u] = b[u] - a[u]; h[u] = q[u] + q[u]);
  QTT_STAGE(hh[u] = h[u] * h[u]; ab[u] = fabs(a[u] * b[u]));
  QTT_STAGE(q2[u] = fma(d[u], d[u], hh[u]));
  QTT_STAGE(y[u] = __builtin_amdgcn_rsq(q2[u]); h[u] = sign_of(h[u], d[u]));
  QTT_STAGE(t[u] = fma(q2[u], y[u], fabs(d[u])));
  QTT_STAGE(t[u] = __builtin_amdgcn_rcp(t[u]));
  // orthogonal to the rounding already (or zero columns): no rotation
  QTT_STAGE(t[u] = hh[u] > (4.0 * DBL_EPSILON * DBL_EPSILON) * ab[u] ? h[u] * t[u] : 0.0);
  QTT_STAGE(q2[u] = fma(t[u], t[u], 1.0));
  QTT_STAGE(y[u] = __builtin_amdgcn_rsq(q2[u]));
  QTT_STAGE(e[u] = q2[u] * y[u]);
  QTT_STAGE(e[u] = fma(-e[u], y[u], 1.0));
  QTT_STAGE(ab[u] = fma(0.375, e[u], 0.5));
  QTT_STAGE(e[u] = e[u] * ab[u]);
  QTT_STAGE(c[u] = fma(y[u], e[u], y[u]));
  QTT_STAGE(s[u] = t[u] * c[u]);
#undef QTT_STAGE
}

// lane i of 16 <- lane i + 1 mod 16 (CTRL 0x12F) or lane i - 1 (0x121)
template <int CTRL>
__device__ __forceinline__ double row_rotate(double v) {
  const long long b = __double_as_longlong(v);
  int lo = int(b & 0xffffffffLL), hi = int(b >> 32);
  lo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xF, 0xF, false);
  hi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xF, 0xF, false);
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}
__device__ __forceinline__ double next_lane(double v) { return row_rotate<0x12F>(v); }
__device__ __forceinline__ double prev_lane(double v) { return row_rotate<0x121>(v); }

struct SolveLds {
  union {
    struct {
      double g[B2][PT], q[B2][PT];  // operands of the products
      double t[2][B2][B + 2];       // Q_b product, two k-halves
      double h[4][B][B + 2];        // Q_a product, four k-quarters
    };
    struct {  // moving rows and diagonal entries of a step, two slots
      double row[2][4][B][B + 1];
      double app[2][B], aqq[2][B], apq[2][B];
      double none[4 * B2 * B2 / 4];  // where the threads without an entry write theirs
    };
  };
  double da[B], db[B];
};
struct ApplyLds {
  double g[B2][PT], qa[B2][PT], qb[B2][PT];
};

__device__ __forceinline__ v4d mfma(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Store of an application: written through to memory at once (agent scope), so
// that it drains while the solves run.  With plain stores the launch ends with
// the write-back of 13 MB of dirty L2 lines (six sectors, k = 149 .. 492): 15.2
// against 12.9 us a launch.
__device__ __forceinline__ void put(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One pair's 32 x 32 block: assemble, test, one Jacobi sweep, store Q and D.
__device__ __forceinline__ void solve(double* __restrict__ base, const GramRound& w, int round,
                                      int* __restrict__ counters, double tol, SolveLds& S) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nb = w.nb, kp = nb * B;
  const int p = circle(w.a, round, nb), q = circle(nb - 1 - w.a, round, nb);
  const int P = tid >> 4, R = tid & 15;
  const double* G = base + ((round & 1) || round == 0 ? w.g0 : w.g1);  // before round - 1 (round 0: fresh)
  double g00, g01, g10, g11;
  if (round == 0) {
    const double* gp = G + int64_t(p) * B * kp;
    const double* gq = G + int64_t(q) * B * kp;
    g00 = gp[int64_t(P) * kp + p * B + R];
    g01 = gp[int64_t(P) * kp + q * B + R];
    g10 = gq[int64_t(P) * kp + p * B + R];
    g11 = gq[int64_t(P) * kp + q * B + R];
  } else {
    int a, sa, b, sb;
    pair_side(p, round - 1, nb, a, sa);
    pair_side(q, round - 1, nb, b, sb);
    const int a0 = circle(a, round - 1, nb), a1 = circle(nb - 1 - a, round - 1, nb);
    const int b0 = circle(b, round - 1, nb), b1 = circle(nb - 1 - b, round - 1, nb);
    const int prev = (round - 1) & 1;
    const double* Qa = base + w.q + (int64_t(prev) * (nb / 2) + a) * (B2 * B2);  // row-major 32 x 32
    const double* Qb = base + w.q + (int64_t(prev) * (nb / 2) + b) * (B2 * B2);
    const double* Da = base + w.d + (int64_t(prev) * (nb / 2) + a) * (B2 * B2);
    const double* Db = base + w.d + (int64_t(prev) * (nb / 2) + b) * (B2 * B2);
    // every load is issued before the first use
    double gv[4], qav[2], qbv[2];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int row = (tid >> 5) + 8 * u, col = tid & 31;
      const int gr = (row < B ? a0 : a1) * B + (row & 15), gc = (col < B ? b0 : b1) * B + (col & 15);
      gv[u] = G[int64_t(gr) * kp + gc];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = P + 16 * u;
      qav[u] = Qa[row * B2 + sa * B + R];
      qbv[u] = Qb[row * B2 + sb * B + R];
    }
    g00 = Da[(sa * B + P) * B2 + sa * B + R];
    g11 = Db[(sb * B + P) * B2 + sb * B + R];
#pragma unroll
    for (int u = 0; u < 4; ++u) S.g[(tid >> 5) + 8 * u][tid & 31] = gv[u];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      S.q[P + 16 * u][R] = qav[u];
      S.q[P + 16 * u][B + R] = qbv[u];
    }
    __syncthreads();
    const int cl = lane & 15, kq = lane >> 4;
    {  // T = G Q_b: wave = (16-row tile, k-half)
      const int ti = wave & 1, k0 = (wave >> 1) * 16;
      v4d acc = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int kk = 0; kk < 16; kk += 4) acc = mfma(S.g[ti * 16 + cl][k0 + kk + kq], S.q[k0 + kk + kq][B + cl], acc);
#pragma unroll
      for (int r = 0; r < 4; ++r) S.t[wave >> 1][ti * 16 + 4 * r + kq][cl] = acc[r];
    }
    __syncthreads();
    {  // H = Q_a^T T: wave = k-quarter
      v4d acc = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int kk = 0; kk < 8; kk += 4) {
        const int k = wave * 8 + kk + kq;
        acc = mfma(S.q[k][cl], S.t[0][k][cl] + S.t[1][k][cl], acc);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) S.h[wave][4 * r + kq][cl] = acc[r];
    }
    __syncthreads();
    g01 = (S.h[0][P][R] + S.h[1][P][R]) + (S.h[2][P][R] + S.h[3][P][R]);
    g10 = (S.h[0][R][P] + S.h[1][R][P]) + (S.h[2][R][P] + S.h[3][R][P]);
  }
  // ---- test: any pair of the 32 columns over the tolerance ------------------------
  if (P == R) {
    S.da[P] = g00;
    S.db[P] = g11;
  }
  __syncthreads();
  auto over = [&](double g, double x, double y) { return x > 0.0 && y > 0.0 && g * g > (tol * x) * (tol * y); };
  int bad = over(g01, S.da[P], S.db[R]);
  if (P < R) bad += int(over(g00, S.da[P], S.da[R])) + int(over(g11, S.db[P], S.db[R]));
  const int any = __syncthreads_or(bad);
  if (round == 0 && bad) atomicAdd(&counters[w.flag], bad);  // apply(0) counts the pairs across
  double qa0 = P == R ? 1.0 : 0.0, qa1 = 0.0, qb0 = 0.0, qb1 = qa0;
  // Thread (P, R) holds the 2 x 2 block of G at row pair P and column pair R
  // of the step, and Q's rows P and 16 + P in column pair R.  A step: every
  // thread reads the diagonal entries of both pairs, forms both rotations
  // itself (the same bits in every thread that does) and updates; then the
  // moving columns come from the neighbouring lane and the moving rows, with
  // the next step's diagonal entries, go through LDS in the other slot, so a
  // step has one barrier.
  auto publish_diag = [&](int slot, double app, int pi, double aqq, int qi) {
    S.app[slot][pi] = app;
    S.aqq[slot][qi] = aqq;
  };
  double c[2], sn[2];
  auto rotate = [&](const double (&a)[2], const double (&b)[2], const double (&q)[2]) {
    rotations(a, b, q, c, sn);
    const double h00 = c[0] * g00 - sn[0] * g10, h01 = c[0] * g01 - sn[0] * g11;
    const double h10 = c[0] * g10 + sn[0] * g00, h11 = c[0] * g11 + sn[0] * g01;
    g00 = c[1] * h00 - sn[1] * h01;
    g01 = c[1] * h01 + sn[1] * h00;
    g10 = c[1] * h10 - sn[1] * h11;
    g11 = c[1] * h11 + sn[1] * h10;
  };
  auto rotate_q = [&] {
    const double a1 = c[1] * qa1 + sn[1] * qa0, b1 = c[1] * qb1 + sn[1] * qb0;
    qa0 = c[1] * qa0 - sn[1] * qa1;
    qb0 = c[1] * qb0 - sn[1] * qb1;
    qa1 = a1;
    qb1 = b1;
  };
  if (any) {
    if (P == R) {
      publish_diag(0, g00, P, g11, P);
      S.apq[0][P] = g01;
    }
    __syncthreads();
  }
  if (any && round > 0) {
    // The 256 pairs across the two blocks in 16 steps: row pair P is (P, 16 +
    // (P + r) mod 16), so the first member stays and the second moves on by
    // one pair a step (rows through LDS from thread row P + 1).
    // The diagonal entries of the next pair i: G[i][i] and the product stay
    // with thread (i, i); the second member's arrives with row i + 1.
    double* const own = P == R ? &S.app[0][P] : &S.none[tid];  // app and apq, 2 B apart
#pragma unroll 2
    for (int r = 0; r < B; ++r) {
      const int sl = r & 1;
      if (r > 0) {
        g10 = S.row[sl][0][(P + 1) & 15][R];
        g11 = S.row[sl][1][(P + 1) & 15][R];
      }
      const double a[2] = {S.app[sl][P], S.app[sl][R]}, q[2] = {S.apq[sl][P], S.apq[sl][R]};
      const double b[2] = {r > 0 ? S.row[sl][1][(P + 1) & 15][P] : S.aqq[0][P],
                           r > 0 ? S.row[sl][1][(R + 1) & 15][R] : S.aqq[0][R]};
      rotate(a, b, q);
      S.row[sl ^ 1][0][P][R] = g10;
      S.row[sl ^ 1][1][P][R] = next_lane(g11);
      g01 = next_lane(g01);
      own[(sl ^ 1) * B] = g00;
      own[(sl ^ 1) * B + 4 * B] = g01;
      rotate_q();
      qa1 = next_lane(qa1);
      qb1 = next_lane(qb1);
      __syncthreads();
    }
    g10 = S.row[0][0][(P + 1) & 15][R];  // after 16 steps every value is back at its first place
    g11 = S.row[0][1][(P + 1) & 15][R];
  } else if (any) {
    // Round 0 of a sweep holds every block once and takes all 496 pairs of its
    // 32 columns in 31 steps: the members of pairs 1 .. 15 and the second of
    // pair 0 travel round a ring (first members to the next pair, the second
    // of pair 0 to the first of pair 1, second members to the previous pair,
    // the first of pair 15 to its own second), the first of pair 0 stays.
    const int top = P == 0 ? 0 : P == 1 ? 0 : P - 1, bot = P == 15 ? 15 : P + 1;
    const int ts = P == 1 ? 2 : 0, bs = P == 15 ? 0 : 2;  // row kinds (0: first, 2: second) they come from
    auto ring = [&](double& f, double& g) {  // the columns' travel
      const double f1 = prev_lane(f), g0 = prev_lane(g), g1 = next_lane(g);
      const double nf = R == 0 ? f : R == 1 ? g0 : f1;
      g = R == 15 ? f : g1;
      f = nf;
    };
    // the thread that holds an entry of the next step's pairs writes it (wa:
    // first members' diagonal, wb: second members', wq: products)
    double* const wa = P != R ? &S.none[tid] : P == 15 ? &S.aqq[0][15] : &S.app[0][P == 0 ? 0 : P + 1];
    double* const wb = P != R ? &S.none[tid] : P == 0 ? &S.app[0][1] : &S.aqq[0][P - 1];
    double* const wq = R == P + 2               ? &S.apq[0][P + 1]
                       : P == 0 && R == 1   ? &S.apq[0][0]
                       : P == 14 && R == 15 ? &S.apq[0][15]
                                            : &S.none[tid];
#pragma unroll 2
    for (int r = 0; r < B2 - 1; ++r) {
      const int sl = r & 1;
      if (r > 0) {
        g00 = S.row[sl][ts][top][R];
        g01 = S.row[sl][ts + 1][top][R];
        g10 = S.row[sl][bs][bot][R];
        g11 = S.row[sl][bs + 1][bot][R];
      }
      const double a[2] = {S.app[sl][P], S.app[sl][R]}, b[2] = {S.aqq[sl][P], S.aqq[sl][R]};
      const double q[2] = {S.apq[sl][P], S.apq[sl][R]};
      rotate(a, b, q);
      const int nx = sl ^ 1;
      wa[nx * B] = g00;
      wb[nx * B] = g11;
      wq[nx * B] = P == 0 && R == 2 ? g11 : P == 14 && R == 15 ? g00 : g01;
      ring(g00, g01);
      ring(g10, g11);
      S.row[nx][0][P][R] = g00;
      S.row[nx][1][P][R] = g01;
      S.row[nx][2][P][R] = g10;
      S.row[nx][3][P][R] = g11;
      rotate_q();
      ring(qa0, qa1);
      ring(qb0, qb1);
      __syncthreads();
    }
    // 31 steps later every member is back at its first place
    g00 = S.row[1][ts][top][R];
    g01 = S.row[1][ts + 1][top][R];
    g10 = S.row[1][bs][bot][R];
    g11 = S.row[1][bs + 1][bot][R];
  }
  double* Q = base + w.q + (int64_t(round & 1) * (nb / 2) + w.a) * (B2 * B2);
  double* D = base + w.d + (int64_t(round & 1) * (nb / 2) + w.a) * (B2 * B2);
  Q[P * B2 + R] = qa0;
  Q[P * B2 + B + R] = qa1;
  Q[(B + P) * B2 + R] = qb0;
  Q[(B + P) * B2 + B + R] = qb1;
  D[P * B2 + R] = g00;
  D[P * B2 + B + R] = g01;
  D[(B + P) * B2 + R] = g10;
  D[(B + P) * B2 + B + R] = g11;
}

// Tile (pair a, pair b), a < b, of G under the rotations of `round`, written
// with its mirror image; a == b: the rotated block that the solve left.
__device__ __forceinline__ void apply_g(double* __restrict__ base, const GramRound& w, int round,
                                        int* __restrict__ counters, double tol, ApplyLds& S) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nb = w.nb, kp = nb * B;
  const double* G = base + ((round & 1) ? w.g1 : w.g0);
  double* O = base + ((round & 1) ? w.g0 : w.g1);
  const int a0 = circle(w.a, round, nb), a1 = circle(nb - 1 - w.a, round, nb);
  const int b0 = circle(w.b, round, nb), b1 = circle(nb - 1 - w.b, round, nb);
  const int r8 = tid >> 5, c32 = tid & 31;
  const int gc = (c32 < B ? b0 : b1) * B + (c32 & 15);
  auto grow = [&](int row) { return (row < B ? a0 : a1) * B + (row & 15); };
  if (w.a == w.b) {
    const double* D = base + w.d + (int64_t(round & 1) * (nb / 2) + w.a) * (B2 * B2);
#pragma unroll
    for (int u = 0; u < 4; ++u) put(O + int64_t(grow(r8 + 8 * u)) * kp + gc, D[(r8 + 8 * u) * B2 + c32]);
    return;
  }
  const double* Qa = base + w.q + (int64_t(round & 1) * (nb / 2) + w.a) * (B2 * B2);
  const double* Qb = base + w.q + (int64_t(round & 1) * (nb / 2) + w.b) * (B2 * B2);
  double gv[4], qa[4], qb[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = r8 + 8 * u;
    gv[u] = G[int64_t(grow(row)) * kp + gc];
    qa[u] = Qa[row * B2 + c32];
    qb[u] = Qb[row * B2 + c32];
  }
  if (round == 0) {  // the convergence test of the pairs across (fresh G)
    const double dc = G[int64_t(gc) * kp + gc];
    int bad = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int gr = grow(r8 + 8 * u);
      const double dr = G[int64_t(gr) * kp + gr];
      bad += dr > 0.0 && dc > 0.0 && gv[u] * gv[u] > (tol * dr) * (tol * dc);
    }
    if (bad) atomicAdd(&counters[w.flag], bad);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = r8 + 8 * u;
    S.g[row][c32] = gv[u];
    S.qa[row][c32] = qa[u];
    S.qb[row][c32] = qb[u];
  }
  __syncthreads();
  const int cl = lane & 15, kq = lane >> 4, ti = wave >> 1, tj = wave & 1;
  v4d acc = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int kk = 0; kk < B2; kk += 4) acc = mfma(S.g[ti * 16 + cl][kk + kq], S.qb[kk + kq][tj * 16 + cl], acc);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) S.g[ti * 16 + 4 * r + kq][tj * 16 + cl] = acc[r];
  __syncthreads();
  acc = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int kk = 0; kk < B2; kk += 4) acc = mfma(S.qa[kk + kq][ti * 16 + cl], S.g[kk + kq][tj * 16 + cl], acc);
  const int oc = (tj == 0 ? b0 : b1) * B + cl;
#pragma unroll
  for (int r = 0; r < 4; ++r) put(O + int64_t((ti == 0 ? a0 : a1) * B + 4 * r + kq) * kp + oc, acc[r]);
  // the mirror image through LDS, so that its rows are written contiguously
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) S.qa[ti * 16 + 4 * r + kq][tj * 16 + cl] = acc[r];
  __syncthreads();
  const int mc = grow(c32);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = r8 + 8 * u;
    put(O + int64_t((row < B ? b0 : b1) * B + (row & 15)) * kp + mc, S.qa[c32][row]);
  }
}

// Rows [64 b, 64 b + 64) of X's column pair a under the rotations of `round`,
// in place: (X Q)^T = Q^T X^T tile by tile, so that a store writes 16
// consecutive rows of a column per 16 lanes.
__device__ __forceinline__ void apply_x(double* __restrict__ base, const GramRound& w, int round, double (*qs)[PT]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nb = w.nb, k = w.k;
  const int c0 = circle(w.a, round, nb) * B, c1 = circle(nb - 1 - w.a, round, nb) * B;
  const double* Q = base + w.q + (int64_t(round & 1) * (nb / 2) + w.a) * (B2 * B2);
  double* X = base + w.x;
  const int cl = lane & 15, kq = lane >> 4;
  const int row = w.b * 64 + wave * 16 + cl;
  const int rr = row < k ? row : k - 1;
  double xv[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int c = 4 * u + kq;
    xv[u] = X[int64_t(c < B ? c0 + c : c1 + c - B) * k + rr];
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) qs[(tid >> 5) + 8 * u][tid & 31] = Q[((tid >> 5) + 8 * u) * B2 + (tid & 31)];
  __syncthreads();
  v4d o0 = v4d{0.0, 0.0, 0.0, 0.0}, o1 = o0;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    o0 = mfma(qs[4 * u + kq][cl], xv[u], o0);
    o1 = mfma(qs[4 * u + kq][B + cl], xv[u], o1);
  }
  if (row < k) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      put(X + int64_t(c0 + 4 * r + kq) * k + row, o0[r]);
      put(X + int64_t(c1 + 4 * r + kq) * k + row, o1[r]);
    }
  }
}

}  // namespace

__global__ __launch_bounds__(256) void k_gram_round(double* __restrict__ base, const GramRound* __restrict__ work,
                                                    int round, int* __restrict__ counters,
                                                    const int* __restrict__ skip, double tol) {
  __shared__ union Lds {
    SolveLds s;
    ApplyLds a;
    __device__ Lds() {}
  } lds;
  const GramRound w = work[blockIdx.x];
  if (skip && skip[w.flag] == 0) return;          // converged in an earlier sweep
  if (round > 1 && counters[w.flag] == 0) return;  // converged: this sweep's test is complete
  if (w.kind == kGramSolve) {
    if (round < w.nb - 1) solve(base, w, round, counters, tol, lds.s);
  } else if (round > 0 && round < w.nb) {
    if (w.kind == kGramApplyX)
      apply_x(base, w, round - 1, lds.a.qa);
    else if (round < w.nb - 1)  // the sweep's last rotations leave no G to carry on
      apply_g(base, w, round - 1, counters, tol, lds.a);
  }
}

void gram_round(hipStream_t st, double* base, const GramRound* work, int nwork, int round, int* counters,
                const int* skip, double tol) {
  if (nwork <= 0) return;
  hipLaunchKernelGGL(k_gram_round, dim3(nwork), dim3(256), 0, st, base, work, round, counters, skip, tol);
}

}  // namespace kern
}  // namespace qtt
