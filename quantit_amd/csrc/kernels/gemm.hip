// Grouped block-sparse GEMM for gfx950 (CDNA4).
//
// One work-group computes one tile of one output block and walks that
// block's list of (A_p, B_p) pairs in order, so every output block is written
// exactly once with a fixed accumulation order (no atomics: results do not
// depend on what else runs on the device).  The permute gather of the
// reference's permute_bl (sources/btensor.cpp:1843-1894) is folded into the
// tile loads through per-pair (row, column) element strides.
//
// The split-FP32 kernel's waves own 32x32 quadrants = 2x2 MFMA tiles; LDS holds
// a 64x16 A tile and a 16x64 B tile (k-major, row pitch 80).
#include <map>
#include <mutex>
#include <type_traits>

#include "../kernels.hpp"

namespace qtt {
namespace kern {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int BM = 64, BN = 64, BK = 16;
constexpr int LDP = BM + 16;  // LDS row pitch (doubles)

// Loads the A tile (BM x BK, element (m,k) at A[m*rs + k*cs]) into As[k][m]
// and the B tile (BK x BN, element (k,n) at B[k*rs + n*cs]) into Bs[k][n], as
// high parts and, in As2 and Bs2, what they leave.
__device__ __forceinline__ void load_tiles(const double* __restrict__ A, const double* __restrict__ B,
                                           const GemmPair& pr, int M, int N, int m0, int n0, int k0, int tid,
                                           float (*As)[LDP], float (*Bs)[LDP], float (*As2)[LDP],
                                           float (*Bs2)[LDP]) {
  const int K = pr.K;
  if (pr.a_cs == 1) {  // row-major A: 4 consecutive k per thread
    const int m = tid >> 2, kq = (tid & 3) * 4;
    const int gm = m0 + m;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gk = k0 + kq + j;
      double v = (gm < M && gk < K) ? A[int64_t(gm) * pr.a_rs + gk] : 0.0;
      float hi = float(v);
      As[kq + j][m] = hi;
      As2[kq + j][m] = float(v - double(hi));
    }
  } else {  // column-major or general strides: 4 consecutive m per thread
    const int k = tid >> 4, mq = (tid & 15) * 4;
    const int gk = k0 + k;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gm = m0 + mq + j;
      double v = (gm < M && gk < K) ? A[int64_t(gm) * pr.a_rs + int64_t(gk) * pr.a_cs] : 0.0;
      float hi = float(v);
      As[k][mq + j] = hi;
      As2[k][mq + j] = float(v - double(hi));
    }
  }
  if (pr.b_cs == 1) {  // row-major B: 4 consecutive n per thread
    const int k = tid >> 4, nq = (tid & 15) * 4;
    const int gk = k0 + k;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gn = n0 + nq + j;
      double v = (gn < N && gk < K) ? B[int64_t(gk) * pr.b_rs + gn] : 0.0;
      float hi = float(v);
      Bs[k][nq + j] = hi;
      Bs2[k][nq + j] = float(v - double(hi));
    }
  } else {  // column-major or general: 4 consecutive k per thread
    const int n = tid >> 2, kq = (tid & 3) * 4;
    const int gn = n0 + n;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gk = k0 + kq + j;
      double v = (gn < N && gk < K) ? B[int64_t(gk) * pr.b_rs + int64_t(gn) * pr.b_cs] : 0.0;
      float hi = float(v);
      Bs[kq + j][n] = hi;
      Bs2[kq + j][n] = float(v - double(hi));
    }
  }
}

// Output element (row, col) of 16x16 MFMA tile register r in lane l:
//   v_mfma_f64_16x16x4_f64: row = 4*r + l/16, col = l%16
//   v_mfma_f32_16x16x4_f32: row = 4*(l/16) + r, col = l%16
// (measured on gfx950; the two layouts differ).  This stores the second.
__device__ __forceinline__ void store_tile(double* __restrict__ C, const GemmOut& o, int m0, int n0, int wm, int wn,
                                           int lane, const v4d (&acc)[2][2], double alpha, double beta) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + i * 16 + 4 * (lane >> 4) + r;
        const int col = n0 + wn + j * 16 + (lane & 15);
        if (row < o.M && col < o.N) {
          double* p = C + int64_t(row) * o.ldc + col;
          double v = alpha * acc[i][j][r];
          if (beta != 0.0) v += beta * (*p);
          *p = v;
        }
      }
}

// ---- FP64 grouped GEMM, contiguous operands -----------------------------------
// One work-group computes a T x T tile (4 waves in 2 x 2); k in steps of 16
// through a double-buffered LDS, one barrier a step, the next step's loads in
// flight under the MFMAs of the current one.  An operand is contiguous in k
// (KC) or in its rows, the same for every pair of the launch, so a thread
// loads 16 bytes at a time (8-byte aligned: a global load needs 4) and the LDS
// tile keeps the operand's own order: row by row (pitch 18) or k by k (pitch
// T + 16), both free of bank conflicts for the MFMA reads.
//
// v_mfma_f64_16x16x4 takes 64 cycles and shares the FP64 units with every
// vector instruction, so the loop keeps those out: loads are a scalar base
// that moves with k and per-thread offsets fixed for a pair, the two LDS
// buffers are unrolled to immediate offsets, and edges are dealt with only in
// the steps that have one.  A thread's pair of rows (or of k) past the edge is
// moved back inside the block; what it holds is put right on the way to LDS,
// after the loads have been waited for.
//
// Products of a ragged tile that have no element in the block are left out:
// 8101 tiles over blocks of 1 .. 1000 rows 188 us against 214, 5707 tiles of a
// matvec 107 against 112 (a tile still loads whole, so its time does not fall
// with its products when few tiles are in flight: 225 tiles 245 us against 216,
// which run at T = 32 below kTile64Min).
//
// 2048^3 product: 53.6 TFLOP/s (at about 2.1 GHz; 47.7 with the offsets formed
// every step, 40.1 for the general kernel below, which loads 8 bytes at a time
// with a bounds check each).  T = 32 for launches with few tiles: a quarter of
// the matrix work per step and four times the work-groups (two 146^3 Gram
// products 6.3 us against 10.4 for T = 64, six of 149 .. 492: 23.7 against 28.8).
//
// Every output element accumulates over k in the same order whatever the tile
// (4-wide MFMA chunks from each pair's k = 0, pairs in list order), so all
// tiles give the same bits.
typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v2d8 __attribute__((ext_vector_type(2), aligned(8)));
constexpr int KS = 16;      // k per step
constexpr int PK = KS + 2;  // LDS pitch of a row kept in k order

template <int T, bool KC>
struct GemmOperand {
  static constexpr int kElems = KC ? T * PK : KS * (T + 16);
  static constexpr int kRow = KC ? PK : 1, kK = KC ? 1 : T + 16;  // LDS strides
  static constexpr int E = T * KS / 512;         // 16-byte loads per thread and step
  static constexpr int L = T / 2, KR = 256 / L;  // row order: threads per k, k per pass
  v2d v[E];
  uint32_t off[E];  // byte offsets from (row 0, first k of the step)
  bool edge = false, swap = false;

  static __device__ __forceinline__ int first_row(int R, int r0, int tid) {
    return min(r0 + (tid % L) * 2, R < 2 ? 0 : R - 2);
  }
  static __device__ __forceinline__ int64_t step(int64_t ld) { return KC ? KS * 8 : KS * 8 * ld; }
  // a new pair: element (r, k) at r * ld + k (KC) or k * ld + r
  __device__ __forceinline__ void begin(int64_t ld, int R, int r0, int tid) {
    if constexpr (KC) {
#pragma unroll
      for (int u = 0; u < E; ++u)
        off[u] = (uint32_t(min(r0 + (tid >> 3) + 32 * u, R - 1)) * uint32_t(ld) + (tid & 7) * 2) * 8u;
    } else {
      edge = r0 + T > R;
      const int r = first_row(R, r0, tid);
      swap = r0 + (tid % L) * 2 != r;  // the block's last row, second of its pair here
#pragma unroll
      for (int u = 0; u < E; ++u) off[u] = (uint32_t(tid / L + KR * u) * uint32_t(ld) + uint32_t(r)) * 8u;
    }
  }
  // p: (row 0, first k of the step); kleft: valid k from there
  __device__ __forceinline__ void fetch(const char* __restrict__ p, int64_t ld, int R, int r0, int kleft, int tid) {
    if (kleft >= KS && (KC || R >= 2)) {
#pragma unroll
      for (int u = 0; u < E; ++u) v[u] = *reinterpret_cast<const v2d8*>(p + off[u]);
      return;
    }
    uint32_t o[E];
    if constexpr (KC) {
      const int k = min((tid & 7) * 2, kleft < 2 ? 0 : kleft - 2);
#pragma unroll
      for (int u = 0; u < E; ++u)
        o[u] = (uint32_t(min(r0 + (tid >> 3) + 32 * u, R - 1)) * uint32_t(ld) + uint32_t(k)) * 8u;
    } else {
      const int r = first_row(R, r0, tid);
#pragma unroll
      for (int u = 0; u < E; ++u)
        o[u] = (uint32_t(min(tid / L + KR * u, kleft - 1)) * uint32_t(ld) + uint32_t(r)) * 8u;
    }
    if (KC ? kleft < 2 : R < 2) {  // a single k or row: nothing beside it to load
#pragma unroll
      for (int u = 0; u < E; ++u) v[u].x = v[u].y = *reinterpret_cast<const double*>(p + o[u]);
    } else {
#pragma unroll
      for (int u = 0; u < E; ++u) v[u] = *reinterpret_cast<const v2d8*>(p + o[u]);
    }
  }
  __device__ __forceinline__ void stash(double* __restrict__ s, int kleft, int tid) const {
    constexpr int step = KC ? 32 * PK : KR * (T + 16);
    double* d = s + (KC ? (tid >> 3) * PK + (tid & 7) * 2 : (tid / L) * (T + 16) + (tid % L) * 2);
    if (kleft >= KS && !edge) {
#pragma unroll
      for (int u = 0; u < E; ++u) *reinterpret_cast<v2d*>(d + u * step) = v[u];
      return;
    }
#pragma unroll
    for (int u = 0; u < E; ++u) {
      v2d x = v[u];
      if constexpr (KC) {
        const int k = (tid & 7) * 2;
        if (k + 1 >= kleft) {
          x.x = k < kleft ? x.y : 0.0;
          x.y = 0.0;
        }
      } else {
        if (swap) x.x = x.y;
        if (tid / L + KR * u >= kleft) x = v2d{0.0, 0.0};
      }
      *reinterpret_cast<v2d*>(d + u * step) = x;
    }
  }
};

// AK: A contiguous in k (else in m); BN: B contiguous in n (else in k).
template <class L, int T, bool AK, bool BN>
__global__ __launch_bounds__(256) void k_gemm_f64c(double* __restrict__ base, L l, uint32_t at_tiles,
                                                   uint32_t at_outs, uint32_t at_pairs, double alpha, double beta) {
  const GemmTile* tiles = l.template list<GemmTile>(at_tiles);
  const GemmOut* outs = l.template list<GemmOut>(at_outs);
  const GemmPair* pairs = l.template list<GemmPair>(at_pairs);
  using OpA = GemmOperand<T, AK>;
  using OpB = GemmOperand<T, !BN>;
  constexpr int F = T / 32;  // 16 x 16 MFMA tiles per wave and dimension
  __shared__ __align__(16) double As[2 * OpA::kElems];
  __shared__ __align__(16) double Bs[2 * OpB::kElems];
  const GemmTile t = tiles[blockIdx.x];
  const GemmOut o = outs[t.out];
  const int m0 = t.tm * T, n0 = t.tn * T;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // a wave takes every other 16 x 16 product of the tile in each dimension, so
  // what a ragged edge leaves of a tile is spread over all four; mi x nj of
  // its F x F have elements in the block
  const int wm = (wave >> 1) * 16, wn = (wave & 1) * 16;
  const int mi = __builtin_amdgcn_readfirstlane(min(F, (o.M - m0 - wm + 31) / 32));
  const int nj = __builtin_amdgcn_readfirstlane(min(F, (o.N - n0 - wn + 31) / 32));
  const int cl = lane & 15, kq = lane >> 4;
  v4d acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  int p = o.pair_begin;
  while (p < o.pair_end && pairs[p].K <= 0) ++p;
  if (p < o.pair_end) {
    OpA ga;
    OpB gb;
    const char *pa, *pb;
    int64_t lda, ldb;
    int kleft;
    auto begin = [&] {
      const GemmPair pr = pairs[p];
      pa = reinterpret_cast<const char*>(base + pr.a_off);
      pb = reinterpret_cast<const char*>(base + pr.b_off);
      lda = AK ? pr.a_rs : pr.a_cs;
      ldb = BN ? pr.b_rs : pr.b_cs;
      kleft = pr.K;
      ga.begin(lda, o.M, m0, tid);
      gb.begin(ldb, o.N, n0, tid);
    };
    auto fetch = [&] {
      ga.fetch(pa, lda, o.M, m0, kleft, tid);
      gb.fetch(pb, ldb, o.N, n0, kleft, tid);
    };
    begin();
    fetch();
    const int ao = (wm + cl) * OpA::kRow + kq * OpA::kK, bo = (wn + cl) * OpB::kRow + kq * OpB::kK;
    auto step = [&](auto buf, auto whole) {
      double* sa = As + decltype(buf)::value * OpA::kElems;
      double* sb = Bs + decltype(buf)::value * OpB::kElems;
      const int have = kleft;
      // this buffer's last readers passed the barrier of the step between
      ga.stash(sa, have, tid);
      gb.stash(sb, have, tid);
      bool more = true;
      kleft -= KS;
      pa += OpA::step(lda);
      pb += OpB::step(ldb);
      if (kleft <= 0) {
        ++p;
        while (p < o.pair_end && pairs[p].K <= 0) ++p;
        more = p < o.pair_end;
        if (more) begin();
      }
      if (more) fetch();
      __syncthreads();
      const double *ap = sa + ao, *bp = sb + bo;
      auto multiply = [&](auto fi, auto fj) {
        constexpr int FI = decltype(fi)::value, FJ = decltype(fj)::value;
#pragma unroll
        for (int kk = 0; kk < KS; kk += 4)
          if (kk < have) {  // uniform: chunks past a pair's end are zeros
            double a[FI], b[FJ];
#pragma unroll
            for (int i = 0; i < FI; ++i) a[i] = ap[i * 32 * OpA::kRow + kk * OpA::kK];
#pragma unroll
            for (int j = 0; j < FJ; ++j) b[j] = bp[j * 32 * OpB::kRow + kk * OpB::kK];
#pragma unroll
            for (int i = 0; i < FI; ++i)
#pragma unroll
              for (int j = 0; j < FJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
          }
      };
      constexpr std::integral_constant<int, F> all{};
      constexpr std::integral_constant<int, 1> one{};
      if (decltype(whole)::value || (mi == F && nj == F)) {
        multiply(all, all);
      } else if constexpr (F == 2) {
        if (mi == 1 && nj == 2)
          multiply(one, all);
        else if (mi == 2 && nj == 1)
          multiply(all, one);
        else if (mi == 1 && nj == 1)
          multiply(one, one);
      }
      return more;
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    // a loop of their own for tiles inside the block: the choice of products
    // in every step costs them 7 %
    if (o.M - m0 >= T && o.N - n0 >= T) {
      while (step(even, std::true_type{}) && step(odd, std::true_type{})) {
      }
    } else {
      while (step(even, std::false_type{}) && step(odd, std::false_type{})) {
      }
    }
  }
  double* C = base + o.c_off;
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + i * 32 + 4 * r + kq;  // f64 MFMA output layout
        const int col = n0 + wn + j * 32 + cl;
        if (row < o.M && col < o.N) {
          double* pc = C + int64_t(row) * o.ldc + col;
          double v = alpha * acc[i][j][r];
          if (beta != 0.0) v += beta * (*pc);
          *pc = v;
        }
      }
}

// ---- FP64 grouped GEMM, any strides --------------------------------------------
// The same tile for launches whose pairs are not contiguous in one common way
// (blocks with unit-length legs beside permuted ones): 8-byte loads with a
// bounds check each, double-buffered LDS k by k.
struct TileRegs {
  double a[BM * BK / 256], b[BN * BK / 256];
};

__device__ __forceinline__ void fetch_t(const double* __restrict__ base, const GemmPair& pr, int M, int N, int m0,
                                        int n0, int k0, int tid, TileRegs& r) {
  constexpr int EA = BM * BK / 256, EB = BN * BK / 256;  // elements per thread
  const double* A = base + pr.a_off;
  const double* B = base + pr.b_off;
  const int K = pr.K;
  if (pr.a_cs == 1) {  // k contiguous: BK/EA threads per row, EA consecutive k each
    constexpr int TPR = BK / EA;
    const int m = tid / TPR, kq = (tid % TPR) * EA, gm = m0 + m;
#pragma unroll
    for (int j = 0; j < EA; ++j) {
      const int gk = k0 + kq + j;
      r.a[j] = (gm < M && gk < K) ? A[int64_t(gm) * pr.a_rs + gk] : 0.0;
    }
  } else {  // m contiguous (or general): BM/EA threads per k, EA consecutive m each
    constexpr int TPK = BM / EA;
    const int k = tid / TPK, mq = (tid % TPK) * EA, gk = k0 + k;
#pragma unroll
    for (int j = 0; j < EA; ++j) {
      const int gm = m0 + mq + j;
      r.a[j] = (gm < M && gk < K) ? A[int64_t(gm) * pr.a_rs + int64_t(gk) * pr.a_cs] : 0.0;
    }
  }
  if (pr.b_cs == 1) {  // n contiguous: BN/EB threads per k, EB consecutive n each
    constexpr int TPK = BN / EB;
    const int k = tid / TPK, nq = (tid % TPK) * EB, gk = k0 + k;
#pragma unroll
    for (int j = 0; j < EB; ++j) {
      const int gn = n0 + nq + j;
      r.b[j] = (gn < N && gk < K) ? B[int64_t(gk) * pr.b_rs + gn] : 0.0;
    }
  } else {  // k contiguous (or general): BK/EB threads per column
    constexpr int TPC = BK / EB;
    const int n = tid / TPC, kq = (tid % TPC) * EB, gn = n0 + n;
#pragma unroll
    for (int j = 0; j < EB; ++j) {
      const int gk = k0 + kq + j;
      r.b[j] = (gn < N && gk < K) ? B[int64_t(gk) * pr.b_rs + int64_t(gn) * pr.b_cs] : 0.0;
    }
  }
}

__device__ __forceinline__ void stash_t(const GemmPair& pr, int tid, const TileRegs& r,
                                        double (*As)[LDP], double (*Bs)[LDP]) {
  constexpr int EA = BM * BK / 256, EB = BN * BK / 256;
  if (pr.a_cs == 1) {
    constexpr int TPR = BK / EA;
    const int m = tid / TPR, kq = (tid % TPR) * EA;
#pragma unroll
    for (int j = 0; j < EA; ++j) As[kq + j][m] = r.a[j];
  } else {
    constexpr int TPK = BM / EA;
    const int k = tid / TPK, mq = (tid % TPK) * EA;
#pragma unroll
    for (int j = 0; j < EA; ++j) As[k][mq + j] = r.a[j];
  }
  if (pr.b_cs == 1) {
    constexpr int TPK = BN / EB;
    const int k = tid / TPK, nq = (tid % TPK) * EB;
#pragma unroll
    for (int j = 0; j < EB; ++j) Bs[k][nq + j] = r.b[j];
  } else {
    constexpr int TPC = BK / EB;
    const int n = tid / TPC, kq = (tid % TPC) * EB;
#pragma unroll
    for (int j = 0; j < EB; ++j) Bs[kq + j][n] = r.b[j];
  }
}

template <class L>
__global__ __launch_bounds__(256) void k_gemm_f64t(double* __restrict__ base, L l, uint32_t at_tiles,
                                                   uint32_t at_outs, uint32_t at_pairs, double alpha, double beta) {
  const GemmTile* tiles = l.template list<GemmTile>(at_tiles);
  const GemmOut* outs = l.template list<GemmOut>(at_outs);
  const GemmPair* pairs = l.template list<GemmPair>(at_pairs);
  constexpr int WM = BM / 2, WN = BN / 2, FI = WM / 16, FJ = WN / 16;
  __shared__ double As[2][BK][LDP];
  __shared__ double Bs[2][BK][LDP];
  const GemmTile t = tiles[blockIdx.x];
  const GemmOut o = outs[t.out];
  const int m0 = t.tm * BM, n0 = t.tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
  v4d acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

  int p = o.pair_begin;
  while (p < o.pair_end && pairs[p].K <= 0) ++p;
  if (p < o.pair_end) {
    GemmPair pr = pairs[p];
    int k0 = 0, buf = 0;
    TileRegs regs;
    fetch_t(base, pr, o.M, o.N, m0, n0, 0, tid, regs);
    stash_t(pr, tid, regs, As[0], Bs[0]);
    __syncthreads();
    // the step after (p, k0)
    auto advance = [&](int& q, int& k, GemmPair& g) {
      k += BK;
      if (k >= g.K) {
        k = 0;
        ++q;
        while (q < o.pair_end && pairs[q].K <= 0) ++q;
        if (q < o.pair_end) g = pairs[q];
      }
    };
    int np = p, nk = k0;
    GemmPair npr = pr;
    advance(np, nk, npr);
    bool more = np < o.pair_end;
    if (more) fetch_t(base, npr, o.M, o.N, m0, n0, nk, tid, regs);
    while (true) {
#pragma unroll
      for (int kk = 0; kk < BK; kk += 4) {
        const int kr = kk + (lane >> 4), c = lane & 15;
        double a[FI], b[FJ];
#pragma unroll
        for (int i = 0; i < FI; ++i) a[i] = As[buf][kr][wm + i * 16 + c];
#pragma unroll
        for (int j = 0; j < FJ; ++j) b[j] = Bs[buf][kr][wn + j * 16 + c];
#pragma unroll
        for (int i = 0; i < FI; ++i)
#pragma unroll
          for (int j = 0; j < FJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      if (!more) break;
      // regs hold step (np, nk): into the other buffer (its last readers
      // passed the barrier of the previous step), then fetch the step after
      stash_t(npr, tid, regs, As[buf ^ 1], Bs[buf ^ 1]);
      int q = np, k = nk;
      advance(q, k, npr);
      more = q < o.pair_end;
      np = q;
      nk = k;
      if (more) fetch_t(base, npr, o.M, o.N, m0, n0, nk, tid, regs);
      __syncthreads();
      buf ^= 1;
      // the step in buffer buf is complete; one more compute round if it
      // was the last one loaded
      if (!more) {
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
          const int kr = kk + (lane >> 4), c = lane & 15;
          double a[FI], b[FJ];
#pragma unroll
          for (int i = 0; i < FI; ++i) a[i] = As[buf][kr][wm + i * 16 + c];
#pragma unroll
          for (int j = 0; j < FJ; ++j) b[j] = Bs[buf][kr][wn + j * 16 + c];
#pragma unroll
          for (int i = 0; i < FI; ++i)
#pragma unroll
            for (int j = 0; j < FJ; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        break;
      }
    }
  }
  double* C = base + o.c_off;
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + i * 16 + 4 * r + (lane >> 4);
        const int col = n0 + wn + j * 16 + (lane & 15);
        if (row < o.M && col < o.N) {
          double* pc = C + int64_t(row) * o.ldc + col;
          double v = alpha * acc[i][j][r];
          if (beta != 0.0) v += beta * (*pc);
          *pc = v;
        }
      }
}

template <class L>
__global__ __launch_bounds__(256) void k_gemm_split(double* __restrict__ base, L l, uint32_t at_tiles,
                                                   uint32_t at_outs, uint32_t at_pairs, double alpha, double beta) {
  const GemmTile* tiles = l.template list<GemmTile>(at_tiles);
  const GemmOut* outs = l.template list<GemmOut>(at_outs);
  const GemmPair* pairs = l.template list<GemmPair>(at_pairs);
  __shared__ float Ah[BK][LDP], Al[BK][LDP];
  __shared__ float Bh[BK][LDP], Bl[BK][LDP];
  const GemmTile t = tiles[blockIdx.x];
  const GemmOut o = outs[t.out];
  const int m0 = t.tm * BM, n0 = t.tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  v4d acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

  for (int p = o.pair_begin; p < o.pair_end; ++p) {
    const GemmPair pr = pairs[p];
    const double* A = base + pr.a_off;
    const double* B = base + pr.b_off;
    for (int k0 = 0; k0 < pr.K; k0 += BK) {
      load_tiles(A, B, pr, o.M, o.N, m0, n0, k0, tid, Ah, Bh, Al, Bl);
      __syncthreads();
      v4f hh[2][2], cr[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          hh[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
          cr[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
      for (int kk = 0; kk < BK; kk += 4) {
        const int kr = kk + (lane >> 4), c = lane & 15;
        float ah[2] = {Ah[kr][wm + c], Ah[kr][wm + 16 + c]};
        float al[2] = {Al[kr][wm + c], Al[kr][wm + 16 + c]};
        float bh[2] = {Bh[kr][wn + c], Bh[kr][wn + 16 + c]};
        float bl[2] = {Bl[kr][wn + c], Bl[kr][wn + 16 + c]};
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            hh[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[i], bh[j], hh[i][j], 0, 0, 0);
            cr[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah[i], bl[j], cr[i][j], 0, 0, 0);
            cr[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(al[i], bh[j], cr[i][j], 0, 0, 0);
          }
      }
      // fold this K chunk into the FP64 accumulators
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] += double(hh[i][j][r]) + double(cr[i][j][r]);
      __syncthreads();
    }
  }
  store_tile(base + o.c_off, o, m0, n0, wm, wn, lane, acc, alpha, beta);
}

// Narrow outputs (N <= kRowsMaxN, summed K <= kRowsMaxK): an MFMA tile of the
// kernels above would be mostly padding there, and these launches are short:
// the chain of dependent loads decides, then the streaming of A.  A wave takes
// RT x 16 rows and all columns as v_mfma_f64_16x16x4 products of the transposed
// operands (a store then holds four columns of 16 rows, contiguous for N <= 4),
// the operands straight from global memory, the next two chunks in flight.  The
// k of all pairs form one list, so a pair of one or two k wastes nothing; where
// each k lives goes to LDS first.  A group takes its rows 64 RT at a time.
// Twelve blocks of 4 .. 15 rows and columns, K 48: 4.7 us against 34.7 for a
// thread per row with B in LDS, whose loads came four at a time.
// Every element is one chain over the pairs in order, k ascending.
struct RowK {
  int64_t a_off, a_rs, b_off, b_cs;
};
template <class L, int RT>
__global__ __launch_bounds__(256) void k_gemm_rows(double* __restrict__ base, L l, uint32_t at_tasks,
                                                   uint32_t at_outs, uint32_t at_pairs, int rows, double alpha,
                                                   double beta) {
  const RowTask* tasks = l.template list<RowTask>(at_tasks);
  const GemmOut* outs = l.template list<GemmOut>(at_outs);
  const GemmPair* pairs = l.template list<GemmPair>(at_pairs);
  __shared__ RowK ks[kRowsMaxK];
  const RowTask t = tasks[blockIdx.x];
  const GemmOut o = outs[t.out];
  const int tid = threadIdx.x, lane = tid & 63;
  const int np = o.pair_end - o.pair_begin;
  int ksum = 0;
  if (np > 0) {
    const GemmPair last = pairs[o.pair_end - 1];
    ksum = last.k0 + last.K;
  }
  for (int q = tid >> 4; q < np; q += 16) {
    const GemmPair pr = pairs[o.pair_begin + q];
    for (int k = tid & 15; k < pr.K; k += 16)
      ks[pr.k0 + k] = {pr.a_off + k * pr.a_cs, pr.a_rs, pr.b_off + k * pr.b_rs, pr.b_cs};
  }
  __syncthreads();
  if (o.N <= 0) return;
  const int cl = lane & 15, kq = lane >> 4;
  const int64_t n = min(cl, o.N - 1);
  const int64_t end = min(int64_t(t.row0) + rows, int64_t(o.M));
  for (int64_t first = t.row0; first < end; first += 64 * RT) {
    const int m0 = int(first) + (tid >> 6) * 16 * RT;
    if (m0 >= o.M) return;
    int64_t m[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) m[i] = min(m0 + 16 * i + cl, o.M - 1);
    v4d acc[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] = v4d{0.0, 0.0, 0.0, 0.0};
    // chunk c: k = 4 c .. 4 c + 3 of the list, one per lane quarter; loads past
    // the list's end repeat its last k, and their values are dropped
    auto load = [&](int c, double (&a)[RT], double& b) {
      const RowK e = ks[min(4 * c + kq, ksum - 1)];
      b = base[e.b_off + n * e.b_cs];
#pragma unroll
      for (int i = 0; i < RT; ++i) a[i] = base[e.a_off + m[i] * e.a_rs];
    };
    auto multiply = [&](int c, double (&a)[RT], double b) {
      if (4 * c + 4 > ksum) {
        const bool in = 4 * c + kq < ksum;
        b = in ? b : 0.0;
#pragma unroll
        for (int i = 0; i < RT; ++i) a[i] = in ? a[i] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(b, a[i], acc[i], 0, 0, 0);
    };
    if (ksum > 0) {
      const int nc = (ksum + 3) / 4;
      double a0[RT], a1[RT], b0, b1;
      load(0, a0, b0);
      load(1, a1, b1);
      if (nc <= 2) {
        multiply(0, a0, b0);
        if (nc == 2) multiply(1, a1, b1);
      } else {
        for (int c = 0; c < nc; c += 2) {
          multiply(c, a0, b0);
          load(c + 2, a0, b0);
          if (c + 1 < nc) multiply(c + 1, a1, b1);
          load(c + 3, a1, b1);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int row = m0 + 16 * i + cl;
      double* C = base + o.c_off + int64_t(row) * o.ldc;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = 4 * r + kq;  // f64 MFMA output layout, transposed
        if (row < o.M && col < o.N) {
          double v = alpha * acc[i][r];
          if (beta != 0.0) v += beta * C[col];
          C[col] = v;
        }
      }
    }
  }
}

void gemm_rows(hipStream_t s, double* base, const Lists& l, int ntasks, int task_rows, double alpha, double beta) {
  if (ntasks <= 0) return;
  if (task_rows % 128 == 0)
    launch_lists(k_gemm_rows<DevLists, 2>, k_gemm_rows<ArgLists, 2>, l, dim3(ntasks), dim3(256), 0, s, base, l.at[3],
                 l.at[1], l.at[2], task_rows, alpha, beta);
  else
    launch_lists(k_gemm_rows<DevLists, 1>, k_gemm_rows<ArgLists, 1>, l, dim3(ntasks), dim3(256), 0, s, base, l.at[3],
                 l.at[1], l.at[2], task_rows, alpha, beta);
}

GemmLayout gemm_layout(const GemmPair* pairs, size_t n, const GemmOut* outs, size_t nouts) {
  bool ak = true, am = true, bk = true, bn = true;
  for (size_t o = 0; o < nouts; ++o)
    for (int32_t q = outs[o].pair_begin; q < outs[o].pair_end && size_t(q) < n; ++q) {
      const GemmPair& p = pairs[q];
      if (p.K <= 0) continue;
      // one k or one row: that dimension's stride is never used; the threads'
      // offsets are 32-bit byte counts (whole rows, or 16 k of all rows)
      const int64_t M = outs[o].M, N = outs[o].N, lim = int64_t(1) << 29;
      ak &= (p.a_cs == 1 || p.K == 1) && M * p.a_rs + KS < lim;
      am &= (p.a_rs == 1 || M == 1) && KS * p.a_cs + M < lim;
      bk &= (p.b_rs == 1 || p.K == 1) && N * p.b_cs + KS < lim;
      bn &= (p.b_cs == 1 || N == 1) && KS * p.b_rs + N < lim;
    }
  if (!(ak || am) || !(bk || bn)) return kLayoutAny;
  return GemmLayout((ak ? 1 : 0) | (bn ? 2 : 0));
}

template <int T, bool AK, bool BN>
static void gemm_contiguous(hipStream_t s, double* base, const Lists& l, int ntiles, double alpha, double beta) {
  launch_lists(k_gemm_f64c<DevLists, T, AK, BN>, k_gemm_f64c<ArgLists, T, AK, BN>, l, dim3(ntiles), dim3(256), 0, s,
               base, l.at[0], l.at[1], l.at[2], alpha, beta);
}

template <int T>
static void gemm_contiguous(hipStream_t s, GemmLayout lay, double* base, const Lists& l, int ntiles, double alpha,
                            double beta) {
  switch (int(lay)) {
    case 0: gemm_contiguous<T, false, false>(s, base, l, ntiles, alpha, beta); break;
    case 1: gemm_contiguous<T, true, false>(s, base, l, ntiles, alpha, beta); break;
    case 2: gemm_contiguous<T, false, true>(s, base, l, ntiles, alpha, beta); break;
    default: gemm_contiguous<T, true, true>(s, base, l, ntiles, alpha, beta); break;
  }
}

void gemm_f64(hipStream_t s, int tile, GemmLayout lay, double* base, const Lists& l, int ntiles, double alpha,
              double beta) {
  if (ntiles <= 0) return;
  if (lay == kLayoutAny)
    launch_lists(k_gemm_f64t<DevLists>, k_gemm_f64t<ArgLists>, l, dim3(ntiles), dim3(256), 0,
                 s, base, l.at[0], l.at[1], l.at[2], alpha, beta);
  else if (tile == 32)
    gemm_contiguous<32>(s, lay, base, l, ntiles, alpha, beta);
  else
    gemm_contiguous<64>(s, lay, base, l, ntiles, alpha, beta);
}

void gemm_split(hipStream_t s, double* base, const Lists& l, int ntiles, double alpha, double beta) {
  if (ntiles <= 0) return;
  launch_lists(k_gemm_split<DevLists>, k_gemm_split<ArgLists>, l, dim3(ntiles), dim3(256), 0, s, base, l.at[0],
               l.at[1], l.at[2], alpha, beta);
}

// Scratch of the allocation-free contraction (packed operands, split-K
// partials, launch descriptors).  Every GPU the library runs on holds its
// own copy for the life of the process.  In host code this name stands for
// the variable, not for a device address: host code uses only the address
// hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) char scratch[kNoAllocScratchBytes];

hipError_t noalloc_scratch_address(int device, void** out) {
  static std::mutex mu;
  static std::map<int, void*> addr;
  std::lock_guard<std::mutex> lk(mu);
  auto it = addr.find(device);
  if (it != addr.end()) {
    *out = it->second;
    return hipSuccess;
  }
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  addr[device] = p;
  *out = p;
  return hipSuccess;
}

}  // namespace kern
}  // namespace qtt
