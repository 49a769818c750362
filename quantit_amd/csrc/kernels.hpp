// Host-side launchers of the gfx950 kernels.  Every device pointer is the
// context arena base plus an element (double) offset, so descriptor lists are
// plain integer records.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <memory>
#include <string>
#include <vector>

#include "qtt_common.hpp"

namespace qtt {
namespace kern {

// ---- descriptor lists of a launch --------------------------------------------
// A launch reads its descriptors either from device memory or, when they are
// short, from its own arguments (a kernel takes up to 4 KB).  An upload is a
// dispatch of its own in front of every launch: upload and a small kernel 5.2
// us back to back (4.8 of the host), with 3 KB of arguments 3.0 (2.7), without
// descriptors 2.7 (2.3).
constexpr size_t kArgListBytes = 3584;
struct ArgLists {
  alignas(16) char b[kArgListBytes];
  template <class T>
  __device__ __forceinline__ const T* list(uint32_t at = 0) const {
    return reinterpret_cast<const T*>(b + at);
  }
};
struct DevLists {
  const char* p;
  // constant while the kernel runs: uniform reads stay scalar loads
  template <class T>
  __device__ __forceinline__ const T* list(uint32_t at = 0) const {
    using Const = const __attribute__((address_space(4))) char;
    return (const T*)((Const*)p + at);
  }
};
// The lists of one launch, list i at byte at[i].
struct Lists {
  const char* dev = nullptr;  // null: in arg
  std::shared_ptr<void> own;  // device memory of their own, until the launches are enqueued
  uint32_t at[6] = {0, 0, 0, 0, 0, 0};
  ArgLists arg;
  Lists() {}
};
// Launches the DevLists or the ArgLists instance of a kernel over its lists.
template <class D, class A, class... X>
void launch_lists(D dev, A arg, const Lists& l, dim3 grid, dim3 block, size_t lds, hipStream_t s, double* base,
                  X... x) {
  if (l.dev)
    hipLaunchKernelGGL(dev, grid, block, lds, s, base, DevLists{l.dev}, x...);
  else
    hipLaunchKernelGGL(arg, grid, block, lds, s, base, l.arg, x...);
}
// Copy of pinned host memory into device memory by a kernel (both 16-byte
// aligned): the runtime's own copy takes 20 us from 64 KB on, this 6.
void stage_copy(hipStream_t s, void* dst, const void* src, size_t bytes);

// ---- grouped block GEMM ---------------------------------------------------
// C_out = alpha * sum_p A_p * B_p + beta * C_out for every output block, the
// pairs of one output block taken in list order (the reference's mm +
// addmm_ order, sources/btensor.cpp:2095-2102).  A_p[m,k] =
// base[a_off + m*a_rs + k*a_cs], B_p[k,n] = base[b_off + k*b_rs + n*b_cs];
// C is row-major M x N at c_off with row pitch ldc.
struct GemmOut {
  int64_t c_off;
  int32_t M, N;
  int32_t pair_begin, pair_end;
  int32_t ldc, pad;  // row pitch of C (N for a packed block)
};
struct GemmPair {
  int64_t a_off, b_off;
  int64_t a_rs, a_cs, b_rs, b_cs;
  int32_t K, k0;  // k0: summed K of the output's pairs before this one (gemm_rows)
};
struct GemmTile {
  int32_t out;
  uint16_t tm, tn;  // tile coordinates inside the output block
};
constexpr int kGemmTile = 64;
// Rows or columns of an output block that tiles of edge T can address: 2.1 M
// for T = 32, 4.2 M for 64.
constexpr int64_t gemm_tile_reach(int T) { return int64_t(T) << 16; }
// Adds the tiles of one M x N output block to a list, row by row.
inline void add_tiles(std::vector<GemmTile>& tiles, int out, int64_t M, int64_t N, int T) {
  if (std::max(M, N) > gemm_tile_reach(T))
    throw InvalidArgument("output block of " + std::to_string(M) + " x " + std::to_string(N) +
                          " elements: more than " + std::to_string(gemm_tile_reach(T)) + " rows or columns");
  const int64_t tm = (M + T - 1) / T, tn = (N + T - 1) / T;
  for (int64_t i = 0; i < tm; ++i)
    for (int64_t j = 0; j < tn; ++j) tiles.push_back({int32_t(out), uint16_t(i), uint16_t(j)});
}
// How the operands of a launch are contiguous: bit 0 A in k (else in m), bit 1
// B in n (else in k), common to all its pairs; kLayoutAny: in no common way.
enum GemmLayout : int { kLayoutAny = -1 };
GemmLayout gemm_layout(const GemmPair* pairs, size_t n, const GemmOut* outs, size_t nouts);
// Lists of the GEMM launches: GemmTile, GemmOut, GemmPair, RowTask.
// The grouped FP64 GEMM with 64 x 64 or 32 x 32 tiles (tile; a tile's tm, tn
// count in its own units).  Launches of kLayoutAny take 64 x 64 tiles.
void gemm_f64(hipStream_t s, int tile, GemmLayout lay, double* base, const Lists& l, int ntiles, double alpha,
              double beta);
// Tile choices of the tuning table and of QTT_GEMM_VARIANT, by number: 5 is
// the 32 x 32 tile, every other number the 64 x 64 one (0 the general kernel;
// 2 to 4 are numbers of wider tiles in tables of older builds, whose 0 and 5
// are not taken over).
enum GemmVariant : int { kTileAny = 0, kTile64 = 1, kTile32 = 5, kGemmVariants = 6 };
inline int variant_tile(int v) { return v == kTile32 ? 32 : 64; }
// Tile of a launch that is not timed: 32 x 32 below this many 64 x 64 tiles
// (three per CU), where the longest tile and the idle CUs decide: 225 tiles
// 161 us against 245, 218 tiles 24.4 against 33.1; from 1024 tiles on the 64 x
// 64 tile is ahead (323 us against 430 at 1024, 107 against 136 at 5707).
constexpr int64_t kTile64Min = 768;

// Size of the file-scope device scratch (kernels/gemm.hip) that the
// allocation-free contraction takes its packed operands, split-K partials
// and descriptors from.
// 128 MiB beside what lists need: a task of 64 or 128 rows, of a tile of 1024
// permuted elements or of a 32 x 32 product takes 8 bytes, so that 32 MiB hold
// those of 2^29 rows.
constexpr size_t kNoAllocScratchBytes = size_t(160) << 20;
// Device address of that scratch on `device` (which must be current):
// hipGetSymbolAddress on the first call per device, cached afterwards.
hipError_t noalloc_scratch_address(int device, void** out);
// hi/lo split FP32 MFMA: each operand x = hi + lo (hi = fp32(x), lo =
// fp32(x - hi)); products hi*hi + hi*lo + lo*hi accumulate in FP32 per K
// chunk and are folded into FP64 accumulators after every chunk.
void gemm_split(hipStream_t s, double* base, const Lists& l, int ntiles, double alpha, double beta);
// Output blocks with at most kRowsMaxN columns and a short summed K.  A task is
// 64, 128 or a multiple of 128 (task_rows) consecutive rows of one output
// block: 64 while the work-groups all fit on the chip at once (30 blocks of 300
// rows, K 128: 8.6 us against 9.9; 72 k rows 4.1 against 4.2), above that 128,
// whose longer streams hide more (760 k rows of 7 and 12 columns, K 33: 46.8 us
// against 52.3, 85.6 for one thread a row).  Up to K = 16 the rows are soon done
// and the list of tasks counts, so from 2^19 rows on a task takes several 128,
// about 4096 tasks in all: 1 M rows, N 3, K 5 26 us a call against 39, 8 M rows,
// N 2, K 2 72 against 99.  (Longer K: 600 k rows, N 16, K 100 133 us against 124.)
constexpr int kRowsMaxN = 16, kRowsMaxK = 128;
struct RowTask {
  int32_t out, row0;
};
inline int rows_per_task(int64_t rows, int64_t longest_k) {
  if (rows < 64 * 2048) return 64;
  return longest_k > 16 ? 128 : 128 * int(std::min<int64_t>((rows + (int64_t(1) << 19) - 1) >> 19, 64));
}
void gemm_rows(hipStream_t s, double* base, const Lists& l, int ntasks, int task_rows, double alpha, double beta);

// ---- data movement ----------------------------------------------------------
// Row-major copy of a permuted view: dst element with multi-index j over
// dims[0..rank) (row-major) reads src[sum_k j_k * sstride[k]].
struct PermDesc {
  int64_t src_off, dst_off, numel;
  int32_t rank;
  int32_t tj, tn;  // set by permute_plan: tiled dim (-1: none) and its tiles' length along the last dim
  int32_t dims[8];
  int64_t sstride[8];
};
// Merges the dims of a descriptor where it can, chooses how it is copied and
// returns its number of tasks (chunks 0 .. of the descriptor).
int64_t permute_plan(PermDesc& d);
struct ChunkTask {
  int32_t desc;
  int32_t chunk;
};
// Elements per work-group task of the element-wise kernels: 8 per thread of
// a 256-thread group, loaded together, so a task is one memory round trip and
// a launch spreads over many work-groups.
constexpr int kChunk = 2048;
// The lists of these launches: descriptors, ChunkTasks.
void permute_copy(hipStream_t s, double* base, const Lists& l, int ntasks);

// 2-D strided copy dst[r*dst_rs + c*dst_cs] = alpha * src[r*src_rs + c*src_cs];
// src_off < 0 fills the destination with the value alpha.
struct Copy2D {
  int64_t src_off, dst_off;
  int64_t src_rs, src_cs, dst_rs, dst_cs;
  int32_t rows, cols;
  double alpha;
};
void copy2d(hipStream_t s, double* base, const Lists& l, int ntasks);
struct SumParts {
  int64_t dst_off, src_off, n;
  int32_t parts, pad;
};
// dst = sum of `parts` consecutive arrays of n doubles at src (fixed order).
// The two lists are those from `first` on.
void sum_parts(hipStream_t s, double* base, const Lists& l, int ntasks, int first = 0);

// ---- elementwise / reductions ---------------------------------------------
// out = x (op) y with y broadcast: mode 0 y scalar, 1 y vector along the last
// dim (x viewed as rows x ncol), 2 y same shape.  op 0 = mul, 1 = div.
// For op 1 with mode 0 and min_abs > 0 the division is skipped (plain copy)
// when |y| < min_abs.
struct EwDesc {
  int64_t x_off, y_off, out_off, numel;
  int32_t ncol, mode;
};
void ew_binary(hipStream_t s, double* base, const Lists& l, int ntasks, int op,
               double min_abs);
// out = a*x + b*y; x_off or y_off < 0 means that operand is absent.  a and b
// are read from device scalars when a_off/b_off >= 0, else the host values.
struct AxpbyDesc {
  int64_t x_off, y_off, out_off, numel;
};
void axpby(hipStream_t s, double* base, const Lists& l, int ntasks, int64_t a_off,
           double a, int64_t b_off, double b);
// Deterministic dot product over matched block pairs: one partial per chunk
// task, then a fixed-order tree reduction into base[out_off].  With sqrt_out
// the square root is stored instead.
struct DotDesc {
  int64_t x_off, y_off, numel;
};
void dot(hipStream_t s, double* base, const Lists& l, int ntasks, int64_t partial_off, int64_t out_off, bool sqrt_out,
         int* done);
// Adds a descriptor to a list.  Where it continues the last one in every
// operand it lengthens it: the blocks of a tensor lie packed, so a pass over
// tensors of the same blocks is one run, with full tasks in place of one short
// task a block and lists short enough for the kernel's arguments: a Lanczos
// step on the D = 1024 cylinder 693 us -> 681, with six uploads fewer.
inline bool continues(const EwDesc& p, const EwDesc& d) {
  return p.mode == d.mode && d.mode != 1 && p.x_off + p.numel == d.x_off && p.out_off + p.numel == d.out_off &&
         p.y_off + (d.mode == 2 ? p.numel : 0) == d.y_off;
}
inline bool continues(const AxpbyDesc& p, const AxpbyDesc& d) {
  auto next = [&p](int64_t a, int64_t b) { return a < 0 || b < 0 ? a < 0 && b < 0 : a + p.numel == b; };
  return next(p.x_off, d.x_off) && next(p.y_off, d.y_off) && p.out_off + p.numel == d.out_off;
}
inline bool continues(const DotDesc& p, const DotDesc& d) {
  return p.x_off + p.numel == d.x_off && p.y_off + p.numel == d.y_off;
}
inline bool continues(const Copy2D& p, const Copy2D& d) {
  auto flat = [](const Copy2D& c) { return c.rows == 1 && c.dst_cs == 1 && (c.src_off < 0 || c.src_cs == 1); };
  return flat(p) && flat(d) && p.alpha == d.alpha && int64_t(p.cols) + d.cols <= INT32_MAX &&
         (p.src_off < 0 ? d.src_off < 0 : p.src_off + p.cols == d.src_off) && p.dst_off + p.cols == d.dst_off;
}
inline void lengthen(Copy2D& p, const Copy2D& d) { p.cols += d.cols; }
template <class D>
void lengthen(D& p, const D& d) {
  p.numel += d.numel;
}
template <class D>
void add_run(std::vector<D>& descs, const D& d) {
  if (!descs.empty() && continues(descs.back(), d))
    lengthen(descs.back(), d);
  else
    descs.push_back(d);
}
// The tasks of a list of descriptors.
inline int64_t elements(const Copy2D& d) { return int64_t(d.rows) * d.cols; }
template <class D>
int64_t elements(const D& d) {
  return d.numel;
}
template <class D>
std::vector<ChunkTask> chunk_tasks(const std::vector<D>& descs) {
  std::vector<ChunkTask> tasks;
  for (size_t i = 0; i < descs.size(); ++i)
    for (int64_t c = 0; c * kChunk < elements(descs[i]); ++c) tasks.push_back({int32_t(i), int32_t(c)});
  return tasks;
}
// eig2x2Mat (sources/dmrg.cpp:543-572) on device scalars a0, a1, b; writes
// E, o, n to out[0..3) and 1 to flags[0] on NaN, else 0.
void eig2x2(hipStream_t s, double* base, int64_t a0_off, int64_t a1_off, int64_t b_off, int64_t out_off,
            int* flags);
// d /= sqrt(sum d^2) over n contiguous values.
void normalize(hipStream_t s, double* base, int64_t off, int64_t n);

// ---- k-step Lanczos (kernels/lanczos.hip) -----------------------------------
// Krylov vectors are the rows of V (row pitch ld doubles, n used).
constexpr int kMaxKrylov = 64;
constexpr int kKrylovPerThread = 8;
constexpr int kKrylovChunk = 256 * kKrylovPerThread;
// out[i] = <V[i], w> for i < m (partials: m * ceil(n / kKrylovChunk) doubles).
void krylov_dot(hipStream_t s, double* base, int64_t v_off, int64_t ld, int m, int64_t w_off, int64_t n,
                int64_t partial_off, int64_t out_off);
// dst = src + sign * sum_i coef[i] V[i] (src_off < 0: no src term), divided by
// sqrt(base[scale_off]) when scale_off >= 0.
void krylov_axpy(hipStream_t s, double* base, int64_t v_off, int64_t ld, int m, int64_t coef_off, double sign,
                 int64_t src_off, int64_t dst_off, int64_t n, int64_t scale_off);
// alpha[j] = c1[j] + c2[j], beta[j] = sqrt(nrm2) into T (alpha T[0..K), beta
// T[K..2K)), then the lowest eigenpair of the leading (j+1)-square
// tridiagonal: out = {eigenvalue, residual beta[j] |y[j]|, beta[j], y...};
// host (pinned): the first three, then 1 when a NaN appeared, else 0.
void lanczos_tridiag(hipStream_t s, double* base, int64_t t_off, int K, int j, int64_t c1_off, int64_t c2_off,
                     int64_t nrm2_off, int64_t out_off, double* host);
// A Lanczos step after the matvec in one launch, for short vectors
// (kKrylovStepMaxN): w orthogonalised twice against rows 0 .. j of V, nrm2 =
// |w|^2, row j + 1 = w / |w| (when j + 1 < K), and lanczos_tridiag's results.  w
// itself is left as it was.
constexpr int kKrylovStepMaxN = 8192;
void krylov_step(hipStream_t s, double* base, int64_t v_off, int64_t ld, int j, int K, int64_t w_off, int64_t n,
                 int64_t t_off, int64_t nrm2_off, int64_t out_off, double* host);

// ---- block SVD ----------------------------------------------------------
// Sector work matrices: Y (ell x k, column-major, ld = ell) is orthogonalised
// in place by block one-sided Jacobi; W (k x k, column-major) accumulates the
// rotations.  See svd_jacobi.hip.
struct SvdSector {
  int64_t y_off, w_off;     // work matrices
  int64_t u_off, v_off;     // outputs: U (m x k) and V (n x k) row-major
  int64_t s_off;            // singular values (k), descending
  int32_t m, n, ell, k;     // ell = max(m,n), k = min(m,n)
  int32_t nb;               // number of column blocks (even)
  int32_t transposed;       // 1 when Y = A^T (m < n)
  int32_t flag_idx;         // rotation counter slot
  int32_t eig_shift;        // 1: eigh via shifted SVD (A + c I), values written ascending
  int64_t shift_off;        // device double holding c (eigh mode)
};
constexpr int kSvdBlock = 16;  // columns per Jacobi block
// Start of a decomposition: the work matrices Y (ell x kp) and their partners
// zero, W (kp x kp) and its partner the identity (offsets < 0: none).
struct SvdPrep {
  int64_t y_off, w_off, y2_off, w2_off;
  int32_t ell, kp;
};
void svd_prepare(hipStream_t s, double* base, const Lists& secs, int nsec, int64_t max_elems);
// One round of the block Jacobi tournament; max_ell = largest row count
// among the sectors (picks the LDS-resident kernel when the block pair fits).
// cross_after0: rounds after the first of a sweep rotate only the pairs
// across the two blocks (the first round takes every pair of its blocks).
// skip (may be null): the previous sweep's counters; a sector whose entry is
// 0 has converged and its work-groups return at once.  A work item carries
// the sector fields a round needs, so a work-group starts with one load.
struct RoundWork {
  int64_t y_off, w_off;
  int32_t ell, nb, flag_idx, pair;
};
void svd_round(hipStream_t s, double* base, const RoundWork* work, int nwork, int round, int* counters,
               const int* skip, double tol, int inner_sweeps, int max_ell, int cross_after0);
// norms + ranks (one work-group per sector) and the tiled transposed scatter
// of the (sector, part, row0, col0) tasks into U / V.
void svd_finalize(hipStream_t s, double* base, const Lists& l, const SvdSector* host_secs, int nsec, int ntasks);
// Orthonormal completion of the Z-side columns (Z: ell x k row-major, values
// S descending) whose singular value is numerically zero, for columns
// t < limit only: a truncation that keeps `limit` columns never reads the
// others.  Scratch: v (ell doubles) and p (k doubles).
struct CompleteTask {
  int64_t z_off, s_off, v_off, p_off;
  int32_t ell, k, limit, pad;
};
void svd_complete(hipStream_t s, double* base, const Lists& tasks, int n);
// eigh mode: Y += c I per sector, c = ||A||_F (norm: stored at shift_off) or
// what shift_off holds.
void svd_shift(hipStream_t s, double* base, const Lists& secs, int nsec, bool norm);
void fill_i32(hipStream_t s, int32_t* p, int n, int32_t v);

// One k x k matrix of the one-work-group kernels.
struct SmallJacobi {
  int64_t y_off, w_off;  // input (ell x k, column-major, ld ldy), output (ldw x ldw, column-major)
  int32_t ell, k, ldy, ldw;
  int32_t flag_idx;       // flags[flag_idx]: result count of the kernel (-1: none)
  int32_t aux_idx;        // flags[aux_idx]: second count (gram_eig; -1: none)
  int64_t shift_off = -1;  // >= 0: an eigh, G any symmetric matrix; receives the shift used (gram_eig)
};
size_t gram_eig_lds_limit();  // largest dynamic LDS per work-group (bytes)
// Eigenvectors of k x k Gram matrices (SmallJacobi with ell = k): W written
// k x k at w_off with leading dimension ldw; flags[flag_idx] = pairs of G
// failing the orthogonality test (0: W = I).  precond: pivoted-Cholesky
// preconditioning.
constexpr int kGramEigMaxK = 140;
// Up to kGramEigFew sectors of more than kGramEigFewK columns in an SVD take the
// rounds of gram_rounds.hip instead: one work-group each leaves the chip idle,
// while a round's launches cost the same for one sector as for several.  One
// work-group against rounds (values over 3 and 10 decades, us): 7 sectors of
// k = 140 1941 / 1496 and 3002 / 2592, of 113 1322 / 1227 and 2110 / 2101, of
// 105 1363 / 1448 and 1617 / 1911; 10 of 121 over 8 decades 1951 / 2012; 24 of
// 121 over 12 decades 2334 / 2506.
constexpr int kGramEigFewK = 112, kGramEigFew = 8;
void gram_eig(hipStream_t s, double* base, const Lists& descs, int n, int* flags, double tol, int max_sweeps,
              int precond, size_t lds_bytes);
size_t gram_eig_lds_bytes(int k);
// First-order Gram-Schmidt factor T (k x k at w_off) from the Gram matrix at
// y_off (SmallJacobi; ell: rows of the matrix whose columns they are).
void gs_step(hipStream_t s, double* base, const Lists& descs, int n, int kmax);

// ---- Gram eigenvectors for wide sectors (G in device memory) ---------------
// Orthogonality test of G (SmallJacobi: y_off = G, k, ldy; flag_idx/aux_idx
// as for gram_eig).
void gram_check(hipStream_t s, double* base, const Lists& descs, int n, int* flags, double tol, int kmax);
// Work item of one round of the two-sided block Jacobi on G (gram_rounds.hip):
// the solve of block pair a, tile (a, b) of G (a <= b), or rows
// [64 b, 64 b + 64) of X's column pair a.
enum GramKind : int32_t { kGramSolve = 0, kGramApplyG = 1, kGramApplyX = 2 };
struct GramRound {
  int64_t g0, g1;  // two kp x kp buffers; a sweep starts from the Gram matrix in g0
  int64_t x;       // X, k x kp column-major, leading dimension k
  int64_t q, d;    // 2 x (nb / 2) row-major 32 x 32 blocks each: rotations and rotated blocks, by round parity
  int32_t k, nb, flag, kind;
  int32_t a, b;
};
// Launch `round` (0 .. max nb - 1) of a sweep.  counters[flag] receives the
// pairs of the fresh G over the tolerance (complete after round 1: a sector
// left at 0 has converged and takes no further part); skip: the previous
// sweep's counters or null.
void gram_round(hipStream_t s, double* base, const GramRound* work, int nwork, int round, int* counters,
                const int* skip, double tol);
struct CholPanel {
  int64_t g_off;      // G (k x k, ld k), updated between panels
  int64_t l_off;      // L (k x k, ld k, zeroed), rows in the original order
  int64_t lp_off;     // panel copy (k x nb)
  int64_t state_off;  // ints: [0] rank (k while running), [1 + i] index i pivoted
  int32_t k, pad;
};
// One panel of nb columns starting at j0; LDS kmax * nb doubles.
void pchol_panel(hipStream_t s, double* base, const void* descs, int n, int j0, int nb, int kmax);
// state of every factorisation: [0] = k (running), [1 .. k] = 0 (none pivoted)
void pchol_init(hipStream_t s, double* base, const void* descs, int n);
constexpr int kPcholExtra = 2;  // panel LDS per index besides the columns: running diagonal, flag
size_t pchol_lds_limit();
struct GramVec {
  int64_t x_off, w_off, scratch_off;  // scratch: 3k doubles
  int32_t k, ldx, ldw, pad;
};
void gram_vectors(hipStream_t s, double* base, const Lists& descs, int n, int kmax);

// Global truncation (sources/btensor_linalg.cpp:657-755,
// sources/LinearAlgebra.cpp:57-75): singular values of nsec sectors stored
// descending at s_off[i] with k[i] entries, s_pos[i] = k[0] + ... + k[i-1];
// writes kept[i], and to kept[nsec] whether some sector keeps a value that is
// not above null_scale times its first.
// lists: s_off, s_pos, k
void truncate_select(hipStream_t s, double* base, const Lists& l, int nsec, int64_t scratch_off, int64_t total, double tol, double pow, int64_t min_size,
                     int64_t max_size, double null_scale, int32_t* kept, double* thr_out);

}  // namespace kern
}  // namespace qtt
