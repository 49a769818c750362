// Data movement, elementwise and reduction kernels (HBM-bound).  Work is
// split into (descriptor, chunk) tasks of kChunk elements so a launch always
// has many work-groups regardless of how uneven the blocks are.
#include <algorithm>

#include "../kernels.hpp"

namespace qtt {
namespace kern {

// A permuted copy whose last dim is not the contiguous one of the source goes
// through LDS in tiles of up to 32 elements along the source's contiguous dim
// and as many along the last as make 2048, so that both sides are read and
// written in order (a tile is read in the source's order: where its two dims
// are the source's last two that is one piece of memory).  The others copy
// element by element in the destination's order, offsets by 32-bit divisions.
// 121 MB in blocks of up to 272 x 272 x 12 with the last two dims exchanged: 22
// us, against 83 with a 64-bit division per element and dim.
//
// A tile is a work-group with a task of its own, however little it holds, so
// tiles are taken where they hold kPermTileMin elements on average.  8 M
// elements, last dims m and n exchanged, list upload included, tiles against
// element by element (us): m 4, n 16 617 / 35; 8, 32 77 / 36; 16, 32 46 / 40; 16,
// 48 35 .. 47 / 41; 8, 128 29 .. 38 / 37; 16, 64 29 .. 38 / 43; 32, 64 26 / 44 (the
// larger ones where the staging ring's pages are read for the first time).
constexpr int kPermTile = 32, kPermElems = 2048, kPermTileMin = 1024;
int64_t permute_plan(PermDesc& d) {
  int r = 0;
  for (int i = 0; i < d.rank; ++i) {
    if (d.dims[i] == 1) continue;
    if (r && d.sstride[r - 1] == d.sstride[i] * d.dims[i] && int64_t(d.dims[r - 1]) * d.dims[i] <= INT32_MAX) {
      d.dims[r - 1] *= d.dims[i];
      d.sstride[r - 1] = d.sstride[i];
    } else {
      d.dims[r] = d.dims[i];
      d.sstride[r++] = d.sstride[i];
    }
  }
  if (r == 0) {
    d.dims[0] = 1;
    d.sstride[r++] = 1;
  }
  d.rank = r;
  d.tj = -1;
  d.tn = 0;
  const int n = d.dims[r - 1];
  if (d.sstride[r - 1] != 1 && n >= 16)
    for (int j = 0; j + 1 < r; ++j)
      if (d.sstride[j] == 1 && d.dims[j] >= 4) d.tj = j;
  if (d.tj >= 0) {
    const int m = d.dims[d.tj];
    d.tn = kPermElems / std::min(m, kPermTile) / 64 * 64;
    const int64_t tiles = (int64_t(m) + kPermTile - 1) / kPermTile * ((int64_t(n) + d.tn - 1) / d.tn);
    if (int64_t(m) * n >= tiles * kPermTileMin) return d.numel / m / n * tiles;
    d.tj = -1;
  }
  return (d.numel + kChunk - 1) / kChunk;
}

template <class L>
__global__ __launch_bounds__(256) void k_permute(double* __restrict__ base, L l, uint32_t tasks) {
  __shared__ double tile[kPermElems + kPermTile];
  const ChunkTask t = l.template list<ChunkTask>(tasks)[blockIdx.x];
  const PermDesc* d = l.template list<PermDesc>() + t.desc;
  const double* src = base + d->src_off;
  double* dst = base + d->dst_off;
  const int rank = d->rank;
  if (d->tj < 0) {
    const int64_t start = int64_t(t.chunk) * kChunk;
    const int64_t end = min(start + int64_t(kChunk), d->numel);
    const bool small = d->numel < (int64_t(1) << 31);
    for (int64_t e = start + threadIdx.x; e < end; e += blockDim.x) {
      int64_t off = 0;
      if (small) {
        uint32_t rem = uint32_t(e);
        for (int k = rank - 1; k > 0; --k) {
          const uint32_t q = rem / uint32_t(d->dims[k]);
          off += int64_t(rem - q * uint32_t(d->dims[k])) * d->sstride[k];
          rem = q;
        }
        off += int64_t(rem) * d->sstride[0];
      } else {
        int64_t rem = e;
        for (int k = rank - 1; k > 0; --k) {
          const int64_t q = rem / d->dims[k];
          off += (rem - q * d->dims[k]) * d->sstride[k];
          rem = q;
        }
        off += rem * d->sstride[0];
      }
      dst[e] = src[off];
    }
    return;
  }
  const int m = d->dims[d->tj], n = d->dims[rank - 1], tn = d->tn;
  const int64_t sn = d->sstride[rank - 1];
  const int nm = (m + kPermTile - 1) / kPermTile, nn = (n + tn - 1) / tn;
  int c = t.chunk;
  const int n0 = (c % nn) * tn;
  c /= nn;
  const int j0 = (c % nm) * kPermTile;
  c /= nm;
  int64_t dj = 0, ds = n;  // destination stride of the tiled dim, of the dim at hand
  src += j0 + n0 * sn;
  dst += n0;
  for (int k = rank - 2; k >= 0; --k) {
    if (k == d->tj) {
      dj = ds;
    } else {
      const int q = c / d->dims[k], i = c - q * d->dims[k];
      src += i * d->sstride[k];
      dst += i * ds;
      c = q;
    }
    ds *= d->dims[k];
  }
  dst += j0 * dj;
  const int mj = min(kPermTile, m - j0), nj = min(tn, n - n0), pitch = tn + 1;
  const uint32_t inv = ((1u << 20) + mj - 1) / mj;  // x / mj for x < 2^11 + 2^5
  for (int x = threadIdx.x; x < mj * nj; x += blockDim.x) {
    const int i = int((uint32_t(x) * inv) >> 20), j = x - i * mj;
    tile[j * pitch + i] = src[j + i * sn];
  }
  __syncthreads();
  for (int j = threadIdx.x >> 6; j < mj; j += 4)
    for (int i = threadIdx.x & 63; i < nj; i += 64) dst[j * dj + i] = tile[j * pitch + i];
}

void permute_copy(hipStream_t s, double* base, const Lists& l, int ntasks) {
  if (ntasks <= 0) return;
  launch_lists(k_permute<DevLists>, k_permute<ArgLists>, l, dim3(ntasks), dim3(256), 0, s, base, l.at[1]);
}

// A task's elements: thread i takes start + i, + 256, ...  Its kPer loads are
// issued before the first result is used (an element past the end repeats the
// last): one after the other they are a chain of memory latencies, which is
// what bounds launches of this size.  At the products of a D = 1024 cylinder
// site sum_parts took 18.9 us and takes 9.0, copies and sums 5.2 -> 4.9 and a
// dot's partials 5.7 -> 4.5; a dot of 20 k elements in one launch 7.4 -> 5.3
// (together with block_sum, whose tree in LDS had eight barriers).
// No task has no elements: a descriptor of numel elements has ceil(numel /
// kChunk) of them.
constexpr int kPer = kChunk / 256;
struct Chunk {
  int64_t first, end;
  __device__ Chunk(const ChunkTask& t, int64_t numel)
      : first(int64_t(t.chunk) * kChunk + threadIdx.x), end(min(int64_t(t.chunk + 1) * kChunk, numel)) {}
  __device__ bool has(int u) const { return first + u * 256 < end; }
  __device__ int64_t at(int u) const { return min(first + u * 256, end - 1); }
};

template <class L>
__global__ __launch_bounds__(256) void k_copy2d(double* __restrict__ base, L l, uint32_t tasks) {
  const ChunkTask t = l.template list<ChunkTask>(tasks)[blockIdx.x];
  const Copy2D d = l.template list<Copy2D>()[t.desc];
  const int64_t numel = int64_t(d.rows) * d.cols;
  const Chunk c(t, numel);
  double* dst = base + d.dst_off;
  const double* src = base + (d.src_off < 0 ? 0 : d.src_off);
  int64_t to[kPer];
  double v[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int64_t e = c.at(u);
    int64_t r = 0;
    if (d.rows > 1) r = numel < (int64_t(1) << 31) ? int64_t(uint32_t(e) / uint32_t(d.cols)) : e / d.cols;
    const int64_t q = e - r * d.cols;
    to[u] = r * d.dst_rs + q * d.dst_cs;
    v[u] = d.src_off < 0 ? 1.0 : src[r * d.src_rs + q * d.src_cs];
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u)
    if (c.has(u)) dst[to[u]] = d.alpha * v[u];
}

// dst[i] = sum over s < parts of src[s * n + i] (fixed order): the reduction of
// split-K partial products.  desc = {dst_off, src_off, n, parts}.
template <class L>
__global__ __launch_bounds__(256) void k_sum_parts(double* __restrict__ base, L l, uint32_t descs,
                                                   uint32_t tasks) {
  const ChunkTask t = l.template list<ChunkTask>(tasks)[blockIdx.x];
  const SumParts d = l.template list<SumParts>(descs)[t.desc];
  const Chunk c(t, d.n);
  double v[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) v[u] = 0.0;
  const double* src = base + d.src_off;
#pragma unroll 2
  for (int p = 0; p < d.parts; ++p, src += d.n) {
    double x[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) x[u] = src[c.at(u)];
#pragma unroll
    for (int u = 0; u < kPer; ++u) v[u] += x[u];
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u)
    if (c.has(u)) base[d.dst_off + c.at(u)] = v[u];
}

void sum_parts(hipStream_t s, double* base, const Lists& l, int ntasks, int first) {
  if (ntasks <= 0) return;
  launch_lists(k_sum_parts<DevLists>, k_sum_parts<ArgLists>, l, dim3(ntasks), dim3(256), 0, s, base, l.at[first],
               l.at[first + 1]);
}

void copy2d(hipStream_t s, double* base, const Lists& l, int ntasks) {
  if (ntasks <= 0) return;
  launch_lists(k_copy2d<DevLists>, k_copy2d<ArgLists>, l, dim3(ntasks), dim3(256), 0, s, base, l.at[1]);
}

template <class L>
__global__ __launch_bounds__(256) void k_ew_binary(double* __restrict__ base, L l, uint32_t tasks, int op, double min_abs) {
  const ChunkTask t = l.template list<ChunkTask>(tasks)[blockIdx.x];
  const EwDesc d = l.template list<EwDesc>()[t.desc];
  const Chunk c(t, d.numel);
  const double* x = base + d.x_off;
  const double* y = base + d.y_off;
  double* out = base + d.out_off;
  double xv[kPer], yv[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int64_t e = c.at(u);
    xv[u] = x[e];
    if (d.mode == 0)
      yv[u] = y[0];
    else if (d.mode == 1)
      yv[u] = y[d.numel < (int64_t(1) << 31) ? int64_t(uint32_t(e) % uint32_t(d.ncol)) : e % d.ncol];
    else
      yv[u] = y[e];
  }
  const bool skip = d.mode == 0 && op == 1 && fabs(yv[0]) < min_abs;
#pragma unroll
  for (int u = 0; u < kPer; ++u)
    if (c.has(u)) out[c.at(u)] = skip ? xv[u] : op == 0 ? xv[u] * yv[u] : xv[u] / yv[u];
}

void ew_binary(hipStream_t s, double* base, const Lists& l, int ntasks, int op,
               double min_abs) {
  if (ntasks <= 0) return;
  launch_lists(k_ew_binary<DevLists>, k_ew_binary<ArgLists>, l, dim3(ntasks), dim3(256), 0, s, base, l.at[1], op, min_abs);
}

template <class L>
__global__ __launch_bounds__(256) void k_axpby(double* __restrict__ base, L l, uint32_t tasks, int64_t a_off, double a,
                                               int64_t b_off, double b) {
  const ChunkTask t = l.template list<ChunkTask>(tasks)[blockIdx.x];
  const AxpbyDesc d = l.template list<AxpbyDesc>()[t.desc];
  const Chunk c(t, d.numel);
  const double av = a_off >= 0 ? base[a_off] : a;
  const double bv = b_off >= 0 ? base[b_off] : b;
  double* out = base + d.out_off;
  const double* x = d.x_off >= 0 ? base + d.x_off : nullptr;
  const double* y = d.y_off >= 0 ? base + d.y_off : nullptr;
  double xv[kPer], yv[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int64_t e = c.at(u);
    xv[u] = x ? x[e] : 0.0;
    yv[u] = y ? y[e] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const double px = av * xv[u], py = bv * yv[u];
    if (c.has(u)) out[c.at(u)] = x && y ? px + py : x ? px : py;
  }
}

void axpby(hipStream_t s, double* base, const Lists& l, int ntasks, int64_t a_off,
           double a, int64_t b_off, double b) {
  if (ntasks <= 0) return;
  launch_lists(k_axpby<DevLists>, k_axpby<ArgLists>, l, dim3(ntasks), dim3(256), 0, s, base, l.at[1], a_off, a, b_off, b);
}

// Block-wide sum in fixed order (deterministic): the waves' sums by lane
// exchanges, then the four of them.
__device__ double block_sum(double v, double* sh) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const double r = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return r;
}

// A thread's part of a task of a dot product.
__device__ __forceinline__ double chunk_dot(const double* __restrict__ base, const DotDesc& d, const ChunkTask& t) {
  const Chunk c(t, d.numel);
  double x[kPer], y[kPer], acc = 0.0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    x[u] = base[d.x_off + c.at(u)];
    y[u] = base[d.y_off + c.at(u)];
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u)
    if (c.has(u)) acc += x[u] * y[u];
  return acc;
}

template <class L>
__global__ __launch_bounds__(256) void k_dot_partial(double* __restrict__ base, L l, uint32_t tasks, int64_t partial_off) {
  __shared__ double sh[4];
  const ChunkTask t = l.template list<ChunkTask>(tasks)[blockIdx.x];
  const DotDesc d = l.template list<DotDesc>()[t.desc];
  const double acc = chunk_dot(base, d, t);
  const double r = block_sum(acc, sh);
  if (threadIdx.x == 0) base[partial_off + blockIdx.x] = r;
}

__global__ __launch_bounds__(256) void k_dot_final(double* __restrict__ base, int64_t partial_off, int n,
                                                   int64_t out_off, int sqrt_out) {
  __shared__ double sh[4];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) acc += base[partial_off + i];
  const double r = block_sum(acc, sh);
  if (threadIdx.x == 0) base[out_off] = sqrt_out ? sqrt(r) : r;
}

// The same in one launch: the work-group that finishes last sums the partials,
// in the same order.  *done: zero between launches; partials pass through
// memory at agent scope, and each group's release writes back its cache, so the
// second launch is ahead from 64 tasks on (1, 32, 64, 128 tasks: 5.2, 5.7, 6.2,
// 7.7 us against 5.4, 6.0, 6.0, 6.2 for two launches, which also take the host
// 2.3 us more).
constexpr int kDotOneLaunch = 64;
template <class L>
__global__ __launch_bounds__(256) void k_dot(double* __restrict__ base, L l, uint32_t tasks, int64_t partial_off,
                                             int64_t out_off, int sqrt_out, int* __restrict__ done) {
  __shared__ double sh[4];
  __shared__ int last;
  const int n = gridDim.x;
  double* partial = base + partial_off;
  {
    const ChunkTask t = l.template list<ChunkTask>(tasks)[blockIdx.x];
    const DotDesc d = l.template list<DotDesc>()[t.desc];
    const double acc = chunk_dot(base, d, t);
    const double r = block_sum(acc, sh);
    if (n == 1) {  // uniform
      if (threadIdx.x == 0) base[out_off] = sqrt_out ? sqrt(r) : r;
      return;
    }
    if (threadIdx.x == 0) {
      __hip_atomic_store(&partial[blockIdx.x], r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = __hip_atomic_fetch_add(done, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    }
    __syncthreads();
    if (!last) return;
  }
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x)
    acc += __hip_atomic_load(&partial[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const double r = block_sum(acc, sh);
  if (threadIdx.x == 0) {
    base[out_off] = sqrt_out ? sqrt(r) : r;
    __hip_atomic_store(done, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

void dot(hipStream_t s, double* base, const Lists& l, int ntasks, int64_t partial_off, int64_t out_off, bool sqrt_out,
         int* done) {
  if (ntasks > 0 && ntasks <= kDotOneLaunch) {
    launch_lists(k_dot<DevLists>, k_dot<ArgLists>, l, dim3(ntasks), dim3(256), 0, s, base, l.at[1], partial_off,
                 out_off, int(sqrt_out), done);
    return;
  }
  if (ntasks > 0)
    launch_lists(k_dot_partial<DevLists>, k_dot_partial<ArgLists>, l, dim3(ntasks), dim3(256), 0, s, base, l.at[1],
                 partial_off);
  hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(256), 0, s, base, partial_off, ntasks, out_off, int(sqrt_out));
}

__global__ void k_eig2x2(double* __restrict__ base, int64_t a0_off, int64_t a1_off, int64_t b_off, int64_t out_off,
                         int* flags) {
  if (threadIdx.x != 0) return;
  const double a0 = base[a0_off], a1 = base[a1_off], b = base[b_off];
  const double d = a0 - a1;
  const double crit = sqrt(d * d + 4.0 * (b * b));
  const double E0 = (a0 + a1 - crit) / 2.0;
  const double delt = E0 - a1;
  double o = sqrt(delt / (-crit));
  double n = (b * o) / delt;
  const bool zero_o = ((o + E0) == E0) || isnan(o);
  if (zero_o) {
    n = 1.0;
    o = 0.0;
  }
  flags[0] = isnan(o) || isnan(n);
  base[out_off + 0] = E0;
  base[out_off + 1] = o;
  base[out_off + 2] = n;
}

void eig2x2(hipStream_t s, double* base, int64_t a0_off, int64_t a1_off, int64_t b_off, int64_t out_off,
            int* flags) {
  hipLaunchKernelGGL(k_eig2x2, dim3(1), dim3(64), 0, s, base, a0_off, a1_off, b_off, out_off, flags);
}

__global__ __launch_bounds__(256) void k_normalize(double* __restrict__ base, int64_t off, int64_t n) {
  __shared__ double sh[4];
  double* d = base + off;
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) acc += d[i] * d[i];
  const double nrm = sqrt(block_sum(acc, sh));
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) d[i] = d[i] / nrm;
}

void normalize(hipStream_t s, double* base, int64_t off, int64_t n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_normalize, dim3(1), dim3(256), 0, s, base, off, n);
}

// The last thread of the grid copies what is left of a whole 16 bytes.
__global__ __launch_bounds__(256) void k_stage_copy(uint4* __restrict__ dst, const uint4* __restrict__ src, size_t n,
                                                    int tail) {
  const size_t step = size_t(gridDim.x) * blockDim.x, i0 = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  for (size_t i = i0; i < n; i += step) dst[i] = src[i];
  if (i0 == step - 1)
    for (int b = 0; b < tail; ++b) reinterpret_cast<char*>(dst + n)[b] = reinterpret_cast<const char*>(src + n)[b];
}

void stage_copy(hipStream_t s, void* dst, const void* src, size_t bytes) {
  const size_t n = bytes / 16, g = (n + 255) / 256;
  hipLaunchKernelGGL(k_stage_copy, dim3(unsigned(std::min<size_t>(std::max<size_t>(g, 1), 1024))), dim3(256), 0, s,
                     static_cast<uint4*>(dst), static_cast<const uint4*>(src), n, int(bytes % 16));
}

}  // namespace kern
}  // namespace qtt
