// Host arithmetic of the launch lists (kernels.hpp), checked without a device:
// every assertion that fails is printed, the exit status is their number.
#include <cstdio>

#include "kernels.hpp"

using namespace qtt;
static int failed = 0;
#define CHECK(x) \
  if (!(x)) ++failed, std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x)

// The tiles cover the block once, in order, inside it.
static void tiles_of(int64_t M, int64_t N, int T) {
  std::vector<kern::GemmTile> t;
  kern::add_tiles(t, 7, M, N, T);
  const int64_t tm = (M + T - 1) / T, tn = (N + T - 1) / T;
  CHECK(int64_t(t.size()) == tm * tn);
  bool right = true;
  for (size_t q = 0; q < t.size(); ++q)
    right &= t[q].out == 7 && t[q].tm * T == int64_t(q) / tn * T && t[q].tn * T == int64_t(q) % tn * T;
  CHECK(right);
}

static bool refused(int64_t M, int64_t N, int T) {
  try {
    std::vector<kern::GemmTile> t;
    kern::add_tiles(t, 0, M, N, T);
  } catch (const InvalidArgument&) {
    return true;
  }
  return false;
}

// Tasks of a copy of (a, n, m) with its last dims exchanged: no more than one
// for 1024 elements, or one for 2048 where the copy is not tiled.
static void permute_tasks(int a, int n, int m) {
  kern::PermDesc d{};
  d.numel = int64_t(a) * n * m;
  d.rank = 3;
  const int dims[3] = {a, m, n};
  const int64_t st[3] = {int64_t(n) * m, 1, m};
  for (int i = 0; i < 3; ++i) d.dims[i] = dims[i], d.sstride[i] = st[i];
  const int64_t tasks = kern::permute_plan(d);
  CHECK(d.tj < 0 ? tasks == (d.numel + 2047) / 2048 : tasks * 1024 <= d.numel);
}

int main() {
  for (int n : {1, 15, 16, 17, 63, 64, 65, 100, 128, 255, 256, 257, 512, 1000})
    for (int m : {1, 3, 4, 5, 8, 15, 16, 17, 31, 32, 33, 63, 64, 65, 300}) permute_tasks(1000, n, m);
  for (int T : {32, 64}) {
    const int64_t reach = kern::gemm_tile_reach(T);
    for (int64_t m : {int64_t(1), int64_t(T), int64_t(T + 1), int64_t(32767) * T, int64_t(32768) * T,
                      int64_t(32768) * T + 1, reach - 1, reach}) {
      tiles_of(m, T, T);
      tiles_of(T + 1, m, T);
    }
    CHECK(refused(reach + 1, 1, T));
    CHECK(refused(1, reach + 1, T));
  }
  return failed;
}
