// Replays the operand loads of the LDS-staged FP64 / FP32 tiles on the host:
// every thread, load and K step of every tile of a block, with the buffer's
// range check dword by dword.  A byte outside the block that the check lets
// through, an element that arrives wrong, or a nonzero past K is an error.
#include <cstdio>
#include <initializer_list>

#include "tile_loads.hpp"

using namespace vmps;

static long errors = 0;
static void fail(const char* what, int bt, int size, int M, int N, int K, int kb, int tid) {
  if (++errors <= 10)
    std::printf("%s: tile %d, element %d bytes, M %d N %d K %d, kb %d, thread %d\n", what, bt, size, M, N, K, kb, tid);
}

// element `at` (from the load's base, `base` elements into the block of `len`)
// passes the range check; inside the block?
static bool arrives(int64_t at, int range) { return at >= 0 && at < range; }

template <int BT>
static void check(int size, int M, int N, int K) {
  typedef BigRole<BT> Role;
  const int last = (K + kBigKd - 1) / kBigKd * kBigKd + kBigKd;  // the loads run ahead of the product
  for (int kb = 0; kb <= last; kb += kBigKd)
    for (int tid = 0; tid < 256; ++tid) {
      Role t;
      t.init(tid);
      for (int m0 = 0; m0 < M; m0 += BT) {
        const int range = big_a_range(M, K, kb, m0);
        for (int q = 0; q < Role::kNA; ++q) {
          const int64_t at = (int64_t)big_a_first(t.ak, t.ai, M, m0) + big_a_next(Role::kDA, q, M);
          const int k = kb + t.ak + Role::kDA * q, i = lesser(m0 + t.ai, M - 1);
          const int64_t e = (int64_t)kb * M + m0 + at;
          if (arrives(at, range) && (e < 0 || e >= (int64_t)M * K)) fail("A: read outside the block", BT, size, M, N, K, kb, tid);
          if (arrives(at, range) != (k < K)) fail("A: k within K arrives, zero past it", BT, size, M, N, K, kb, tid);
          if (k < K && e != (int64_t)k * M + i) fail("A: another element", BT, size, M, N, K, kb, tid);
        }
      }
      for (int n0 = 0; n0 < N; n0 += BT) {
        const int range = big_b_range(big_b_panel(BT, N, K, n0, size), K, kb);
        for (int h = 0; h < Role::kNB; ++h) {
          const bool in0 = big_b_in(kb, t.bk, K);
          for (int u = 0; u < 2; ++u) {
            const int64_t at = (int64_t)big_b_pair(t.bj, h, t.bk, N, K, n0) + u;
            const int k = kb + t.bk + u, j = lesser(n0 + t.bj + 32 * h, N - 1);
            const int64_t e = (int64_t)n0 * K + kb + at;
            const bool got = in0 && arrives(at, range);
            if (got && (e < 0 || e >= (int64_t)K * N)) fail("B: read outside the block", BT, size, M, N, K, kb, tid);
            if (k < K && (!got || e != (int64_t)j * K + k)) fail("B: another element", BT, size, M, N, K, kb, tid);
            if (u == 0 && k >= K && got) fail("B: nonzero past K", BT, size, M, N, K, kb, tid);
          }
        }
      }
    }
}

int main() {
  const int dims[] = {1, 2, 3, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 200};
  const int depths[] = {1, 2, 3, 4, 7, 8, 15, 16, 17, 18, 31, 32, 33, 47};
  for (int K : depths)
    for (int M : dims)
      for (int size : {4, 8}) {
        const int N = 201 - M;  // both operands run over every dimension
        check<64>(size, M, N, K);
        check<128>(size, M, N, K);
      }
  // ranges fit the descriptor's size field
  if ((int64_t)big_b_panel(128, 128, 1 << 21, 0, 8) * 8 > kMaxRangeBytes) ++errors;
  std::printf("%ld errors\n", errors);
  return errors ? 1 : 0;
}
