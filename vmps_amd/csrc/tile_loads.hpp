// Which elements the operand loads of the LDS-staged FP64 / FP32 tiles touch:
// offsets, masks and buffer ranges in one place, for the kernels (engine.hip)
// and for the host check of every address.
//
// A raw buffer load returns zero for every dword at or past the buffer's range,
// scalar offset included (as measured on gfx950; a 16-byte load across the
// range's end returns its dwords before it).
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define VMPS_HD __host__ __device__ __forceinline__
#else
#define VMPS_HD inline
#endif

namespace vmps {

constexpr int kBigKd = 16;                      // k depth of a step (work items count in it too)
constexpr uint32_t kNoLoad = 0x80000000u;       // a byte offset past every range
constexpr int64_t kMaxRangeBytes = 0x7fffffff;  // of a buffer descriptor

// Staging roles of a thread: A elements (row ai, k = ak + kDA q, q < kNA), B pairs
// (k = bk and bk + 1, column bj + 32 h, h < kNB) of a BT x kBigKd / kBigKd x BT tile.
template <int BT>
struct BigRole {
  static constexpr int kNA = kBigKd * BT / 256, kNB = kNA / 2, kDA = 256 / BT;
  int ai, ak, bj, bk;
  VMPS_HD void init(int tid) {
    ai = tid % BT;
    ak = tid / BT;
    bj = tid >> 3;
    bk = (tid & 7) * 2;
  }
};

VMPS_HD int lesser(int a, int b) { return a < b ? a : b; }

// Elements from (row m0, k = kb) of a column-major M x K block to the end of the
// step, or of the block
VMPS_HD int big_a_range(int M, int K, int kb, int m0) {
  const int r = lesser(K - kb, kBigKd) * M - m0;
  return r > 0 ? r : 0;
}
// a thread's A element q is big_a_first + big_a_next of it, from that element on;
// rows past the block repeat its last one
VMPS_HD int big_a_first(int ak, int ai, int M, int m0) { return ak * M + lesser(ai, M - 1 - m0); }
VMPS_HD int big_a_next(int kda, int q, int M) { return kda * q * M; }

// Elements of a tile's columns n0, n0 + 1, .. of a column-major K x N block, and
// the range left from k = kb on: a pair that starts at k = K - 1 (K odd) reads the
// next column's first element, and behind the last column nothing
VMPS_HD int big_b_panel(int bt, int N, int K, int n0, int elem_size) {
  const int64_t r = (int64_t)lesser(bt, N - n0) * K, most = kMaxRangeBytes / elem_size;
  return (int)(r < most ? r : most);
}
VMPS_HD int big_b_range(int panel, int K, int kb) { return kb < K ? panel - kb : 0; }
// a thread's pair h, from that element on; columns past the block repeat its last one
VMPS_HD int big_b_pair(int bj, int h, int bk, int N, int K, int n0) { return lesser(bj + 32 * h, N - 1 - n0) * K + bk; }
VMPS_HD bool big_b_in(int kb, int bk, int K) { return kb + bk < K; }

}  // namespace vmps
