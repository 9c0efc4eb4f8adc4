// Split-BF16 x3 path of the staged effective-Hamiltonian application.
//
// Every FP64 operand x is carried as hi = bf16(x), lo = bf16(x - hi); a
// product a.b is formed as a_hi.b_hi + a_hi.b_lo + a_lo.b_hi by three
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation (relative error ~1e-5).
// Operands are k-contiguous with k padded to a multiple of 8 and stored in groups
// of [8 hi | 8 lo] (32 bytes; the zero padding ends K): an MFMA lane's 8 k values
// are one aligned 16-byte load for hi and the next one for lo, and a 32-deep step
// of a row is one 128-byte line:
//   L^T (row-major M x Kp), V and R (column-major Kp x N); T is FP32 (row-major
//   M x Np), and so is U unless stage B is explicit, which stores U split.
// Offsets into a split array count padded elements: element (row, k) of a block
// at `off` is at 2 (off + row Kp) + 16 (k / 8) + k % 8, its lo part 8 further.
// Work decomposition as in the FP64 kernels: stage A one wave per 32 x 32
// tile, stage C one workgroup per tile with the combine sum_j c_j T_j done on
// the operand load and a 4-way split of the K iterations reduced through LDS.
#include "engine.hpp"
#include "combine.hpp"
#include "wave.hpp"

namespace vmps {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

namespace {

// Operand roles as in the FP64 kernels: the MFMA computes C^T = B^T A^T, so the
// MFMA A operand is B[k..k+7][j] and the MFMA B operand is A[i][k..k+7];
// accumulator element v of lane l then holds C[i = l%16][j = 4(l/16) + v].
__device__ inline v4f mac3(const v8bf& bh, const v8bf& bl, const v8bf& ah, const v8bf& al, v4f c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl, ah, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh, al, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh, ah, c, 0, 0, 0);
  return c;
}

__device__ inline v8bf ld8(const __bf16* p) { return *reinterpret_cast<const v8bf*>(p); }

__device__ inline void split8(const float (&x)[8], v8bf& hi, v8bf& lo) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const __bf16 h = (__bf16)x[e];
    hi[e] = h;
    lo[e] = (__bf16)(x[e] - (float)h);
  }
}

__device__ inline void st8(__bf16* p, const v8bf& x) { *reinterpret_cast<v8bf*>(p) = x; }

// Packed FP64 V columns -> padded split-BF16 copies (one workgroup per task of
// at most 4096 padded elements, a group of 8 k per thread and round).
__global__ __launch_bounds__(256) void k_split_v(const VConv* __restrict__ tasks, const double* __restrict__ vin,
                                                 __bf16* __restrict__ Vs) {
  const VConv t = tasks[blockIdx.x];
  const int g8 = t.Kp / 8, n = g8 * t.N;
  for (int e = threadIdx.x; e < n; e += 256) {
    const int j = e / g8, k = 8 * (e - j * g8);
    const double* __restrict__ src = vin + t.src_off + (int64_t)j * t.K + k;
    v8bf hi, lo;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const double x = k + u < t.K ? src[u] : 0.0;
      const __bf16 h = (__bf16)(float)x;
      hi[u] = h;
      lo[u] = (__bf16)(float)(x - (double)(float)h);
    }
    __bf16* __restrict__ dst = Vs + 2 * (t.dst_off + (int64_t)e * 8);
    st8(dst, hi);
    st8(dst + 8, lo);
  }
}

// FP64 L blocks (column-major M x K, ld M) -> row-major M x Kp split-BF16
// copies (L^T in the layout of k_split_v's output); one workgroup per task of
// at most 4096 padded elements, task rows r read src[src_off + k M + r].
__global__ __launch_bounds__(256) void k_split_lt(const VConv* __restrict__ tasks, const double* __restrict__ L,
                                                  __bf16* __restrict__ Ls) {
  const VConv t = tasks[blockIdx.x];
  const int g8 = t.Kp / 8, n = g8 * t.N;
  for (int e = threadIdx.x; e < n; e += 256) {
    const int r = e / g8, k = 8 * (e - r * g8);
    const double* __restrict__ src = L + t.src_off + (int64_t)k * t.pad + r;
    v8bf hi, lo;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const double x = k + u < t.K ? src[(int64_t)u * t.pad] : 0.0;
      const __bf16 h = (__bf16)(float)x;
      hi[u] = h;
      lo[u] = (__bf16)(float)(x - (double)(float)h);
    }
    __bf16* __restrict__ dst = Ls + 2 * (t.dst_off + (int64_t)e * 8);
    st8(dst, hi);
    st8(dst + 8, lo);
  }
}

// Explicit stage B: U = sum_j c_j T_j, stored split (U's k is T's column), so
// that stage C's tiles of one row of blocks load it instead of each splitting it
// again.  One workgroup per task; a thread takes groups of 8 elements, the task's
// terms come 64 at a time, one descriptor per lane, two terms per round.
__global__ __launch_bounds__(256) void k_combine_split(const CombTask* __restrict__ tasks,
                                                       const TermC16* __restrict__ terms,
                                                       const float* __restrict__ Tbuf, __bf16* __restrict__ Us) {
  constexpr int NV = kCombTaskElems / 256 / 8;
  const CombTask t = tasks[blockIdx.x];
  const int lane = threadIdx.x & 63;
  const v4f zf = {0, 0, 0, 0};
  v4f acc[NV][2];
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v][0] = acc[v][1] = zf;
  auto load = [&](const float* __restrict__ src, v4f (&x)[NV][2]) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int e = 8 * ((int)threadIdx.x + 256 * v);
      x[v][0] = e < t.n ? *reinterpret_cast<const v4f*>(src + e) : zf;
      x[v][1] = e < t.n ? *reinterpret_cast<const v4f*>(src + e + 4) : zf;
    }
  };
  for (int g = t.term_begin; g < t.term_end; g += 64) {
    const int nt = min(64, t.term_end - g);
    int64_t my_off = 0;
    float my_c = 0.f;
    if (lane < nt) {
      const TermC16 tm = terms[g + lane];
      my_off = tm.t_off;
      my_c = tm.c;
    }
    int j = 0;
    for (; j + 1 < nt; j += 2) {
      const float c0 = readlane_f(my_c, j), c1 = readlane_f(my_c, j + 1);
      v4f x0[NV][2], x1[NV][2];
      load(Tbuf + readlane64(my_off, j) + t.e0, x0);
      load(Tbuf + readlane64(my_off, j + 1) + t.e0, x1);
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[v][q] += c0 * x0[v][q] + c1 * x1[v][q];
    }
    if (j < nt) {
      const float c0 = readlane_f(my_c, j);
      v4f x0[NV][2];
      load(Tbuf + readlane64(my_off, j) + t.e0, x0);
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[v][q] += c0 * x0[v][q];
    }
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int e = 8 * ((int)threadIdx.x + 256 * v);
    if (e >= t.n) continue;
    const float u[8] = {acc[v][0][0], acc[v][0][1], acc[v][0][2], acc[v][0][3],
                        acc[v][1][0], acc[v][1][1], acc[v][1][2], acc[v][1][3]};
    v8bf hi, lo;
    split8(u, hi, lo);
    __bf16* __restrict__ dst = Us + 2 * (t.u_off + t.e0 + e);
    st8(dst, hi);
    st8(dst + 8, lo);
  }
}

// The split operands of one 32-deep K block of a 32 x 32 wave tile:
// A rows i0 = m0 + lane%16 and i0 + 16, B columns j0 = n0 + lane%16 and j0 + 16,
// k = kb + 8 (lane/16) .. +7.
struct WaveOps {
  v8bf a0h, a0l, a1h, a1l, b0h, b0l, b1h, b1l;
};

__device__ inline void wave_mac(const WaveOps& o, bool has_m1, bool has_n1, v4f& c00, v4f& c01, v4f& c10,
                                v4f& c11) {
  c00 = mac3(o.b0h, o.b0l, o.a0h, o.a0l, c00);
  if (has_m1) c10 = mac3(o.b0h, o.b0l, o.a1h, o.a1l, c10);
  if (has_n1) {
    c01 = mac3(o.b1h, o.b1l, o.a0h, o.a0l, c01);
    if (has_m1) c11 = mac3(o.b1h, o.b1l, o.a1h, o.a1l, c11);
  }
}

// Stage A, small problems: Tp (row-major M x Np) = L (Lt row-major M x Kp) . V (col-major Kp x N).
// Most of these tiles need one or two 32-deep K blocks, so a wave that took a
// single tile would spend its life waiting: for the descriptor, then for the
// operands.  Instead each wave walks the tiles w, w + W, w + 2W, ... (W = waves
// in the grid): their descriptors arrive 64 at a time, one per lane, and are
// broadcast with readlane, and the operand loads of the next K block -- of the
// same tile or of the wave's next tile -- are issued before the MFMAs of the
// current one.
struct TileCursor {
  int64_t a_off, b_off, c_off;
  int M, N, Kp, Np, m0, n0;
};

__device__ inline TileCursor tile_at(const TileA16& d, int src) {
  TileCursor c;
  c.a_off = readlane64(d.a_off, src);
  c.b_off = readlane64(d.b_off, src);
  c.c_off = readlane64(d.c_off, src);
  c.M = readlane32(d.M, src);
  c.N = readlane32(d.N, src);
  c.Kp = readlane32(d.Kp, src);
  c.Np = readlane32(d.Np, src);
  c.m0 = readlane32((int)d.mt, src) * kTile;
  c.n0 = readlane32((int)d.nt, src) * kTile;
  return c;
}

__global__ __launch_bounds__(256) void k_stage_a_bf16x3(const TileA16* __restrict__ tiles, int ntiles,
                                                        const __bf16* __restrict__ Ls, const __bf16* __restrict__ Vs,
                                                        float* __restrict__ Tp) {
  const int nwaves = gridDim.x * 4;
  const int w0 = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (w0 >= ntiles) return;
  const int nmine = (ntiles - 1 - w0) / nwaves + 1;  // tiles w0 + j * nwaves, j < nmine
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lg = lane >> 4;
  const v8bf z = {};
  auto load = [&](const TileCursor& t, int kb, WaveOps& o) {
    const int k = kb + 8 * lg;
    const bool kin = k < t.Kp;
    const int i0 = t.m0 + li, i1 = i0 + 16, j0 = t.n0 + li, j1 = j0 + 16;
    const bool ra = kin && i0 < t.M, rb = kin && i1 < t.M, qa = kin && j0 < t.N, qb = kin && j1 < t.N;
    const __bf16* __restrict__ pa0 = Ls + 2 * (t.a_off + (int64_t)i0 * t.Kp + k);
    o.a0h = ra ? ld8(pa0) : z;
    o.a0l = ra ? ld8(pa0 + 8) : z;
    const __bf16* __restrict__ pa1 = Ls + 2 * (t.a_off + (int64_t)i1 * t.Kp + k);
    o.a1h = rb ? ld8(pa1) : z;
    o.a1l = rb ? ld8(pa1 + 8) : z;
    const __bf16* __restrict__ pb0 = Vs + 2 * (t.b_off + (int64_t)j0 * t.Kp + k);
    o.b0h = qa ? ld8(pb0) : z;
    o.b0l = qa ? ld8(pb0 + 8) : z;
    const __bf16* __restrict__ pb1 = Vs + 2 * (t.b_off + (int64_t)j1 * t.Kp + k);
    o.b1h = qb ? ld8(pb1) : z;
    o.b1l = qb ? ld8(pb1 + 8) : z;
  };
  auto store = [&](const TileCursor& t, const v4f& c00, const v4f& c01, const v4f& c10, const v4f& c11) {
    const int i0 = t.m0 + li, i1 = i0 + 16;
    float* __restrict__ C = Tp + t.c_off;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int ja = t.n0 + 4 * lg + v, jb = ja + 16;
      if (i0 < t.M) {
        if (ja < t.N) C[(int64_t)i0 * t.Np + ja] = c00[v];
        if (jb < t.N) C[(int64_t)i0 * t.Np + jb] = c01[v];
      }
      if (i1 < t.M) {
        if (ja < t.N) C[(int64_t)i1 * t.Np + ja] = c10[v];
        if (jb < t.N) C[(int64_t)i1 * t.Np + jb] = c11[v];
      }
    }
  };
  for (int g = 0; g < nmine; g += 64) {
    const int n = min(64, nmine - g);
    TileA16 d = {};
    if (lane < n) d = tiles[w0 + (int64_t)(g + lane) * nwaves];
    // load cursor (lt, lj, lk) runs one K block ahead of the compute cursor (ct, cj, ck);
    // a tile has max(1, Kp / 32) K blocks (Kp is a multiple of 8)
    TileCursor lt = tile_at(d, 0), ct = lt;
    int lj = 0, lk = 0, cj = 0, ck = 0;
    auto advance_load = [&]() {
      lk += 32;
      if (lk >= max(lt.Kp, 1)) {
        lk = 0;
        if (++lj < n) lt = tile_at(d, lj);
      }
    };
    WaveOps o0, o1;
    load(lt, 0, o0);
    advance_load();
    v4f c00 = {0, 0, 0, 0}, c01 = c00, c10 = c00, c11 = c00;
    // one pipeline step: prefetch into `nx`, multiply `cur`; false when the group is done
    auto step = [&](const WaveOps& cur, WaveOps& nx) -> bool {
      if (lj < n) {
        load(lt, lk, nx);
        advance_load();
      }
      wave_mac(cur, ct.m0 + 16 < ct.M, ct.n0 + 16 < ct.N, c00, c01, c10, c11);
      ck += 32;
      if (ck >= max(ct.Kp, 1)) {
        store(ct, c00, c01, c10, c11);
        c00 = v4f{0, 0, 0, 0};
        c01 = c00;
        c10 = c00;
        c11 = c00;
        ck = 0;
        if (++cj == n) return false;
        ct = tile_at(d, cj);
      }
      return true;
    };
    while (step(o0, o1) && step(o1, o0)) {
    }
  }
}

// Stage C, small problems: Vout (FP64 col-major M x N) = sum over chunks (sum_j c_j T_j) . R.
// kSplitU (explicit stage B): every chunk reads one split block of unit weight from Us.
template <bool kSplitU>
__global__ __launch_bounds__(256) void k_stage_c_bf16x3(const TileC* __restrict__ tiles, int ntiles,
                                                        const ChunkC16* __restrict__ chunks,
                                                        const TermC16* __restrict__ terms, const float* __restrict__ Tp,
                                                        const __bf16* __restrict__ Us, const __bf16* __restrict__ Rs,
                                                        double* __restrict__ Vout) {
  __shared__ v4f red[3][4][64];
  if ((int)blockIdx.x >= ntiles) return;  // workgroup-uniform
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const TileC t = tiles[blockIdx.x];
  const int m0 = t.mt * kTile, n0 = t.nt * kTile;
  const int li = lane & 15, lg = lane >> 4;
  const int i0 = m0 + li, i1 = i0 + 16, j0 = n0 + li, j1 = j0 + 16;
  const bool has_m1 = m0 + 16 < t.M, has_n1 = n0 + 16 < t.N;
  const bool r0 = i0 < t.M, r1 = i1 < t.M, q0 = j0 < t.N, q1 = j1 < t.N;
  const v8bf z = {};
  v4f c00 = {0, 0, 0, 0}, c01 = c00, c10 = c00, c11 = c00;
  int it = 0;
  for (int g = t.chunk_begin; g < t.chunk_end; g += 64) {
    // chunk descriptors, one per lane, broadcast with readlane
    const int nch = min(64, t.chunk_end - g);
    int64_t my_r = 0;
    int my_K = 0, my_tb = 0, my_te = 0;
    if (lane < nch) {
      const ChunkC16 cd = chunks[g + lane];
      my_r = cd.r_off;
      my_K = cd.Kp;
      my_tb = cd.term_begin;
      my_te = cd.term_end;
    }
    for (int ci = 0; ci < nch; ++ci) {
      const int Kp = readlane32(my_K, ci);
      const int nkb = (Kp + 31) >> 5;
      // K blocks of this chunk handled by this wave: it + q with (it + q) % 4 == wave
      const int first = (wave - (it & 3)) & 3;
      if (first >= nkb) {
        it += nkb;
        continue;
      }
      const int64_t roff = readlane64(my_r, ci);
      const int tb = readlane32(my_tb, ci);
      const int nt = readlane32(my_te, ci) - tb;
      // the chunk's terms (at most 64), one per lane
      int64_t my_toff = 0;
      float my_c = 0.f;
      if (lane < nt) {
        const TermC16 tm = terms[tb + lane];
        my_toff = tm.t_off;
        my_c = tm.c;
      }
      for (int q = first; q < nkb; q += 4) {
        const int k = q * 32 + 8 * lg;
        const bool kin = k < Kp;
        const bool a0 = kin && r0, a1 = kin && r1;
        const __bf16* __restrict__ p0 = Rs + 2 * (roff + (int64_t)j0 * Kp + k);
        const __bf16* __restrict__ p1 = Rs + 2 * (roff + (int64_t)j1 * Kp + k);
        WaveOps o;
        o.b0h = (kin && q0) ? ld8(p0) : z;
        o.b0l = (kin && q0) ? ld8(p0 + 8) : z;
        o.b1h = (kin && q1) ? ld8(p1) : z;
        o.b1l = (kin && q1) ? ld8(p1 + 8) : z;
        if constexpr (kSplitU) {
          const int64_t u = readlane64(my_toff, 0) + k;
          const __bf16* __restrict__ u0 = Us + 2 * (u + (int64_t)i0 * Kp);
          const __bf16* __restrict__ u1 = Us + 2 * (u + (int64_t)i1 * Kp);
          o.a0h = a0 ? ld8(u0) : z;
          o.a0l = a0 ? ld8(u0 + 8) : z;
          o.a1h = a1 ? ld8(u1) : z;
          o.a1l = a1 ? ld8(u1 + 8) : z;
          wave_mac(o, has_m1, has_n1, c00, c01, c10, c11);
          continue;
        }
        float u0[8], u1[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          u0[e] = 0.f;
          u1[e] = 0.f;
        }
        // U rows i0, i1 at k..k+7 = sum_j c_j T_j, two terms per round with all loads first
        int jt = 0;
        for (; jt + 1 < nt; jt += 2) {
          const float* __restrict__ T0 = Tp + readlane64(my_toff, jt) + k;
          const float* __restrict__ T1 = Tp + readlane64(my_toff, jt + 1) + k;
          const float c0 = readlane_f(my_c, jt), c1 = readlane_f(my_c, jt + 1);
          const v4f zf = {0, 0, 0, 0};
          const v4f x00 = a0 ? *reinterpret_cast<const v4f*>(T0 + (int64_t)i0 * Kp) : zf;
          const v4f x01 = a0 ? *reinterpret_cast<const v4f*>(T0 + (int64_t)i0 * Kp + 4) : zf;
          const v4f x10 = a1 ? *reinterpret_cast<const v4f*>(T0 + (int64_t)i1 * Kp) : zf;
          const v4f x11 = a1 ? *reinterpret_cast<const v4f*>(T0 + (int64_t)i1 * Kp + 4) : zf;
          const v4f y00 = a0 ? *reinterpret_cast<const v4f*>(T1 + (int64_t)i0 * Kp) : zf;
          const v4f y01 = a0 ? *reinterpret_cast<const v4f*>(T1 + (int64_t)i0 * Kp + 4) : zf;
          const v4f y10 = a1 ? *reinterpret_cast<const v4f*>(T1 + (int64_t)i1 * Kp) : zf;
          const v4f y11 = a1 ? *reinterpret_cast<const v4f*>(T1 + (int64_t)i1 * Kp + 4) : zf;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            u0[e] += c0 * x00[e] + c1 * y00[e];
            u0[e + 4] += c0 * x01[e] + c1 * y01[e];
            u1[e] += c0 * x10[e] + c1 * y10[e];
            u1[e + 4] += c0 * x11[e] + c1 * y11[e];
          }
        }
        if (jt < nt) {
          const float* __restrict__ T0 = Tp + readlane64(my_toff, jt) + k;
          const float c0 = readlane_f(my_c, jt);
          const v4f zf = {0, 0, 0, 0};
          const v4f x00 = a0 ? *reinterpret_cast<const v4f*>(T0 + (int64_t)i0 * Kp) : zf;
          const v4f x01 = a0 ? *reinterpret_cast<const v4f*>(T0 + (int64_t)i0 * Kp + 4) : zf;
          const v4f x10 = a1 ? *reinterpret_cast<const v4f*>(T0 + (int64_t)i1 * Kp) : zf;
          const v4f x11 = a1 ? *reinterpret_cast<const v4f*>(T0 + (int64_t)i1 * Kp + 4) : zf;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            u0[e] += c0 * x00[e];
            u0[e + 4] += c0 * x01[e];
            u1[e] += c0 * x10[e];
            u1[e + 4] += c0 * x11[e];
          }
        }
        split8(u0, o.a0h, o.a0l);
        split8(u1, o.a1h, o.a1l);
        wave_mac(o, has_m1, has_n1, c00, c01, c10, c11);
      }
      it += nkb;
    }
  }
  if (wave > 0) {
    red[wave - 1][0][lane] = c00;
    red[wave - 1][1][lane] = c01;
    red[wave - 1][2][lane] = c10;
    red[wave - 1][3][lane] = c11;
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int w = 0; w < 3; ++w) {
      c00 += red[w][0][lane];
      c01 += red[w][1][lane];
      c10 += red[w][2][lane];
      c11 += red[w][3][lane];
    }
    double* __restrict__ C = Vout + t.c_off;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int ja = n0 + 4 * lg + v, jb = ja + 16;
      if (ja < t.N) {
        if (r0) C[(int64_t)ja * t.M + i0] = (double)c00[v];
        if (r1) C[(int64_t)ja * t.M + i1] = (double)c10[v];
      }
      if (jb < t.N) {
        if (r0) C[(int64_t)jb * t.M + i0] = (double)c01[v];
        if (r1) C[(int64_t)jb * t.M + i1] = (double)c11[v];
      }
    }
  }
}

// ---- LDS-staged 128 x 128 workgroup tiles for large blocks -------------------
// 4 waves in a 2 x 2 grid (8 in a 2 x 4 grid on 128 x 256), sub-blocks of 16 rows and columns dealt to the waves
// alternately as in the FP64 kernels, and one of 16 instances NX x NY for the
// tiles at a block's edge.  32-deep K steps, two LDS buffers: while a wave
// multiplies step i from registers it reads step i + 1's operands from one buffer,
// writes step i + 2's (loaded a step ago) to the other and issues the loads of
// step i + 3, each between MFMAs; one barrier per step.
//
// What bounds it (12 products of 1152 x 1152 x 11520): MFMAs and barriers alone
// run at 537 TFLOP/s of products (a third of the BF16 rate), with the LDS reads
// 472, with the LDS writes 359; the loads then set the pace, by the number of
// 64-byte requests to the L2, not by bytes: 246 with hi and lo in separate arrays
// (64 bytes per row and step), 312 with the interleaved layout, whose rows are
// whole 128-byte lines.  (A single-buffered 64-deep form with masked loads and
// separate arrays: 278.)
constexpr int kBT = kBigTile;
constexpr int kBKs = kBigK;         // k depth of a step, in which the work items count
static_assert(kBKs == 32, "a row of a step is 8 pieces of 16 bytes, one per thread");
constexpr int kLR = 2 * kBKs + 8;   // LDS row: 4 groups of [8 hi | 8 lo], 144 bytes: no bank conflicts

// NW: waves of the workgroup, and 32-column strips of its tile.  Stage C of pivots
// with enough tiles takes NW = 8, 128 x 256 tiles: its K loops run hundreds of
// steps and the workgroups drift apart, so the L2 seldom serves a panel twice, and
// with 128 columns it fetched 16 GB in 2.8 ms on C60 at M = 4096, more than a
// copy's rate.  Wider tiles fetch a quarter less; HxV there 6.1 -> 5.4 ms.
template <int NW>
struct BigSmem {  // 4 waves: 72 KB, two workgroups per CU; 8 waves: 108 KB
  __bf16 A[2][kBT * kLR], B[2][32 * NW * kLR];
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t bf_buffer(const __bf16* p, bool on) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(p), (short)0, on ? 0x7fffffff : 0, 0x00020000);
}

template <int NW>
struct BigTile16 {
  static constexpr int kBN = 32 * NW;   // columns of the tile
  static constexpr int kCS = 8 * NW;    // columns between a wave's sub-blocks
  static constexpr int kRS = 8 * NW;    // rows between a thread's pieces
  static constexpr int kPA = kBT / kRS, kPB = kBN / kRS;
  uint32_t offA[kPA], offB[kPB];  // byte offsets of this thread's pieces at k = 0
  v8bf ra[kPA], rb[kPB];
  const __bf16 *A, *B;        // wave-uniform: the tile's first row / column
  int Kp, M, N, m0, n0;
  int row, c8, kk;            // staging role: row, offset in the LDS row, first k of the piece
  int kb;                     // k of the load cursor
  int wm, wn, li, lg;

  __device__ __forceinline__ void init(int M_, int N_, int mt, int nt, int tid) {
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    M = M_;
    N = N_;
    m0 = mt * kBT;
    n0 = nt * kBN;
    li = lane & 15;
    lg = lane >> 4;
    wm = (wave & 1) * 16;
    wn = (wave >> 1) * 16;
    row = tid >> 3;
    c8 = (tid & 7) * 8;
    kk = (tid & 6) * 4;
  }
  __device__ __forceinline__ int nx() const { return min(4, (M - m0 + 31) / 32); }  // workgroup-uniform
  __device__ __forceinline__ int ny() const { return min(4, (N - n0 + kCS - 1) / kCS); }
  // rows and columns past the block are clamped to its last one (not stored)
  __device__ __forceinline__ void set(const __bf16* Ablk, const __bf16* Bblk, int Kp_) {
    Kp = Kp_;
    A = Ablk + 2 * (int64_t)m0 * Kp;
    B = Bblk + 2 * (int64_t)n0 * Kp;
#pragma unroll
    for (int h = 0; h < kPA; ++h) offA[h] = 2u * (uint32_t)(min(row + kRS * h, M - 1 - m0) * 2 * Kp + c8);
#pragma unroll
    for (int h = 0; h < kPB; ++h) offB[h] = 2u * (uint32_t)(min(row + kRS * h, N - 1 - n0) * 2 * Kp + c8);
  }
  // K step at kb: pieces at k >= Kp (a multiple of 8) load zeros
  __device__ __forceinline__ void load_a(int kb) {
    const auto r = bf_buffer(A + 2 * kb, kb < Kp);
    const bool in = kb + kk < Kp;
#pragma unroll
    for (int h = 0; h < kPA; ++h)
      ra[h] = __builtin_bit_cast(v8bf, __builtin_amdgcn_raw_buffer_load_b128(r, in ? offA[h] : 0x80000000u, 0, 0));
  }
  __device__ __forceinline__ void load_b(int kb) {
    const auto r = bf_buffer(B + 2 * kb, kb < Kp);
    const bool in = kb + kk < Kp;
#pragma unroll
    for (int h = 0; h < kPB; ++h)
      rb[h] = __builtin_bit_cast(v8bf, __builtin_amdgcn_raw_buffer_load_b128(r, in ? offB[h] : 0x80000000u, 0, 0));
  }
  __device__ __forceinline__ void stage_a(BigSmem<NW>& s, int buf) const {
#pragma unroll
    for (int h = 0; h < kPA; ++h) st8(&s.A[buf][(row + kRS * h) * kLR + c8], ra[h]);
  }
  __device__ __forceinline__ void stage_b(BigSmem<NW>& s, int buf) const {
#pragma unroll
    for (int h = 0; h < kPB; ++h) st8(&s.B[buf][(row + kRS * h) * kLR + c8], rb[h]);
  }
};

template <int NW, int NX, int NY>
struct BigAcc16 {
  typedef BigTile16<NW> Tile;
  v4f acc[NX][NY];
  v8bf a[2][NX][2], b[2][NY][2];  // [step parity][sub-block][hi, lo]

  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
      for (int y = 0; y < NY; ++y) acc[x][y] = v4f{0, 0, 0, 0};
  }
  __device__ __forceinline__ void read(const Tile& g, const BigSmem<NW>& s, int buf, int p) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
      for (int x = 0; x < NX; ++x) a[p][x][q] = ld8(&s.A[buf][(g.wm + 32 * x + g.li) * kLR + 16 * g.lg + 8 * q]);
#pragma unroll
      for (int y = 0; y < NY; ++y) b[p][y][q] = ld8(&s.B[buf][(g.wn + Tile::kCS * y + g.li) * kLR + 16 * g.lg + 8 * q]);
    }
  }
  __device__ __forceinline__ void mac(int p) {  // lo.hi, hi.lo, hi.hi, as mac3 adds them
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[p][y][q == 0], a[p][x][q == 1], acc[x][y], 0, 0, 0);
  }
  // one step from registers p; buffer p ^ 1 holds the next one
  template <class Next>
  __device__ __forceinline__ void step(Tile& g, BigSmem<NW>& s, int p, Next&& next) {
    next(g);          // the load cursor moves on
    __syncthreads();  // the next step is staged, and this one's buffer no longer read
    __builtin_amdgcn_sched_barrier(0);
    read(g, s, p ^ 1, p ^ 1);
    g.stage_a(s, p);
    g.stage_b(s, p);
    g.load_a(g.kb);
    g.load_b(g.kb);
    mac(p);
#pragma unroll
    for (int i = 0; i < 2 * (NX + NY); ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
    }
#pragma unroll
    for (int i = 0; i < Tile::kPA + Tile::kPB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
    }
#pragma unroll
    for (int i = 0; i < Tile::kPA + Tile::kPB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // global load
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // `steps` K steps; next(g) sets the operands and k of the following load (g.kb)
  template <class Next>
  __device__ __forceinline__ void run(Tile& g, BigSmem<NW>& s, int steps, Next&& next) {
    zero();
    if (steps <= 0) return;  // workgroup-uniform
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (i) {
        g.stage_a(s, i - 1);
        g.stage_b(s, i - 1);
      }
      next(g);
      g.load_a(g.kb);
      g.load_b(g.kb);
    }
    __syncthreads();
    read(g, s, 0, 0);
    for (int i = 0; i < steps; i += 2) {
      step(g, s, 0, next);
      if (i + 1 < steps) step(g, s, 1, next);
    }
  }
};

// f(BigAcc16 of the instance covering the tile); workgroup-uniform
template <int NW, class F>
__device__ __forceinline__ void with_big_acc16(const BigTile16<NW>& g, F&& f) {
  const int nx = g.nx(), ny = g.ny();
#define VMPS_BIG_ACC(X, Y)     \
  if (nx == X && ny == Y) {    \
    BigAcc16<NW, X, Y> acc;    \
    f(acc);                    \
    return;                    \
  }
#define VMPS_BIG_ACC_ROW(X) VMPS_BIG_ACC(X, 1) VMPS_BIG_ACC(X, 2) VMPS_BIG_ACC(X, 3) VMPS_BIG_ACC(X, 4)
  VMPS_BIG_ACC_ROW(1)
  VMPS_BIG_ACC_ROW(2)
  VMPS_BIG_ACC_ROW(3)
  VMPS_BIG_ACC_ROW(4)
#undef VMPS_BIG_ACC_ROW
#undef VMPS_BIG_ACC
}

// Stage A, large problems: Tp (row-major M x Np) = Lt (row-major M x Kp) . V (col-major Kp x N)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_stage_a_bf16x3_big(
    const TileA16* __restrict__ tiles, int ntiles, const __bf16* __restrict__ Ls, const __bf16* __restrict__ Vs,
    float* __restrict__ Tp) {
  __shared__ BigSmem<4> s;
  if ((int)blockIdx.x >= ntiles) return;  // workgroup-uniform
  const TileA16 t = tiles[blockIdx.x];
  if (t.Kp <= 0) return;  // a padding slot of the launch order (workgroup-uniform)
  typedef BigTile16<4> Tile;
  Tile g;
  g.init(t.M, t.N, t.mt, t.nt, threadIdx.x);
  g.set(Ls + 2 * t.a_off, Vs + 2 * t.b_off, t.Kp);
  float* __restrict__ C = Tp + t.c_off;
  with_big_acc16(g, [&](auto& acc) __attribute__((always_inline)) {
    g.kb = -kBKs;
    acc.run(g, s, (t.Kp + kBKs - 1) / kBKs, [](Tile& h) __attribute__((always_inline)) { h.kb += kBKs; });
    constexpr int NX = sizeof(acc.acc) / sizeof(acc.acc[0]), NY = sizeof(acc.acc[0]) / sizeof(v4f);
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int i = g.m0 + g.wm + 32 * x + g.li;
      if (i >= t.M) continue;
#pragma unroll
      for (int y = 0; y < NY; ++y) {
        const int j = g.n0 + g.wn + 32 * y + 4 * g.lg;  // Np and c_off are multiples of 8: 16-byte aligned
        float* __restrict__ c = C + (int64_t)i * t.Np + j;
        if (j + 4 <= t.N) {
          *reinterpret_cast<v4f*>(c) = acc.acc[x][y];
        } else {  // the padding columns keep their zeros
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (j + v < t.N) c[v] = acc.acc[x][y][v];
        }
      }
    }
  });
}

// Stage C, large output blocks: Vout (FP64 col-major M x N) = sum_chunks (sum_j c_j T_j) . R.
// Work items as in the FP64 kernel (BigItemC, in steps of kBKs k); partial
// tiles are FP32, column-major, of 128 x 32 NW.
// kSplitU (explicit stage B): every chunk reads one split block of unit weight
// from Us, the loads running ahead across the chunks' boundaries; otherwise U
// is formed and split on the operand load.
template <bool kSplitU, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void k_stage_c_bf16x3_big(
    const TileC* __restrict__ tiles, const BigItemC* __restrict__ items, int nitems,
    const ChunkC16* __restrict__ chunks, const TermC16* __restrict__ terms, const float* __restrict__ Tp,
    const __bf16* __restrict__ Us, const __bf16* __restrict__ Rs, double* __restrict__ Vout,
    float* __restrict__ partial) {
  typedef BigTile16<NW> Tile;
  __shared__ BigSmem<NW> s;
  if ((int)blockIdx.x >= nitems) return;  // workgroup-uniform
  const BigItemC w = items[blockIdx.x];
  if (w.tile < 0) return;  // a padding slot of the launch order (workgroup-uniform)
  const TileC t = tiles[w.tile];
  Tile g;
  g.init(t.M, t.N, t.mt, t.nt, threadIdx.x);
  int left = w.nsteps, c = w.chunk, kb = w.step * kBKs;
  auto store = [&](auto& acc) __attribute__((always_inline)) {
    constexpr int NX = sizeof(acc.acc) / sizeof(acc.acc[0]), NY = sizeof(acc.acc[0]) / sizeof(v4f);
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int r = g.wm + 32 * x + g.li;
      if (g.m0 + r >= t.M) continue;
#pragma unroll
      for (int y = 0; y < NY; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int cl = g.wn + Tile::kCS * y + 4 * g.lg + v;
          if (g.n0 + cl >= t.N) continue;
          if (w.slot < 0)
            Vout[t.c_off + (int64_t)(g.n0 + cl) * t.M + g.m0 + r] = (double)acc.acc[x][y][v];
          else
            partial[w.slot * (int64_t)(kBT * Tile::kBN) + cl * kBT + r] = acc.acc[x][y][v];
        }
    }
  };
  if constexpr (kSplitU) {
    g.kb = kb - kBKs;
    auto enter = [&](Tile& h) __attribute__((always_inline)) {
      const ChunkC16 ch = chunks[c];
      h.set(Us + 2 * terms[ch.term_begin].t_off, Rs + 2 * ch.r_off, ch.Kp);
    };
    if (left > 0) enter(g);
    with_big_acc16(g, [&](auto& acc) __attribute__((always_inline)) {
      acc.run(g, s, w.nsteps, [&](Tile& h) __attribute__((always_inline)) {
        h.kb += kBKs;
        while (h.kb >= h.Kp && left > 0) {
          ++c;
          h.kb = 0;
          enter(h);
        }
        --left;
      });
      store(acc);
    });
  } else {
    const int lane = threadIdx.x & 63;
    static_assert(NW == 4, "the fused form stages U with 256 threads");
    BigAcc16<NW, 4, 4> acc;
    acc.zero();
    const int row = threadIdx.x >> 2, k8 = (threadIdx.x & 3) * 8;  // U pieces: rows row, row + 64, 8 k each
    for (; left > 0; ++c, kb = 0) {
      const ChunkC16 ch = chunks[c];
      const int nt = ch.term_end - ch.term_begin;
      int64_t my_toff = 0;
      float my_c = 0.f;
      if (lane < nt) {
        const TermC16 tm = terms[ch.term_begin + lane];
        my_toff = tm.t_off;
        my_c = tm.c;
      }
      g.set(Rs, Rs + 2 * ch.r_off, ch.Kp);  // A is not used
      for (; kb < ch.Kp && left > 0; kb += kBKs, --left) {
        const v4f zf = {0, 0, 0, 0};
        v4f u[2][2] = {{zf, zf}, {zf, zf}};
        bool in[2];
        int64_t at[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          in[h] = g.m0 + row + 64 * h < t.M && kb + k8 < ch.Kp;
          at[h] = (int64_t)(g.m0 + row + 64 * h) * ch.Kp + kb + k8;
        }
        g.load_b(kb);
        for (int jt = 0; jt < nt; ++jt) {
          const float* __restrict__ T0 = Tp + readlane64(my_toff, jt);
          const float c0 = readlane_f(my_c, jt);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            u[h][0] += c0 * (in[h] ? *reinterpret_cast<const v4f*>(T0 + at[h]) : zf);
            u[h][1] += c0 * (in[h] ? *reinterpret_cast<const v4f*>(T0 + at[h] + 4) : zf);
          }
        }
        __syncthreads();  // the previous step's LDS reads are done
        g.stage_b(s, 0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float x[8] = {u[h][0][0], u[h][0][1], u[h][0][2], u[h][0][3],
                              u[h][1][0], u[h][1][1], u[h][1][2], u[h][1][3]};
          v8bf hi, lo;
          split8(x, hi, lo);
          st8(&s.A[0][(row + 64 * h) * kLR + 2 * k8], hi);
          st8(&s.A[0][(row + 64 * h) * kLR + 2 * k8 + 8], lo);
        }
        __syncthreads();
        acc.read(g, s, 0, 0);
        acc.mac(0);
      }
    }
    store(acc);
  }
}

}  // namespace

void DevPlan::ensure_bf16_buffers() {
  if (bf16_ready || (H.tilesA.empty() && H.tilesC.empty())) return;
  Bf16Layout B;
  build_bf16_layout(H, B);  // work lists; the operands are split on the device
  Ls.alloc(std::max<int64_t>(1, 2 * B.L_size));
  Rs.alloc(std::max<int64_t>(1, 2 * B.R_size));
  {
    DevBuf<VConv> lc, rc;  // freed after the synchronisation below
    lc.upload(B.lconv, stream);
    rc.upload(B.rconv, stream);
    if (lc.n)
      hipLaunchKernelGGL(k_split_lt, dim3((unsigned)lc.n), dim3(256), 0, stream, lc.p, L.p, (__bf16*)Ls.p);
    if (rc.n)
      hipLaunchKernelGGL(k_split_v, dim3((unsigned)rc.n), dim3(256), 0, stream, rc.p, R.p, (__bf16*)Rs.p);
    VMPS_HIP_CHECK(hipGetLastError());
    VMPS_HIP_CHECK(hipStreamSynchronize(stream));
  }
  Vs.alloc(std::max<int64_t>(1, 2 * B.V_size));
  Tp.alloc(std::max<int64_t>(1, B.T_size));
  VMPS_HIP_CHECK(hipMemsetAsync(Tp.p, 0, Tp.n * sizeof(float), stream));  // padding columns stay zero
  upload_bf16_lists(B);
  VMPS_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ_a16, k_stage_a_bf16x3, 256, 0));
  VMPS_HIP_CHECK(hipStreamSynchronize(stream));
  bf16_ready = true;
  ++gen;
}

void DevPlan::upload_bf16_lists(const Bf16Layout& B) {
  bfA.upload(B.tilesA, stream);
  bfAbig.upload(B.tilesA_big, stream);
  bfCsmall.upload(B.tilesC_small, stream);
  bfCbig.upload(B.tilesC_big, stream);
  itemsC16.upload(B.itemsC, stream);
  redsC16.upload(B.redsC, stream);
  c16_wide = B.wideC;
  const size_t part = (size_t)(B.slotsC * kBigTile * kBigTile * (B.wideC ? 2 : 1));
  if (Cpart.n < part) Cpart.alloc(part);
  bfC.upload(B.chunksC, stream);
  bfT.upload(B.termsC, stream);
  vconv.upload(B.vconv, stream);
  bfCombTasks.upload(B.comb_tasks, stream);
  bfCombTerms.upload(B.comb_terms, stream);
  if (H.explicit_u)
    Us.alloc(std::max<int64_t>(1, 2 * B.U_size));
  else
    Us.release();
}

void DevPlan::retile(int wave_edge, int big_min, int big_min64, bool explicit_u) {
  if (wave_edge == H.wave_edge && big_min == H.big_min && big_min64 == H.big_min64 && explicit_u == H.explicit_u)
    return;  // the lists on the device are already these
  ++gen;
  const bool bf16_lists = bf16_ready && (big_min != H.big_min || explicit_u != H.explicit_u);
  if (explicit_u != H.explicit_u) {
    H.explicit_u = explicit_u;
    build_tiles(H);  // chunk / term tables and every tile list
  }
  set_wave_edge(H, wave_edge, big_min64);
  H.big_min = big_min;
  upload_lists();
  if (bf16_lists) {  // split-BF16 work lists; the split operands stay
    VMPS_HIP_CHECK(hipStreamSynchronize(stream));
    Bf16Layout B;
    build_bf16_layout(H, B);
    upload_bf16_lists(B);
  }
  VMPS_HIP_CHECK(hipStreamSynchronize(stream));
}

void DevPlan::launch_stage_bf16x3(int stage, const double* d_vin, double* d_vout, hipStream_t s) {
  const int nA = (int)bfA.n, nAb = (int)bfAbig.n, nC = (int)bfCsmall.n, nW = (int)itemsC16.n, nR = (int)redsC16.n;
  const __bf16 *l = (const __bf16*)Ls.p, *r = (const __bf16*)Rs.p, *v = (const __bf16*)Vs.p, *u = (const __bf16*)Us.p;
  if (stage == 0) {
    if (vconv.n)
      hipLaunchKernelGGL(k_split_v, dim3((unsigned)vconv.n), dim3(256), 0, s, vconv.p, d_vin, (__bf16*)Vs.p);
    if (nAb)
      hipLaunchKernelGGL(k_stage_a_bf16x3_big, dim3((unsigned)nAb), dim3(256), 0, s, bfAbig.p, nAb, l, v, Tp.p);
    if (nA)
      hipLaunchKernelGGL(k_stage_a_bf16x3, dim3((unsigned)persistent_blocks(nA, occ_a16)), dim3(256), 0, s, bfA.p, nA,
                         l, v, Tp.p);
  } else if (stage == 2) {
    if (H.explicit_u && bfCombTasks.n)  // stage B: U = sum c T, then stage C reads U
      hipLaunchKernelGGL(k_combine_split, dim3((unsigned)bfCombTasks.n), dim3(256), 0, s, bfCombTasks.p,
                         bfCombTerms.p, Tp.p, (__bf16*)Us.p);
    if (nW && c16_wide)
      hipLaunchKernelGGL((k_stage_c_bf16x3_big<true, 8>), dim3((unsigned)nW), dim3(512), 0, s, bfCbig.p, itemsC16.p,
                         nW, bfC.p, bfT.p, Tp.p, u, r, d_vout, Cpart.p);
    else if (nW && H.explicit_u)
      hipLaunchKernelGGL((k_stage_c_bf16x3_big<true, 4>), dim3((unsigned)nW), dim3(256), 0, s, bfCbig.p, itemsC16.p,
                         nW, bfC.p, bfT.p, Tp.p, u, r, d_vout, Cpart.p);
    else if (nW)
      hipLaunchKernelGGL((k_stage_c_bf16x3_big<false, 4>), dim3((unsigned)nW), dim3(256), 0, s, bfCbig.p, itemsC16.p,
                         nW, bfC.p, bfT.p, Tp.p, u, r, d_vout, Cpart.p);
    if (nR && c16_wide)
      hipLaunchKernelGGL((k_reduce_big<float, double, kBigTile, 2 * kBigTile>), dim3((unsigned)(4 * nR)), dim3(256), 0,
                         s, bfCbig.p, redsC16.p, Cpart.p, d_vout);
    else if (nR)
      hipLaunchKernelGGL((k_reduce_big<float, double, kBigTile, kBigTile>), dim3((unsigned)(4 * nR)), dim3(256), 0, s,
                         bfCbig.p, redsC16.p, Cpart.p, d_vout);
    if (nC && H.explicit_u)
      hipLaunchKernelGGL(k_stage_c_bf16x3<true>, dim3((unsigned)nC), dim3(256), 0, s, bfCsmall.p, nC, bfC.p, bfT.p,
                         Tp.p, u, r, d_vout);
    else if (nC)
      hipLaunchKernelGGL(k_stage_c_bf16x3<false>, dim3((unsigned)nC), dim3(256), 0, s, bfCsmall.p, nC, bfC.p, bfT.p,
                         Tp.p, u, r, d_vout);
  }
  VMPS_HIP_CHECK(hipGetLastError());
}

}  // namespace vmps
