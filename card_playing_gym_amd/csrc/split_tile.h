// The main loop of the large projections: one block's TM x 128 tile of C = A B from fp32
// operands of any layout, on v_mfma_f32_16x16x32_bf16 (gfx950).
//
// PLANES 3: fp32 products in three bf16 parts (split.h); PLANES 1: operands rounded to bf16
// (autocast).  Four waves as 2 x 2, each TM / 2 x 64.  A stage is KS = 32 NK values of k: its
// fp32 values go global -> registers (while the previous stage multiplies) -> bf16 parts ->
// LDS, converted once per block and read by the two waves that share them.  LDS holds each
// 16-row block of a part as [k / 8][row][8 k], rows exclusive-or'ed with 4 (k / 8 mod 4): an
// operand fragment is 64 consecutive 16-byte reads, and the four-row, four-k-group writes of
// 16 lanes start 64 bytes apart, so neither conflicts on banks.
#pragma once

#include <type_traits>

#include "split.h"

namespace cg {

constexpr int ST_N = 128;

// Operand layouts of element (r, k) at p[r * sr + k * sk].  1: k contiguous (16-byte aligned
// rows, k extent a multiple of 4); 2: rows contiguous (16-byte aligned, row extent a multiple
// of 4); 0: any strides.
template <int MODE, int ROWS, int NK>
struct TileRegs {
  static constexpr int N = ROWS * NK / 8;  // values per thread
  float v[N];
};

__device__ __forceinline__ int tile_offset(int row, int kg) {  // bytes inside one 32-k part
  return (row >> 4) * 1024 + kg * 256 + (((row & 15) ^ (kg * 4)) << 4);
}

// A thread's place in a tile: byte offsets from the tile's first row at a stage's first k (32 bits
// beside a uniform pointer, so a load costs no vector address arithmetic).  MODE 1: one per
// 64 rows; MODE 2: one, its eight k a uniform stride apart.
template <int MODE, int ROWS>
struct TilePlace {
  unsigned at[ROWS / 64];
};
template <int MODE, int ROWS>
__device__ __forceinline__ TilePlace<MODE, ROWS> tile_place(int64_t sr, int64_t sk, int rows_left, int tid) {
  TilePlace<MODE, ROWS> t{};
  if constexpr (MODE == 2) {
    constexpr int W = ROWS / 64;  // consecutive rows per thread
    const int row = W * (tid & 63);
    t.at[0] = 4u * (unsigned(8 * (tid >> 6)) * unsigned(sk) +
                    unsigned(W == 2 ? max(0, min(row, rows_left - 2)) : min(row, rows_left - 1)));
  } else if constexpr (MODE == 1) {
#pragma unroll
    for (int e = 0; e < ROWS / 64; ++e)
      t.at[e] = 4u * (unsigned(min((tid + e * 256) >> 2, rows_left - 1)) * unsigned(sr) + unsigned(8 * (tid & 3)));
  }
  return t;
}

// A whole stage (p at its first k): rows past the tile's are read from its last row and their
// results never stored.
template <int MODE, int ROWS, int NK>
__device__ __forceinline__ void tile_load(TileRegs<MODE, ROWS, NK> &t, const TilePlace<MODE, ROWS> &place,
                                          const float *__restrict__ p, int64_t sk) {
  auto at = [](const float *q, unsigned bytes) { return reinterpret_cast<const char *>(q) + bytes; };
#pragma unroll
  for (int s = 0; s < NK; ++s) {
    if constexpr (MODE == 2) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const char *q = at(p + int64_t(32 * s + i) * sk, place.at[0]);
        if constexpr (ROWS == 128) {
          const split_f32x2 x = *reinterpret_cast<const split_f32x2 *>(q);
          t.v[(s * 2 + 0) * 8 + i] = x[0];
          t.v[(s * 2 + 1) * 8 + i] = x[1];
        } else {
          t.v[s * 8 + i] = *reinterpret_cast<const float *>(q);
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < ROWS / 64; ++e) {
        const char *q = at(p + 32 * s, place.at[e]);
        const split_f32x4 x = *reinterpret_cast<const split_f32x4 *>(q), y = *reinterpret_cast<const split_f32x4 *>(q + 16);
        float *o = t.v + (s * (ROWS / 64) + e) * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = x[i], o[4 + i] = y[i];
      }
    }
  }
}

// The last stage of a ragged k, and every stage of MODE 0: clamped, always valid addresses with
// no branches; k >= k_left is zeroed at the LDS write.
template <int MODE, int ROWS, int NK>
__device__ __forceinline__ void tile_load_tail(TileRegs<MODE, ROWS, NK> &t, const float *__restrict__ p, int64_t sr,
                                               int64_t sk, int rows_left, int k_left, int tid) {
#pragma unroll
  for (int s = 0; s < NK; ++s) {
    if constexpr (MODE == 2) {
      constexpr int W = ROWS / 64;
      const int row = W * (tid & 63), kg = tid >> 6;
      const int rc = W == 2 ? max(0, min(row, rows_left - 2)) : min(row, rows_left - 1);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float *q = p + int64_t(min(32 * s + 8 * kg + i, k_left - 1)) * sk + rc;
        if constexpr (W == 2) {
          const split_f32x2 x = *reinterpret_cast<const split_f32x2 *>(q);
          t.v[(s * 2 + 0) * 8 + i] = x[0];
          t.v[(s * 2 + 1) * 8 + i] = x[1];
        } else {
          t.v[s * 8 + i] = *q;
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < ROWS / 64; ++e) {
        const int slot = tid + e * 256, row = slot >> 2, k = 32 * s + 8 * (slot & 3);
        const float *q = p + int64_t(min(row, rows_left - 1)) * sr;
        float *o = t.v + (s * (ROWS / 64) + e) * 8;
        if constexpr (MODE == 1) {
          const split_f32x4 x = *reinterpret_cast<const split_f32x4 *>(q + max(0, min(k, k_left - 4)));
          const split_f32x4 y = *reinterpret_cast<const split_f32x4 *>(q + max(0, min(k + 4, k_left - 4)));
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = x[i], o[4 + i] = y[i];
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) o[i] = q[int64_t(min(k + i, k_left - 1)) * sk];
        }
      }
    }
  }
}

// The largest row stride (MODE 1) or k stride (MODE 2) whose offsets inside a tile fit 32 bits.
constexpr int64_t TILE_MAX_STRIDE = int64_t(1) << 22;

// Converts the stage's values and writes them to `lds`: part p of k step s at byte
// (s PLANES + p) plane.  TAIL: k >= k_left is zeroed (the last stage of a ragged k).
// `sums` (one per row of the thread, or NULL) receives the values as multiplied.
template <int MODE, int ROWS, int NK, int PLANES, bool TAIL>
__device__ __forceinline__ void tile_store(char *lds, int plane, const TileRegs<MODE, ROWS, NK> &t, int k_left, int tid,
                                           CarriedSum *sums = nullptr) {
#pragma unroll
  for (int s = 0; s < NK; ++s)
#pragma unroll
    for (int e = 0; e < ROWS / 64; ++e) {
      int row, kg;
      if constexpr (MODE == 2) {
        row = (ROWS / 64) * (tid & 63) + e;
        kg = tid >> 6;
      } else {
        row = (tid + e * 256) >> 2;
        kg = tid & 3;
      }
      const float *v = t.v + (s * (ROWS / 64) + e) * 8;
      split_f32x4 x, y;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 32 * s + 8 * kg + i;
        x[i] = !TAIL || k < k_left ? v[i] : 0.f;
        y[i] = !TAIL || k + 4 < k_left ? v[4 + i] : 0.f;
      }
      char *o = lds + s * PLANES * plane + tile_offset(row, kg);
      if constexpr (PLANES == 3) {
        const Split8 p = split8(x, y);
        *reinterpret_cast<split_u32x4 *>(o) = p.hi;
        *reinterpret_cast<split_u32x4 *>(o + plane) = p.mid;
        *reinterpret_cast<split_u32x4 *>(o + 2 * plane) = p.lo;
        if (sums) sums[e].add(((x[0] + x[1]) + (x[2] + x[3])) + ((y[0] + y[1]) + (y[2] + y[3])));
      } else {
        const split_u32x4 p = {split_pack(x[0], x[1]), split_pack(x[2], x[3]), split_pack(y[0], y[1]),
                               split_pack(y[2], y[3])};
        *reinterpret_cast<split_u32x4 *>(o) = p;
        if (sums) {
          auto two = [&](int i) { return __uint_as_float(p[i] << 16) + __uint_as_float(p[i] & 0xffff0000u); };
          sums[e].add((two(0) + two(1)) + (two(2) + two(3)));
        }
      }
    }
}

// Stages of LDS: two blocks share a CU at either height, so TM 64 can hold the next stage beside
// the current one (one barrier per stage), TM 128 cannot.
template <int TM>
constexpr int tile_buffers() {
  return TM == 64 ? 2 : 1;
}
template <int TM, int PLANES, int NK>
constexpr int tile_lds_bytes() {
  return tile_buffers<TM>() * (TM + ST_N) * 64 * PLANES * NK;
}

// acc[i][j] = the wave's 16 x 16 tiles of A[m0 .., kbeg .. kend) B: lane (li, lg) holds rows
// 16 i + 4 lg + r, column 16 j + li of the wave's TM / 2 x 64 part.  a / b point at the tile's
// first row and column; ma / nb are the rows and columns left there.  All 256 threads call it.
// With SUMS and `row_sums` set, row_sums[r] = sum over k of A's row r as it was multiplied (r < ma).
template <int AM, int BM, int TM, int PLANES, int NK, bool SUMS = false>
__device__ __forceinline__ void tile_product(const float *__restrict__ a, int64_t sam, int64_t sak, int ma,
                                             const float *__restrict__ b, int64_t sbk, int64_t sbn, int nb, int kbeg,
                                             int kend, char *lds, split_f32x4 (&acc)[TM / 32][4],
                                             float *__restrict__ row_sums = nullptr) {
  constexpr int FM = TM / 32, KS = 32 * NK;
  constexpr int PLANE = (TM + ST_N) * 64;  // bytes of one part of one 32-k step, A rows then B rows
  constexpr int STAGE = PLANE * PLANES * NK;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1, li = lane & 15, lg = lane >> 4;
  const int frag = lg * 256 + ((li ^ (lg * 4)) << 4);
  split_f32x4 cor[FM][4];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = cor[i][j] = split_f32x4{0.f, 0.f, 0.f, 0.f};
  if (kbeg >= kend) return;  // (never with SUMS: slices are not empty)
  CarriedSum sums[TM / 64];
  TileRegs<AM, TM, NK> ra;
  TileRegs<BM, ST_N, NK> rb;
  const int last = kbeg + (kend - kbeg - 1) / KS * KS;  // first k of the last stage
  const TilePlace<AM, TM> pa = tile_place<AM, TM>(sam, sak, ma, tid);
  const TilePlace<BM, ST_N> pb = tile_place<BM, ST_N>(sbn, sbk, nb, tid);
  auto load = [&](int k0) {
    k0 = min(k0, last);
    if (AM != 0 && k0 + KS <= kend) {
      tile_load<AM, TM, NK>(ra, pa, a + int64_t(k0) * sak, sak);
      tile_load<BM, ST_N, NK>(rb, pb, b + int64_t(k0) * sbk, sbk);
    } else {
      tile_load_tail<AM, TM, NK>(ra, a + int64_t(k0) * sak, sam, sak, ma, kend - k0, tid);
      tile_load_tail<BM, ST_N, NK>(rb, b + int64_t(k0) * sbk, sbn, sbk, nb, kend - k0, tid);
    }
  };
  auto store = [&](auto tail, char *to, int k_left) {
    if constexpr (SUMS) {
      if (row_sums) tile_store<AM, TM, NK, PLANES, decltype(tail)::value>(to, PLANE, ra, k_left, tid, sums);
      else tile_store<AM, TM, NK, PLANES, decltype(tail)::value>(to, PLANE, ra, k_left, tid);
    } else {
      tile_store<AM, TM, NK, PLANES, decltype(tail)::value>(to, PLANE, ra, k_left, tid);
    }
    tile_store<BM, ST_N, NK, PLANES, decltype(tail)::value>(to + TM * 64, PLANE, rb, k_left, tid);
  };
  auto multiply = [&](const char *from) {
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const char *ta = from + s * PLANES * PLANE + wm * (TM / 2) * 64 + frag;
      const char *tb = from + s * PLANES * PLANE + (TM + wn * 64) * 64 + frag;
      auto part = [&](const char *t, int i, int p) {
        return *reinterpret_cast<const split_u32x4 *>(t + p * PLANE + i * 1024);
      };
      if constexpr (PLANES == 3) {
        Split8 fb[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[j] = Split8{part(tb, j, 0), part(tb, j, 1), part(tb, j, 2)};
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const Split8 fa{part(ta, i, 0), part(ta, i, 1), part(ta, i, 2)};
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] = split_mma1(fa.hi, fb[j].hi, acc[i][j]);
#pragma unroll
          for (int j = 0; j < 4; ++j) cor[i][j] = split_mma1(fa.lo, fb[j].hi, cor[i][j]);
#pragma unroll
          for (int j = 0; j < 4; ++j) cor[i][j] = split_mma1(fa.hi, fb[j].lo, cor[i][j]);
#pragma unroll
          for (int j = 0; j < 4; ++j) cor[i][j] = split_mma1(fa.mid, fb[j].mid, cor[i][j]);
#pragma unroll
          for (int j = 0; j < 4; ++j) cor[i][j] = split_mma1(fa.mid, fb[j].hi, cor[i][j]);
#pragma unroll
          for (int j = 0; j < 4; ++j) cor[i][j] = split_mma1(fa.hi, fb[j].mid, cor[i][j]);
        }
      } else {
        split_u32x4 fb[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[j] = part(tb, j, 0);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const split_u32x4 fa = part(ta, i, 0);
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] = split_mma1(fa, fb[j], acc[i][j]);
        }
      }
    }
  };
  constexpr std::integral_constant<bool, true> tail{};
  constexpr std::integral_constant<bool, false> full{};
  load(kbeg);
  store(tail, lds, kend - kbeg);
  load(kbeg + KS);
  __syncthreads();
  char *cur = lds, *nxt = lds + (tile_buffers<TM>() - 1) * STAGE;
  for (int k0 = kbeg; k0 + KS < kend; k0 += KS) {
    if constexpr (tile_buffers<TM>() == 1) {
      multiply(cur);
      __syncthreads();
    }
    if (k0 + 2 * KS <= kend) store(full, nxt, KS);
    else store(tail, nxt, kend - k0 - KS);
    load(k0 + 2 * KS);
    if constexpr (tile_buffers<TM>() == 2) multiply(cur);
    __syncthreads();
    char *t = cur;
    cur = nxt;
    nxt = t;
  }
  multiply(cur);
  if constexpr (SUMS) {
    if (row_sums) {  // a row's four k groups meet: four lanes (MODE 0, 1) or four waves (MODE 2)
      if constexpr (AM == 2) {
        __syncthreads();
        float *meet = reinterpret_cast<float *>(lds);  // [4][TM]
#pragma unroll
        for (int e = 0; e < TM / 64; ++e) meet[wave * TM + (TM / 64) * lane + e] = sums[e].value();
        __syncthreads();
        if (tid < TM && tid < ma) row_sums[tid] = (meet[tid] + meet[TM + tid]) + (meet[2 * TM + tid] + meet[3 * TM + tid]);
      } else {
#pragma unroll
        for (int e = 0; e < TM / 64; ++e) {
          float v = sums[e].value();
          v += __shfl_xor(v, 1);
          v += __shfl_xor(v, 2);
          const int row = (tid + e * 256) >> 2;
          if ((tid & 3) == 0 && row < ma) row_sums[row] = v;
        }
      }
    }
  }
  if constexpr (PLANES == 3) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] += cor[i][j];
  }
}

// Recomputes the tile's results that do not hold (split.h) as plain fp32 sums.  m0 / n0: the
// first row and column of the wave's part; a and b point at element k = 0 of the sum.
template <int FM>
__device__ __forceinline__ void tile_repair(split_f32x4 (&acc)[FM][4], const float *__restrict__ a, int64_t sam,
                                            int64_t sak, const float *__restrict__ b, int64_t sbk, int64_t sbn, int m0,
                                            int n0, int M, int N, int k) {
  unsigned least = SPLIT_LEAST, most = 0;  // (two instructions a result; zeros take the test below)
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const unsigned u = __float_as_uint(acc[i][j][r]) & 0x7fffffffu;
        least = min(least, u);
        most = max(most, u);
      }
  if (!__any(least < SPLIT_LEAST || most >= SPLIT_INF)) return;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + i * 16 + 4 * lg + r, n = n0 + j * 16 + li;
        if (split_holds(acc[i][j][r]) || m >= M || n >= N) continue;
        const float *ar = a + int64_t(m) * sam, *bc = b + int64_t(n) * sbn;
        CarriedSum v;
#pragma unroll 1
        for (int e = 0; e < k; ++e) v.add(ar[int64_t(e) * sak] * bc[int64_t(e) * sbk]);
        acc[i][j][r] = v.value();
      }
}

}  // namespace cg
