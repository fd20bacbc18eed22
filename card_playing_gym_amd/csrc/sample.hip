// Masked softmax and inverse-CDF sampling of policy rows on the device (gfx950):
// cardgym/rl/ppo.py:75-94 (masked_probabilities, sample_rows), which the reference runs
// in numpy on the host after copying each wave's logits back (cardgym/rl/selfplay.py:
// 532-567).  One wave per row, reproducing numpy's float32 arithmetic order:
//   probabilities: max over the legal entries (NaN propagates), exp(x - max) on legal
//     entries and 0 elsewhere, the normaliser summed in numpy's pairwise order (blocks of
//     at most 128 with eight running sums, halves split at multiples of 8), and a
//     correctly rounded division.  Only the float32 exp can differ from numpy's (by an
//     ulp; numpy's exp is CPU-specific code).
//   sampling: the running float32 sum of each row in index order, compared as float64
//     with the row's uniform; the count of entries below it, clamped to the last legal
//     index and replaced by it when the entry is illegal.  Given the same probabilities
//     and uniforms the result is the reference's, bit for bit.
#include <cmath>

#include "common.h"

namespace cg {
namespace {

constexpr int ROWS_PER_BLOCK = 4;  // one wave per row
constexpr int MAX_WIDTH = 4096;    // six halvings leave blocks of at most 128 entries

__device__ __forceinline__ float wave_max(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// numpy's float32 pairwise sum of w[0 .. n): a block of at most 128 keeps eight running sums
// r[j] = w[j] + w[j + 8] + ..., combined as ((r0 + r1) + (r2 + r3)) + ((r4 + r5) + (r6 + r7)) and
// followed by the n % 8 remaining entries one by one; larger ranges split at n / 2 rounded down
// to a multiple of 8.  The wave sums its leaf blocks eight at a time, eight lanes a block (one
// running sum per lane; the adds of a butterfly commute, so its order is numpy's), then adds them
// up along the tree.  Rounds of eight leaves: two up to 1024 entries, eight up to 4096.

// Visits the leaves of a range in order; leaf(index, offset, length) with wave-uniform arguments.
template <int LEVEL, typename F>
__device__ __forceinline__ void pairwise_leaves(int off, int n, int &index, const F &leaf) {
  if constexpr (LEVEL > 0) {
    if (n > 128) {
      const int n2 = n / 2 - n / 2 % 8;
      pairwise_leaves<LEVEL - 1>(off, n2, index, leaf);
      pairwise_leaves<LEVEL - 1>(off + n2, n - n2, index, leaf);
      return;
    }
  }
  leaf(index++, off, n);
}

template <int LEVEL, int ROUNDS>
__device__ __forceinline__ float pairwise_tree(int n, int &index, const float (&leaf)[ROUNDS]) {
  if constexpr (LEVEL > 0) {
    if (n > 128) {
      const int n2 = n / 2 - n / 2 % 8;
      const float left = pairwise_tree<LEVEL - 1>(n2, index, leaf);
      return left + pairwise_tree<LEVEL - 1>(n - n2, index, leaf);
    }
  }
  float v = leaf[0];
#pragma unroll
  for (int r = 1; r < ROUNDS; ++r) v = index >> 3 == r ? leaf[r] : v;
  return __shfl(v, 8 * (index++ & 7), 64);
}

// STEPS: the most entries of a leaf that one running sum takes (8 for rows of at most 64 entries).
template <int LEVEL, int ROUNDS, int STEPS = 16>
__device__ __forceinline__ float pairwise_sum(const float *w, int n, int lane) {
  int at[ROUNDS], len[ROUNDS], count = 0;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) at[r] = len[r] = 0;
  pairwise_leaves<LEVEL>(0, n, count, [&](int index, int off, int length) {
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const bool mine = index == 8 * r + (lane >> 3);
      at[r] = mine ? off : at[r];
      len[r] = mine ? length : len[r];
    }
  });
  float leaf[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    leaf[r] = 0.f;
    if (8 * r >= count) continue;
    const float *a = w + at[r];
    const int body = len[r] - len[r] % 8, j = lane & 7;
    if (body > 0) {
      float v[STEPS];
#pragma unroll
      for (int i = 0; i < STEPS; ++i) v[i] = a[min(8 * i, body - 8) + j];
      float s = v[0];
#pragma unroll
      for (int i = 1; i < STEPS; ++i) s = 8 * i < body ? s + v[i] : s;
      s += __shfl_xor(s, 1, 64);
      s += __shfl_xor(s, 2, 64);
      s += __shfl_xor(s, 4, 64);
      leaf[r] = s;
    }
    for (int i = body; i < len[r]; ++i) leaf[r] += a[i];
  }
  int index = 0;
  return pairwise_tree<LEVEL>(n, index, leaf);
}

// E > 0: rows of up to 64 E entries, held in registers from the one pass over them, E per lane
// (four consecutive ones with VEC: 16-byte aligned rows, 4-byte aligned masks).  E 0: any width.
template <int E, bool VEC>
__global__ __launch_bounds__(64 * ROWS_PER_BLOCK) void masked_probabilities_kernel(
    const float *__restrict__ logits, int64_t ld_logits, const uint8_t *__restrict__ mask, int64_t ld_mask,
    int32_t rows, int32_t width, float *__restrict__ probs, int64_t ld_probs) {
  extern __shared__ float wrow[];  // [ROWS_PER_BLOCK][width]: the row's weights
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = blockIdx.x * ROWS_PER_BLOCK + wave;
  if (row >= rows) return;  // whole wave
  const float *x = logits + int64_t(row) * ld_logits;
  const uint8_t *legal = mask + int64_t(row) * ld_mask;
  float *p = probs + int64_t(row) * ld_probs;
  float *w = wrow + wave * width;
  // max over the legal entries; a NaN among them makes it NaN, as numpy's max does
  float m = -INFINITY;
  int nan = 0;
  auto see = [&](float v) {
    if (v != v) nan = 1;
    else m = fmaxf(m, v);
  };
  auto settle = [&] {
    m = wave_max(m);
    if (__any(nan)) m = NAN;
  };
  auto visible = [] {  // the wave's LDS writes to its own reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  if constexpr (E == 0) {
    for (int i = lane; i < width; i += 64) see(legal[i] ? x[i] : -INFINITY);
    settle();
    for (int i = lane; i < width; i += 64) w[i] = legal[i] ? expf(x[i] - m) : 0.f;
    visible();
    const float total = pairwise_sum<6, 8>(w, width, lane);
    for (int i = lane; i < width; i += 64) p[i] = w[i] / total;
  } else {
    float v[E];
    bool on[E];
    // Entry of v[e]: with VEC 256 (e / 4) + 4 lane + e % 4, else 64 e + lane.
    auto index = [&](int e) { return VEC ? 256 * (e >> 2) + 4 * lane + (e & 3) : 64 * e + lane; };
    if constexpr (VEC) {
#pragma unroll
      for (int q = 0; q < E / 4; ++q) {
        const int i = 256 * q + 4 * lane, at = i < width ? i : 0;
        const float4 f = *reinterpret_cast<const float4 *>(x + at);
        const uchar4 l = *reinterpret_cast<const uchar4 *>(legal + at);
        const bool in = i < width;
        v[4 * q] = f.x, v[4 * q + 1] = f.y, v[4 * q + 2] = f.z, v[4 * q + 3] = f.w;
        on[4 * q] = in && l.x, on[4 * q + 1] = in && l.y, on[4 * q + 2] = in && l.z, on[4 * q + 3] = in && l.w;
      }
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = index(e), at = i < width ? i : 0;
        v[e] = x[at];
        on[e] = i < width && legal[at];
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) see(on[e] ? v[e] : -INFINITY);
    settle();
#pragma unroll
    for (int e = 0; e < E; ++e) {
      v[e] = on[e] ? expf(v[e] - m) : 0.f;
      if (index(e) < width) w[index(e)] = v[e];
    }
    visible();
    // Leaves of at most 128: one up to 128 entries, four (two halvings) up to 256.
    const float total = E == 1   ? pairwise_sum<0, 1, 8>(w, width, lane)
                        : E == 4 ? pairwise_sum<2, 1>(w, width, lane)
                       : E == 2 ? pairwise_sum<0, 1>(w, width, lane)
                                 : pairwise_sum<4, 2>(w, width, lane);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] /= total;
    if constexpr (VEC) {
#pragma unroll
      for (int q = 0; q < E / 4; ++q)
        if (256 * q + 4 * lane < width)
          *reinterpret_cast<float4 *>(p + 256 * q + 4 * lane) = float4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (index(e) < width) p[index(e)] = v[e];
    }
  }
}

// The running sums of a row are a serial chain (np.cumsum's order), so the block's rows walk it
// side by side, one lane each, with the next 16 entries already in registers; loading the rows
// and counting the sums below each uniform is the whole block's work.  `pitch` (floats, 4 mod 64)
// keeps 16 rows' accesses to one column on different LDS banks; its tail past the width is walked
// but not counted.
template <int PER_WAVE>
__global__ __launch_bounds__(256) void sample_rows_kernel(
    const float *__restrict__ probs, int64_t ld_probs, const uint8_t *__restrict__ mask, int64_t ld_mask,
    const double *__restrict__ uniforms, int32_t rows, int32_t width, int32_t pitch, int64_t *__restrict__ sampled) {
  extern __shared__ __align__(16) float prow[];  // [4 PER_WAVE][pitch]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = blockIdx.x * 4 * PER_WAVE, mine = row0 + wave * PER_WAVE;
  const float *p[PER_WAVE];
  const uint8_t *legal[PER_WAVE];
  int last[PER_WAVE];
  double u[PER_WAVE];
#pragma unroll
  for (int r = 0; r < PER_WAVE; ++r) {  // rows past the end are read (not written) as the last one
    const int64_t row = min(mine + r, rows - 1);
    p[r] = probs + row * ld_probs;
    legal[r] = mask + row * ld_mask;
    last[r] = -1;
    u[r] = uniforms[row];  // (in flight while the running sums form)
  }
#pragma unroll 4
  for (int i = lane; i < width; i += 64) {
#pragma unroll
    for (int r = 0; r < PER_WAVE; ++r) {
      prow[(wave * PER_WAVE + r) * pitch + i] = p[r][i];
      if (legal[r][i]) last[r] = i;
    }
  }
  __syncthreads();
  if (threadIdx.x < 4 * PER_WAVE) {
    float *pr = prow + threadIdx.x * pitch;
    float4 q[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) q[k] = *reinterpret_cast<const float4 *>(pr + 4 * k);
    float c = -0.f;  // -0 + x is x, bit for bit
    for (int i = 0; i < width; i += 16) {
      float4 n[4];
      const int next = i + 16 < width ? i + 16 : i;
#pragma unroll
      for (int k = 0; k < 4; ++k) n[k] = *reinterpret_cast<const float4 *>(pr + next + 4 * k);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        c += q[k].x;
        q[k].x = c;
        c += q[k].y;
        q[k].y = c;
        c += q[k].z;
        q[k].z = c;
        c += q[k].w;
        q[k].w = c;
        *reinterpret_cast<float4 *>(pr + i + 4 * k) = q[k];
        q[k] = n[k];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < PER_WAVE; ++r) {
    const int row = mine + r;
    if (row >= rows) break;  // whole wave
    // float c < double u  <=>  c < t, t the least float >= u (NaN and +-inf included).
    float t = float(u[r]);
    if (double(t) < u[r]) t = nextafterf(t, INFINITY);
    const float *pr = prow + (wave * PER_WAVE + r) * pitch;
    int below = 0, top = last[r];
    for (int i = lane; i < width; i += 64) below += pr[i] < t;
    for (int o = 32; o > 0; o >>= 1) {
      below += __shfl_xor(below, o, 64);
      top = max(top, __shfl_xor(top, o, 64));
    }
    if (lane != 0) continue;
    if (top < 0) top = width - 1;
    int s = below < top ? below : top;
    if (!legal[r][s]) s = top;
    sampled[row] = s;
  }
}

}  // namespace
}  // namespace cg

using namespace cg;

extern "C" {

int cg_masked_probabilities(const float *logits, int64_t ld_logits, const uint8_t *mask, int64_t ld_mask,
                            int32_t rows, int32_t width, float *probs, int64_t ld_probs, void *stream) {
  return guarded([&] {
    CG_REQUIRE(rows >= 0 && width >= 0, CG_ERR_INVALID, "rows and width must be non-negative");
    if (rows == 0 || width == 0) return;
    CG_REQUIRE(logits && mask && probs, CG_ERR_INVALID, "logits, mask and probs are required");
    CG_REQUIRE(ld_logits >= width && ld_mask >= width && ld_probs >= width, CG_ERR_INVALID,
               "row strides must be at least the width");
    CG_REQUIRE(width <= MAX_WIDTH, CG_ERR_UNSUPPORTED, "masked_probabilities: rows wider than 4096");
    const size_t lds = size_t(ROWS_PER_BLOCK) * width * 4;
    const unsigned grid = unsigned((int64_t(rows) + ROWS_PER_BLOCK - 1) / ROWS_PER_BLOCK);
    const uintptr_t at = reinterpret_cast<uintptr_t>(logits) | reinterpret_cast<uintptr_t>(probs);
    const bool vec = width % 4 == 0 && (at & 15) == 0 && (reinterpret_cast<uintptr_t>(mask) & 3) == 0 &&
                     ((ld_logits | ld_mask | ld_probs) & 3) == 0;
    // Entries per lane by width: a lane of 16 does the exponentials and divisions of 1024 entries
    // whatever the width (65536 rows of 8, 64 and 128 entries: 55 us; 16, 17 and 25 so).
    const auto kernel = width > 1024  ? masked_probabilities_kernel<0, false>
                        : width > 256 ? (vec ? masked_probabilities_kernel<16, true> : masked_probabilities_kernel<16, false>)
                        : width > 128 ? (vec ? masked_probabilities_kernel<4, true> : masked_probabilities_kernel<4, false>)
                        : width > 64  ? masked_probabilities_kernel<2, false>
                                      : masked_probabilities_kernel<1, false>;
    kernel<<<grid, 64 * ROWS_PER_BLOCK, lds, as_stream(stream)>>>(logits, ld_logits, mask, ld_mask, rows, width, probs,
                                                                  ld_probs);
    CG_LAUNCHED();
  });
}

int cg_sample_rows(const float *probs, int64_t ld_probs, const uint8_t *mask, int64_t ld_mask,
                   const double *uniforms, int32_t rows, int32_t width, int64_t *sampled, void *stream) {
  return guarded([&] {
    CG_REQUIRE(rows >= 0 && width >= 0, CG_ERR_INVALID, "rows and width must be non-negative");
    if (rows == 0) return;
    CG_REQUIRE(width > 0, CG_ERR_INVALID, "cannot sample from rows of width 0");
    CG_REQUIRE(probs && mask && uniforms && sampled, CG_ERR_INVALID, "probs, mask, uniforms and sampled are required");
    CG_REQUIRE(ld_probs >= width && ld_mask >= width, CG_ERR_INVALID, "row strides must be at least the width");
    CG_REQUIRE(width <= MAX_WIDTH, CG_ERR_UNSUPPORTED, "sample_rows: rows wider than 4096");
    // Rows per block: 4 while that leaves few wavefronts to a CU or the rows are short (us for 4, 8 and 16
    // rows: 64 x 8 2.6, 3.1, 4.4; 4096 x 64 3.5, 3.9, 4.9; 8192 x 256 7.7, 6.8, 7.7), 16 for many entries
    // of rows that leave a CU four blocks of LDS (16384 x 256 14.6, 9.7, 8.9; 65536 x 512 84, 56, 52; but
    // 65536 x 600 100, 67, 76), 8 between.  A row of 4096 entries takes 16 KB of 64.
    const int pitch = width > 4032 ? (width + 15) / 16 * 16 : (width + 63) / 64 * 64 + 4;
    const int64_t entries = int64_t(rows) * width;
    const int per_wave = rows <= 1024 || entries <= (rows <= 4096 ? 1 << 20 : 1 << 19)        ? 1
                         : rows >= 16384 && entries >= 1 << 21 && 64 * pitch <= 40960 ? 4
                         : 32 * pitch <= 65536                                        ? 2
                                                                                      : 1;
    const auto kernel = per_wave == 4 ? sample_rows_kernel<4> : per_wave == 2 ? sample_rows_kernel<2> : sample_rows_kernel<1>;
    kernel<<<unsigned((int64_t(rows) + 4 * per_wave - 1) / (4 * per_wave)), 256, size_t(4 * per_wave) * pitch * 4,
             as_stream(stream)>>>(probs, ld_probs, mask, ld_mask, uniforms, rows, width, pitch, sampled);
    CG_LAUNCHED();
  });
}

}  // extern "C"
