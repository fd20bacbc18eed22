// Training side of the trunk (gfx950, fp32): the pieces of a packed-row forward that keeps
// what its backward needs, and that backward (cardgym/nn/trunk.py:124-181, 285-374 under
// autograd; packed rows as in cardgym/nn/packing.py:36-40).
//
//   * gemm_strided_kernel   C = alpha op(A) op(B) + beta C for any strides: the weight
//                           gradients (dW = dY^T X) and input gradients (dX = dY W) of
//                           every projection (split_tile.h);
//   * layernorm_fwd / _bwd  LayerNorm keeping (mean, rstd) per row; the backward's input
//                           gradient per row and per-block partial sums of dw / db;
//   * rmsnorm_bwd           the input RMSNorm's backward (gain only);
//   * gelu_fwd / _bwd       erf GELU and its derivative;
//   * attn_fwd              causal attention inside each packed sequence (GQA), keeping
//                           the log-sum-exp of every (token, head);
//   * attn_bwd_dq / _dkv    its backward: dQ (and D = rowsum(dO * O)) per (token, head),
//                           dK / dV per (token, KV head) summed over the head group.
// The attention kernels work on 16 x 16 (query, key) tiles; head_dim is a template parameter
// (8 to 64).
#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "common.h"
#include "split_tile.h"

namespace cg {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;

// bf16 (autocast) precision: values are kept in fp32 storage holding bf16 numbers.  A pair of
// fp32 values to packed bf16, round to nearest even (v_cvt_pk_bf16_f32): a in the low half.
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
// The bf16 value nearest x, as fp32.
__device__ __forceinline__ float round_bf16(float x) { return __builtin_bit_cast(float, pack_bf16(0.f, x) & 0xffff0000u); }

// erf by Abramowitz & Stegun, Handbook of Mathematical Functions, formula 7.1.26:
// erf(x) = 1 - (a1 t + a2 t^2 + a3 t^3 + a4 t^4 + a5 t^5) e^(-x^2), t = 1 / (1 + p x) for x >= 0
// (odd in x), |error| <= 1.5e-7.  `gauss` receives e^(-x^2), which GELU's derivative reuses.
__device__ __forceinline__ float erf_as(float x, float &gauss) {
  const float ax = fabsf(x);
  const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, ax, 1.0f));
  const float poly =
      t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, 1.061405429f, -1.453152027f), 1.421413741f), -0.284496736f), 0.254829592f);
  gauss = __expf(-ax * ax);
  return copysignf(1.0f - poly * gauss, x);
}

// erf GELU, u Phi(u), and its derivative Phi(u) + u phi(u) (phi(u) = e^(-u^2 / 2) / sqrt(2 pi)).
__device__ __forceinline__ float gelu_exact(float u) {
  float gauss;
  return 0.5f * u * (1.0f + erf_as(u * 0.70710678118654752f, gauss));
}
__device__ __forceinline__ float gelu_grad(float u) {
  float gauss;
  const float cdf = 0.5f * (1.0f + erf_as(u * 0.70710678118654752f, gauss));
  return fmaf(u * 0.3989422804014327f, gauss, cdf);
}

// What a GEMM does with each result v = alpha (A B)[m, n] on its way out: add bias[n], round
// to bf16 when `round` (autocast: a bf16 product's output), add beta times the prior value
// (read from `cin` when set, else from C itself: the fp32 residual), then either multiply by
// gelu'(aux_in[m, n]) (GELU_GRAD: the MLP's backward; rounded again under `round`) or also
// write gelu(v) to aux_out[m, n] (GELU: the MLP's forward; rounded under `round`).
// aux_in / aux_out / cin share C's row stride.
enum EpiMode : int32_t { EPI_PLAIN = 0, EPI_GELU = 1, EPI_GELU_GRAD = 2 };
struct Epi {
  const float *bias = nullptr;
  const float *cin = nullptr;
  const float *aux_in = nullptr;
  float *aux_out = nullptr;
  float *row_sum = nullptr;  // [M]: also the sums of A's rows over k (a weight gradient's bias gradient;
                             // under `round` of the rounded operands, rounded)
  int32_t mode = EPI_PLAIN;
  int32_t round = 0;  // bf16 operands (the GEMM rounds them as it stages) and bf16 outputs
};

__device__ __forceinline__ float epi_value(const Epi &e, float v, float beta, float prior, float bias, float aux) {
  v += bias;
  if (e.round) v = round_bf16(v);
  if (beta != 0.f) v += beta * prior;
  if (e.mode == EPI_GELU_GRAD) {
    v *= gelu_grad(aux);
    if (e.round) v = round_bf16(v);
  }
  return v;
}

__device__ __forceinline__ void epilogue(const Epi &e, float v, float beta, float *__restrict__ C, int64_t ldc,
                                         int64_t m, int64_t n) {
  const int64_t i = m * ldc + n;
  v = epi_value(e, v, beta, beta != 0.f ? (e.cin ? e.cin[i] : C[i]) : 0.f, e.bias ? e.bias[n] : 0.f,
                e.mode == EPI_GELU_GRAD ? e.aux_in[i] : 0.f);
  C[i] = v;
  if (e.mode == EPI_GELU) e.aux_out[i] = e.round ? round_bf16(gelu_exact(v)) : gelu_exact(v);
}

// ---- strided GEMM ---------------------------------------------------------------------
// A(m, k) = A[m * sam + k * sak], B(k, n) = B[k * sbk + n * sbn]; TM x 128 tiles through
// tile_product (split_tile.h): fp32 products in three bf16 parts, bf16 (autocast) ones with
// operands rounded as they are staged.  Split K (grid.z > 1): slice z covers k in
// [z kc, (z + 1) kc) and writes its partial product to part[z] ([m, n]); a second pass sums
// them.
constexpr int GT_M = 128, GT_N = ST_N, GT_K = 32;

template <int AM, int BM, int TM, bool BF, bool SUMS>
__global__ __launch_bounds__(256, 2) void gemm_strided_kernel(int32_t M, int32_t N, int32_t K, int32_t kc, float alpha,
                                                           const float *__restrict__ A, int64_t sam, int64_t sak,
                                                           const float *__restrict__ B, int64_t sbk, int64_t sbn,
                                                           float beta, float *__restrict__ C, int64_t ldc,
                                                           float *__restrict__ part, const Epi epi) {
  constexpr int FM = TM / 32;  // 16-row MFMA blocks per wave: a wave takes TM / 2 rows x 64 columns
  constexpr int PLANES = BF ? 1 : 3, NK = BF ? 2 : 1;
  __shared__ __align__(16) char lds[tile_lds_bytes<TM, PLANES, NK>()];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lg = lane >> 4;
  int mt = blockIdx.y, nt = blockIdx.x;
  if (gridDim.z == 1) {  // XCD-aware order: XCD k (block ids = k mod 8) takes a contiguous run of
                         // tiles, N fastest, so the rows of A it reads stay in its own L2
    const int tiles = gridDim.x * gridDim.y, b = blockIdx.x + gridDim.x * blockIdx.y;
    const int xcd = b & 7, per = tiles >> 3, extra = tiles & 7;
    const int t = xcd * per + min(xcd, extra) + (b >> 3);
    mt = t / gridDim.x;
    nt = t % gridDim.x;
  }
  const int m0 = mt * TM, n0 = nt * GT_N;
  const int kbeg = blockIdx.z * kc, kend = min(K, kbeg + kc);
  f32x4 acc[FM][4];
  // Row sums: the first column of tiles leaves them beside its slice's partial products.
  float *sums = nullptr;
  if constexpr (SUMS)
    if (nt == 0) sums = part ? part + int64_t(gridDim.z) * M * N + int64_t(blockIdx.z) * M + m0 : epi.row_sum + m0;
  tile_product<AM, BM, TM, PLANES, NK, SUMS>(A + int64_t(m0) * sam, sam, sak, M - m0, B + int64_t(n0) * sbn, sbk, sbn,
                                             N - n0, kbeg, kend, lds, acc, sums);
  if constexpr (SUMS && BF)
    if (sums && !part) {  // the sums' own threads wrote them
      __syncthreads();
      if (int(threadIdx.x) < min(TM, M - m0)) sums[threadIdx.x] = round_bf16(sums[threadIdx.x]);
    }
  if constexpr (!BF)
    tile_repair<FM>(acc, A + int64_t(kbeg) * sak, sam, sak, B + int64_t(kbeg) * sbk, sbk, sbn, m0 + wm * (TM / 2),
                    n0 + wn * 64, M, N, kend - kbeg);
  if (part) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + wm * (TM / 2) + i * 16 + 4 * lg + r, n = n0 + wn * 64 + j * 16 + li;
          if (m < M && n < N) part[(int64_t(blockIdx.z) * M + m) * N + n] = acc[i][j][r];
        }
    return;
  }
  // Epilogue, a 16-row block at a time: every operand it reads (prior C or cin, bias, aux_in; only
  // those this product has) is loaded at once, from addresses a uniform pointer plus 32 bits per
  // lane; tiles that hang over an edge clamp them.
  const bool prior = beta != 0.f, grad = epi.mode == EPI_GELU_GRAD, fwd_gelu = epi.mode == EPI_GELU;
  const float *pin = epi.cin ? epi.cin : C;
  float bj[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = min(n0 + wn * 64 + j * 16 + li, N - 1);
    bj[j] = epi.bias ? epi.bias[n] : 0.f;
  }
  const bool inside = m0 + TM <= M && n0 + GT_N <= N && ldc >= 0 && ldc <= TILE_MAX_STRIDE;
  auto finish = [&](auto whole) {
    constexpr bool WHOLE = decltype(whole)::value;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int64_t base = int64_t(m0 + i * 16) * ldc + n0;
      unsigned at[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) at[r] = 4u * (unsigned(wm * (TM / 2) + 4 * lg + r) * unsigned(ldc) + unsigned(wn * 64 + li));
      auto place = [&](auto *p, int j, int r) {
        using T = std::remove_pointer_t<decltype(p)>;
        if constexpr (WHOLE) {
          using B = std::conditional_t<std::is_const_v<T>, const char, char>;
          return reinterpret_cast<T *>(reinterpret_cast<B *>(p + base + 16 * j) + at[r]);
        } else {
          const int64_t m = min(m0 + wm * (TM / 2) + i * 16 + 4 * lg + r, M - 1), n = min(n0 + wn * 64 + j * 16 + li, N - 1);
          return p + m * ldc + n;
        }
      };
      float pv[4][4], av[4][4];
      if (prior) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) pv[j][r] = *place(pin, j, r);
      }
      if (grad) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) av[j][r] = *place(epi.aux_in, j, r);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + wm * (TM / 2) + i * 16 + 4 * lg + r, n = n0 + wn * 64 + j * 16 + li;
          const float v = epi_value(epi, alpha * acc[i][j][r], beta, prior ? pv[j][r] : 0.f, bj[j], grad ? av[j][r] : 0.f);
          if (WHOLE || (m < M && n < N)) {
            *place(C, j, r) = v;
            if (fwd_gelu) *place(epi.aux_out, j, r) = epi.round ? round_bf16(gelu_exact(v)) : gelu_exact(v);
          }
        }
    }
  };
  if (inside) finish(std::true_type{});
  else finish(std::false_type{});
}

// ---- products of few rows --------------------------------------------------------------
// A microbatch of hundreds of rows is bound by launches and by the latency of each: a staged product
// split over k takes a second launch for its slices (792 x 256 x 512: 11.4 us, 7.1 here).  Here one launch
// spreads k over the eight waves of a 32 x 32 tile's block, each reading its operand fragments straight
// from global memory (lane (li, lg): row li, k 8 lg .. 8 lg + 7 of a 32-k step) and the partial tiles
// meeting in LDS.
template <int MODE>
__device__ __forceinline__ void rows_frag(const float *__restrict__ p, int64_t sk, int k0, int K, split_f32x4 (&v)[2]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int k = k0 + 4 * h;
    if constexpr (MODE == 1) {  // K is a multiple of 4
      const split_f32x4 x = *reinterpret_cast<const split_f32x4 *>(p + min(k, K - 4));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[h][e] = k < K ? x[e] : 0.f;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = p[int64_t(min(k + e, K - 1)) * sk];
        v[h][e] = k + e < K ? x : 0.f;
      }
    }
  }
}

// Up to 512 tiles (two blocks a CU) and k of 1024: us here and through staged tiles, x w^T fp32 2040 x 256 x
// 256 6.6, 12.7, at k 1024 19.7, 24.4; 64 x 256 x 1024 10.3, 11.5, bf16 there 9.4, 8.7, all in one launch.
// Weight gradients in bf16 read both operands a value at a time here (2040 x 256 over 1024 26.0, 22.7; 792 x
// 512 16.2, 20.4), so the longest of them with the most tiles stay staged.
constexpr int ROWS_K = 1024;
constexpr int64_t ROWS_TILES = 512, ROWS_GRAD_WORK = 448 * 1024;
bool few_rows(int32_t m, int32_t n, int32_t k, bool bf16_gradient) {
  const int64_t tiles = int64_t((m + 31) / 32) * ((n + 31) / 32);
  return k > 0 && k <= ROWS_K && tiles <= ROWS_TILES && (!bf16_gradient || tiles * k <= ROWS_GRAD_WORK);
}

template <int AM, int BM, bool BF, bool SUMS>
__global__ __launch_bounds__(512) void gemm_rows_kernel(int32_t M, int32_t N, int32_t K, float alpha,
                                                        const float *__restrict__ A, int64_t sam, int64_t sak,
                                                        const float *__restrict__ B, int64_t sbk, int64_t sbn, float beta,
                                                        float *__restrict__ C, int64_t ldc, const Epi epi) {
  constexpr int T = 32, PITCH = T + 4, WAVES = 8, PARTS = BF ? 1 : 3;
  __shared__ float red[WAVES][T * PITCH];
  __shared__ float sums[SUMS ? WAVES : 1][T];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  const float *ar[2], *br[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    ar[i] = A + int64_t(min(m0 + 16 * i + li, M - 1)) * sam;
    br[i] = B + int64_t(min(n0 + 16 * i + li, N - 1)) * sbn;
  }
  f32x4 acc[2][2], cor[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = cor[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float rs[2] = {0.f, 0.f};
  for (int k0 = 32 * wave; k0 < K; k0 += 2 * 32 * WAVES) {
    split_f32x4 a[2][2][2], b[2][2][2];  // two steps' operands in flight
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int k = k0 + t * 32 * WAVES;
      if (k >= K) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        rows_frag<AM>(ar[i], sak, k + 8 * lg, K, a[t][i]);
        rows_frag<BM>(br[i], sbk, k + 8 * lg, K, b[t][i]);
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (k0 + t * 32 * WAVES >= K) continue;
      if constexpr (BF) {
        split_u32x4 af[2], bf[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            af[i][e] = split_pack(a[t][i][e >> 1][2 * (e & 1)], a[t][i][e >> 1][2 * (e & 1) + 1]);
            bf[i][e] = split_pack(b[t][i][e >> 1][2 * (e & 1)], b[t][i][e >> 1][2 * (e & 1) + 1]);
            if constexpr (SUMS) rs[i] += __uint_as_float(af[i][e] << 16) + __uint_as_float(af[i][e] & 0xffff0000u);
          }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = split_mma1(af[i], bf[j], acc[i][j]);
      } else {
        Split8 as[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          as[i] = split8(a[t][i][0], a[t][i][1]);
          if constexpr (SUMS) {
            const split_f32x4 s = a[t][i][0] + a[t][i][1];
            rs[i] += (s[0] + s[1]) + (s[2] + s[3]);
          }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const Split8 bs = split8(b[t][j][0], b[t][j][1]);
#pragma unroll
          for (int i = 0; i < 2; ++i) split_mma(as[i], bs, acc[i][j], cor[i][j]);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[wave][(16 * i + 4 * lg + r) * PITCH + 16 * j + li] = PARTS == 3 ? acc[i][j][r] + cor[i][j][r] : acc[i][j][r];
  if constexpr (SUMS) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      rs[i] += __shfl_xor(rs[i], 16);
      rs[i] += __shfl_xor(rs[i], 32);
      if (lg == 0) sums[wave][16 * i + li] = rs[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = tid; e < T * T; e += 64 * WAVES) {
    const int r = e / T, c = e % T, m = m0 + r, n = n0 + c;
    float v = red[0][r * PITCH + c];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += red[w][r * PITCH + c];
    if (m >= M || n >= N) continue;
    if (!BF && __builtin_expect(!split_holds(v), 0)) {  // see split.h
      CarriedSum sum;
#pragma unroll 1
      for (int k = 0; k < K; ++k) sum.add(A[m * sam + k * sak] * B[k * sbk + n * sbn]);
      v = sum.value();
    }
    epilogue(epi, alpha * v, beta, C, ldc, m, n);
  }
  if constexpr (SUMS) {
    if (blockIdx.x == 0 && tid < T && m0 + tid < M) {
      float v = sums[0][tid];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) v += sums[w][tid];
      epi.row_sum[m0 + tid] = BF ? round_bf16(v) : v;
    }
  }
}

// C[m, n] = epilogue(alpha * sum_z part[z][m, n]).  A block takes 64 times four consecutive entries
// (float4 loads when N is a multiple of 4); its wave w sums the slices z = w mod 4, four at a time, and the
// waves' sums meet in LDS, so that few entries of many slices still fill the chip with loads in flight.
__global__ __launch_bounds__(256) void gemm_reduce_kernel(int32_t M, int32_t N, int32_t slices, float alpha,
                                                          const float *__restrict__ part, float beta,
                                                          float *__restrict__ C, int64_t ldc, const Epi epi) {
  __shared__ __align__(16) float red[4][256];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t total = int64_t(M) * N, first = 256 * int64_t(blockIdx.x), i0 = first + 4 * lane;
  f32x4 s[4] = {};
  if ((N & 3) == 0) {
    if (i0 < total) {
      int z = wave;
      for (; z + 12 < slices; z += 16)
#pragma unroll
        for (int u = 0; u < 4; ++u) s[u] += *reinterpret_cast<const f32x4 *>(part + int64_t(z + 4 * u) * total + i0);
      for (; z < slices; z += 4) s[0] += *reinterpret_cast<const f32x4 *>(part + int64_t(z) * total + i0);
    }
  } else {
    for (int z = wave; z < slices; z += 4)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i0 + e < total) s[0][e] += part[int64_t(z) * total + i0 + e];
  }
  *reinterpret_cast<f32x4 *>(&red[wave][4 * lane]) = (s[0] + s[1]) + (s[2] + s[3]);
  __syncthreads();
  const int64_t i = first + tid;
  if (i < total) {
    const float v = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
    epilogue(epi, alpha * v, beta, C, ldc, i / N, i % N);
  }
  if (epi.row_sum) {
    const float *sums = part + int64_t(slices) * total;
    for (int64_t m0 = 64 * int64_t(blockIdx.x); m0 < M; m0 += 64 * int64_t(gridDim.x)) {
      CarriedSum t;
      const int64_t m = min<int64_t>(m0 + lane, M - 1);
#pragma unroll 4
      for (int z = wave; z < slices; z += 4) t.add(sums[int64_t(z) * M + m]);
      __syncthreads();
      red[wave][lane] = t.sum;
      red[wave][64 + lane] = t.lost;
      __syncthreads();
      if (wave == 0 && m0 + lane < M) {
        for (int w = 1; w < 4; ++w) t.add(red[w][lane]);
        t.lost += (red[1][64 + lane] + red[2][64 + lane]) + red[3][64 + lane];
        const float v = t.value();
        epi.row_sum[m0 + lane] = epi.round ? round_bf16(v) : v;
      }
    }
  }
}

// Launch plan: row tile TM and split K.  Products of few 128-row tiles take 64-row tiles (twice the
// blocks): with a short reduction, or up to sixteen of them, three parts over 8192 and more up to eight
// (dY^T X 1024 x 256, us in 64-row and 128-row tiles: bf16 over 16384 tokens 39.8, 45.4, fp32 over 4096
// 25.6, 28.6, over 8192 40.4, 39.8, over 16384 66.8, 62.4; 256 x 256 over 16384 fp32 27.4, 28.2).  A
// reduction whose tiles leave most of the chip idle is split over k into enough (tile, slice) blocks to
// fill it, and a second pass sums the slices.
struct GemmPlan {
  int tm, slices, kc;
};
GemmPlan gemm_plan(int32_t m, int32_t n, int32_t k, bool generic, bool bf16) {
  const int64_t nt = (n + GT_N - 1) / GT_N, tiles128 = int64_t((m + GT_M - 1) / GT_M) * nt;
  int tm = GT_M;
  if (!generic && (m <= 64 || tiles128 <= (bf16 || k < 8192 ? 16 : 8) || (tiles128 < 512 && !(k >= 1024 && tiles128 < 128)))) tm = 64;
  const int64_t tiles = int64_t((m + tm - 1) / tm) * nt;
  // Split K toward the 512 blocks that the chip holds at once (256 CUs x 2), never past them: 408
  // tiles split in two would run as a full wave plus a tail, slower than unsplit (13041-token
  // packed batches hit this).  A slice keeps four 32-k stages, two where four would leave most of the
  // chip idle (us at two and four, fp32: 256 x 256 over 1100 11.4, 13.4, 512 x 256 12.6, 13.9, 64 x 64
  // over 2048 8.8, 10.8, but 384 x 256 16.9, 14.1).  At most 64 slices in three parts, 32 in one, whose
  // slices are shorter against the second pass (256 x 256 over 16384, at 32 and 64: fp32 32.0, 27.4,
  // bf16 23.4, 24.6).
  const int stages = tiles <= 8 || k < 2048 ? 2 : 4;
  int slices = 1;
  if (tiles <= 256 && k >= 2 * stages * GT_K) {
    slices = int(std::min<int64_t>(512 / tiles, k / (stages * GT_K)));
    slices = std::max(1, std::min(slices, bf16 ? 32 : 64));
  }
  const int kc = std::max((k + slices - 1) / slices + GT_K - 1, GT_K) / GT_K * GT_K;  // (k 0: one empty slice)
  slices = std::max((k + kc - 1) / kc, 1);
  return {tm, slices, kc};
}

// ---- LayerNorm / RMSNorm -----------------------------------------------------------------
// One wave per row.
__global__ void layernorm_fwd_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                     const float *__restrict__ b, float eps, float *__restrict__ y,
                                     float *__restrict__ mean, float *__restrict__ rstd, int32_t n, int32_t d) {
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= n) return;
  const float *xr = x + int64_t(row) * d;
  float s = 0.f;
  for (int k = lane; k < d; k += 64) s += xr[k];
  const float mu = wave_sum(s) / float(d);
  float v = 0.f;
  for (int k = lane; k < d; k += 64) {
    const float c = xr[k] - mu;
    v = fmaf(c, c, v);
  }
  const float r = 1.0f / sqrtf(wave_sum(v) / float(d) + eps);
  float *yr = y + int64_t(row) * d;
  for (int k = lane; k < d; k += 64) yr[k] = (xr[k] - mu) * r * w[k] + b[k];
  if (lane == 0) {
    mean[row] = mu;
    rstd[row] = r;
  }
}

// The same for d <= 256 NV, d a multiple of 4, 16-byte aligned rows: lane l owns the float4
// columns 4 l + 256 v of a row (two-pass mean and variance from registers), wave w takes rows
// r0 + w, r0 + w + 4, ... of its block's 16, loading the next row while it reduces this one.
template <int NV>
__global__ __launch_bounds__(256) void layernorm_rows_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                             const float *__restrict__ b, float eps,
                                                             float *__restrict__ y, float *__restrict__ mean,
                                                             float *__restrict__ rstd, int32_t n, int32_t d) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r0 = blockIdx.x * 16, r1 = min(n, r0 + 16);
  const float4 zero = {0.f, 0.f, 0.f, 0.f};
  float4 wv[NV], bv[NV], xa[NV];
  bool in[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int c = 4 * lane + 256 * v;
    in[v] = c < d;
    wv[v] = in[v] ? *reinterpret_cast<const float4 *>(w + c) : zero;
    bv[v] = in[v] ? *reinterpret_cast<const float4 *>(b + c) : zero;
  }
  auto load = [&](int row, float4 (&xs)[NV]) {
#pragma unroll
    for (int v = 0; v < NV; ++v)
      xs[v] = in[v] ? *reinterpret_cast<const float4 *>(x + int64_t(row) * d + 4 * lane + 256 * v) : zero;
  };
  int row = r0 + wave;
  if (row < r1) load(row, xa);
  for (; row < r1; row += 4) {
    float4 xc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) xc[v] = xa[v];
    if (row + 4 < r1) load(row + 4, xa);
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) s += (xc[v].x + xc[v].y) + (xc[v].z + xc[v].w);
    const float mu = wave_sum(s) / float(d);
    float q = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (!in[v]) continue;
      const float a0 = xc[v].x - mu, a1 = xc[v].y - mu, a2 = xc[v].z - mu, a3 = xc[v].w - mu;
      q += (a0 * a0 + a1 * a1) + (a2 * a2 + a3 * a3);
    }
    const float r = 1.0f / sqrtf(wave_sum(q) / float(d) + eps);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (!in[v]) continue;
      *reinterpret_cast<float4 *>(y + int64_t(row) * d + 4 * lane + 256 * v) =
          float4{(xc[v].x - mu) * r * wv[v].x + bv[v].x, (xc[v].y - mu) * r * wv[v].y + bv[v].y,
                 (xc[v].z - mu) * r * wv[v].z + bv[v].z, (xc[v].w - mu) * r * wv[v].w + bv[v].w};
    }
    if (lane == 0) {
      mean[row] = mu;
      rstd[row] = r;
    }
  }
}

// dx = rstd (g - mean(g) - xhat mean(g xhat)) (+ residual), g = dy * w; per block of
// `rows_per_block` rows, partial dw = sum dy xhat and db = sum dy into part[blockIdx][0 / 1][d].
// A NULL mean selects RMSNorm (no centring, no bias).  Any d (norm_bwd_rows_kernel takes the
// common shapes).
__global__ void norm_bwd_kernel(const float *__restrict__ x, const float *__restrict__ dy,
                                const float *__restrict__ w, const float *__restrict__ mean,
                                const float *__restrict__ rstd, const float *__restrict__ residual,
                                float *__restrict__ dx, float *__restrict__ part, int32_t n, int32_t d,
                                int32_t rows_per_block) {
  extern __shared__ float acc_lds[];  // [2][d]
  const int waves = blockDim.x >> 6, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int k = threadIdx.x; k < 2 * d; k += blockDim.x) acc_lds[k] = 0.f;
  __syncthreads();
  const int r0 = blockIdx.x * rows_per_block;
  for (int row = r0 + wave; row < min(n, r0 + rows_per_block); row += waves) {
    const float *xr = x + int64_t(row) * d, *gr = dy + int64_t(row) * d;
    const float mu = mean ? mean[row] : 0.f, r = rstd[row];
    float sg = 0.f, sgx = 0.f;
    for (int k = lane; k < d; k += 64) {
      const float xh = (xr[k] - mu) * r, g = gr[k] * w[k];
      sg += g;
      sgx = fmaf(g, xh, sgx);
    }
    const float mg = mean ? wave_sum(sg) / float(d) : 0.f, mgx = wave_sum(sgx) / float(d);
    float *dxr = dx + int64_t(row) * d;
    for (int k = lane; k < d; k += 64) {
      const float xh = (xr[k] - mu) * r;
      dxr[k] = r * (gr[k] * w[k] - mg - xh * mgx) + (residual ? residual[int64_t(row) * d + k] : 0.f);
      atomicAdd(&acc_lds[k], gr[k] * xh);  // LDS atomics: order within a block only
      atomicAdd(&acc_lds[d + k], gr[k]);
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < 2 * d; k += blockDim.x) part[int64_t(blockIdx.x) * 2 * d + k] = acc_lds[k];
}

// The same for d <= 256 NV, d a multiple of 4, 16-byte aligned rows: lane l owns the float4
// columns 4 l + 256 v (v < NV) and keeps them, the gain and its dw / db partials in registers;
// wave w of a block takes rows r0 + w, r0 + w + 4, ... of its NORM_ROWS, loading the next row
// while it reduces the current one.
constexpr int NORM_ROWS = 16;

__device__ __forceinline__ float4 f4_fma(float4 a, float4 b, float4 c) {
  return float4{fmaf(a.x, b.x, c.x), fmaf(a.y, b.y, c.y), fmaf(a.z, b.z, c.z), fmaf(a.w, b.w, c.w)};
}

template <int NV>
__global__ __launch_bounds__(256) void norm_bwd_rows_kernel(const float *__restrict__ x, const float *__restrict__ dy,
                                                            const float *__restrict__ w, const float *__restrict__ mean,
                                                            const float *__restrict__ rstd,
                                                            const float *__restrict__ residual, float *__restrict__ dx,
                                                            float *__restrict__ part, int32_t n, int32_t d) {
  __shared__ float4 red[4][2 * 64 * NV];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r0 = blockIdx.x * NORM_ROWS, r1 = min(n, r0 + NORM_ROWS);
  const float4 zero = {0.f, 0.f, 0.f, 0.f};
  float4 wv[NV], pw[NV], pb[NV], xa[NV], ga[NV];
  bool in[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int c = 4 * lane + 256 * v;
    in[v] = c < d;
    wv[v] = in[v] ? *reinterpret_cast<const float4 *>(w + c) : zero;
    pw[v] = zero;
    pb[v] = zero;
  }
  auto load = [&](int row, float4 (&xs)[NV], float4 (&gs)[NV]) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int64_t i = int64_t(row) * d + 4 * lane + 256 * v;
      xs[v] = in[v] ? *reinterpret_cast<const float4 *>(x + i) : zero;
      gs[v] = in[v] ? *reinterpret_cast<const float4 *>(dy + i) : zero;
    }
  };
  int row = r0 + wave;
  float mu_n = 0.f, r_n = 0.f;
  if (row < r1) {
    load(row, xa, ga);
    mu_n = mean ? mean[row] : 0.f;
    r_n = rstd[row];
  }
  for (; row < r1; row += 4) {
    float4 xc[NV], gc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      xc[v] = xa[v];
      gc[v] = ga[v];
    }
    const float mu = mu_n, r = r_n;
    if (row + 4 < r1) {
      load(row + 4, xa, ga);
      mu_n = mean ? mean[row + 4] : 0.f;
      r_n = rstd[row + 4];
    }
    float4 xh[NV], g[NV];
    float sg = 0.f, sgx = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      xh[v] = float4{(xc[v].x - mu) * r, (xc[v].y - mu) * r, (xc[v].z - mu) * r, (xc[v].w - mu) * r};
      g[v] = float4{gc[v].x * wv[v].x, gc[v].y * wv[v].y, gc[v].z * wv[v].z, gc[v].w * wv[v].w};
      sg += (g[v].x + g[v].y) + (g[v].z + g[v].w);
      sgx += (g[v].x * xh[v].x + g[v].y * xh[v].y) + (g[v].z * xh[v].z + g[v].w * xh[v].w);
    }
    const float mg = mean ? wave_sum(sg) / float(d) : 0.f, mgx = wave_sum(sgx) / float(d);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (!in[v]) continue;
      const int64_t i = int64_t(row) * d + 4 * lane + 256 * v;
      float4 o = {r * (g[v].x - mg - xh[v].x * mgx), r * (g[v].y - mg - xh[v].y * mgx),
                  r * (g[v].z - mg - xh[v].z * mgx), r * (g[v].w - mg - xh[v].w * mgx)};
      if (residual) {
        const float4 a = *reinterpret_cast<const float4 *>(residual + i);
        o = float4{o.x + a.x, o.y + a.y, o.z + a.z, o.w + a.w};
      }
      *reinterpret_cast<float4 *>(dx + i) = o;
      pw[v] = f4_fma(gc[v], xh[v], pw[v]);
      pb[v] = float4{pb[v].x + gc[v].x, pb[v].y + gc[v].y, pb[v].z + gc[v].z, pb[v].w + gc[v].w};
    }
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    red[wave][v * 64 + lane] = pw[v];
    red[wave][(NV + v) * 64 + lane] = pb[v];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 2 * 64 * NV; i += 256) {
    const int which = i / (64 * NV), v = (i / 64) % NV, c = 4 * (i % 64) + 256 * v;
    if (c >= d) continue;
    const float4 a = red[0][i], b = red[1][i], e = red[2][i], f = red[3][i];
    *reinterpret_cast<float4 *>(part + int64_t(blockIdx.x) * 2 * d + which * d + c) =
        float4{(a.x + b.x) + (e.x + f.x), (a.y + b.y) + (e.y + f.y), (a.z + b.z) + (e.z + f.z),
               (a.w + b.w) + (e.w + f.w)};
  }
}

// dw[c] (+)= sum_p part[p][0][c] and db[c] (+)= sum_p part[p][1][c] (db NULL: RMSNorm): 64 of
// the 2 d columns per block, its 16 waves splitting the partial rows.
__global__ __launch_bounds__(1024) void norm_params_kernel(const float *__restrict__ part, int32_t parts, int32_t d,
                                                           float *__restrict__ dw, float *__restrict__ db,
                                                           int32_t accumulate) {
  __shared__ float red[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  if (c < 2 * d) {
    int p = wave;
    for (; p + 48 < parts; p += 64) {
      s0 += part[int64_t(p) * 2 * d + c];
      s1 += part[int64_t(p + 16) * 2 * d + c];
      s2 += part[int64_t(p + 32) * 2 * d + c];
      s3 += part[int64_t(p + 48) * 2 * d + c];
    }
    for (; p < parts; p += 16) s0 += part[int64_t(p) * 2 * d + c];
  }
  red[wave][lane] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (wave != 0 || c >= 2 * d) return;
  float s = 0.f;
#pragma unroll
  for (int q = 0; q < 16; ++q) s += red[q][lane];
  float *o = c < d ? dw + c : (db ? db + (c - d) : nullptr);
  if (o) *o = accumulate ? *o + s : s;
}

// out[c] = sum_r in[r * ld + c] (+ out[c] when accumulate): column sums of per-block
// partials and bias gradients.  A block takes 64 columns x `chunk` rows: its four waves
// split the rows, each lane one column (coalesced rows), and meet in LDS; blockIdx.y's
// chunk lands in out[y][c] (a second pass sums the chunks).
__global__ __launch_bounds__(256) void column_sum_kernel(const float *__restrict__ in, int32_t rows, int32_t cols,
                                                         int64_t ld, float *__restrict__ out, int32_t accumulate,
                                                         int32_t chunk) {
  __shared__ float red[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  const int r0 = blockIdx.y * chunk, r1 = min(rows, r0 + chunk);
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  if (c < cols) {
    int r = r0 + wave;
    auto at = [&](int rr) { return in[int64_t(rr) * ld + c]; };
    for (; r + 12 < r1; r += 16) {
      s0 += at(r);
      s1 += at(r + 4);
      s2 += at(r + 8);
      s3 += at(r + 12);
    }
    for (; r < r1; r += 4) s0 += at(r);
  }
  red[wave][lane] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (wave == 0 && c < cols) {
    float s = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
    float *o = out + int64_t(blockIdx.y) * cols + c;
    *o = accumulate ? *o + s : s;
  }
}

// ---- GELU -------------------------------------------------------------------------------

__global__ void gelu_fwd_kernel(const float *__restrict__ u, float *__restrict__ g, int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
    g[i] = gelu_exact(u[i]);
}

// du = dg * (Phi(u) + u phi(u)).
__global__ void gelu_bwd_kernel(const float *__restrict__ u, const float *__restrict__ dg, float *__restrict__ du,
                                int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    du[i] = dg[i] * gelu_grad(u[i]);
  }
}

// ---- attention ------------------------------------------------------------------------------
// Packed rows: token t belongs to sequence s with seq_start[s] <= t < seq_start[s + 1];
// seq_of[t] = s.  q [N, H, D], k / v [N, KVH, D] (row strides ldq / ldk / ldv floats; the
// gradients dq / dk / dv use the same strides, so they land in a [q | k | v] row buffer
// like their inputs), o and do [N, H, D] dense, lse / dsum [N, H].  Query t of a sequence
// sees its keys start .. t.
struct AttnTrain {
  int32_t n, H, KVH;
  float scale;
  const int64_t *seq_start;
  const int32_t *seq_of;
  const float *q, *k, *v;
  int64_t ldq, ldk, ldv;
  const float *o, *dout, *lse;
  float *out, *lse_out, *dsum, *dq, *dk, *dv;
  int32_t round;  // bf16 outputs (o, dq, dk, dv), as SDPA on bf16 operands returns them
  int32_t vec;    // output rows start 16-byte aligned
  // dK / dV of `splits` parts of each head group, [split][n][dk | dv of every KV head], summed (and
  // rounded) by merge_dkv_kernel; NULL: one part, written to dk / dv.
  float *parts;
  int32_t splits;
};

__device__ __forceinline__ float attn_out(const AttnTrain &a, float v) { return a.round ? round_bf16(v) : v; }

// The three kernels work on 16 x 16 tiles of (query, key) pairs with v_mfma_f32_16x16x32_bf16.
// PARTS 3: fp32 operands in three bf16 parts (split.h); PARTS 1: operands that hold bf16 numbers
// (the bf16 trunk's q, k, v and dO), so one part is exact.  Probabilities and dS are fp32 and
// always multiplied in three parts.  A contraction over head_dim (padded to 32) takes both
// operands with lane (li, lg) holding d = 8 lg .. 8 lg + 7.  A score tile leaves its MFMA with
// lane (li, lg) holding rows 4 lg + r, column li; a contraction over those rows (keys or queries)
// takes 32 of them, two score tiles, with lane group lg's k the rows {4 lg + r} of the one and
// {16 + 4 lg + r} of the other, so scores never leave the lane.  Staged tiles are therefore kept
// in up to two LDS layouts: by rows (a lane's eight d of a row) and by columns (a lane's eight
// rows of a d).  Outputs over d come out transposed ([d][row]): each lane stores four consecutive
// d.  What bounds them is the VALU work per score (exp, masks, splitting), so masks are only
// evaluated in tiles that some query sees partly.
constexpr int KT = 64;  // rows (keys, or queries of a dK / dV unit) per staged tile

template <int D, int PARTS>
struct AttnDims {
  static constexpr int DK = (D + 31) / 32;  // 32-wide d slices of a contraction over d
  static constexpr int DT = (D + 15) / 16;  // 16-wide d tiles of an output
  static constexpr int C4 = D / 4;
  static constexpr int SLOTS = 32 * C4;                 // a slot: two rows x four d
  static constexpr int PER = (SLOTS + 255) / 256;       // slots per thread
  static constexpr int ROW_PART = 4096 * DK, COL_PART = 2048 * DT;  // bytes of one part of a tile
  static constexpr int ROWS = PARTS * ROW_PART, COLS = PARTS * COL_PART;
};

// The parts of one MFMA operand.
template <int PARTS>
struct Operand {
  split_u32x4 p[PARTS];
};
template <int D, int PARTS>
using DimOperand = Operand<PARTS>[AttnDims<D, PARTS>::DK];
// A thread's slots of a staged tile: two rows' four d each.
template <int D, int PARTS>
using SlotRegs = float4[AttnDims<D, PARTS>::PER][2];

template <int PARTS>
__device__ __forceinline__ Operand<PARTS> operand_of(const float (&v)[8]) {
  Operand<PARTS> o;
  const f32x4 x = {v[0], v[1], v[2], v[3]}, y = {v[4], v[5], v[6], v[7]};
  if constexpr (PARTS == 3) {
    const Split8 s = split8(x, y);
    o.p[0] = s.hi, o.p[1] = s.mid, o.p[2] = s.lo;
  } else {
    o.p[0] = split_u32x4{split_pack(x[0], x[1]), split_pack(x[2], x[3]), split_pack(y[0], y[1]), split_pack(y[2], y[3])};
  }
  return o;
}

// c + a b, smallest products first; of one order the last part of `b` first, or with `A_FIRST` of `a`:
// mma_parts(a, b) and mma_parts<.., true>(b, a) add the same terms in the same order.
template <int PA, int PB, bool A_FIRST = false>
__device__ __forceinline__ f32x4 mma_parts(const Operand<PA> &a, const Operand<PB> &b, f32x4 c) {
#pragma unroll
  for (int order = 2; order >= 0; --order)
#pragma unroll
    for (int i = 0; i <= order; ++i) {
      const int ia = A_FIRST ? order - i : i, ib = order - ia;
      if (ia < PA && ib < PB) c = split_mma1(a.p[ia], b.p[ib], c);
    }
  return c;
}

// A sum over rows: the leading products, and (fp32 operands) the corrections apart from them.  Small
// terms added to a large sum lose their low bits downwards in the matrix unit, every term the same way:
// with one sum the gradients' column sums were three times as far off (64 x 256 tokens: dq 9.5e-7
// relative, 2.7e-7 so; dk and dv themselves 6.1e-7, 3.4e-7).  bf16 results hide it (sum in one).
template <int PARTS>
struct RowSum {
  f32x4 part[PARTS == 3 ? 2 : 1];
  __device__ __forceinline__ void scale(float x) {
#pragma unroll
    for (f32x4 &v : part) v *= x;
  }
  __device__ __forceinline__ f32x4 total() const { return PARTS == 3 ? part[0] + part[PARTS == 3] : part[0]; }
};

template <int PARTS>
__device__ __forceinline__ void mma_add(const Operand<PARTS> &a, const Operand<3> &b, RowSum<PARTS> &sum) {
#pragma unroll
  for (int order = 2; order >= 0; --order)
#pragma unroll
    for (int i = 0; i <= order; ++i)
      if (i < PARTS) {
        f32x4 &to = sum.part[PARTS == 3 && order != 0];
        to = split_mma1(a.p[i], b.p[order - i], to);
      }
}

// A score tile in natural units: three parts hold scaled queries already; bf16 queries are scaled
// here, rounded before anything is subtracted.  The backward forms a score with the forward's own
// operations, so that P = exp(score - lse) carries the rounding of lse alone: a score of any size that
// the forward took as its maximum comes back as exp(0).
template <int PARTS>
__device__ __forceinline__ f32x4 natural_score(f32x4 c, float scale) {
#pragma clang fp contract(off)
  if constexpr (PARTS == 1) c = c * scale;
  return c;
}
__device__ __forceinline__ float4 scaled_query(const float4 &q, float scale) {
#pragma clang fp contract(off)
  return float4{q.x * scale, q.y * scale, q.z * scale, q.w * scale};
}

constexpr float LOG2E = 1.4426950408889634f;

// e^x (v_exp_f32 is 2^x).
__device__ __forceinline__ float exp_natural(float x) { return __builtin_amdgcn_exp2f(x * LOG2E); }

__device__ __forceinline__ float max_over_rows(float x) {  // over lanes li, li + 16, li + 32, li + 48
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}

__device__ __forceinline__ float sum_over_rows(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}

// Clears LDS once: the d >= D padding of a staged tile is read (times zero or into output rows
// that are never stored) and never written.
__device__ __forceinline__ void clear_lds(char *lds, int bytes) {
  for (int i = threadIdx.x * 16; i < bytes; i += 256 * 16) *reinterpret_cast<split_u32x4 *>(lds + i) = split_u32x4{0, 0, 0, 0};
}

// Rows [r0, r0 + 64) of p (row stride ld floats, D used columns) into registers; rows past `last` are
// read as the last (their scores are masked).  The row base is uniform, the rest 32 bits where the
// stride allows.
template <int D, int PARTS>
__device__ __forceinline__ void rows_load(SlotRegs<D, PARTS> &r, const float *__restrict__ p, int64_t ld, int64_t r0,
                                          int64_t last) {
  using S = AttnDims<D, PARTS>;
  const char *base = reinterpret_cast<const char *>(p + r0 * ld);
  const bool near = ld >= 0 && ld <= TILE_MAX_STRIDE;
  const int left = int(min<int64_t>(last - r0, KT - 1));
#pragma unroll
  for (int e = 0; e < S::PER; ++e) {
    const int slot = min(int(threadIdx.x) + 256 * e, S::SLOTS - 1), row = 2 * (slot / S::C4), c = (slot % S::C4) * 4;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = min(row + h, left);
      if (near)
        r[e][h] = *reinterpret_cast<const float4 *>(base + 4u * (unsigned(at) * unsigned(ld) + unsigned(c)));
      else
        r[e][h] = *reinterpret_cast<const float4 *>(base + 4 * (at * ld + c));
    }
  }
}

// The parts of a slot: per row (h), per part, its four d packed.
template <int PARTS>
__device__ __forceinline__ void slot_parts(const float4 (&v)[2], unsigned (&out)[2][PARTS][2]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if constexpr (PARTS == 3) {
      split_pair(v[h].x, v[h].y, out[h][0][0], out[h][1][0], out[h][2][0]);
      split_pair(v[h].z, v[h].w, out[h][0][1], out[h][1][1], out[h][2][1]);
    } else {
      out[h][0][0] = split_pack(v[h].x, v[h].y);
      out[h][0][1] = split_pack(v[h].z, v[h].w);
    }
  }
}

// Registers -> LDS: by rows (tile_offset per 32-d slice) and / or by columns: row kappa of a
// 32-row half u is value (kappa & 3) + 4 (kappa >> 4) of lane group (kappa >> 2) & 3, [u][16-d
// tile][lane group][d, exclusive-or'ed with the lane group][8 rows].
template <int D, int PARTS, bool BY_ROWS, bool BY_COLS>
__device__ __forceinline__ void rows_store(char *rows, char *cols, const SlotRegs<D, PARTS> &r) {
  using S = AttnDims<D, PARTS>;
#pragma unroll
  for (int e = 0; e < S::PER; ++e) {
    const int slot = threadIdx.x + 256 * e;
    if (slot >= S::SLOTS) continue;
    const int c = (slot % S::C4) * 4, row = 2 * (slot / S::C4);
    unsigned v[2][PARTS][2];
    slot_parts<PARTS>(r[e], v);
    if constexpr (BY_ROWS) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        char *to = rows + (c >> 5) * 4096 + tile_offset(row + h, (c >> 3) & 3) + (c & 4) * 2;
#pragma unroll
        for (int q = 0; q < PARTS; ++q) *reinterpret_cast<u32x2 *>(to + q * S::ROW_PART) = u32x2{v[h][q][0], v[h][q][1]};
      }
    }
    if constexpr (BY_COLS) {
      const int u = row >> 5, kappa = row & 31, lg = (kappa >> 2) & 3, at = (kappa & 3) + 4 * (kappa >> 4);
      char *to = cols + u * 1024 * S::DT + (c >> 4) * 1024 + lg * 256 + at * 2;
#pragma unroll
      for (int q = 0; q < PARTS; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned a = v[0][q][i >> 1], b = v[1][q][i >> 1];
          const unsigned w = i & 1 ? (a >> 16) | (b & 0xffff0000u) : (a & 0xffffu) | (b << 16);
          *reinterpret_cast<unsigned *>(to + q * S::COL_PART + ((((c + i) & 15) ^ lg) << 4)) = w;
        }
    }
  }
}

// A operand fragments: 16 rows `sub` of slice dk by rows; 16 d `dt` over the 32 rows `u` by columns.
template <int D, int PARTS>
__device__ __forceinline__ Operand<PARTS> row_frag(const char *rows, int sub, int dk, int li, int lg) {
  Operand<PARTS> o;
#pragma unroll
  for (int q = 0; q < PARTS; ++q)
    o.p[q] = *reinterpret_cast<const split_u32x4 *>(rows + q * AttnDims<D, PARTS>::ROW_PART + dk * 4096 +
                                                    tile_offset(16 * sub + li, lg));
  return o;
}
template <int D, int PARTS>
__device__ __forceinline__ Operand<PARTS> col_frag(const char *cols, int u, int dt, int li, int lg) {
  using S = AttnDims<D, PARTS>;
  Operand<PARTS> o;
#pragma unroll
  for (int q = 0; q < PARTS; ++q)
    o.p[q] = *reinterpret_cast<const split_u32x4 *>(cols + q * S::COL_PART + (u * S::DT + dt) * 1024 + lg * 256 +
                                                    ((li ^ lg) << 4));
  return o;
}

// A lane's eight d of one row (d = 32 dk + 8 lg ..) as a B operand; zero when !live or past D.
template <int D, int PARTS>
__device__ __forceinline__ void row_operand(DimOperand<D, PARTS> &o, const float *__restrict__ p, bool live, int lg,
                                            float scale = 1.0f) {
#pragma unroll
  for (int dk = 0; dk < AttnDims<D, PARTS>::DK; ++dk) {
    float v[8];
    const int d = 32 * dk + 8 * lg;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float4 x = scaled_query(
          live && d < D ? *reinterpret_cast<const float4 *>(p + d + 4 * h) : float4{0.f, 0.f, 0.f, 0.f}, scale);
      v[4 * h] = x.x, v[4 * h + 1] = x.y, v[4 * h + 2] = x.z, v[4 * h + 3] = x.w;
    }
    o[dk] = operand_of<PARTS>(v);
  }
}

// Two score tiles' values as the B operand of a contraction over their 32 rows.
__device__ __forceinline__ Operand<3> score_operand(const f32x4 &a, const f32x4 &b) {
  const float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  return operand_of<3>(v);
}

// Four consecutive d of an output row.
__device__ __forceinline__ void store4(const AttnTrain &a, float *p, const f32x4 &v, float scale) {
  const float4 o = {attn_out(a, v[0] * scale), attn_out(a, v[1] * scale), attn_out(a, v[2] * scale),
                    attn_out(a, v[3] * scale)};
  if (a.vec) {
    *reinterpret_cast<float4 *>(p) = o;
  } else {
    p[0] = o.x;
    p[1] = o.y;
    p[2] = o.z;
    p[3] = o.w;
  }
}

// Block of the forward and dQ kernels: 256 threads; wave w takes a strip of 16 tokens
// (strip w / gpb) of head g = gpb blockIdx.z + w % gpb of KV head blockIdx.y, gpb =
// min(G, 4) heads and 4 / gpb strips per block, so all waves share every staged K / V tile.
struct QueryStrip {
  int h;
  bool active;     // the wave has a head and tokens
  int64_t t0;      // first token of the wave's strip
  int64_t base;    // first token of the block
  int64_t b_last;  // last token of the block
};

__device__ __forceinline__ QueryStrip query_strip(const AttnTrain &a, int tid) {
  const int G = a.H / a.KVH, gpb = min(G, 4), tpb = 4 / gpb, wave = tid >> 6;
  const int strip = wave / gpb, g = blockIdx.z * gpb + wave % gpb;
  QueryStrip q;
  q.base = int64_t(blockIdx.x) * 16 * tpb;
  q.b_last = min<int64_t>(a.n - 1, q.base + 16 * tpb - 1);
  q.t0 = q.base + 16 * strip;
  q.active = strip < tpb && g < G && q.t0 < a.n;
  q.h = blockIdx.y * G + min(g, G - 1);
  return q;
}

// Plain fp32 forms of the three kernels' results, one lane's query (or key) and d = 16 dt + 4 lg + r at
// a time, over the rows that it sees alone.  A part of an infinity or of a value past bf16's largest
// number is not finite, and a hidden row's zero weight times it is NaN, so results that are not finite
// are formed again here (split.h); finite ones never come here.  The callers find their lane's place
// again from `fresh_thread`, so that the main loops keep nothing alive for this.
__device__ __forceinline__ int fresh_thread() {
  int tid = threadIdx.x;
  asm("" : "+v"(tid));
  return tid;
}

template <int D>
__device__ __forceinline__ float plain_dot(const float *__restrict__ x, const float *__restrict__ y) {
  float s = 0.f;
#pragma unroll 1  // (few registers: the kernels' occupancy is the main loops')
  for (int d = 0; d < D; d += 4) {
    const float4 a = *reinterpret_cast<const float4 *>(x + d), b = *reinterpret_cast<const float4 *>(y + d);
    s = fmaf(a.x, b.x, fmaf(a.y, b.y, fmaf(a.z, b.z, fmaf(a.w, b.w, s))));
  }
  return s;
}

template <int DT>
__device__ __forceinline__ bool all_finite(const f32x4 (&v)[DT]) {
  bool ok = true;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) ok = ok && split_finite(v[dt][r]);
  return ok;
}

// acc += w x[d] over the lane's d.
template <int D, int DT>
__device__ __forceinline__ void plain_add(f32x4 (&acc)[DT], float w, const float *__restrict__ x, int lg) {
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    if (dt * 16 + 4 * lg >= D) continue;
    const float4 v = *reinterpret_cast<const float4 *>(x + dt * 16 + 4 * lg);
    acc[dt] = f32x4{fmaf(w, v.x, acc[dt][0]), fmaf(w, v.y, acc[dt][1]), fmaf(w, v.z, acc[dt][2]), fmaf(w, v.w, acc[dt][3])};
  }
}

template <int DT>
__device__ __forceinline__ void clear(f32x4 (&v)[DT]) {
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) v[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
}

template <int D>
__device__ __forceinline__ float plain_score(const AttnTrain &a, int64_t t, int64_t j, int h, int hk) {
#pragma clang fp contract(off)
  return plain_dot<D>(a.q + t * a.ldq + h * D, a.k + j * a.ldk + hk * D) * a.scale;
}

// Softmax over keys start .. t: the maximum m, the sum l and the sums of V.
template <int D, int DT>
__device__ __forceinline__ void plain_forward(const AttnTrain &a, int64_t t, int64_t start, int h, int hk, int lg,
                                              float &m, float &l, f32x4 (&acc)[DT]) {
  m = -1e30f;
#pragma unroll 1
  for (int64_t j = start; j <= t; ++j) m = fmaxf(m, plain_score<D>(a, t, j, h, hk));
  l = 0.f;
  clear(acc);
#pragma unroll 1
  for (int64_t j = start; j <= t; ++j) {
    const float p = exp_natural(plain_score<D>(a, t, j, h, hk) - m);
    l += p;
    plain_add<D>(acc, p, a.v + j * a.ldv + hk * D, lg);
  }
}

// P and dS of one (query, key) pair.
template <int D>
__device__ __forceinline__ void plain_pair(const AttnTrain &a, int64_t t, int64_t j, int h, int hk, float dsum, float &p,
                                           float &ds) {
  const int64_t row = t * a.H + h;
  p = exp_natural(plain_score<D>(a, t, j, h, hk) - a.lse[row]);
  ds = p * (plain_dot<D>(a.dout + row * D, a.v + j * a.ldv + hk * D) - dsum);
}

// Forward: online softmax over K / V tiles staged KT keys at a time.  S^T = K Q^T (keys on
// the rows, the lane's query li on the column), row statistics per query across the four
// lanes li + 16 lg, O^T += V^T P^T.
template <int D, int PARTS>
__global__ __launch_bounds__(256, D <= 32 ? (PARTS == 1 ? 5 : 4) : 3) void attn_fwd_kernel(const AttnTrain a) {
  using S = AttnDims<D, PARTS>;
  __shared__ __align__(16) char lds[S::ROWS + S::COLS];
  char *const kr = lds, *const vc = lds + S::ROWS;
  const int hk = blockIdx.y, lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const QueryStrip w = query_strip(a, threadIdx.x);
  const int64_t t = w.t0 + li, w_last = min<int64_t>(a.n - 1, w.t0 + 15);
  const bool live = w.active && t < a.n;
  const int64_t start = live ? a.seq_start[a.seq_of[t]] : 0;
  const int64_t w_first = w.active ? a.seq_start[a.seq_of[w.t0]] : 0;  // first key any query of the strip sees
  const int64_t k_lo = a.seq_start[a.seq_of[w.base]];
  clear_lds(lds, S::ROWS + S::COLS);
  Operand<PARTS> qf[S::DK];  // (scaling bf16 queries would take more than one part)
  row_operand<D, PARTS>(qf, a.q + t * a.ldq + w.h * D, live, lg, PARTS == 3 ? a.scale : 1.0f);
  RowSum<PARTS> sum[S::DT] = {};
  float m = -1e30f, l = 0.f;
  float4 kp[S::PER][2], vp[S::PER][2];
  rows_load<D, PARTS>(kp, a.k + hk * D, a.ldk, k_lo, w.b_last);
  rows_load<D, PARTS>(vp, a.v + hk * D, a.ldv, k_lo, w.b_last);
  for (int64_t j0 = k_lo; j0 <= w.b_last; j0 += KT) {
    __syncthreads();  // the tile before (and the clearing) is done with
    rows_store<D, PARTS, true, false>(kr, nullptr, kp);
    rows_store<D, PARTS, false, true>(nullptr, vc, vp);
    __syncthreads();
    if (j0 + KT <= w.b_last) {  // the next tile's loads fly during this one's products
      rows_load<D, PARTS>(kp, a.k + hk * D, a.ldk, j0 + KT, w.b_last);
      rows_load<D, PARTS>(vp, a.v + hk * D, a.ldv, j0 + KT, w.b_last);
    }
    if (!(w.active && j0 <= w_last && j0 + KT - 1 >= w_first)) continue;
    // The lane's query sees the tile's keys lo .. hi.
    const int lo = live ? int(max<int64_t>(start - j0, 0)) : KT, hi = live ? int(min<int64_t>(t - j0, KT - 1)) : -1;
    const unsigned seen = unsigned(max(hi - lo + 1, 0));
    const bool whole = __all(seen == KT);
    f32x4 s[4];
    bool any[4];
    float mt = -INFINITY;
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) {
      const int64_t jb = j0 + 16 * sub;
      any[sub] = jb <= w_last && jb + 15 >= w_first;
      s[sub] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (!any[sub]) continue;
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dk = 0; dk < S::DK; ++dk) c = mma_parts<PARTS, PARTS>(row_frag<D, PARTS>(kr, sub, dk, li, lg), qf[dk], c);
      s[sub] = natural_score<PARTS>(c, a.scale);
      if (!whole) {
#pragma unroll
        for (int r = 0; r < 4; ++r) s[sub][r] = unsigned(4 * lg - lo + 16 * sub + r) < seen ? s[sub][r] : -INFINITY;
      }
      mt = fmaxf(fmaxf(mt, fmaxf(s[sub][0], s[sub][1])), fmaxf(s[sub][2], s[sub][3]));
    }
    mt = max_over_rows(mt);
    const float mn = fmaxf(m, mt);
    const float corr = exp_natural(m - mn);
    m = mn;
    l *= corr;
#pragma unroll
    for (int dt = 0; dt < S::DT; ++dt) sum[dt].scale(corr);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (!any[2 * u] && !any[2 * u + 1]) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[2 * u + h][r] = exp_natural(s[2 * u + h][r] - mn);
          l += s[2 * u + h][r];
        }
      const Operand<3> p = score_operand(s[2 * u], s[2 * u + 1]);
#pragma unroll
      for (int dt = 0; dt < S::DT; ++dt) mma_add<PARTS>(col_frag<D, PARTS>(vc, u, dt, li, lg), p, sum[dt]);
    }
  }
  l = sum_over_rows(l);
  if (!live) return;
  f32x4 acc[S::DT];
#pragma unroll
  for (int dt = 0; dt < S::DT; ++dt) acc[dt] = sum[dt].total();
  if (!(split_finite(l) && all_finite(acc))) {
    const int tid = fresh_thread();
    const QueryStrip z = query_strip(a, tid);
    const int64_t tz = z.t0 + (tid & 15);
    plain_forward<D>(a, tz, a.seq_start[a.seq_of[tz]], z.h, blockIdx.y, (tid & 63) >> 4, m, l, acc);
  }
  float *orow = a.out + (t * a.H + w.h) * D;
#pragma unroll
  for (int dt = 0; dt < S::DT; ++dt)
    if (dt * 16 + 4 * lg < D) store4(a, orow + dt * 16 + 4 * lg, acc[dt], 1.0f / l);
  if (lg == 0) a.lse_out[t * a.H + w.h] = m + logf(l);
}

// dQ (and D = rowsum(dO * O)) with the forward's blocks: S^T = K Q^T and dP^T = V dO^T per
// 16-key tile, P from the saved log-sum-exp, dS = P (dP - D), dQ^T += K^T dS^T.
template <int D, int PARTS>
__global__ __launch_bounds__(256, D <= 32 ? (PARTS == 1 ? 5 : 4) : 2) void attn_bwd_dq_kernel(const AttnTrain a) {
  using S = AttnDims<D, PARTS>;
  __shared__ __align__(16) char lds[2 * S::ROWS + S::COLS];
  char *const kr = lds, *const vr = lds + S::ROWS, *const kc = lds + 2 * S::ROWS;
  const int hk = blockIdx.y, lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const QueryStrip w = query_strip(a, threadIdx.x);
  const int64_t t = w.t0 + li, w_last = min<int64_t>(a.n - 1, w.t0 + 15);
  const bool live = w.active && t < a.n;
  const int64_t row = t * a.H + w.h;
  const int64_t start = live ? a.seq_start[a.seq_of[t]] : 0;
  const int64_t w_first = w.active ? a.seq_start[a.seq_of[w.t0]] : 0;
  const int64_t k_lo = a.seq_start[a.seq_of[w.base]];
  clear_lds(lds, 2 * S::ROWS + S::COLS);
  Operand<PARTS> qf[S::DK], gf[S::DK];
  row_operand<D, PARTS>(qf, a.q + t * a.ldq + w.h * D, live, lg, PARTS == 3 ? a.scale : 1.0f);
  row_operand<D, PARTS>(gf, a.dout + row * D, live, lg);
  float part = 0.f;
#pragma unroll
  for (int dk = 0; dk < S::DK; ++dk)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int d = 32 * dk + 8 * lg + 4 * h;
      if (!live || d >= D) continue;
      const float4 g = *reinterpret_cast<const float4 *>(a.dout + row * D + d);
      const float *o = a.o + row * D + d;
      part = fmaf(g.x, o[0], fmaf(g.y, o[1], fmaf(g.z, o[2], fmaf(g.w, o[3], part))));
    }
  const float dsum = sum_over_rows(part);
  const float lse = live ? a.lse[row] : 0.f;
  RowSum<PARTS> sum[S::DT] = {};
  float4 kp[S::PER][2], vp[S::PER][2];
  rows_load<D, PARTS>(kp, a.k + hk * D, a.ldk, k_lo, w.b_last);
  rows_load<D, PARTS>(vp, a.v + hk * D, a.ldv, k_lo, w.b_last);
  for (int64_t j0 = k_lo; j0 <= w.b_last; j0 += KT) {
    __syncthreads();
    rows_store<D, PARTS, true, true>(kr, kc, kp);
    rows_store<D, PARTS, true, false>(vr, nullptr, vp);
    __syncthreads();
    if (j0 + KT <= w.b_last) {
      rows_load<D, PARTS>(kp, a.k + hk * D, a.ldk, j0 + KT, w.b_last);
      rows_load<D, PARTS>(vp, a.v + hk * D, a.ldv, j0 + KT, w.b_last);
    }
    if (!(w.active && j0 <= w_last && j0 + KT - 1 >= w_first)) continue;
    const int lo = live ? int(max<int64_t>(start - j0, 0)) : KT, hi = live ? int(min<int64_t>(t - j0, KT - 1)) : -1;
    const unsigned seen = unsigned(max(hi - lo + 1, 0));
    const bool whole = __all(seen == KT);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t jb = j0 + 32 * u;
      if (!(jb <= w_last && jb + 31 >= w_first)) continue;
      f32x4 ds[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int sub = 2 * u + h;
        f32x4 st = {0.f, 0.f, 0.f, 0.f}, dp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dk = 0; dk < S::DK; ++dk) {
          st = mma_parts<PARTS, PARTS>(row_frag<D, PARTS>(kr, sub, dk, li, lg), qf[dk], st);
          dp = mma_parts<PARTS, PARTS>(row_frag<D, PARTS>(vr, sub, dk, li, lg), gf[dk], dp);
        }
        st = natural_score<PARTS>(st, a.scale);
        f32x4 p;
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = exp_natural(st[r] - lse);
        if (!whole) {
#pragma unroll
          for (int r = 0; r < 4; ++r) p[r] = unsigned(4 * lg - lo + 16 * sub + r) < seen ? p[r] : 0.f;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) ds[h][r] = p[r] * (dp[r] - dsum);
      }
      const Operand<3> dso = score_operand(ds[0], ds[1]);
#pragma unroll
      for (int dt = 0; dt < S::DT; ++dt) mma_add<PARTS>(col_frag<D, PARTS>(kc, u, dt, li, lg), dso, sum[dt]);
    }
  }
  if (!live) return;
  f32x4 acc[S::DT];
#pragma unroll
  for (int dt = 0; dt < S::DT; ++dt) acc[dt] = sum[dt].total();
  if (!all_finite(acc)) {
    const int tid = fresh_thread();
    const QueryStrip z = query_strip(a, tid);
    const int64_t tz = z.t0 + (tid & 15);
    clear(acc);
#pragma unroll 1
    for (int64_t j = a.seq_start[a.seq_of[tz]]; j <= tz; ++j) {
      float p, ds;
      plain_pair<D>(a, tz, j, z.h, blockIdx.y, dsum, p, ds);
      plain_add<D>(acc, ds, a.k + j * a.ldk + blockIdx.y * D, (tid & 63) >> 4);
    }
  }
  float *dqrow = a.dq + t * a.ldq + w.h * D;
#pragma unroll
  for (int dt = 0; dt < S::DT; ++dt)
    if (dt * 16 + 4 * lg < D) store4(a, dqrow + dt * 16 + 4 * lg, acc[dt], a.scale);
  if (lg == 0) a.dsum[row] = dsum;
}

// dK / dV: a block holds 64 keys of KV head blockIdx.y, wave w keys j0 + 16 w + li in
// registers, and walks the units (KT tokens of one head of the group) that can see them,
// staged through LDS.  S = Q K^T and dP = dO V^T (queries on the rows), P and dS per lane,
// dV^T += dO^T P and dK^T += Q^T dS.  A block's walk is its critical path (the first keys of a
// 256-token sequence see 16 units of four heads), so the heads of a group may be split over
// blockIdx.z.
template <int D, int PARTS>
__global__ __launch_bounds__(256) void attn_bwd_dkv_kernel(const AttnTrain a) {
  using S = AttnDims<D, PARTS>;
  __shared__ __align__(16) char lds[2 * S::ROWS + 2 * S::COLS];
  __shared__ __align__(16) float ls[2 * KT];
  char *const qr = lds, *const gr = lds + S::ROWS, *const qc = lds + 2 * S::ROWS, *const gc = qc + S::COLS;
  const int G = a.H / a.KVH / a.splits, hk = blockIdx.y, h0 = hk * (a.H / a.KVH) + blockIdx.z * G;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  // Early keys of a sequence are seen by more queries: odd KV heads walk the key blocks backwards,
  // so that the CU that got a long block first gets a short one next.
  const int64_t jb = hk & 1 ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
  const int64_t j0 = jb * 64, jw = j0 + 16 * wave, j = jw + li;
  const bool live = j < a.n, wave_live = jw < a.n;
  const int64_t end = live ? a.seq_start[a.seq_of[j] + 1] : 0;
  const int64_t w_hi = wave_live ? a.seq_start[a.seq_of[min<int64_t>(a.n - 1, jw + 15)] + 1] : 0;
  const int64_t q_hi = a.seq_start[a.seq_of[min<int64_t>(a.n - 1, j0 + 63)] + 1];
  const int units = int((q_hi - j0 + KT - 1) / KT) * G;
  clear_lds(lds, 2 * S::ROWS + 2 * S::COLS);
  Operand<PARTS> kf[S::DK], vf[S::DK];
  row_operand<D, PARTS>(kf, a.k + j * a.ldk + hk * D, live, lg);
  row_operand<D, PARTS>(vf, a.v + j * a.ldv + hk * D, live, lg);
  RowSum<PARTS> dk_sum[S::DT] = {}, dv_sum[S::DT] = {};
  float4 qp[S::PER][2], gp[S::PER][2];
  float sp = 0.f;
  auto load = [&](int u) {
    const int h = h0 + u % G;
    const int64_t t0 = j0 + KT * (u / G), last = min<int64_t>(a.n, q_hi) - 1;
    rows_load<D, PARTS>(qp, a.q + h * D, a.ldq, t0, last);
    rows_load<D, PARTS>(gp, a.dout + h * D, int64_t(a.H) * D, t0, last);
    const int64_t t = t0 + (threadIdx.x & (KT - 1));
    if (threadIdx.x < 2 * KT)
      sp = t > last ? 0.f : threadIdx.x < KT ? a.lse[t * a.H + h] : a.dsum[t * a.H + h];
  };
  load(0);
  for (int u = 0; u < units; ++u) {
    __syncthreads();
    if constexpr (PARTS == 3) {
#pragma unroll
      for (int e = 0; e < S::PER; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h) qp[e][h] = scaled_query(qp[e][h], a.scale);
    }
    rows_store<D, PARTS, true, true>(qr, qc, qp);
    rows_store<D, PARTS, true, true>(gr, gc, gp);
    if (threadIdx.x < 2 * KT) ls[threadIdx.x] = sp;  // [0, KT) lse, [KT, 2 KT) D
    __syncthreads();
    if (u + 1 < units) load(u + 1);
    const int64_t t0 = j0 + KT * (u / G);
    if (!(wave_live && t0 + KT - 1 >= jw && t0 < w_hi)) continue;
    // The lane's key is seen by the unit's queries lo .. hi.
    const int lo = live ? int(max<int64_t>(j - t0, 0)) : KT, hi = live ? int(min<int64_t>(end - t0, KT)) - 1 : -1;
    const unsigned seen = unsigned(max(hi - lo + 1, 0));
    const bool whole = __all(seen == KT);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int64_t tb = t0 + 32 * half;
      if (!(tb + 31 >= jw && tb < w_hi)) continue;
      f32x4 p[2], ds[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int sub = 2 * half + x;
        f32x4 sc = {0.f, 0.f, 0.f, 0.f}, dp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < S::DK; ++k) {
          sc = mma_parts<PARTS, PARTS, true>(row_frag<D, PARTS>(qr, sub, k, li, lg), kf[k], sc);
          dp = mma_parts<PARTS, PARTS>(row_frag<D, PARTS>(gr, sub, k, li, lg), vf[k], dp);
        }
        sc = natural_score<PARTS>(sc, a.scale);
        const f32x4 lse = *reinterpret_cast<const f32x4 *>(ls + 16 * sub + 4 * lg);
        const f32x4 dsum = *reinterpret_cast<const f32x4 *>(ls + KT + 16 * sub + 4 * lg);
#pragma unroll
        for (int r = 0; r < 4; ++r) p[x][r] = exp_natural(sc[r] - lse[r]);
        if (!whole) {
#pragma unroll
          for (int r = 0; r < 4; ++r) p[x][r] = unsigned(4 * lg - lo + 16 * sub + r) < seen ? p[x][r] : 0.f;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) ds[x][r] = p[x][r] * (dp[r] - dsum[r]);
      }
      const Operand<3> po = score_operand(p[0], p[1]), dso = score_operand(ds[0], ds[1]);
#pragma unroll
      for (int dt = 0; dt < S::DT; ++dt) {
        mma_add<PARTS>(col_frag<D, PARTS>(gc, half, dt, li, lg), po, dv_sum[dt]);
        mma_add<PARTS>(col_frag<D, PARTS>(qc, half, dt, li, lg), dso, dk_sum[dt]);
      }
    }
  }
  if (!live) return;
  f32x4 dk[S::DT], dv[S::DT];
#pragma unroll
  for (int dt = 0; dt < S::DT; ++dt) {
    dk[dt] = dk_sum[dt].total();
    dv[dt] = dv_sum[dt].total();
  }
  float dk_scale = PARTS == 3 ? 1.0f : a.scale;  // (of the staged queries)
  if (!(all_finite(dk) && all_finite(dv))) {
    const int tid = fresh_thread(), lz = tid & 63;
    const int64_t jz = j0 + 16 * (tid >> 6) + (lz & 15), stop = a.seq_start[a.seq_of[jz] + 1];
    clear(dk);
    clear(dv);
    dk_scale = a.scale;
#pragma unroll 1
    for (int h = h0; h < h0 + G; ++h)
#pragma unroll 1
      for (int64_t t = jz; t < stop; ++t) {
        float p, ds;
        plain_pair<D>(a, t, jz, h, hk, a.dsum[t * a.H + h], p, ds);
        plain_add<D>(dk, ds, a.q + t * a.ldq + h * D, lz >> 4);
        plain_add<D>(dv, p, a.dout + (t * a.H + h) * D, lz >> 4);
      }
  }
  if (a.parts) {
    float *row = a.parts + (int64_t(blockIdx.z) * a.n + j) * 2 * a.KVH * D + hk * D;
#pragma unroll
    for (int dt = 0; dt < S::DT; ++dt)
      if (dt * 16 + 4 * lg < D) {
        *reinterpret_cast<f32x4 *>(row + dt * 16 + 4 * lg) = dk[dt] * dk_scale;
        *reinterpret_cast<f32x4 *>(row + a.KVH * D + dt * 16 + 4 * lg) = dv[dt];
      }
    return;
  }
  float *dkrow = a.dk + j * a.ldk + hk * D, *dvrow = a.dv + j * a.ldv + hk * D;
#pragma unroll
  for (int dt = 0; dt < S::DT; ++dt)
    if (dt * 16 + 4 * lg < D) {
      store4(a, dkrow + dt * 16 + 4 * lg, dk[dt], dk_scale);
      store4(a, dvrow + dt * 16 + 4 * lg, dv[dt], 1.0f);
    }
}

// dk / dv = the sum of the head parts (width = KVH * D columns each, a multiple of 4), rounded like the
// attention's other outputs.
__global__ void merge_dkv_kernel(const AttnTrain a, int32_t width) {
  const int quads = 2 * width / 4;
  const int64_t total = int64_t(a.n) * quads;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t t = i / quads;
    const int c = int(i % quads) * 4;
    f32x4 v = *reinterpret_cast<const f32x4 *>(a.parts + t * 2 * width + c);
    for (int z = 1; z < a.splits; ++z) v += *reinterpret_cast<const f32x4 *>(a.parts + (z * int64_t(a.n) + t) * 2 * width + c);
    store4(a, c < width ? a.dk + t * a.ldk + c : a.dv + t * a.ldv + c - width, v, 1.0f);
  }
}

// dst[i] = 0: clears the accumulated gradients (a kernel rather than a memset node, so a
// captured backward replays it like any other launch).
__global__ void zero_fill_kernel(float *__restrict__ dst, int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
    dst[i] = 0.0f;
}

// dst[r, c] += alpha * src[r * ld_src + c] (ld_src 0 broadcasts one row: bias adds).
__global__ void add_strided_kernel(int32_t rows, int32_t cols, float alpha, const float *__restrict__ src,
                                   int64_t ld_src, float *__restrict__ dst, int64_t ld_dst) {
  const int64_t total = int64_t(rows) * cols;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t r = i / cols;
    const int c = int(i % cols);
    dst[r * ld_dst + c] += alpha * src[r * ld_src + c];
  }
}

// The per-layer embedding's update of the stream, x[r, c] += scale * ple[r, c % pd]
// (Trunk._add_ple), and its gradient, dple[r, k] = scale * (dx[r, k] + dx[r, k + pd] + ...).
__global__ void ple_add_kernel(int32_t rows, int32_t d, int32_t pd, float scale, const float *__restrict__ ple,
                               int64_t ld_ple, float *__restrict__ x) {
  const int64_t total = int64_t(rows) * d;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t r = i / d;
    x[i] += scale * ple[r * ld_ple + int(i % d) % pd];
  }
}
__global__ void ple_grad_kernel(int32_t rows, int32_t d, int32_t pd, float scale, const float *__restrict__ dx,
                                float *__restrict__ dple, int64_t ld_ple) {
  const int64_t total = int64_t(rows) * pd;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t r = i / pd;
    const int k = int(i % pd);
    float s = 0.f;
    for (int c = k; c < d; c += pd) s += scale * dx[r * d + c];
    dple[r * ld_ple + k] = s;
  }
}

// dst[r, c] = src[r * ld_src + c].
__global__ void copy_strided_kernel(int32_t rows, int32_t cols, const float *__restrict__ src, int64_t ld_src,
                                    float *__restrict__ dst, int64_t ld_dst) {
  const int64_t total = int64_t(rows) * cols;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.x) * blockDim.x)
    dst[i / cols * ld_dst + i % cols] = src[i / cols * ld_src + i % cols];
}

// Gain-only RMSNorm keeping rstd per row (one wave per row).
__global__ void rmsnorm_fwd_kernel(const float *__restrict__ x, const float *__restrict__ w, float eps,
                                   float *__restrict__ y, float *__restrict__ rstd, int32_t n, int32_t d) {
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= n) return;
  const float *xr = x + int64_t(row) * d;
  float s = 0.f;
  for (int k = lane; k < d; k += 64) s = fmaf(xr[k], xr[k], s);
  const float r = 1.0f / sqrtf(wave_sum(s) / float(d) + eps);
  float *yr = y + int64_t(row) * d;
  for (int k = lane; k < d; k += 64) yr[k] = xr[k] * r * w[k];
  if (lane == 0) rstd[row] = r;
}

// seq_of[t] for packed rows.
__global__ void seq_of_kernel(const int64_t *__restrict__ seq_start, int32_t n_seqs, int32_t *__restrict__ seq_of) {
  const int s = blockIdx.x;
  if (s >= n_seqs) return;
  for (int64_t t = seq_start[s] + threadIdx.x; t < seq_start[s + 1]; t += blockDim.x) seq_of[t] = s;
}

unsigned blocks_of(int64_t items, int per_block) { return unsigned((items + per_block - 1) / per_block); }
unsigned grid_1d(int64_t n) { return unsigned(std::min<int64_t>((n + 255) / 256, 8192)); }

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Operand checks shared by the attention launchers: the kernels load rows of q / k / v as
// float4, so rows start 16-byte aligned.
void check_attn_train(const cg_attn_train *p) {
  CG_REQUIRE(p && p->H > 0 && p->KVH > 0 && p->H % p->KVH == 0 && p->H / p->KVH <= 16, CG_ERR_INVALID,
             "training attention: H a multiple of KVH, at most 16 heads per KV head");
  CG_REQUIRE(p->q && p->k && p->v && p->seq_start && p->seq_of, CG_ERR_INVALID,
             "attention q, k, v, seq_start and seq_of are required");
  CG_REQUIRE(aligned16(p->q) && aligned16(p->k) && aligned16(p->v) && p->ldq % 4 == 0 && p->ldk % 4 == 0 &&
                 p->ldv % 4 == 0,
             CG_ERR_INVALID, "attention q / k / v: 16-byte aligned rows (pointers and row strides)");
}

// Operand mode (rows, k) of a GEMM input: 1 k contiguous, 2 rows contiguous, 0 any strides.
int operand_mode(const float *p, int64_t sr, int64_t sk, int32_t rows, int32_t kk) {
  if (!aligned16(p)) return 0;
  if (sk == 1 && sr % 4 == 0 && kk % 4 == 0 && sr >= 0 && sr <= TILE_MAX_STRIDE) return 1;
  if (sr == 1 && sk % 4 == 0 && rows % 4 == 0 && sk >= 0 && sk <= TILE_MAX_STRIDE) return 2;
  return 0;
}

// A split product's partial results and partial row sums.
size_t slice_bytes(const GemmPlan &pl, int32_t m, int32_t n) { return size_t(pl.slices) * size_t(m) * (size_t(n) + 1) * 4; }

GemmPlan plan_of(int32_t m, int32_t n, int32_t k, const float *a, int64_t sam, int64_t sak, const float *b,
                 int64_t sbk, int64_t sbn, bool bf16, int *am, int *bm) {
  *am = operand_mode(a, sam, sak, m, k);
  *bm = operand_mode(b, sbn, sbk, n, k);
  if (*am == 0 || *bm == 0) *am = *bm = 0;
  return gemm_plan(m, n, k, *am == 0, bf16);
}

void rows_launch(int32_t m, int32_t n, int32_t k, float alpha, const float *a, int64_t sam, int64_t sak, const float *b,
                 int64_t sbk, int64_t sbn, float beta, float *c, int64_t ldc, const Epi &epi, int am, int bm,
                 hipStream_t s) {
  const dim3 grid(unsigned((n + 31) / 32), unsigned((m + 31) / 32));
  const bool bf = epi.round != 0, sums = epi.row_sum != nullptr;
#define CG_ROWS_RUN(A_, B_, BF_, S_) \
  gemm_rows_kernel<A_, B_, BF_, S_><<<grid, 512, 0, s>>>(m, n, k, alpha, a, sam, sak, b, sbk, sbn, beta, c, ldc, epi)
#define CG_ROWS_CASE(A_, B_, S_)               \
  if (sums == S_ && am == A_ && bm == B_) {    \
    if (bf) CG_ROWS_RUN(A_, B_, true, S_);     \
    else CG_ROWS_RUN(A_, B_, false, S_);       \
  }
  CG_REQUIRE(!sums || (am == 2 && bm == 2) || (am == 0 && bm == 0), CG_ERR_UNSUPPORTED, "GEMM: row sums of this layout");
  CG_ROWS_CASE(1, 1, false)
  CG_ROWS_CASE(1, 2, false)
  CG_ROWS_CASE(2, 1, false)
  CG_ROWS_CASE(2, 2, false)
  CG_ROWS_CASE(0, 0, false)
  CG_ROWS_CASE(2, 2, true)
  CG_ROWS_CASE(0, 0, true)
#undef CG_ROWS_CASE
#undef CG_ROWS_RUN
  CG_LAUNCHED();
}

void gemm_launch(int32_t m, int32_t n, int32_t k, float alpha, const float *a, int64_t sam, int64_t sak,
                 const float *b, int64_t sbk, int64_t sbn, float beta, float *c, int64_t ldc, void *workspace,
                 size_t workspace_size, const Epi &epi, void *stream) {
  CG_REQUIRE(m >= 0 && n >= 0 && k >= 0, CG_ERR_INVALID, "negative GEMM size");
  if (m == 0 || n == 0) return;
  CG_REQUIRE(a && b && c, CG_ERR_INVALID, "a, b and c are required");
  CG_REQUIRE((epi.mode != EPI_GELU || epi.aux_out) && (epi.mode != EPI_GELU_GRAD || epi.aux_in), CG_ERR_INVALID,
             "GEMM epilogue: GELU needs its second output, GELU' its pre-activation");
  int am, bm;
  const bool bf = epi.round != 0, sums = epi.row_sum != nullptr;
  const GemmPlan pl = plan_of(m, n, k, a, sam, sak, b, sbk, sbn, bf, &am, &bm);
  if (few_rows(m, n, k, bf && am == 2 && bm == 2)) {
    rows_launch(m, n, k, alpha, a, sam, sak, b, sbk, sbn, beta, c, ldc, epi, am, bm, as_stream(stream));
    return;
  }
  const size_t need = pl.slices > 1 ? slice_bytes(pl, m, n) : 0;
  CG_REQUIRE(k > 0 || !epi.row_sum, CG_ERR_INVALID, "GEMM: row sums of an empty product");
  CG_REQUIRE(need == 0 || (workspace && workspace_size >= need), CG_ERR_INVALID,
             "GEMM: workspace too small, need " + std::to_string(need) + " bytes");
  const dim3 grid(unsigned((n + GT_N - 1) / GT_N), unsigned((m + pl.tm - 1) / pl.tm), unsigned(pl.slices));
  CG_REQUIRE(grid.y <= 65535, CG_ERR_UNSUPPORTED, "GEMM: too many row tiles");
  hipStream_t s = as_stream(stream);
  float *part = pl.slices > 1 ? static_cast<float *>(workspace) : nullptr;
  const int32_t kc = pl.kc;
  CG_REQUIRE(!sums || (am == 2 && bm == 2) || (am == 0 && bm == 0), CG_ERR_UNSUPPORTED, "GEMM: row sums of this layout");
#define CG_GEMM_RUN(A_, B_, T_, BF_, S_)                                                                        \
  gemm_strided_kernel<A_, B_, T_, BF_, S_><<<grid, 256, 0, s>>>(m, n, k, kc, alpha, a, sam, sak, b, sbk, sbn, beta, c, \
                                                                ldc, part, epi)
#define CG_GEMM_CASE(A_, B_, T_)                     \
  if (!sums && am == A_ && bm == B_ && pl.tm == T_) { \
    if (bf) CG_GEMM_RUN(A_, B_, T_, true, false);    \
    else CG_GEMM_RUN(A_, B_, T_, false, false);      \
  }
#define CG_GEMM_SUMS(A_, B_, T_)                    \
  if (sums && am == A_ && bm == B_ && pl.tm == T_) { \
    if (bf) CG_GEMM_RUN(A_, B_, T_, true, true);    \
    else CG_GEMM_RUN(A_, B_, T_, false, true);      \
  }
  CG_GEMM_CASE(1, 1, 128)
  CG_GEMM_CASE(1, 2, 128)
  CG_GEMM_CASE(2, 1, 128)
  CG_GEMM_CASE(2, 2, 128)
  CG_GEMM_CASE(1, 1, 64)
  CG_GEMM_CASE(1, 2, 64)
  CG_GEMM_CASE(2, 1, 64)
  CG_GEMM_CASE(2, 2, 64)
  CG_GEMM_CASE(0, 0, 128)
  CG_GEMM_SUMS(2, 2, 128)  // weight gradients: A = dY^T, B = X, both token-major
  CG_GEMM_SUMS(2, 2, 64)
  CG_GEMM_SUMS(0, 0, 128)
#undef CG_GEMM_RUN
#undef CG_GEMM_SUMS
#undef CG_GEMM_CASE
  CG_LAUNCHED();
  if (part) {
    gemm_reduce_kernel<<<blocks_of(int64_t(m) * n, 256), 256, 0, s>>>(m, n, pl.slices, alpha, part, beta, c, ldc, epi);
    CG_LAUNCHED();
  }
}

// Split-K partials of a GEMM (the most over the operand layouts and precisions).
size_t gemm_workspace_bytes(int32_t m, int32_t n, int32_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  size_t most = 0;
  for (bool generic : {false, true})
    for (bool bf16 : {false, true}) {
      const GemmPlan pl = gemm_plan(m, n, k, generic, bf16);
      if (pl.slices > 1) most = std::max(most, slice_bytes(pl, m, n));
    }
  return most;
}

size_t column_sum_ws(int32_t rows, int32_t cols) {
  return rows > 2048 ? size_t((rows + 255) / 256) * size_t(std::max(cols, 0)) * 4 : 0;
}

// out[c] (+)= sum_r x[r * ld + c].
void column_sum_launch(const float *x, int32_t rows, int32_t cols, int64_t ld, float *out, int32_t accumulate,
                       void *workspace, size_t workspace_size, void *stream) {
  if (cols == 0) return;
  CG_REQUIRE(x && out && rows >= 0, CG_ERR_INVALID, "column sum operands are required");
  hipStream_t s = as_stream(stream);
  if (rows <= 2048) {
    column_sum_kernel<<<dim3(blocks_of(cols, 64), 1), 256, 0, s>>>(x, rows, cols, ld, out, accumulate, rows);
    CG_LAUNCHED();
    return;
  }
  const size_t need = column_sum_ws(rows, cols);
  CG_REQUIRE(workspace && workspace_size >= need, CG_ERR_INVALID, "column sum: workspace too small");
  const int chunks = (rows + 255) / 256;
  float *part = static_cast<float *>(workspace);
  column_sum_kernel<<<dim3(blocks_of(cols, 64), unsigned(chunks)), 256, 0, s>>>(x, rows, cols, ld, part, 0, 256);
  CG_LAUNCHED();
  column_sum_kernel<<<dim3(blocks_of(cols, 64), 1), 256, 0, s>>>(part, chunks, cols, cols, out, accumulate, chunks);
  CG_LAUNCHED();
}

// dst[r, c] = bf16(dst[r, c] + src[r * ld_src + c]): the value embedding added to v in fp32 and
// rounded once (the attention reads bf16 v).
__global__ void add_round_kernel(int32_t rows, int32_t cols, const float *__restrict__ src, int64_t ld_src,
                                 float *__restrict__ dst, int64_t ld_dst) {
  const int64_t total = int64_t(rows) * cols;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t r = i / cols;
    const int c = int(i % cols);
    float *d = dst + r * ld_dst + c;
    *d = round_bf16(*d + src[r * ld_src + c]);
  }
}

// Grid of the forward and dQ kernels: blocks of 16 tokens x four heads of a group, or more
// tokens per block when the group has fewer heads.
dim3 query_grid(const cg_attn_train &p) {
  const int G = p.H / p.KVH, gpb = std::min(G, 4), tpb = 4 / gpb;
  return dim3(blocks_of(p.n, 16 * tpb), unsigned(p.KVH), unsigned((G + gpb - 1) / gpb));
}

// Attention launches; bf16_operands: q, k, v (and dout) hold bf16 numbers, so one part of each is
// exact.
void attn_fwd_launch(const cg_attn_train *p, bool bf16_operands, hipStream_t s) {
  check_attn_train(p);
  if (p->n == 0) return;
  AttnTrain a{p->n, p->H, p->KVH, p->scale, p->seq_start, p->seq_of, p->q, p->k, p->v, p->ldq, p->ldk, p->ldv,
              nullptr, nullptr, nullptr, p->o, p->lse, nullptr, nullptr, nullptr, nullptr, p->round_bf16, 1, nullptr, 1};
  CG_REQUIRE(a.out && a.lse_out, CG_ERR_INVALID, "attention forward outputs are required");
  CG_REQUIRE(aligned16(a.out), CG_ERR_INVALID, "attention output: 16-byte aligned");
  const dim3 grid = query_grid(*p);
  switch (p->head_dim) {
#define CG_FWD_CASE(DD)                                                   \
  case DD:                                                                \
    if (bf16_operands) attn_fwd_kernel<DD, 1><<<grid, 256, 0, s>>>(a);    \
    else attn_fwd_kernel<DD, 3><<<grid, 256, 0, s>>>(a);                  \
    break;
    CG_FWD_CASE(8)
    CG_FWD_CASE(16)
    CG_FWD_CASE(24)
    CG_FWD_CASE(32)
    CG_FWD_CASE(64)
#undef CG_FWD_CASE
    default: throw Error(CG_ERR_UNSUPPORTED, "training attention: head_dim 8, 16, 24, 32 or 64");
  }
  CG_LAUNCHED();
}

// Backward; `parts` (16-byte aligned, part_floats floats; NULL: none) lets few key blocks split their head
// groups.
void attn_bwd_launch(const cg_attn_train *p, const float *dout, float *dsum, float *dq, float *dk, float *dv,
                     bool bf16_operands, hipStream_t s, float *parts = nullptr, int64_t part_floats = 0) {
  check_attn_train(p);
  if (p->n == 0) return;
  AttnTrain a{p->n, p->H, p->KVH, p->scale, p->seq_start, p->seq_of, p->q, p->k, p->v, p->ldq, p->ldk, p->ldv,
              p->o, dout, p->lse, nullptr, nullptr, dsum, dq, dk, dv, p->round_bf16,
              aligned16(dq) && aligned16(dk) && aligned16(dv), nullptr, 1};
  CG_REQUIRE(a.o && a.dout && a.lse && dsum && dq && dk && dv, CG_ERR_INVALID,
             "attention backward operands are required");
  CG_REQUIRE(aligned16(dout), CG_ERR_INVALID, "attention dO: 16-byte aligned");
  // Heads split while the blocks stay within eight per CU (13.8 k ragged tokens fp32: 432 blocks 77 us,
  // 1728 blocks 52 and the merge 9), with one-part operands, whose walk is shorter, within two (64 x 256
  // tokens: 512 blocks 39.5 us, 2048 blocks 32.9 and the merge 9.7).
  const int64_t blocks = int64_t(blocks_of(p->n, 64)) * p->KVH, width = int64_t(p->KVH) * p->head_dim;
  for (int z = 4; z > 1 && parts; z /= 2)
    if (p->H / p->KVH % z == 0 && blocks * z <= (bf16_operands ? 512 : 2048) && z * 2 * width * p->n <= part_floats) {
      a.splits = z;
      a.parts = parts;
      break;
    }
  const dim3 grid = query_grid(*p), grid_kv(blocks_of(p->n, 64), unsigned(p->KVH), unsigned(a.splits));
  switch (p->head_dim) {
#define CG_BWD_CASE(DD)                                                      \
  case DD:                                                                   \
    if (bf16_operands) attn_bwd_dq_kernel<DD, 1><<<grid, 256, 0, s>>>(a);    \
    else attn_bwd_dq_kernel<DD, 3><<<grid, 256, 0, s>>>(a);                  \
    CG_LAUNCHED();                                                           \
    if (bf16_operands) attn_bwd_dkv_kernel<DD, 1><<<grid_kv, 256, 0, s>>>(a); \
    else attn_bwd_dkv_kernel<DD, 3><<<grid_kv, 256, 0, s>>>(a);              \
    break;
    CG_BWD_CASE(8)
    CG_BWD_CASE(16)
    CG_BWD_CASE(24)
    CG_BWD_CASE(32)
    CG_BWD_CASE(64)
#undef CG_BWD_CASE
    default: throw Error(CG_ERR_UNSUPPORTED, "training attention: head_dim 8, 16, 24, 32 or 64");
  }
  CG_LAUNCHED();
  if (a.parts) {
    merge_dkv_kernel<<<grid_1d(int64_t(p->n) * width / 2), 256, 0, s>>>(a, int32_t(width));
    CG_LAUNCHED();
  }
}

}  // namespace
}  // namespace cg

using namespace cg;

extern "C" {

size_t cg_gemm_workspace_size(int32_t m, int32_t n, int32_t k) { return gemm_workspace_bytes(m, n, k); }

int cg_gemm_strided(int32_t m, int32_t n, int32_t k, float alpha, const float *a, int64_t sam, int64_t sak,
                    const float *b, int64_t sbk, int64_t sbn, float beta, float *c, int64_t ldc,
                    int32_t compute_dtype, void *workspace, size_t workspace_size, void *stream) {
  return guarded([&] {
    CG_REQUIRE(compute_dtype == CG_F32 || compute_dtype == CG_BF16, CG_ERR_UNSUPPORTED,
               "GEMM compute dtype: CG_F32 or CG_BF16");
    Epi e;
    e.round = compute_dtype == CG_BF16;
    gemm_launch(m, n, k, alpha, a, sam, sak, b, sbk, sbn, beta, c, ldc, workspace, workspace_size, e, stream);
  });
}

int cg_layernorm_fwd(const float *x, const float *w, const float *b, float eps, float *y, float *mean, float *rstd,
                     int32_t n, int32_t d, void *stream) {
  return guarded([&] {
    if (n == 0) return;
    CG_REQUIRE(x && w && b && y && mean && rstd && d > 0, CG_ERR_INVALID, "LayerNorm operands are required");
    hipStream_t s = as_stream(stream);
    if (d % 4 == 0 && d <= 1024 && aligned16(x) && aligned16(w) && aligned16(b) && aligned16(y)) {
      switch ((d + 255) / 256) {
#define CG_LN_CASE(NV)                                                                                        \
  case NV:                                                                                                    \
    layernorm_rows_kernel<NV><<<blocks_of(n, 16), 256, 0, s>>>(x, w, b, eps, y, mean, rstd, n, d); \
    break;
        CG_LN_CASE(1)
        CG_LN_CASE(2)
        CG_LN_CASE(3)
        CG_LN_CASE(4)
#undef CG_LN_CASE
      }
    } else {
      layernorm_fwd_kernel<<<blocks_of(n, 4), 256, 0, s>>>(x, w, b, eps, y, mean, rstd, n, d);
    }
    CG_LAUNCHED();
  });
}

size_t cg_norm_bwd_workspace_size(int32_t n, int32_t d) {
  return n > 0 && d > 0 ? size_t((int64_t(n) + NORM_ROWS - 1) / NORM_ROWS) * 2 * size_t(d) * 4 : 0;
}

int cg_norm_bwd(const float *x, const float *dy, const float *w, const float *mean, const float *rstd, float *dx,
                const float *residual, float *dw, float *db, int32_t n, int32_t d, void *workspace,
                size_t workspace_size, int32_t accumulate, void *stream) {
  return guarded([&] {
    if (n == 0) return;
    CG_REQUIRE(x && dy && w && rstd && dx && dw && d > 0, CG_ERR_INVALID, "norm backward operands are required");
    CG_REQUIRE(mean == nullptr || db != nullptr, CG_ERR_INVALID, "LayerNorm backward needs db");
    CG_REQUIRE(workspace && workspace_size >= cg_norm_bwd_workspace_size(n, d), CG_ERR_INVALID,
               "norm backward: workspace too small");
    hipStream_t s = as_stream(stream);
    float *part = static_cast<float *>(workspace);
    const bool vec = d % 4 == 0 && d <= 1024 && aligned16(x) && aligned16(dy) && aligned16(w) && aligned16(dx) &&
                     (residual == nullptr || aligned16(residual)) && aligned16(part);
    const int32_t parts = int32_t((int64_t(n) + NORM_ROWS - 1) / NORM_ROWS);
    if (vec) {
      switch ((d + 255) / 256) {
#define CG_NORM_CASE(NV)                                                                                        \
  case NV:                                                                                                      \
    norm_bwd_rows_kernel<NV><<<unsigned(parts), 256, 0, s>>>(x, dy, w, mean, rstd, residual, dx, part, n, d); \
    break;
        CG_NORM_CASE(1)
        CG_NORM_CASE(2)
        CG_NORM_CASE(3)
        CG_NORM_CASE(4)
#undef CG_NORM_CASE
      }
    } else {
      norm_bwd_kernel<<<unsigned(parts), 256, 2 * d * sizeof(float), s>>>(x, dy, w, mean, rstd, residual, dx, part, n,
                                                                         d, NORM_ROWS);
    }
    CG_LAUNCHED();
    norm_params_kernel<<<blocks_of(2 * int64_t(d), 64), 1024, 0, s>>>(part, parts, d, dw, db, accumulate);
    CG_LAUNCHED();
  });
}

size_t cg_column_sum_workspace_size(int32_t rows, int32_t cols) { return column_sum_ws(rows, cols); }

int cg_column_sum(const float *x, int32_t rows, int32_t cols, int64_t ld, float *out, int32_t accumulate,
                  void *workspace, size_t workspace_size, void *stream) {
  return guarded([&] { column_sum_launch(x, rows, cols, ld, out, accumulate, workspace, workspace_size, stream); });
}

int cg_gelu_fwd(const float *u, float *g, int64_t n, void *stream) {
  return guarded([&] {
    if (n == 0) return;
    CG_REQUIRE(u && g, CG_ERR_INVALID, "GELU operands are required");
    gelu_fwd_kernel<<<grid_1d(n), 256, 0, as_stream(stream)>>>(u, g, n);
    CG_LAUNCHED();
  });
}

int cg_gelu_bwd(const float *u, const float *dg, float *du, int64_t n, void *stream) {
  return guarded([&] {
    if (n == 0) return;
    CG_REQUIRE(u && dg && du, CG_ERR_INVALID, "GELU backward operands are required");
    gelu_bwd_kernel<<<grid_1d(n), 256, 0, as_stream(stream)>>>(u, dg, du, n);
    CG_LAUNCHED();
  });
}

int cg_add_strided(int32_t rows, int32_t cols, float alpha, const float *src, int64_t ld_src, float *dst,
                   int64_t ld_dst, void *stream) {
  return guarded([&] {
    if (int64_t(rows) * cols == 0) return;
    CG_REQUIRE(src && dst && rows > 0 && cols > 0, CG_ERR_INVALID, "add operands are required");
    add_strided_kernel<<<grid_1d(int64_t(rows) * cols), 256, 0, as_stream(stream)>>>(rows, cols, alpha, src, ld_src,
                                                                                     dst, ld_dst);
    CG_LAUNCHED();
  });
}

int cg_rmsnorm_fwd(const float *x, const float *w, float eps, float *y, float *rstd, int32_t n, int32_t d,
                   void *stream) {
  return guarded([&] {
    if (n == 0) return;
    CG_REQUIRE(x && w && y && rstd && d > 0, CG_ERR_INVALID, "RMSNorm operands are required");
    rmsnorm_fwd_kernel<<<blocks_of(n, 4), 256, 0, as_stream(stream)>>>(x, w, eps, y, rstd, n, d);
    CG_LAUNCHED();
  });
}

int cg_seq_of(const int64_t *seq_start, int32_t n_seqs, int32_t *seq_of, void *stream) {
  return guarded([&] {
    if (n_seqs == 0) return;
    CG_REQUIRE(seq_start && seq_of, CG_ERR_INVALID, "seq_start and seq_of are required");
    seq_of_kernel<<<unsigned(n_seqs), 256, 0, as_stream(stream)>>>(seq_start, n_seqs, seq_of);
    CG_LAUNCHED();
  });
}

int cg_attn_train_fwd(const cg_attn_train *p, void *stream) {
  return guarded([&] { attn_fwd_launch(p, false, as_stream(stream)); });
}

int cg_attn_train_bwd(const cg_attn_train *p, const float *dout, float *dsum, float *dq, float *dk, float *dv,
                      void *stream) {
  return guarded([&] { attn_bwd_launch(p, dout, dsum, dq, dk, dv, false, as_stream(stream)); });
}

}  // extern "C"

// ---- the whole trunk: forward keeping activations, and backward -------------------------------
namespace {

void ok(int status) {
  if (status == CG_OK) return;
  char buf[512];
  cg_last_error(buf, sizeof(buf));
  throw Error(status, "training step: " + std::string(buf));
}

struct TrainDims {
  int64_t n, d, F, H, KVH, D, Q, KVW, QKV, L, P, V, pd;
  bool bf;  // bf16 autocast precision
};

TrainDims dims_of(const cg_train_config &c, int32_t n) {
  TrainDims t{};
  t.n = n;
  t.bf = c.bf16 != 0;
  t.d = c.d_model;
  t.F = c.d_ff;
  t.H = c.n_heads;
  t.KVH = c.n_kv_heads;
  t.D = c.d_model / c.n_heads;
  t.Q = t.H * t.D;
  t.KVW = t.KVH * t.D;
  t.QKV = t.Q + 2 * t.KVW;
  t.L = c.n_layers;
  t.P = c.ple_width;
  t.V = c.value_width;
  t.pd = c.per_layer_dim;
  return t;
}

// Per layer, in floats of n rows: xl, h1 (d), m1, r1 (1), qkv (QKV), o (Q), lse (H), x1, h2 (d),
// m2, r2 (1), u, g (F: the MLP's pre-activation and its GELU); then x_last (d), mf, rf (1) and
// seq_of (n int32).  Every array starts on a
// 256-byte boundary (the attention kernels load rows of qkv as float4).
struct SavedLayer {
  float *xl, *h1, *m1, *r1, *qkv, *o, *lse, *x1, *h2, *m2, *r2, *u, *g;
};

int64_t span_of(const TrainDims &t, int64_t cols) { return (t.n * cols + 63) / 64 * 64; }

int64_t layer_floats(const TrainDims &t) {
  return 4 * span_of(t, t.d) + 4 * span_of(t, 1) + span_of(t, t.QKV) + span_of(t, t.Q) + span_of(t, t.H) +
         2 * span_of(t, t.F);
}

SavedLayer saved_layer(const TrainDims &t, void *saved, int64_t l) {
  float *p = static_cast<float *>(saved) + l * layer_floats(t);
  SavedLayer s{};
  auto take = [&](int64_t cols) {
    float *q = p;
    p += span_of(t, cols);
    return q;
  };
  s.xl = take(t.d);
  s.h1 = take(t.d);
  s.m1 = take(1);
  s.r1 = take(1);
  s.qkv = take(t.QKV);
  s.o = take(t.Q);
  s.lse = take(t.H);
  s.x1 = take(t.d);
  s.h2 = take(t.d);
  s.m2 = take(1);
  s.r2 = take(1);
  s.u = take(t.F);
  s.g = take(t.F);
  return s;
}

struct SavedTail {
  float *x_last, *mf, *rf;
  int32_t *seq_of;
};
SavedTail saved_tail(const TrainDims &t, void *saved) {
  float *p = static_cast<float *>(saved) + t.L * layer_floats(t);
  float *mf = p + span_of(t, t.d), *rf = mf + span_of(t, 1);
  return {p, mf, rf, reinterpret_cast<int32_t *>(rf + span_of(t, 1))};
}

size_t max_gemm_ws(const TrainDims &t) {
  size_t m = 0;
  const int64_t shapes[][3] = {{t.n, t.QKV, t.d}, {t.n, t.d, t.Q}, {t.n, t.F, t.d}, {t.n, t.d, t.F},
                               {t.QKV, t.d, t.n}, {t.d, t.Q, t.n}, {t.F, t.d, t.n}, {t.d, t.F, t.n},
                               {t.n, t.d, t.QKV}, {t.n, t.Q, t.d}, {t.n, t.d, t.F}};
  for (auto &sh : shapes) m = std::max(m, cg_gemm_workspace_size(int32_t(sh[0]), int32_t(sh[1]), int32_t(sh[2])));
  return m;
}

// Scratch of one call: GEMM split-K partials, then (backward) dx, dx1, dh (d each), du (F), do (Q),
// dqkv (QKV), dsum (H), norm partials.
struct Scratch {
  float *gemm_ws;
  size_t gemm_bytes;
  float *dx, *dx1, *dh, *du, *dout, *dqkv, *dsum, *red;
  size_t red_bytes;
};

size_t red_bytes_of(const TrainDims &t) { return cg_norm_bwd_workspace_size(int32_t(t.n), int32_t(t.d)); }

Scratch scratch_of(const TrainDims &t, void *base) {
  Scratch s{};
  char *p = static_cast<char *>(base);
  s.gemm_bytes = (max_gemm_ws(t) + 255) / 256 * 256;
  s.gemm_ws = reinterpret_cast<float *>(p);
  p += s.gemm_bytes;
  float *f = reinterpret_cast<float *>(p);
  auto take = [&](int64_t cols) {
    float *q = f;
    f += (t.n * cols + 63) / 64 * 64;
    return q;
  };
  s.dx = take(t.d);
  s.dx1 = take(t.d);
  s.dh = take(t.d);
  s.du = take(t.F);
  s.dout = take(t.Q);
  s.dqkv = take(t.QKV);
  s.dsum = take(t.H);
  s.red = f;
  s.red_bytes = red_bytes_of(t);
  return s;
}

size_t scratch_bytes(const TrainDims &t) {
  const int64_t cols = 3 * t.d + t.F + t.Q + t.QKV + t.H;
  return (max_gemm_ws(t) + 255) / 256 * 256 + size_t(t.n * cols + 64 * 7) * 4 + red_bytes_of(t) + 256;
}

struct Gemm {
  const Scratch &s;
  hipStream_t st;
  bool bf;  // bf16 operands and outputs (autocast), else fp32
  Epi with(Epi e) const {
    e.round = bf ? 1 : 0;
    return e;
  }
  // out[M, N] = alpha x[M, K] W[N, K]^T (+ the epilogue's terms)
  void nt(int64_t M, int64_t N, int64_t K, const float *x, const float *w, float *out, float beta = 0.f,
          const Epi &e = Epi{}) const {
    gemm_launch(int32_t(M), int32_t(N), int32_t(K), 1.f, x, K, 1, w, 1, K, beta, out, N, s.gemm_ws, s.gemm_bytes,
                with(e), st);
  }
  // out[M, K] = dy[M, N] W[N, K]
  void nn(int64_t M, int64_t N, int64_t K, const float *dy, const float *w, float *out, const Epi &e = Epi{}) const {
    gemm_launch(int32_t(M), int32_t(K), int32_t(N), 1.f, dy, N, 1, w, K, 1, 0.f, out, K, s.gemm_ws, s.gemm_bytes,
                with(e), st);
  }
  // out[N, K] = dy[M, N]^T x[M, K]; dbias[N] (when set) the column sums of dy
  void tn(int64_t M, int64_t N, int64_t K, const float *dy, const float *x, float *out, float *dbias = nullptr) const {
    Epi e;
    e.row_sum = dbias;
    gemm_launch(int32_t(N), int32_t(K), int32_t(M), 1.f, dy, 1, N, x, K, 1, 0.f, out, K, s.gemm_ws, s.gemm_bytes,
                with(e), st);
  }
};

// Scale of each repeat of a per-layer embedding over the model width (trunk.py:318-333).
float ple_scale(int64_t d, int64_t pd) { return pd == d ? 1.0f : 1.0f / std::sqrt(float((d + pd - 1) / pd)); }

cg_attn_train attn_args(const TrainDims &t, const int64_t *seq_start, const int32_t *seq_of, const float *qkv,
                        float *o, float *lse) {
  cg_attn_train a{};
  a.n = int32_t(t.n);
  a.H = int32_t(t.H);
  a.KVH = int32_t(t.KVH);
  a.head_dim = int32_t(t.D);
  a.scale = 1.0f / std::sqrt(float(t.D));
  a.seq_start = seq_start;
  a.seq_of = seq_of;
  a.q = qkv;
  a.k = qkv + t.Q;
  a.v = qkv + t.Q + t.KVW;
  a.ldq = a.ldk = a.ldv = t.QKV;
  a.o = o;
  a.lse = lse;
  a.round_bf16 = t.bf ? 1 : 0;
  return a;
}

}  // namespace

extern "C" {

size_t cg_train_saved_size(const cg_train_config *c, int32_t n) {
  if (!c || n <= 0) return 0;
  const TrainDims t = dims_of(*c, n);
  return size_t(t.L * layer_floats(t) + span_of(t, t.d) + 2 * span_of(t, 1)) * 4 + size_t(t.n) * 4 + 256;
}

size_t cg_train_scratch_size(const cg_train_config *c, int32_t n) {
  if (!c || n <= 0) return 0;
  return scratch_bytes(dims_of(*c, n));
}

int cg_trunk_train_forward(const cg_train_config *c, const cg_train_block *blocks, const float *final_w,
                           const float *final_b, const float *x, const float *ple, const float *values,
                           const int64_t *seq_start, int32_t n_seqs, int32_t n, float *hidden, void *saved,
                           size_t saved_size, void *scratch, size_t scratch_size, void *stream) {
  return guarded([&] {
    CG_REQUIRE(c && blocks && final_w && final_b && x && seq_start && hidden && saved && scratch, CG_ERR_INVALID,
               "training forward: missing operand");
    CG_REQUIRE(n > 0 && n_seqs > 0, CG_ERR_INVALID, "training forward: empty batch");
    CG_REQUIRE(saved_size >= cg_train_saved_size(c, n) && scratch_size >= cg_train_scratch_size(c, n),
               CG_ERR_INVALID, "training forward: buffers too small");
    CG_REQUIRE(aligned16(saved) && aligned16(scratch), CG_ERR_INVALID, "training forward: saved / scratch 16-byte aligned");
    CG_REQUIRE((c->ple_width == 0 || ple) && (c->value_width == 0 || values), CG_ERR_INVALID,
               "training forward: ple / values lookups are required");
    const TrainDims t = dims_of(*c, n);
    hipStream_t st = as_stream(stream);
    const Scratch s = scratch_of(t, scratch);
    const Gemm gm{s, st, t.bf};
    const SavedTail tail = saved_tail(t, saved);
    ok(cg_seq_of(seq_start, n_seqs, tail.seq_of, st));
    CG_HIP(hipMemcpyAsync(saved_layer(t, saved, 0).xl, x, size_t(t.n * t.d) * 4, hipMemcpyDeviceToDevice, st));
    for (int64_t l = 0; l < t.L; ++l) {
      const cg_train_block &w = blocks[l];
      const SavedLayer a = saved_layer(t, saved, l);
      float *x_next = l + 1 < t.L ? saved_layer(t, saved, l + 1).xl : tail.x_last;
      ok(cg_layernorm_fwd(a.xl, w.ln_attn_w, w.ln_attn_b, c->eps, a.h1, a.m1, a.r1, int32_t(t.n), int32_t(t.d), st));
      gm.nt(t.n, t.QKV, t.d, a.h1, w.qkv_w, a.qkv);
      const int32_t vi = c->value_index ? c->value_index[l] : -1;
      if (vi >= 0) {
        if (t.bf) {  // v = bf16(v + value embedding): the attention reads bf16 v
          add_round_kernel<<<grid_1d(t.n * t.KVW), 256, 0, st>>>(int32_t(t.n), int32_t(t.KVW), values + vi * t.KVW,
                                                                 t.V, a.qkv + t.Q + t.KVW, t.QKV);
          CG_LAUNCHED();
        } else {
          ok(cg_add_strided(int32_t(t.n), int32_t(t.KVW), 1.f, values + vi * t.KVW, t.V, a.qkv + t.Q + t.KVW, t.QKV,
                            st));
        }
      }
      const cg_attn_train at = attn_args(t, seq_start, tail.seq_of, a.qkv, a.o, a.lse);
      attn_fwd_launch(&at, t.bf, st);
      Epi res;  // x1 = xl + o W_out^T
      res.cin = a.xl;
      gm.nt(t.n, t.d, t.Q, a.o, w.out_w, a.x1, 1.f, res);
      ok(cg_layernorm_fwd(a.x1, w.ln_mlp_w, w.ln_mlp_b, c->eps, a.h2, a.m2, a.r2, int32_t(t.n), int32_t(t.d), st));
      Epi up;  // u = h2 W_up^T + b_up, g = gelu(u)
      up.bias = w.up_b;
      up.aux_out = a.g;
      up.mode = EPI_GELU;
      gm.nt(t.n, t.F, t.d, a.h2, w.up_w, a.u, 0.f, up);
      Epi down;  // x_next = x1 + g W_down^T + b_down
      down.cin = a.x1;
      down.bias = w.down_b;
      gm.nt(t.n, t.d, t.F, a.g, w.down_w, x_next, 1.f, down);
      if (ple) {
        ple_add_kernel<<<grid_1d(t.n * t.d), 256, 0, st>>>(int32_t(t.n), int32_t(t.d), int32_t(t.pd),
                                                           ple_scale(t.d, t.pd), ple + l * t.pd, t.P, x_next);
        CG_LAUNCHED();
      }
    }
    ok(cg_layernorm_fwd(tail.x_last, final_w, final_b, c->eps, hidden, tail.mf, tail.rf, int32_t(t.n),
                        int32_t(t.d), st));
  });
}

int cg_trunk_train_backward(const cg_train_config *c, const cg_train_block *blocks, const float *final_w,
                            const int64_t *seq_start, int32_t n, const float *dhidden, void *saved,
                            size_t saved_size, void *scratch, size_t scratch_size, const cg_train_grads *grads,
                            float *dx, float *dple, float *dvalues, void *stream) {
  return guarded([&] {
    CG_REQUIRE(c && blocks && final_w && seq_start && dhidden && saved && scratch && grads && dx, CG_ERR_INVALID,
               "training backward: missing operand");
    CG_REQUIRE(n > 0, CG_ERR_INVALID, "training backward: empty batch");
    CG_REQUIRE(saved_size >= cg_train_saved_size(c, n) && scratch_size >= cg_train_scratch_size(c, n),
               CG_ERR_INVALID, "training backward: buffers too small");
    CG_REQUIRE(aligned16(saved) && aligned16(scratch), CG_ERR_INVALID, "training backward: saved / scratch 16-byte aligned");
    const TrainDims t = dims_of(*c, n);
    hipStream_t st = as_stream(stream);
    const Scratch s = scratch_of(t, scratch);
    const Gemm gm{s, st, t.bf};
    const SavedTail tail = saved_tail(t, saved);
    const int32_t N = int32_t(t.n);
    ok(cg_norm_bwd(tail.x_last, dhidden, final_w, tail.mf, tail.rf, s.dx, nullptr, grads->final_dw,
                   grads->final_db, N, int32_t(t.d), s.red, s.red_bytes, 0, st));
    // Every layer writes its own columns of dple, and of dvalues where each slot has one layer; columns
    // that no layer writes, or several add to, start from zero.
    std::vector<int> users(size_t(t.V / std::max<int64_t>(t.KVW, 1)), 0);
    bool own_slots = t.V % t.KVW == 0;
    for (int64_t l = 0; l < t.L; ++l) {
      const int32_t vi = c->value_index ? c->value_index[l] : -1;
      if (vi >= 0 && size_t(vi) < users.size()) ++users[size_t(vi)];
    }
    for (int u : users) own_slots = own_slots && u == 1;
    auto zero = [&](float *p, int64_t cols) {
      zero_fill_kernel<<<grid_1d(t.n * cols), 256, 0, st>>>(p, t.n * cols);
      CG_LAUNCHED();
    };
    if (dple && t.P != t.L * t.pd) zero(dple, t.P);
    if (dvalues && !own_slots) zero(dvalues, t.V);
    for (int64_t l = t.L - 1; l >= 0; --l) {
      const cg_train_block &w = blocks[l];
      const cg_train_block_grads &gw = grads->blocks[l];
      const SavedLayer a = saved_layer(t, saved, l);
      if (dple) {
        ple_grad_kernel<<<grid_1d(t.n * t.pd), 256, 0, st>>>(N, int32_t(t.d), int32_t(t.pd), ple_scale(t.d, t.pd), s.dx,
                                                             dple + l * t.pd, t.P);
        CG_LAUNCHED();
      }
      gm.tn(t.n, t.d, t.F, s.dx, a.g, gw.down_w, gw.down_b);
      Epi dgelu;  // du = (dx W_down) gelu'(u)
      dgelu.aux_in = a.u;
      dgelu.mode = EPI_GELU_GRAD;
      gm.nn(t.n, t.d, t.F, s.dx, w.down_w, s.du, dgelu);
      gm.tn(t.n, t.F, t.d, s.du, a.h2, gw.up_w, gw.up_b);
      gm.nn(t.n, t.F, t.d, s.du, w.up_w, s.dh);
      ok(cg_norm_bwd(a.x1, s.dh, w.ln_mlp_w, a.m2, a.r2, s.dx1, s.dx, gw.ln_mlp_w, gw.ln_mlp_b, N, int32_t(t.d),
                     s.red, s.red_bytes, 0, st));
      gm.tn(t.n, t.d, t.Q, s.dx1, a.o, gw.out_w);
      gm.nn(t.n, t.d, t.Q, s.dx1, w.out_w, s.dout);
      const cg_attn_train at = attn_args(t, seq_start, tail.seq_of, a.qkv, a.o, a.lse);
      attn_bwd_launch(&at, s.dout, s.dsum, s.dqkv, s.dqkv + t.Q, s.dqkv + t.Q + t.KVW, t.bf, st, s.du,
                      t.n * t.F);  // (du has been used up)
      const int32_t vi = c->value_index ? c->value_index[l] : -1;
      if (vi >= 0 && dvalues) {
        const float *dv = s.dqkv + t.Q + t.KVW;
        if (own_slots) {
          copy_strided_kernel<<<grid_1d(t.n * t.KVW), 256, 0, st>>>(N, int32_t(t.KVW), dv, t.QKV, dvalues + vi * t.KVW, t.V);
          CG_LAUNCHED();
        } else {
          ok(cg_add_strided(N, int32_t(t.KVW), 1.f, dv, t.QKV, dvalues + vi * t.KVW, t.V, st));
        }
      }
      gm.tn(t.n, t.QKV, t.d, s.dqkv, a.h1, gw.qkv_w);
      gm.nn(t.n, t.QKV, t.d, s.dqkv, w.qkv_w, s.dh);
      ok(cg_norm_bwd(a.xl, s.dh, w.ln_attn_w, a.m1, a.r1, s.dx, s.dx1, gw.ln_attn_w, gw.ln_attn_b, N, int32_t(t.d),
                     s.red, s.red_bytes, 0, st));
    }
    CG_HIP(hipMemcpyAsync(dx, s.dx, size_t(t.n * t.d) * 4, hipMemcpyDeviceToDevice, st));
  });
}

}  // extern "C"
