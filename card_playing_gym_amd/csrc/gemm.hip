// MFMA projections of the trunk with fused epilogues (gfx950).
//
// C[M, N] = A[M, K] . W[N, K]^T with fp32 accumulation; A and W are stored in the compute
// type (bf16 for the autocast path, fp32 otherwise: the split_* kernels).  The epilogue is one of:
//   * plain store (+bias) or GELU(+bias) store (mlp[0] + nn.GELU, trunk.py:139);
//   * the QKV split that writes q and appends k / v (+ value embedding) straight into the
//     KV pool at each token's slot (trunk.py:141-152 followed by KVCache.write_step,
//     kv_cache.py:84-105) -- the append costs no separate pass over K/V;
//   * residual add into the fp32 stream (+bias, + the per-layer embedding of
//     Trunk._add_ple, trunk.py:318-333), optionally followed by the LayerNorm of the
//     updated row (the next ln_mlp / ln_attn, trunk.py:154-160): with full-row tiles the
//     epilogue owns whole rows, so the norm costs no extra launch or re-read.
//
// bf16 main loop: the workgroup stages 128-byte-wide K chunks of its A rows and W rows in LDS
// (16-byte coalesced global loads, double-buffered: chunk k+1 is in flight while chunk k
// feeds the MFMAs).  Fragments: lane l supplies row (l % 16) of a 16-row A tile and column
// (l % 16) of a 16-column W tile, eight consecutive k values from 8 (l / 16); A and W use
// the same lane -> k assignment, so every k is summed once (v_mfma_f32_16x16x32_bf16).
// The 16x16 fp32 result sits in lane l as rows 4 (l / 16) + r, r < 4, column l % 16.
#include <algorithm>

#include "common.h"
#include "gemm.h"
#include "split_tile.h"

namespace cg {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

constexpr int CHUNK_BYTES = 128;                // K bytes per row per staged chunk
constexpr int LDS_ROW = CHUNK_BYTES + 16;        // padded LDS row (bytes)
constexpr int VPR = CHUNK_BYTES / 16;            // 16-byte vectors per row chunk

template <int BM, int BN, int WM, int WN, int EPI>
__global__ __launch_bounds__(64 * WM * WN) void gemm_kernel(GemmArgs g) {
  constexpr int THREADS = 64 * WM * WN;
  constexpr int ES = 2;
  constexpr int KC = CHUNK_BYTES / ES;  // elements per chunk
  constexpr int VA = (BM * VPR + THREADS - 1) / THREADS;
  constexpr int VW = (BN * VPR + THREADS - 1) / THREADS;
  constexpr int FM = BM / WM / 16, FN = BN / WN / 16;
  static_assert(FM >= 1 && FN >= 1, "tile too small for the wave layout");
  __shared__ __align__(16) unsigned char smem[2 * (BM + BN) * LDS_ROW];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int li = lane & 15, lg = lane >> 4;
  const char *A = static_cast<const char *>(g.A);
  const char *W = static_cast<const char *>(g.W);
  const int64_t lda_b = g.lda * ES, ldw_b = int64_t(g.K) * ES;
  const int k_bytes = g.K * ES;
  const int nchunks = (g.K + KC - 1) / KC;

  uint4 ra[VA], rw[VW];
  auto gload = [&](int kc) {
    const int kb0 = kc * CHUNK_BYTES;
#pragma unroll
    for (int i = 0; i < VA; ++i) {
      const int v = tid + i * THREADS;
      uint4 val = {0u, 0u, 0u, 0u};
      const int r = v / VPR, kb = kb0 + (v % VPR) * 16;
      if (v < BM * VPR && m0 + r < g.M && kb < k_bytes)
        val = *reinterpret_cast<const uint4 *>(A + int64_t(m0 + r) * lda_b + kb);
      ra[i] = val;
    }
#pragma unroll
    for (int i = 0; i < VW; ++i) {
      const int v = tid + i * THREADS;
      uint4 val = {0u, 0u, 0u, 0u};
      const int r = v / VPR, kb = kb0 + (v % VPR) * 16;
      if (v < BN * VPR && n0 + r < g.N && kb < k_bytes)
        val = *reinterpret_cast<const uint4 *>(W + int64_t(n0 + r) * ldw_b + kb);
      rw[i] = val;
    }
  };
  auto sstore = [&](int buf) {
    unsigned char *base = smem + buf * (BM + BN) * LDS_ROW;
#pragma unroll
    for (int i = 0; i < VA; ++i) {
      const int v = tid + i * THREADS;
      if (v < BM * VPR) *reinterpret_cast<uint4 *>(base + (v / VPR) * LDS_ROW + (v % VPR) * 16) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < VW; ++i) {
      const int v = tid + i * THREADS;
      if (v < BN * VPR)
        *reinterpret_cast<uint4 *>(base + (BM + v / VPR) * LDS_ROW + (v % VPR) * 16) = rw[i];
    }
  };

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](int buf) {
    const unsigned char *base = smem + buf * (BM + BN) * LDS_ROW;
#pragma unroll
    for (int ks = 0; ks < KC / 32; ++ks) {
      const int kb = (ks * 32 + 8 * lg) * ES;
      bf16x8 af[FM], wf[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i)
        af[i] = *reinterpret_cast<const bf16x8 *>(base + (wm * FM * 16 + i * 16 + li) * LDS_ROW + kb);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        wf[j] = *reinterpret_cast<const bf16x8 *>(base + (BM + wn * FN * 16 + j * 16 + li) * LDS_ROW + kb);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], wf[j], acc[i][j], 0, 0, 0);
    }
  };

  gload(0);
  sstore(0);
  __syncthreads();
  for (int kc = 0; kc < nchunks; ++kc) {
    const bool more = kc + 1 < nchunks;
    if (more) gload(kc + 1);
    compute(kc & 1);
    if (more) sstore((kc + 1) & 1);
    __syncthreads();
  }

  // ---- epilogue ------------------------------------------------------------------------
  if constexpr (EPI == EPI_RESID || EPI == EPI_RESID_LN) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + wn * FN * 16 + j * 16 + li;
      const bool n_ok = n < g.N;
      const float bias = (n_ok && g.bias) ? g.bias[n] : 0.f;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + wm * FM * 16 + i * 16 + 4 * lg + r;
          float x = 0.f;
          if (n_ok && m < g.M) {
            x = acc[i][j][r] + bias;
            if (g.ple) x = fmaf(g.ple[int64_t(m) * g.ld_ple + g.ple_off + n % g.ple_dim], g.ple_scale, x);
            float *dst = g.resid + int64_t(m) * g.ldr + n;
            x += *dst;
            *dst = x;
          }
          acc[i][j][r] = x;
        }
    }
    if constexpr (EPI == EPI_RESID_LN) {
      // Row statistics: lanes with the same (l / 16) hold the same 4 rows of a tile; their
      // 16 columns reduce by shuffles, then the WN column slices meet in LDS.
      float *red = reinterpret_cast<float *>(smem);  // [2][WN][BM]
      float mean[FM][4], rstd[FM][4];
#pragma unroll
      for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
              const int n = n0 + wn * FN * 16 + j * 16 + li;
              const float v = acc[i][j][r];
              const float d = pass == 0 ? v : v - mean[i][r];
              s += n < g.N ? (pass == 0 ? d : d * d) : 0.f;
            }
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o, 64);
            if (li == 0) red[(pass * WN + wn) * BM + wm * FM * 16 + i * 16 + 4 * lg + r] = s;
          }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = wm * FM * 16 + i * 16 + 4 * lg + r;
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < WN; ++w) s += red[(pass * WN + w) * BM + row];
            if (pass == 0) mean[i][r] = s / float(g.N);
            else rstd[i][r] = rsqrtf(s / float(g.N) + g.eps);
          }
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = n0 + wn * FN * 16 + j * 16 + li;
        if (n >= g.N) continue;
        const float w = g.ln_w[n], b = g.ln_b[n];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int m = m0 + wm * FM * 16 + i * 16 + 4 * lg + r;
            if (m >= g.M) continue;
            const float y = fmaf((acc[i][j][r] - mean[i][r]) * rstd[i][r], w, b);
            const int64_t o = int64_t(m) * g.ldo + n;
            if (g.out_dtype == CG_BF16) static_cast<bf16 *>(g.out)[o] = from_f32<bf16>(y);
            else static_cast<float *>(g.out)[o] = y;
          }
      }
    }
    return;
  }

  const int kvw = g.kv_heads * g.head_dim;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int n = n0 + wn * FN * 16 + j * 16 + li;
    if (n >= g.N) continue;
    const float bias = g.bias ? g.bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm * FM * 16 + i * 16 + 4 * lg + r;
        if (m >= g.M) continue;
        const float c = acc[i][j][r] + bias;
        if constexpr (EPI == EPI_STORE || EPI == EPI_GELU || EPI == EPI_SCALE_ADD) {
          float v = c;
          if constexpr (EPI == EPI_GELU) v = gelu_erf(c);
          if constexpr (EPI == EPI_SCALE_ADD) {
            const float cc = g.round_c ? to_f32(from_f32<bf16>(c)) : c;
            const int64_t ai = int64_t(m) * g.ld_add + n;
            if (g.add_dtype == CG_BF16) {
              const float sum = to_f32(from_f32<bf16>(cc + to_f32(static_cast<const bf16 *>(g.addend)[ai])));
              v = to_f32(from_f32<bf16>(sum * g.scale));
            } else {
              v = (cc + static_cast<const float *>(g.addend)[ai]) * g.scale;
            }
          }
          const int64_t o = int64_t(m) * g.ldo + n;
          if (g.out_dtype == CG_BF16) static_cast<bf16 *>(g.out)[o] = from_f32<bf16>(v);
          else static_cast<float *>(g.out)[o] = v;
        } else {  // EPI_QKV
          if (n < g.q_cols) {
            static_cast<float *>(g.out)[int64_t(m) * g.ldo + n] = c;
          } else {
            const int row = g.tok_row[m];
            if (row < 0) continue;
            const bool is_v = n >= g.q_cols + kvw;
            const int kv = n - g.q_cols - (is_v ? kvw : 0);
            const int h = kv / g.head_dim, d = kv % g.head_dim;
            float v = c;
            if (is_v && g.vemb_off >= 0) v += g.vemb[int64_t(m) * g.ld_vemb + g.vemb_off + kv];
            const int64_t dst =
                ((int64_t(row) * g.kv_heads + h) * g.max_len + g.tok_pos[m]) * g.head_dim + d;
            void *base = is_v ? g.vc : g.kc;
            if (g.kv_dtype == CG_BF16) static_cast<bf16 *>(base)[dst] = from_f32<bf16>(v);
            else if (g.kv_dtype == CG_F16) static_cast<f16 *>(base)[dst] = from_f32<f16>(v);
            else static_cast<float *>(base)[dst] = v;
          }
        }
      }
    }
  }
}

// (C + addend) * scale with the addend's rounding (EPI_SCALE_ADD).
__device__ __forceinline__ float scale_add(const GemmArgs &g, float c, float addend) {
  if (g.round_c) c = to_f32(from_f32<bf16>(c));
  if (g.add_dtype != CG_BF16) return (c + addend) * g.scale;
  return to_f32(from_f32<bf16>(to_f32(from_f32<bf16>(c + addend)) * g.scale));
}

// ---- fp32 products of few rows -----------------------------------------------------------
// What bounds a decode wave's product is latency, not rate: 64 rows x 1024 x 256 is 1 MB of
// weights and 0.03 GFLOP.  So the k of one small output tile is spread over the WK waves of a
// block (32 k a step, waves taking steps in turn), every wave reads its operand fragments
// straight from global memory (lane (li, lg) row li, k 8 lg .. 8 lg + 7: 128 contiguous bytes
// per row and step, no staging and no barrier per step) and multiplies them in three bf16
// parts (split.h); the WK partial tiles meet in LDS, added in a fixed order.  With `LN` the
// rows of A are normalised on the way in (every wave holds its k of the tile's rows, so the
// statistics cost one exchange through LDS), which saves the whole-row tiles, and the launches,
// that a LayerNorm in the producer's epilogue needs.
constexpr int SPLIT_LN_K = 256;  // widest A row that a block normalises by itself

template <int BM, int BN, int WK, int EPI, bool LN>
__global__ __launch_bounds__(64 * WK) void split_rows_kernel(GemmArgs g) {
  constexpr int THREADS = 64 * WK;
  constexpr int FM = BM / 16, FN = BN / 16;
  constexpr int PITCH = BN + 4;  // the four row groups of a wave's stores start 16 banks apart
  constexpr int LN_STEPS = LN ? SPLIT_LN_K / 32 / WK : 1;
  __shared__ float red[WK][BM * PITCH];
  __shared__ float stat[LN ? 2 : 1][LN ? WK : 1][LN ? BM : 1];
  __shared__ float norm[LN ? 2 : 1][LN ? BM : 1];
  const int tid = threadIdx.x, lane = tid & 63, wk = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const float *arow[FM], *wrow[FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
    arow[i] = static_cast<const float *>(g.A) + int64_t(min(m0 + i * 16 + li, g.M - 1)) * g.lda + 8 * lg;
#pragma unroll
  for (int j = 0; j < FN; ++j)
    wrow[j] = static_cast<const float *>(g.W) + int64_t(min(n0 + j * 16 + li, g.N - 1)) * g.K + 8 * lg;
  const split_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // One lane's eight values of step s (K is a multiple of 8: all of them or none are inside).
  auto load = [&](const float *row, int s, split_f32x4 (&v)[2]) {
    const bool in = 32 * s + 8 * lg < g.K;
    const float *p = row + (in ? 32 * s : -8 * lg);
    const split_f32x4 x = *reinterpret_cast<const split_f32x4 *>(p), y = *reinterpret_cast<const split_f32x4 *>(p + 4);
    v[0] = in ? x : zero;
    v[1] = in ? y : zero;
  };
  split_f32x4 acc[FM][FN], cor[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = cor[i][j] = zero;
  auto multiply = [&](const split_f32x4 (&a)[FM][2], const split_f32x4 (&b)[FN][2]) {
    Split8 as[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) as[i] = split8(a[i][0], a[i][1]);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const Split8 bs = split8(b[j][0], b[j][1]);
#pragma unroll
      for (int i = 0; i < FM; ++i) split_mma(as[i], bs, acc[i][j], cor[i][j]);
    }
  };
  const int steps = (g.K + 31) / 32;
  if constexpr (LN) {
    split_f32x4 a[LN_STEPS][FM][2], b[FN][2], lw[LN_STEPS][2], lb[LN_STEPS][2];
#pragma unroll
    for (int t = 0; t < LN_STEPS; ++t) {
#pragma unroll
      for (int i = 0; i < FM; ++i) load(arow[i], wk + t * WK, a[t][i]);
      load(g.a_ln_w + 8 * lg, wk + t * WK, lw[t]);
      load(g.a_ln_b + 8 * lg, wk + t * WK, lb[t]);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) load(wrow[j], wk, b[j]);
    // The wave's own k of each row: exact two-pass mean and centred squares, then Chan et al.'s
    // pairwise merge over the WK waves.
    auto held = [&](int w) {  // how many k wave w holds of a row
      int c = 0;
#pragma unroll
      for (int t = 0; t < LN_STEPS; ++t) c += max(0, min(32, g.K - 32 * (w + t * WK)));
      return c;
    };
    const int count = held(wk);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      float s = 0.f;
#pragma unroll
      for (int t = 0; t < LN_STEPS; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) s += a[t][i][0][e] + a[t][i][1][e];
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      const float mean = count ? s / float(count) : 0.f;
      float q = 0.f;
#pragma unroll
      for (int t = 0; t < LN_STEPS; ++t) {
        if (32 * (wk + t * WK) + 8 * lg >= g.K) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float c0 = a[t][i][0][e] - mean, c1 = a[t][i][1][e] - mean;
          q = fmaf(c0, c0, fmaf(c1, c1, q));
        }
      }
      q += __shfl_xor(q, 16);
      q += __shfl_xor(q, 32);
      if (lg == 0) {
        stat[0][wk][i * 16 + li] = mean;
        stat[1][wk][i * 16 + li] = q;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int r = i * 16 + li;
      float mean = 0.f, q = 0.f;
#pragma unroll
      for (int w = 0; w < WK; ++w) mean += stat[0][w][r] * float(held(w));
      mean /= float(g.K);
#pragma unroll
      for (int w = 0; w < WK; ++w) {
        const float off = stat[0][w][r] - mean;
        q += stat[1][w][r] + off * off * float(held(w));
      }
      const float rstd = rsqrtf(q / float(g.K) + g.a_eps);
      if (wk == 0 && lg == 0) {
        norm[0][r] = mean;
        norm[1][r] = rstd;
      }
#pragma unroll
      for (int t = 0; t < LN_STEPS; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) a[t][i][h][e] = fmaf((a[t][i][h][e] - mean) * rstd, lw[t][h][e], lb[t][h][e]);
    }
    // (Lanes past K hold zero gain and bias, so zero.)
#pragma unroll
    for (int t = 0; t < LN_STEPS; ++t) {
      split_f32x4 nb[FN][2];
      if (t + 1 < LN_STEPS)
#pragma unroll
        for (int j = 0; j < FN; ++j) load(wrow[j], wk + (t + 1) * WK, nb[j]);
      multiply(a[t], b);
      if (t + 1 < LN_STEPS)
#pragma unroll
        for (int j = 0; j < FN; ++j) b[j][0] = nb[j][0], b[j][1] = nb[j][1];
    }
  } else {
    // DEPTH steps' operands in flight at once (one round trip to memory for k <= 1024).
    constexpr int DEPTH = FM * FN == 1 ? 4 : 2;
    for (int s0 = wk; s0 < steps; s0 += WK * DEPTH) {
      split_f32x4 a[DEPTH][FM][2], b[DEPTH][FN][2];
#pragma unroll
      for (int t = 0; t < DEPTH; ++t) {
        if (s0 + t * WK >= steps) continue;
#pragma unroll
        for (int i = 0; i < FM; ++i) load(arow[i], s0 + t * WK, a[t][i]);
#pragma unroll
        for (int j = 0; j < FN; ++j) load(wrow[j], s0 + t * WK, b[t][j]);
      }
#pragma unroll
      for (int t = 0; t < DEPTH; ++t)
        if (s0 + t * WK < steps) multiply(a[t], b[t]);
    }
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[wk][(i * 16 + 4 * lg + r) * PITCH + j * 16 + li] = acc[i][j][r] + cor[i][j][r];
  __syncthreads();
  // A thread's results, then everything their epilogue reads at once, then the epilogue: read
  // element by element, each load waited for the store before it (a 1024-row fp32 decode step of
  // 41 launches: 550 us, 539 so).
  constexpr int E = (BM * BN + THREADS - 1) / THREADS;
  float v[E];
  int mr[E], nc[E];
  bool ok[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int at = min(tid + e * THREADS, BM * BN - 1), r = at / BN, c = at % BN, m = m0 + r, n = n0 + c;
    ok[e] = tid + e * THREADS < BM * BN && m < g.M && n < g.N;
    mr[e] = min(m, g.M - 1);
    nc[e] = min(n, g.N - 1);
    v[e] = red[0][r * PITCH + c];
#pragma unroll
    for (int w = 1; w < WK; ++w) v[e] += red[w][r * PITCH + c];
    if (__builtin_expect(ok[e] & !split_holds(v[e]), 0)) {  // see split.h
      const float *ar = static_cast<const float *>(g.A) + int64_t(m) * g.lda;
      const float *wr = static_cast<const float *>(g.W) + int64_t(n) * g.K;
      CarriedSum sum;
#pragma unroll 1
      for (int k = 0; k < g.K; ++k) {
        float x = ar[k];
        if constexpr (LN) x = fmaf((x - norm[0][r]) * norm[1][r], g.a_ln_w[k], g.a_ln_b[k]);
        sum.add(x * wr[k]);
      }
      v[e] = sum.value();
    }
  }
  if (g.bias) {
    float bias[E];
#pragma unroll
    for (int e = 0; e < E; ++e) bias[e] = g.bias[nc[e]];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] += bias[e];
  }
  if constexpr (EPI == EPI_RESID) {
    if (g.ple) {
      float p[E];
#pragma unroll
      for (int e = 0; e < E; ++e) p[e] = g.ple[int64_t(mr[e]) * g.ld_ple + g.ple_off + nc[e] % g.ple_dim];
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = fmaf(p[e], g.ple_scale, v[e]);
    }
    float x[E];
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = g.resid[int64_t(mr[e]) * g.ldr + nc[e]];
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (ok[e]) g.resid[int64_t(mr[e]) * g.ldr + nc[e]] = x[e] + v[e];
  } else if constexpr (EPI == EPI_QKV) {
    const int kvw = g.kv_heads * g.head_dim;
    int row[E], pos[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      row[e] = g.tok_row[mr[e]];
      pos[e] = g.tok_pos[mr[e]];
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (!ok[e]) continue;
      const int m = mr[e], n = nc[e];
      if (n < g.q_cols) {
        static_cast<float *>(g.out)[int64_t(m) * g.ldo + n] = v[e];
        continue;
      }
      if (row[e] < 0) continue;
      const bool is_v = n >= g.q_cols + kvw;
      const int kv = n - g.q_cols - (is_v ? kvw : 0);
      const int h = kv / g.head_dim, d = kv % g.head_dim;
      float c = v[e];
      if (is_v && g.vemb_off >= 0) c += g.vemb[int64_t(m) * g.ld_vemb + g.vemb_off + kv];
      const int64_t dst = ((int64_t(row[e]) * g.kv_heads + h) * g.max_len + pos[e]) * g.head_dim + d;
      void *base = is_v ? g.vc : g.kc;
      if (g.kv_dtype == CG_BF16) static_cast<bf16 *>(base)[dst] = from_f32<bf16>(c);
      else if (g.kv_dtype == CG_F16) static_cast<f16 *>(base)[dst] = from_f32<f16>(c);
      else static_cast<float *>(base)[dst] = c;
    }
  } else {
    if constexpr (EPI == EPI_GELU) {
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = gelu_erf(v[e]);
    }
    if constexpr (EPI == EPI_SCALE_ADD) {
      float x[E];
      if (g.add_dtype == CG_BF16) {
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = to_f32(static_cast<const bf16 *>(g.addend)[int64_t(mr[e]) * g.ld_add + nc[e]]);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = static_cast<const float *>(g.addend)[int64_t(mr[e]) * g.ld_add + nc[e]];
      }
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = scale_add(g, v[e], x[e]);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (!ok[e]) continue;
      const int64_t o = int64_t(mr[e]) * g.ldo + nc[e];
      if (g.out_dtype == CG_BF16) static_cast<bf16 *>(g.out)[o] = from_f32<bf16>(v[e]);
      else static_cast<float *>(g.out)[o] = v[e];
    }
  }
}

// ---- fp32 products of many rows -----------------------------------------------------------
template <int TM, int EPI>
__global__ __launch_bounds__(256, 2) void split_tile_kernel(GemmArgs g) {
  constexpr int FM = TM / 32;
  __shared__ __align__(16) char lds[tile_lds_bytes<TM, 3, 1>()];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1, li = lane & 15, lg = lane >> 4;
  // XCD k (block ids = k mod 8) takes a contiguous run of tiles, N fastest, so the rows of A it
  // reads stay in its own L2.
  const int tiles = gridDim.x * gridDim.y, b = blockIdx.x + gridDim.x * blockIdx.y;
  const int xcd = b & 7, per = tiles >> 3, extra = tiles & 7;
  const int t = xcd * per + min(xcd, extra) + (b >> 3);
  const int m0 = t / int(gridDim.x) * TM, n0 = t % int(gridDim.x) * ST_N;
  const float *A = static_cast<const float *>(g.A), *W = static_cast<const float *>(g.W);
  split_f32x4 acc[FM][4];
  tile_product<1, 1, TM, 3, 1>(A + int64_t(m0) * g.lda, g.lda, 1, g.M - m0, W + int64_t(n0) * g.K, 1, g.K, g.N - n0, 0,
                               g.K, lds, acc);
  const int mw = m0 + wm * (TM / 2), nw = n0 + wn * 64;
  tile_repair<FM>(acc, A, g.lda, 1, W, 1, g.K, mw, nw, g.M, g.N, g.K);
  // Everything the epilogue reads is loaded for a 16-row block at once, from clamped addresses.
  const int kvw = g.kv_heads * g.head_dim;
  int nj[4];
  bool nok[4];
  float bias[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = nw + j * 16 + li;
    nok[j] = n < g.N;
    nj[j] = min(n, g.N - 1);
    bias[j] = g.bias ? g.bias[nj[j]] : 0.f;
  }
  const bool f32_out = g.out_dtype == CG_F32;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    int64_t mr[4];
    bool ok[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = mw + i * 16 + 4 * lg + r;
      ok[r] = m < g.M;
      mr[r] = min(m, g.M - 1);
    }
    float c[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) c[j][r] = acc[i][j][r] + bias[j];
    if constexpr (EPI == EPI_RESID) {
      float x[4][4], e[4][4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x[j][r] = g.resid[mr[r] * g.ldr + nj[j]];
          e[j][r] = g.ple ? g.ple[mr[r] * g.ld_ple + g.ple_off + nj[j] % g.ple_dim] : 0.f;
        }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (nok[j] && ok[r])
            g.resid[mr[r] * g.ldr + nj[j]] = x[j][r] + (g.ple ? fmaf(e[j][r], g.ple_scale, c[j][r]) : c[j][r]);
    } else if constexpr (EPI == EPI_QKV) {
      int64_t row[4], slot[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        row[r] = ok[r] ? g.tok_row[mr[r]] : -1;
        slot[r] = g.tok_pos[mr[r]];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (!nok[j]) continue;
        if (nj[j] < g.q_cols) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (ok[r]) static_cast<float *>(g.out)[mr[r] * g.ldo + nj[j]] = c[j][r];
          continue;
        }
        const bool is_v = nj[j] >= g.q_cols + kvw;
        const int kv = nj[j] - g.q_cols - (is_v ? kvw : 0);
        const int h = kv / g.head_dim, d = kv % g.head_dim;
        if (is_v && g.vemb_off >= 0) {
          float e[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) e[r] = g.vemb[mr[r] * g.ld_vemb + g.vemb_off + kv];
#pragma unroll
          for (int r = 0; r < 4; ++r) c[j][r] += e[r];
        }
        void *base = is_v ? g.vc : g.kc;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (row[r] < 0) continue;
          const int64_t dst = ((row[r] * g.kv_heads + h) * g.max_len + slot[r]) * g.head_dim + d;
          if (g.kv_dtype == CG_BF16) static_cast<bf16 *>(base)[dst] = from_f32<bf16>(c[j][r]);
          else if (g.kv_dtype == CG_F16) static_cast<f16 *>(base)[dst] = from_f32<f16>(c[j][r]);
          else static_cast<float *>(base)[dst] = c[j][r];
        }
      }
    } else if constexpr (EPI == EPI_SCALE_ADD) {
      float e[4][4];
      if (g.add_dtype == CG_BF16) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) e[j][r] = to_f32(static_cast<const bf16 *>(g.addend)[mr[r] * g.ld_add + nj[j]]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) e[j][r] = static_cast<const float *>(g.addend)[mr[r] * g.ld_add + nj[j]];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (!nok[j] || !ok[r]) continue;
          const float v = scale_add(g, c[j][r], e[j][r]);
          const int64_t o = mr[r] * g.ldo + nj[j];
          if (f32_out) static_cast<float *>(g.out)[o] = v;
          else static_cast<bf16 *>(g.out)[o] = from_f32<bf16>(v);
        }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = EPI == EPI_GELU ? gelu_erf(c[j][r]) : c[j][r];
          if (!nok[j] || !ok[r]) continue;
          const int64_t o = mr[r] * g.ldo + nj[j];
          if (f32_out) static_cast<float *>(g.out)[o] = v;
          else static_cast<bf16 *>(g.out)[o] = from_f32<bf16>(v);
        }
    }
  }
}

enum SplitTile : int { SPLIT_16, SPLIT_32, SPLIT_32x64, SPLIT_TILE_64, SPLIT_TILE_128 };

// Which kernel a fp32 product takes.  16 x 16 tiles of split_rows_kernel while they are two per
// CU or fewer (64 x 256 x 1024: 7.1 us, 32 x 32 tiles 10.5; 512 x 256 x 1024: both 10.9), 32 x 32
// tiles up to four per CU (1024 x 256 x 1024: 12.2 us, 16 x 16 19.6, the 64-row staged tiles 36.9;
// 1024 x 1024 x 256: 15.3 against 17.8; from two per CU and up to k = 256, 32 x 64 tiles with k over
// four waves convert half as much: 12.3), the staged tiles beyond (2048 x 1024 x 256: 26 us in
// 32 x 32 tiles, 18.5 staged; at four per CU and k = 1024 they lead as well, 36 against 42).
// Staged tiles are 128 rows high when that gives two per CU (16384 x 1024 x 256: 76 against
// 84 us), else 64 (16384 x 256 x 1024: 67 against 69).
// (Rows too long for the staged tiles' 32-bit offsets keep the 32 x 32 ones.)
SplitTile split_tile_of(int32_t m, int32_t n, int32_t k, int64_t lda) {
  auto tiles = [&](int64_t tm, int64_t tn) { return ((m + tm - 1) / tm) * ((n + tn - 1) / tn); };
  if (tiles(16, 16) <= 512) return SPLIT_16;
  const int64_t t32 = tiles(32, 32);
  if (t32 > 512 && t32 <= 1024 && k <= SPLIT_LN_K && n >= 64 && lda == k) return SPLIT_32x64;
  if (t32 < 1024 || std::max<int64_t>(k, lda) > TILE_MAX_STRIDE) return SPLIT_32;
  return tiles(128, 128) >= 512 ? SPLIT_TILE_128 : SPLIT_TILE_64;
}

template <int EPI, bool LN>
void launch_split_tile(const GemmArgs &g, hipStream_t s) {
  const SplitTile tile = split_tile_of(g.M, g.N, g.K, g.lda);
  const int tm = tile == SPLIT_16 ? 16 : tile <= SPLIT_32x64 ? 32 : tile == SPLIT_TILE_64 ? 64 : 128;
  const int tn = tile <= SPLIT_32 ? tm : tile == SPLIT_32x64 ? 64 : ST_N;
  const dim3 grid((g.N + tn - 1) / tn, (g.M + tm - 1) / tm);
  CG_REQUIRE(grid.y <= 65535u, CG_ERR_UNSUPPORTED, "too many rows for one launch");
  if (tile == SPLIT_16) {
    split_rows_kernel<16, 16, 8, EPI, LN><<<grid, 512, 0, s>>>(g);
  } else if (tile == SPLIT_32) {
    split_rows_kernel<32, 32, 8, EPI, LN><<<grid, 512, 0, s>>>(g);
  } else if (tile == SPLIT_32x64) {
    split_rows_kernel<32, 64, 4, EPI, LN><<<grid, 256, 0, s>>>(g);
  } else {
    CG_REQUIRE(!LN, CG_ERR_UNSUPPORTED, "the staged product takes rows that are already normalised");
    if (tile == SPLIT_TILE_64) split_tile_kernel<64, EPI><<<grid, 256, 0, s>>>(g);
    else split_tile_kernel<128, EPI><<<grid, 256, 0, s>>>(g);
  }
  CG_LAUNCHED();
}

void launch_split(const GemmArgs &g, hipStream_t s) {
  CG_REQUIRE(!g.a_ln_w || split_gemm_norms(g.M, g.N, g.K, g.a_ln_w, g.a_ln_b), CG_ERR_UNSUPPORTED,
             "this product does not normalise its rows");
  switch (g.epi) {
    case EPI_STORE:
      return launch_split_tile<EPI_STORE, false>(g, s);
    case EPI_GELU:
      if (g.a_ln_w) return launch_split_tile<EPI_GELU, true>(g, s);
      return launch_split_tile<EPI_GELU, false>(g, s);
    case EPI_RESID:
      return launch_split_tile<EPI_RESID, false>(g, s);
    case EPI_QKV:
      if (g.a_ln_w) return launch_split_tile<EPI_QKV, true>(g, s);
      return launch_split_tile<EPI_QKV, false>(g, s);
    case EPI_SCALE_ADD:
      return launch_split_tile<EPI_SCALE_ADD, false>(g, s);
  }
  throw Error(CG_ERR_INVALID, "no such fp32 epilogue");
}

// Tile shapes: 64x64 (2x2 waves of 32x32) for the wide projections, 16 rows x 256
// columns (4 waves side by side) when the epilogue needs whole rows.
template <int EPI>
void launch_tile(const GemmArgs &g, hipStream_t s) {
  dim3 grid((g.N + 63) / 64, (g.M + 63) / 64);
  CG_REQUIRE(grid.y <= 65535u, CG_ERR_UNSUPPORTED, "too many rows for one launch");
  gemm_kernel<64, 64, 2, 2, EPI><<<grid, 256, 0, s>>>(g);
  CG_LAUNCHED();
}

template <int EPI>
void launch_rows(const GemmArgs &g, hipStream_t s) {
  dim3 grid(1, (g.M + 15) / 16);
  CG_REQUIRE(grid.y <= 65535u, CG_ERR_UNSUPPORTED, "too many rows for one launch");
  gemm_kernel<16, 256, 1, 4, EPI><<<grid, 256, 0, s>>>(g);
  CG_LAUNCHED();
}

void launch_bf16(const GemmArgs &g, hipStream_t s) {
  switch (g.epi) {
    case EPI_STORE:
      return launch_tile<EPI_STORE>(g, s);
    case EPI_GELU:
      return launch_tile<EPI_GELU>(g, s);
    case EPI_RESID:
      if (g.N <= 256) return launch_rows<EPI_RESID>(g, s);
      return launch_tile<EPI_RESID>(g, s);
    case EPI_QKV:
      return launch_tile<EPI_QKV>(g, s);
    case EPI_SCALE_ADD:
      return launch_tile<EPI_SCALE_ADD>(g, s);
    case EPI_RESID_LN:
      CG_REQUIRE(g.N <= 256, CG_ERR_UNSUPPORTED, "fused residual LayerNorm needs d_model <= 256");
      return launch_rows<EPI_RESID_LN>(g, s);
  }
  throw Error(CG_ERR_INVALID, "unknown epilogue");
}

// One wave per row; every lane's loads are issued before the reductions.
template <int PER_LANE>
__global__ __launch_bounds__(256) void layernorm_rows_kernel(const float *__restrict__ x,
                                                             const int32_t *__restrict__ index,
                                                             const float *__restrict__ w,
                                                             const float *__restrict__ b, float eps,
                                                             void *__restrict__ y, int32_t y_dtype,
                                                             int32_t n, int32_t d) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= n) return;
  const int src = index ? index[row] : row;
  float v[PER_LANE];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < PER_LANE; ++i) {
    const int k = lane + 64 * i;
    v[i] = (src >= 0 && k < d) ? x[int64_t(src) * d + k] : 0.f;
    s += v[i];
  }
  const float mean = wave_sum(s) / float(d);
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < PER_LANE; ++i) {
    const int k = lane + 64 * i;
    const float t = k < d ? v[i] - mean : 0.f;
    q = fmaf(t, t, q);
  }
  const float rstd = rsqrtf(wave_sum(q) / float(d) + eps);
#pragma unroll
  for (int i = 0; i < PER_LANE; ++i) {
    const int k = lane + 64 * i;
    if (k >= d) continue;
    const float out = src >= 0 ? fmaf((v[i] - mean) * rstd, w[k], b[k]) : 0.f;
    const int64_t o = int64_t(row) * d + k;
    if (y_dtype == CG_BF16) static_cast<bf16 *>(y)[o] = from_f32<bf16>(out);
    else static_cast<float *>(y)[o] = out;
  }
}

// The same for d a multiple of 4 up to 256 and 16-byte aligned rows: a lane holds four consecutive
// columns of a row, a wave four rows with all their loads in flight (16384 x 256: 9.1 -> 8.6 us).
__global__ __launch_bounds__(256) void layernorm_rows4_kernel(const float *__restrict__ x,
                                                              const int32_t *__restrict__ index,
                                                              const float *__restrict__ w,
                                                              const float *__restrict__ b, float eps,
                                                              void *__restrict__ y, int32_t y_dtype, int32_t n,
                                                              int32_t d) {
  const int row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 4, k = 4 * (threadIdx.x & 63);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  const bool in = k < d;
  f32x4 v[4];
  int src[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = min(row0 + r, n - 1);
    src[r] = index ? index[row] : row;
    v[r] = src[r] >= 0 && in ? *reinterpret_cast<const f32x4 *>(x + int64_t(src[r]) * d + k) : zero;
  }
  const f32x4 g = in ? *reinterpret_cast<const f32x4 *>(w + k) : zero, o = in ? *reinterpret_cast<const f32x4 *>(b + k) : zero;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float mean = wave_sum((v[r][0] + v[r][1]) + (v[r][2] + v[r][3])) / float(d);
    float q = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float t = in ? v[r][e] - mean : 0.f;
      q = fmaf(t, t, q);
    }
    const float rstd = rsqrtf(wave_sum(q) / float(d) + eps);
    if (row0 + r >= n || !in) continue;
    f32x4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = src[r] >= 0 ? fmaf((v[r][e] - mean) * rstd, g[e], o[e]) : 0.f;
    const int64_t at = int64_t(row0 + r) * d + k;
    if (y_dtype == CG_BF16) *reinterpret_cast<u32x2 *>(static_cast<bf16 *>(y) + at) = cvt4<bf16>(out);
    else *reinterpret_cast<f32x4 *>(static_cast<float *>(y) + at) = out;
  }
}

__global__ void convert_kernel(const float *__restrict__ x, void *__restrict__ y, int32_t dtype, int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    if (dtype == CG_BF16) static_cast<bf16 *>(y)[i] = from_f32<bf16>(x[i]);
    else static_cast<float *>(y)[i] = x[i];
  }
}

}  // namespace

void launch_gemm(const GemmArgs &g, hipStream_t s) {
  CG_REQUIRE(g.M >= 0 && g.N > 0 && g.K > 0, CG_ERR_INVALID, "GEMM sizes must be positive");
  CG_REQUIRE(g.K % 8 == 0, CG_ERR_UNSUPPORTED, "GEMM inner size must be a multiple of 8");
  CG_REQUIRE(g.lda % 8 == 0, CG_ERR_UNSUPPORTED, "GEMM row stride must be a multiple of 8");
  CG_REQUIRE((reinterpret_cast<uintptr_t>(g.A) | reinterpret_cast<uintptr_t>(g.W)) % 16 == 0,
             CG_ERR_INVALID, "GEMM operands must be 16-byte aligned");
  if (g.M == 0) return;
  if (g.compute == CG_BF16) return launch_bf16(g, s);
  CG_REQUIRE(g.compute == CG_F32, CG_ERR_INVALID, "compute dtype must be CG_F32 or CG_BF16");
  launch_split(g, s);
}

bool split_gemm_norms(int32_t m, int32_t n, int32_t k, const float *w, const float *b) {
  return k <= SPLIT_LN_K && ((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(b)) & 15) == 0 &&
         split_tile_of(m, n, k, k) <= SPLIT_32x64;
}

void launch_layernorm_rows(const float *x, const int32_t *index, const float *w, const float *b,
                           float eps, void *y, int32_t y_dtype, int32_t n, int32_t d,
                           hipStream_t s) {
  if (n <= 0) return;
  const unsigned grid = unsigned((n + 3) / 4);
  const uintptr_t at = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(b) |
                       reinterpret_cast<uintptr_t>(y);
  if (d <= 256 && d % 4 == 0 && (at & 15) == 0)
    layernorm_rows4_kernel<<<unsigned((int64_t(n) + 15) / 16), 256, 0, s>>>(x, index, w, b, eps, y, y_dtype, n, d);
  else if (d <= 256) layernorm_rows_kernel<4><<<grid, 256, 0, s>>>(x, index, w, b, eps, y, y_dtype, n, d);
  else if (d <= 512) layernorm_rows_kernel<8><<<grid, 256, 0, s>>>(x, index, w, b, eps, y, y_dtype, n, d);
  else if (d <= 1024) layernorm_rows_kernel<16><<<grid, 256, 0, s>>>(x, index, w, b, eps, y, y_dtype, n, d);
  else throw Error(CG_ERR_UNSUPPORTED, "LayerNorm width above 1024");
  CG_LAUNCHED();
}

void launch_convert(const float *x, void *y, int32_t dtype, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  convert_kernel<<<unsigned(blocks), 256, 0, s>>>(x, y, dtype, n);
  CG_LAUNCHED();
}

}  // namespace cg

using namespace cg;

extern "C" int cg_linear(const float *x, const float *w, const float *bias, float *y, int32_t m,
                         int32_t n, int32_t k, int32_t act, int32_t compute_dtype, void *stream) {
  return guarded([&] {
    CG_REQUIRE(act == CG_ACT_NONE || act == CG_ACT_GELU, CG_ERR_INVALID, "unknown activation");
    if (m == 0) return;
    CG_REQUIRE(x && w && y, CG_ERR_INVALID, "x, w and y are required");
    CG_REQUIRE(compute_dtype == CG_F32 || compute_dtype == CG_BF16, CG_ERR_INVALID,
               "compute dtype must be CG_F32 or CG_BF16");
    GemmArgs g{};
    g.M = m;
    g.N = n;
    g.K = k;
    g.compute = CG_F32;  // fp32 operands: the product is exact fp32 whatever compute_dtype asks
    g.A = x;
    g.lda = k;
    g.W = w;
    g.bias = bias;
    g.epi = act == CG_ACT_GELU ? EPI_GELU : EPI_STORE;
    g.out = y;
    g.out_dtype = CG_F32;
    g.ldo = n;
    launch_gemm(g, as_stream(stream));
  });
}

extern "C" int cg_linear_add_scale(const float *x, const float *w, const void *addend, int32_t addend_dtype,
                                   float *y, int32_t m, int32_t n, int32_t k, float scale,
                                   int32_t compute_dtype, void *stream) {
  return guarded([&] {
    if (m == 0) return;
    CG_REQUIRE(x && w && addend && y, CG_ERR_INVALID, "x, w, addend and y are required");
    CG_REQUIRE(compute_dtype == CG_F32 || compute_dtype == CG_BF16, CG_ERR_INVALID,
               "compute dtype must be CG_F32 or CG_BF16");
    CG_REQUIRE(addend_dtype == CG_F32 || addend_dtype == CG_BF16, CG_ERR_INVALID,
               "addend dtype must be CG_F32 or CG_BF16");
    GemmArgs g{};
    g.M = m;
    g.N = n;
    g.K = k;
    g.compute = CG_F32;
    g.A = x;
    g.lda = k;
    g.W = w;
    g.epi = EPI_SCALE_ADD;
    g.addend = addend;
    g.add_dtype = addend_dtype;
    g.round_c = compute_dtype == CG_BF16;
    g.ld_add = n;
    g.scale = scale;
    g.out = y;
    g.out_dtype = CG_F32;
    g.ldo = n;
    launch_gemm(g, as_stream(stream));
  });
}
