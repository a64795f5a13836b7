// Host side of the score index (8-bit copy of the A_K rows used by the scan): binding to an A_K
// buffer, building / extending it, and the quantisation kernel.
#include <algorithm>

#include "common.hpp"
#include "ctx.hpp"
#include "prefill_pieces.hpp"

namespace lrqk {

// W of one head from a strided sample of at most kSidxSample of the rows [0, rows): second-moment
// matrix S of the sample (plus a small ridge), Cholesky factor S = L L^T, W = L^-T.  Two launches:
// kSidxParts workgroups per head sum their share of the sample (fixed order: reproducible), then
// one workgroup per head adds the parts and factors.  Anything degenerate (no rows, zero or
// non-finite S, a non-positive pivot) gives W = I.
constexpr int kSidxSample = 4096;
constexpr int kSidxParts = 16;  // workgroups per head in the first launch
typedef float sidx_v16f __attribute__((ext_vector_type(16)));

// Sums over a part's rows on the fp32 matrix pipe (32x32x2, two rows per product): lane (m, kh) holds element m of row
// 2 kk + kh as both operands, so the rows go from memory straight into the product, eight products' worth requested at
// a time.  Bound by the latency of those reads (a part is 256 rows): 158 us as 64-term chains on the vector ALUs with
// two LDS reads each, 18 us here, at 32 heads and R = 64.
template <typename T, int R>
__global__ __launch_bounds__(256) void score_index_moments_kernel(const T* __restrict__ a_k, int64_t head_stride,
                                                                  int64_t rows, float* __restrict__ part) {
  constexpr int NT = (R + 31) / 32, NP = NT * (NT + 1) / 2;  // 32-column tiles; tile pairs on and above the diagonal
  __shared__ float red[4][1024];
  const int h = blockIdx.y, p = blockIdx.x, tid = threadIdx.x;
  const int lane = lane_id(), wave = wave_id(), m = lane & 31, kh = lane >> 5;
  const T* A = a_k + (int64_t)h * head_stride;
  const int64_t step = rows > 0 ? (rows + kSidxSample - 1) / kSidxSample : 1;
  const int64_t n = rows > 0 ? (rows + step - 1) / step : 0;  // sample size
  const int64_t per = (n + kSidxParts - 1) / kSidxParts;
  const int64_t n0 = min(n, p * per), n1 = min(n, n0 + per);
  sidx_v16f acc[NP];
#pragma unroll
  for (int q = 0; q < NP; ++q)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[q][v] = 0.0f;
  constexpr int U = 8;  // products in flight: 16 rows of this wave
  for (int64_t t0 = n0 + wave * 2 * U; t0 < n1; t0 += 4 * 2 * U) {
    float x[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t t = t0 + 2 * u + kh;
#pragma unroll
      for (int c = 0; c < NT; ++c) {
        const float f = ld_f32<T>(A, min(t, n1 - 1) * step * R + min(32 * c + m, R - 1));
        x[u][c] = t < n1 && 32 * c + m < R ? f : 0.0f;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int c = 0; c < NT; ++c)
#pragma unroll
        for (int c2 = 0; c2 <= c; ++c2)
          acc[c * (c + 1) / 2 + c2] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[u][c2], x[u][c], acc[c * (c + 1) / 2 + c2], 0, 0, 0);
  }
  float* out = part + ((int64_t)h * kSidxParts + p) * R * R;
#pragma unroll
  for (int c = 0; c < NT; ++c)
#pragma unroll
    for (int c2 = 0; c2 <= c; ++c2) {
      __syncthreads();
#pragma unroll
      for (int v = 0; v < 16; ++v) red[wave][((v >> 2) * 8 + kh * 4 + (v & 3)) * 32 + m] = acc[c * (c + 1) / 2 + c2][v];
      __syncthreads();
      for (int x = tid; x < 1024; x += 256) {
        const int i = 32 * c2 + (x >> 5), j = 32 * c + (x & 31);
        if (i >= R || j >= R) continue;
        const float sum = (red[0][x] + red[1][x]) + (red[2][x] + red[3][x]);
        out[i * R + j] = sum;
        if (c != c2) out[j * R + i] = sum;
      }
    }
}

// L^-1 by elimination of [S | I]: step c scales row c of the right half by 1 / sqrt(pivot) and takes l_i times it (and
// l_i l_j on the left) off the rows below.  A thread of the 16 x 16 grid keeps rows ti + 16 a, columns tj + 16 b of both
// halves in registers; the pivot column and row go round through LDS, one barrier per step (Cholesky in LDS with three
// barriers per column and a substitution with one column per thread: 140 us at R = 64, 15 us at R = 16; 37 and 7 us here).
template <int R>
__global__ __launch_bounds__(256) void score_index_factor_kernel(const float* __restrict__ part, int64_t rows,
                                                                 float* __restrict__ wm) {
  constexpr int N = R / 16;
  __shared__ float colp[2][R];  // the pivot column of S
  __shared__ float rowx[2][R];  // the pivot row of the right half
  __shared__ float diag[R];
  const int h = blockIdx.x, tid = threadIdx.x;
  const int ti = tid >> 4, tj = tid & 15;
  float* W = wm + (int64_t)h * (R * R + R);
  const int64_t step = rows > 0 ? (rows + kSidxSample - 1) / kSidxSample : 1;
  const int64_t n = rows > 0 ? (rows + step - 1) / step : 0;
  const float inv_n = n > 0 ? 1.0f / (float)n : 0.0f;
  float S[N][N], X[N][N];
  const float* ph = part + (int64_t)h * kSidxParts * R * R;
#pragma unroll
  for (int a = 0; a < N; ++a)
#pragma unroll
    for (int b = 0; b < N; ++b) {
      const int x = (ti + 16 * a) * R + tj + 16 * b;
      float sum = 0.0f;
#pragma unroll
      for (int p = 0; p < kSidxParts; ++p) sum += ph[(int64_t)p * R * R + x];
      S[a][b] = sum * inv_n;
      X[a][b] = ti == tj && a == b ? 1.0f : 0.0f;
      if (ti == tj && a == b) diag[ti + 16 * a] = S[a][b];
    }
  __syncthreads();
  float tr = 0.0f;
  for (int i = 0; i < R; ++i) tr += diag[i];
  // (1 % of the mean diagonal: directions that hold next to nothing are not blown up to unit size, where their
  // quantisation step would only add slack to the bound; 12 % fewer rows to rescore than with 0.01 % on the 128K stream)
  const float ridge = 1e-2f * tr / (float)R;
  bool bad = !(tr > 0.0f && tr < INFINITY);
  if (ti == tj) {
#pragma unroll
    for (int a = 0; a < N; ++a) S[a][a] += ridge;
  }
#pragma unroll
  for (int k = 0; k < N; ++k) {
#pragma unroll 1
    for (int t = 0; t < 16; ++t) {
      const int c = 16 * k + t, buf = t & 1;  // (two slots: whoever passes a step's barrier has read the slot before)
      if (tj == t) {
#pragma unroll
        for (int a = 0; a < N; ++a) colp[buf][ti + 16 * a] = S[a][k];
      }
      if (ti == t) {
#pragma unroll
        for (int b = 0; b < N; ++b) rowx[buf][tj + 16 * b] = X[k][b];
      }
      __syncthreads();
      const float piv = colp[buf][c];
      bad = bad || !(piv > 0.0f && piv < INFINITY);
      const float inv = 1.0f / sqrtf(piv);
      float li[N], lj[N], xr[N];
#pragma unroll
      for (int a = 0; a < N; ++a) {
        li[a] = ti + 16 * a > c ? colp[buf][ti + 16 * a] * inv : 0.0f;
        lj[a] = colp[buf][tj + 16 * a] * inv;
        xr[a] = rowx[buf][tj + 16 * a] * inv;
      }
      if (ti == t) {
#pragma unroll
        for (int b = 0; b < N; ++b) X[k][b] = xr[b];
      }
#pragma unroll
      for (int a = 0; a < N; ++a)
#pragma unroll
        for (int b = 0; b < N; ++b) {
          S[a][b] = fmaf(-li[a], lj[b], S[a][b]);
          X[a][b] = fmaf(-li[a], xr[b], X[a][b]);
        }
    }
  }
#pragma unroll
  for (int a = 0; a < N; ++a)
#pragma unroll
    for (int b = 0; b < N; ++b) {
      const int i = ti + 16 * a, j = tj + 16 * b;
      if (j <= i) bad = bad || !(fabsf(X[a][b]) < INFINITY) || (i == j && !(X[a][b] > 0.0f));
    }
  const bool ident = __syncthreads_or(bad) != 0;
  // W[i][j] = L^-1[j][i] for i <= j, zero below the diagonal; then 1 / W_jj
#pragma unroll
  for (int a = 0; a < N; ++a)
#pragma unroll
    for (int b = 0; b < N; ++b) {
      const int j = ti + 16 * a, i = tj + 16 * b;
      W[i * R + j] = ident ? (i == j ? 1.0f : 0.0f) : (i <= j ? X[a][b] : 0.0f);
      if (i == j) W[R * R + j] = ident ? 1.0f : 1.0f / X[a][b];
    }
}

// One wave per row: lane i holds element i of the row, and column `lane` of W stays in registers.
template <typename T, int R>
__global__ __launch_bounds__(256) void score_index_build_kernel(const T* __restrict__ a_k, int64_t head_stride,
                                                                int64_t row0, int64_t row1, uint8_t* __restrict__ qa,
                                                                uint16_t* __restrict__ qs, const float* __restrict__ wm,
                                                                int64_t head_rows) {
  const int h = blockIdx.y;
  const int lane = lane_id();
  const int64_t wave0 = (int64_t)blockIdx.x * (blockDim.x / kWave) + wave_id();
  const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x / kWave);
  float wcol[R];
  score_index_load_wcol<R>(wm + (int64_t)h * (R * R + R), lane, wcol);
  for (int64_t row = row0 + wave0; row < row1; row += nwaves) {
    const float v = lane < R ? ld_f32<T>(a_k, (int64_t)h * head_stride + row * R + lane) : 0.0f;
    float scale;
    const uint8_t u = score_index_encode_row<R>(v, wcol, &scale);
    if (lane < R) qa[((int64_t)h * head_rows + row) * R + lane] = u;
    if (lane == 0) qs[(int64_t)h * head_rows + row] = sidx_scale_bits(scale);
  }
}

// Many rows at a time: C^T = W^T A^T on the matrix cores, and a second product on absolute values for g.  A lane's
// operand on the right is eight consecutive elements of one row as they lie in memory, and what it receives are 16 of
// the 32 columns of that row's a' (column 8 (v / 4) + 4 (lane / 32) + v % 4 in element v): the maxima over a row are
// taken in the lane, with one exchange between the wave's halves, and the codes leave as words of four.
// bf16 rows: W as three bf16 pieces (products exact in fp32), |W| for g rounded up to one piece; fp32 rows: the fp32
// pipe (32x32x2), a half of the wave taking a half of the row.  Any summation order inside the pipes
// stays within the rounding bound the scale charges for, and a g that is too large by 2^-7 only loosens it.
// Bound by HBM (a row read and R + 2 bytes written): 16384 rows of 64 elements, 32 heads: 101 MB in 46 us (253 us
// with a wave per row); 131072 rows of 32: 411 MB in 111 us (454 us with the rows on the other side of the product
// and two wave reductions per row).
template <typename T, int R>
__global__ __launch_bounds__(256) void score_index_build_rows_kernel(const T* __restrict__ a_k, int64_t head_stride,
                                                                     int64_t row0, int64_t row1, uint8_t* __restrict__ qa,
                                                                     uint16_t* __restrict__ qs, const float* __restrict__ wm,
                                                                     int64_t head_rows) {
  constexpr bool F32 = sizeof(T) == 4;
  constexpr int NT = (R + 31) / 32;               // 32-column tiles of a'
  constexpr int KB = F32 ? R / 2 : R / 16;        // products per tile (and piece)
  constexpr int NV = R < 32 ? R / 2 : 16;         // elements of a tile that a lane uses
  const int h = blockIdx.y;
  const int lane = lane_id(), m = lane & 31, kh = lane >> 5;
  const int64_t ngroups = (row1 - row0 + 31) / 32;
  const int64_t wave0 = (int64_t)blockIdx.x * (blockDim.x / kWave) + wave_id();
  const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x / kWave);
  const T* A = a_k + (int64_t)h * head_stride;
  const float* W = wm + (int64_t)h * (R * R + R);
  // left operands: row j = 32 t + m of W^T
  float wf[F32 ? NT : 1][F32 ? KB : 1];
  gd_bf16x8 wp[F32 ? 1 : NT][F32 ? 1 : KB][3], wg[F32 ? 1 : NT][F32 ? 1 : KB];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = min(32 * t + m, R - 1);
    const bool live = 32 * t + m < R;
    if constexpr (F32) {
#pragma unroll
      for (int k = 0; k < KB; ++k) wf[t][k] = live ? W[(kh * KB + k) * R + j] : 0.0f;
    } else {
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        float f[8];
        uint32_t g[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          f[q] = live ? W[(16 * k + 8 * kh + q) * R + j] : 0.0f;
          g[q] = __float_as_uint(fabsf(f[q]));
          g[q] += g[q] < 0x7f000000u ? 0xffffu : 0u;  // (truncated below: the next bf16 number up)
        }
        gd_split3x8(f, wp[t][k]);
        typedef uint32_t v4u __attribute__((ext_vector_type(4)));
        wg[t][k] = __builtin_bit_cast(gd_bf16x8, v4u{gd_pack2(g[0], g[1]), gd_pack2(g[2], g[3]), gd_pack2(g[4], g[5]),
                                                     gd_pack2(g[6], g[7])});
      }
    }
  }
  constexpr int NLD = F32 ? R / 8 : KB;  // 16-byte loads per lane and group
  gd_u32x4 pre[NLD];
  auto issue = [&](int64_t grp) {
    const T* src = A + min(row0 + grp * 32 + m, row1 - 1) * R;
#pragma unroll
    for (int c = 0; c < NLD; ++c)
      pre[c] = *reinterpret_cast<const gd_u32x4*>(src + (F32 ? kh * (R / 2) + 4 * c : 16 * c + 8 * kh));
  };
  if (wave0 < ngroups) issue(wave0);
  for (int64_t grp = wave0; grp < ngroups; grp += nwaves) {
    gd_u32x4 cur[NLD];
#pragma unroll
    for (int c = 0; c < NLD; ++c) cur[c] = pre[c];
    if (grp + nwaves < ngroups) issue(grp + nwaves);
    sidx_v16f acc[NT], accg[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[t][v] = accg[t][v] = 0.0f;
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        if constexpr (F32) {
          const float x = __uint_as_float(cur[k / 4][k % 4]);
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[t][k], x, acc[t], 0, 0, 0);
          accg[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(fabsf(wf[t][k]), fabsf(x), accg[t], 0, 0, 0);
        } else {
          const gd_bf16x8 x = __builtin_bit_cast(gd_bf16x8, cur[k]);
          const gd_bf16x8 xa = __builtin_bit_cast(gd_bf16x8, cur[k] & 0x7fff7fffu);
#pragma unroll
          for (int p = 2; p >= 0; --p) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wp[t][k][p], x, acc[t], 0, 0, 0);
          accg[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wg[t][k], xa, accg[t], 0, 0, 0);
        }
      }
    }
    float mx = 0.0f, gx = 0.0f;
    bool ok = true;  // false for NaN and infinity anywhere in the row
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        mx = fmaxf(mx, fabsf(acc[t][v]));
        gx = fmaxf(gx, accg[t][v]);
        ok = ok && accg[t][v] < INFINITY;
      }
    if (!ok) gx = INFINITY;
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    gx = fmaxf(gx, __shfl_xor(gx, 32, kWave));
    const float scale = score_index_scale(mx, gx, R);
    const float inv = 1.0f / scale;
    const int64_t row = row0 + grp * 32 + m;
    if (row < row1) {
      uint32_t* dst = reinterpret_cast<uint32_t*>(qa + ((int64_t)h * head_rows + row) * R);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int q = 0; q < NV / 4; ++q) {
          uint32_t w = 0;
#pragma unroll
          for (int b = 0; b < 4; ++b) w |= (uint32_t)score_index_code(acc[t][4 * q + b], inv) << (8 * b);
          dst[8 * t + 2 * q + kh] = w;
        }
      if (kh == 0) qs[(int64_t)h * head_rows + row] = sidx_scale_bits(scale);
    }
  }
}

template <typename T, int R>
static void launch_build(lrqk_ctx* ctx, const void* a_k, int64_t head_stride, int bh, int64_t from, int64_t upto,
                         int64_t head_rows, hipStream_t st) {
  float* wm = (float*)ctx->sidx_wm.p;
  if (from == 0) {  // first rows of this binding: they set W
    float* part = (float*)ctx->sidx_part.p;
    hipLaunchKernelGGL((score_index_moments_kernel<T, R>), dim3(kSidxParts, (unsigned)bh), dim3(256), 0, st,
                       (const T*)a_k, head_stride, upto, part);
    hipLaunchKernelGGL((score_index_factor_kernel<R>), dim3((unsigned)bh), dim3(256), 0, st, (const float*)part, upto, wm);
  }
  if (upto - from >= 32) {
    // (every wave loads and splits W: about four of its 32-row groups per wave, at most what the GPU holds at a time)
    const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>(std::max(1, 2048 / bh), (upto - from + 511) / 512));
    hipLaunchKernelGGL((score_index_build_rows_kernel<T, R>), dim3(blocks, (unsigned)bh), dim3(256), 0, st, (const T*)a_k,
                       head_stride, from, upto, (uint8_t*)ctx->sidx_qa.p, (uint16_t*)ctx->sidx_qs.p, wm, head_rows);
    return;
  }
  const unsigned blocks = (unsigned)std::min<int64_t>(2048, (upto - from + 3) / 4);
  hipLaunchKernelGGL((score_index_build_kernel<T, R>), dim3(blocks, (unsigned)bh), dim3(256), 0, st, (const T*)a_k,
                     head_stride, from, upto, (uint8_t*)ctx->sidx_qa.p, (uint16_t*)ctx->sidx_qs.p, wm, head_rows);
}

int score_index_prepare(lrqk_ctx* ctx, const void* a_k, int64_t head_stride, int bh, int64_t m, int r, int dtype,
                        hipStream_t st, ScoreIndexView* view) {
  if (!ctx->sidx_enabled) return 0;
  if (!(r == 16 || r == 32 || r == 64) || head_stride % r != 0 || ((uintptr_t)a_k % 16 != 0)) return 0;
  const int64_t head_rows = head_stride / r;
  if (m > head_rows) return 0;
  const bool bound = ctx->sidx_a_k == a_k && ctx->sidx_head_rows == head_rows && ctx->sidx_r == r &&
                     ctx->sidx_dtype == dtype && ctx->sidx_bh == bh;
  if (!bound) {
    int rc;
    ctx->sidx_a_k = nullptr;  // (a block that grows loses what was indexed, also where the next one is not to be had)
    if ((rc = ctx->sidx_qa.ensure((size_t)bh * head_rows * r))) return rc;
    if ((rc = ctx->sidx_qs.ensure((size_t)bh * head_rows * sizeof(uint16_t)))) return rc;
    if ((rc = ctx->sidx_wm.ensure((size_t)bh * (r * r + r) * sizeof(float)))) return rc;
    if ((rc = ctx->sidx_part.ensure((size_t)bh * kSidxParts * r * r * sizeof(float)))) return rc;
    ctx->sidx_a_k = a_k;
    ctx->sidx_head_rows = head_rows;
    ctx->sidx_r = r;
    ctx->sidx_dtype = dtype;
    ctx->sidx_bh = bh;
    ctx->sidx_valid = 0;
  }
  if (ctx->sidx_valid < m) {
    // index everything that is known to exist, so that the rows appended from now on stay contiguous
    const int64_t upto = std::min(head_rows, std::max(m, ctx->sidx_rows_hint));
    const int64_t from = ctx->sidx_valid;
#define LRQK_SIDX_BUILD(TT)                                                                   \
  (r == 16 ? launch_build<TT, 16>(ctx, a_k, head_stride, bh, from, upto, head_rows, st)       \
   : r == 32 ? launch_build<TT, 32>(ctx, a_k, head_stride, bh, from, upto, head_rows, st)     \
             : launch_build<TT, 64>(ctx, a_k, head_stride, bh, from, upto, head_rows, st))
    if (dtype == LRQK_F32)
      LRQK_SIDX_BUILD(float);
    else
      LRQK_SIDX_BUILD(bf16_t);
#undef LRQK_SIDX_BUILD
    LRQK_HIP_CHECK(hipGetLastError());
    ctx->sidx_valid = upto;
  }
  view->qa = (const uint8_t*)ctx->sidx_qa.p;
  view->qs = (const uint16_t*)ctx->sidx_qs.p;
  view->wm = (const float*)ctx->sidx_wm.p;
  view->head_rows = head_rows;
  return 1;
}

}  // namespace lrqk

using namespace lrqk;

extern "C" int lrqk_ctx_score_index(lrqk_ctx* ctx, int enable) {
  LRQK_REQUIRE(ctx != nullptr, LRQK_EINVAL, "ctx is null");
  ctx->sidx_enabled = enable != 0;
  ctx->sidx_a_k = nullptr;  // whatever was indexed is dropped; the next scan rebuilds what it needs
  ctx->sidx_valid = 0;
  ctx->sel_bh = 0;  // the bound a scan carries to the next one is in the units of the scan that made it
  return LRQK_OK;
}
