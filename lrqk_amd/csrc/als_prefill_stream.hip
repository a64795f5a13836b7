// The passes over the long axis for the prefill iterations on Gram matrices (the sums of rows of 128 at ranks up to 32 are in
// als_prefill_gram.hip).
//
//   sums   S = X^T X, and over given factors A the sums G = A^T A, C = A^T X
//   apply  A = X M
//
// All on the bf16 matrix cores (32x32x16) with fp32 accuracy: an fp32 operand is the exact sum of three bf16 pieces, a
// product of two pieces is exact in fp32, and all piece pairs but lo x lo (2^-32) are formed.  Both are bound by HBM
// (every input read once), so the shape of the kernels follows the memory: a wave streams 32-row groups of its own
// through a private LDS tile, the next group already requested, and never meets another wave before the end.
// 32 heads of 16384 bf16 rows of 128, rank 64: all sums 193 us (435 MB; two waves' worth of matrix-core and vector work
// on one wave per SIMD, which the accumulators leave room for), A_K 42 us; the row-by-row kernels for this rank took
// 1.3 ms per pass, ten passes for four iterations.
#include <algorithm>

#include "common.hpp"
#include "ctx.hpp"
#include "prefill_pieces.hpp"

namespace lrqk {

constexpr int kStWaves = 4, kStThreads = kStWaves * kWave;

__device__ __forceinline__ void st_wave_sync() {  // orders one wave's LDS writes and reads
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// a x b over piece pairs, smallest first (PB = 1: a bf16 operand as it is), two k blocks, into a fresh accumulator:
// the matrix cores do not round to nearest when they add to a large one, so a 32-row group's sum joins the running
// total by ordinary fp32 additions.
template <int PA, int PB>
__device__ __forceinline__ gd_floatx16 st_product(const gd_bf16x8 (&a)[2][PA], const gd_bf16x8 (&b)[2][PB]) {
  gd_floatx16 t;
#pragma unroll
  for (int v = 0; v < 16; ++v) t[v] = 0.0f;
#pragma unroll
  for (int w = PA + PB - 2; w >= 0; --w)  // (a piece of index p is 2^-8p of its number)
#pragma unroll
    for (int i = PA - 1; i >= 0; --i) {
      const int j = w - i;
      if (j < 0 || j >= PB || (PA == 3 && PB == 3 && w == 4)) continue;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kb][i], b[kb][j], t, 0, 0, 0);
    }
  return t;
}

constexpr int st_sums_smem(int db) {  // bytes of LDS: the waves' tiles, or their sums on the way out
  const int tile = 32 * (32 * db + 16) * (int)sizeof(bf16_t);
  return kStWaves * (tile > 4096 ? tile : 4096);
}

// AT: 32-column tiles of A (ranks up to 32, 64); DB: 32-column blocks of X (64, 128 elements); GIVEN: sums over the
// given factors, a head per query head (X of its kv head); XTX: X^T X, a head per head of X.  Both from one reading of X
// where the accumulators allow it (DB = 2: up to 10 tiles; DB = 4 would need 15 to 21 of 16 registers each beside the
// operands), else by workgroups of their own.
// Split s of S of head h; 4 waves; a split takes every S-th set of 4 x 32 rows, so the workgroups of a head walk its
// rows side by side.  part: [head][S][r][r + d]; xtx_part: [head][S][d][d] (both triangles).
template <int AT, int DB, bool GIVEN, bool XTX>
__device__ __forceinline__ void st_sums_body(char* smem, int h, int s, const bf16_t* __restrict__ X, int xh, int hq,
                                             int64_t l, int r, const float* __restrict__ A, float* __restrict__ part,
                                             float* __restrict__ xtx_part, int S) {
  constexpr int D = 32 * DB;
  constexpr int VEC = Vec16<bf16_t>::N;
  constexpr int LDX = D + 16;  // elements per row of the LDS tile: the transposing reads want successive rows 8 banks apart
  constexpr int NL = 32 * D / (kWave * VEC);
  constexpr int SMEM = st_sums_smem(DB);
  const int tid = threadIdx.x, lane = lane_id(), wave = gd_wave();
  const int col = lane & 31, half = lane >> 5;
  uint16_t* x_s = reinterpret_cast<uint16_t*>(smem + wave * (SMEM / kStWaves));
  const int64_t xhead = GIVEN ? (int64_t)(h / hq) * xh + (h % hq) / (hq / xh) : h;
  const bf16_t* Xh = X + xhead * l * D;
  const float* Ah = A + (int64_t)h * l * r;

  constexpr int NAA = AT * (AT + 1) / 2, NXX = DB * (DB + 1) / 2;
  gd_floatx16 gAA[GIVEN ? NAA : 1], gAX[GIVEN ? AT : 1][GIVEN ? DB : 1], gXX[XTX ? NXX : 1];
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    if constexpr (GIVEN) {
#pragma unroll
      for (int i = 0; i < NAA; ++i) gAA[i][v] = 0.0f;
#pragma unroll
      for (int i = 0; i < AT; ++i)
#pragma unroll
        for (int n = 0; n < DB; ++n) gAX[i][n][v] = 0.0f;
    }
    if constexpr (XTX) {
#pragma unroll
      for (int i = 0; i < NXX; ++i) gXX[i][v] = 0.0f;
    }
  }

  gd_u32x4 pre[NL];
  float arow[GIVEN ? AT : 1][16];
  auto issue = [&](int64_t t0) {
    const int last = (int)min((int64_t)32, l - t0) - 1;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = (i * kWave + lane) * VEC;
      pre[i] = gd_at<gd_u32x4>(Xh + t0 * D, (uint32_t)(min(e / D, last) * D + e % D) * 2u);
    }
    if constexpr (GIVEN) {
#pragma unroll
      for (int at = 0; at < AT; ++at)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          arow[at][v] = gd_factor(Ah + t0 * r, gd_mfma_row(lane, v), last, r, min(32 * at + col, r - 1));
    }
  };
  const int64_t stride = (int64_t)S * kStWaves * 32;
  const int64_t first = ((int64_t)s * kStWaves + wave) * 32;
  if (first < l) issue(first);
  for (int64_t t0 = first; t0 < l; t0 += stride) {
    const int rows = (int)min((int64_t)32, l - t0);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = (i * kWave + lane) * VEC;
      *reinterpret_cast<gd_u32x4*>(&x_s[(e / D) * LDX + e % D]) = e / D < rows ? pre[i] : gd_u32x4{0, 0, 0, 0};
    }
    // the pieces of this group's rows of A: element v of a lane is row gd_mfma_row(lane, v) of its column, so eight at
    // a time are an operand's k elements (X comes out of LDS in the same order)
    gd_bf16x8 cp[GIVEN ? AT : 1][2][3];
    if constexpr (GIVEN) {
#pragma unroll
      for (int at = 0; at < AT; ++at) {
        const int valid = (32 * at + col < r ? rows : 0) - 4 * half;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          float f[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) f[q] = gd_mfma_row0(8 * kb + q) < valid ? arow[at][8 * kb + q] : 0.0f;
          gd_split3x8(f, cp[at][kb]);
        }
      }
    }
    st_wave_sync();
    if (t0 + stride < l) issue(t0 + stride);
    // rows 16 kb + 4 half .. + 3 and the same + 8 of column 32 nb + col
    auto operand = [&](int nb, gd_bf16x8 (&x)[2][1]) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int s16 = lane & 15;
        const uint16_t* p = x_s + (16 * kb + 4 * half + (s16 >> 2)) * LDX + 32 * nb + (col & 16) + 4 * (s16 & 3);
        const gd_v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gd_lds_v4s)p);
        const gd_v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gd_lds_v4s)(p + 8 * LDX));
        x[kb][0] = __builtin_bit_cast(gd_bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    if constexpr (GIVEN) {
#pragma unroll
      for (int ta = 0; ta < AT; ++ta)
#pragma unroll
        for (int tb = ta; tb < AT; ++tb) {
          const gd_floatx16 t = st_product<3, 3>(cp[ta], cp[tb]);
#pragma unroll
          for (int v = 0; v < 16; ++v) gAA[ta + tb][v] += t[v];
        }
    }
    gd_bf16x8 xb[XTX ? DB : 1][2][1];
#pragma unroll
    for (int nb = 0; nb < DB; ++nb) {
      gd_bf16x8(&x)[2][1] = xb[XTX ? nb : 0];
      operand(nb, x);
      if constexpr (GIVEN) {
#pragma unroll
        for (int at = 0; at < AT; ++at) {
          const gd_floatx16 t = st_product<3, 1>(cp[at], x);
#pragma unroll
          for (int v = 0; v < 16; ++v) gAX[at][nb][v] += t[v];
        }
      }
      if constexpr (XTX) {
#pragma unroll
        for (int n2 = 0; n2 <= nb; ++n2) {
          const gd_floatx16 t = st_product<1, 1>(xb[n2], x);
#pragma unroll
          for (int v = 0; v < 16; ++v) gXX[nb * (nb + 1) / 2 + n2][v] += t[v];
        }
      }
    }
    st_wave_sync();  // this wave's reads of the tile precede its next staging writes
  }
  // the four waves' tiles, one at a time: f(row, column, sum)
  float* sm = reinterpret_cast<float*>(smem);
  auto reduce = [&](const gd_floatx16& acc, auto&& f) {
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 16; ++v) sm[wave * 1024 + gd_mfma_row(lane, v) * 32 + col] = acc[v];
    __syncthreads();
#pragma unroll
    for (int o = tid; o < 1024; o += kStThreads)
      f(o >> 5, o & 31, (sm[o] + sm[1024 + o]) + (sm[2048 + o] + sm[3072 + o]));
  };
  if constexpr (GIVEN) {
    const int ld = r + D;
    float* out = part + ((int64_t)h * S + s) * r * ld;
#pragma unroll
    for (int ta = 0; ta < AT; ++ta) {
#pragma unroll
      for (int tb = ta; tb < AT; ++tb)
        reduce(gAA[ta + tb], [&](int m, int n, float v) {
          m += 32 * ta;
          n += 32 * tb;
          if (m < r && n < r) {
            out[m * ld + n] = v;
            if (ta != tb) out[n * ld + m] = v;
          }
        });
#pragma unroll
      for (int nb = 0; nb < DB; ++nb)
        reduce(gAX[ta][nb], [&](int m, int n, float v) {
          if (32 * ta + m < r) out[(32 * ta + m) * ld + r + 32 * nb + n] = v;
        });
    }
  }
  if constexpr (XTX) {
    float* out = xtx_part + ((int64_t)h * S + s) * D * D;
#pragma unroll
    for (int nb = 0; nb < DB; ++nb)
#pragma unroll
      for (int n2 = 0; n2 <= nb; ++n2)
        reduce(gXX[nb * (nb + 1) / 2 + n2], [&](int m, int n, float v) {
          out[(32 * n2 + m) * D + 32 * nb + n] = v;
          if (n2 != nb) out[(32 * nb + n) * D + 32 * n2 + m] = v;
        });
  }
}

// The sums of both sides in one launch: one after the other they were up to four, 15 us each of a short prompt's host
// time, and each with a last round of workgroups that left most of the GPU idle (three prompts of 2531 rows of 64:
// 44 -> 27 us; rank 64, 16K rows: 237 -> 193).  Workgroups in order: Q's sums over the given factors [bh * S], K's
// [bh * S], Q^T Q [bh * S], K^T K [bkv * Sxk]; FUSED_Q / FUSED_K: the side's X^T X comes with its sums.
struct StSums {
  const bf16_t *q, *k;
  const float *a_q, *a_k;
  float *part_q, *part_k, *xq_part, *xk_part;
  int64_t l;
  int hq, hkv, r, S, Sxk, given;  // given: workgroups of one side's sums over the given factors
};
template <int AT, int DB, bool FUSED_Q, bool FUSED_K>
__global__ __launch_bounds__(kStThreads) void pf_stream_sums_kernel(StSums g) {
  __shared__ __align__(16) char smem[st_sums_smem(DB)];
  const bf16_t *q = g.q, *k = g.k;
  int w = blockIdx.x;
  if (w < g.given) {
    st_sums_body<AT, DB, true, FUSED_Q>(smem, w / g.S, w % g.S, q, g.hq, g.hq, g.l, g.r, g.a_q, g.part_q, g.xq_part, g.S);
    return;
  }
  w -= g.given;
  if (w < g.given) {
    st_sums_body<AT, DB, true, FUSED_K>(smem, w / g.S, w % g.S, k, g.hkv, g.hq, g.l, g.r, g.a_k, g.part_k, g.xk_part, g.S);
    return;
  }
  w -= g.given;
  if constexpr (!FUSED_Q) {
    if (w < g.given) {
      st_sums_body<1, DB, false, true>(smem, w / g.S, w % g.S, q, g.hq, g.hq, g.l, g.r, nullptr, nullptr, g.xq_part, g.S);
      return;
    }
    w -= g.given;
  }
  if constexpr (!FUSED_K)
    st_sums_body<1, DB, false, true>(smem, w / g.Sxk, w % g.Sxk, k, g.hkv, g.hq, g.l, g.r, nullptr, nullptr, g.xk_part,
                                        g.Sxk);
}

// A = X M for every query head (its kv head's X): M^T (fp32, [head][r][d]) in LDS as three bf16 pieces, X through the
// wave's private tile.  One launch for both sides (a cache asks for one row of A_Q: alone that is a launch and 8 us), whose
// workgroups alternate where both have as many; else the second side's come last.  The query heads that share a kv head's
// rows lie eight workgroups apart, on one XCD, and walk the same rows at the same time.
// Bound by HBM.  32 heads (8 kv heads), us: 32K rows of 128 at rank 32, both sides 100 (470 MB) -- A_K from rows staged for
// four heads at a time and A_Q in launches of their own: 48 + 64; A_K and one row of A_Q 45 (42 + 8); 16K rows at rank 64 42
// (59 with the heads of a kv head wherever they fell).  With M's pieces in registers and more, smaller workgroups: 106 for 100.
template <typename OUT>
struct StApply {
  const bf16_t* x;
  int S;              // splits of the rows
  int64_t l, x_stride;  // rows; elements between the heads of x
  const float* mt;
  OUT* a;             // heads a_stride elements apart, rows of r
  int64_t a_stride;
  int nh, pairs, chunks;  // heads that share a head of x (one, or as many as the launch's other side has at most); pairs of a
                          // head of x and a split; chunks of workgroups
};
constexpr int kStApplyWaves = 8;
template <int AT, int DB, typename OUT>
__global__ __launch_bounds__(kStApplyWaves * kWave) void pf_stream_apply_kernel(StApply<OUT> first_side,
                                                                               StApply<OUT> second_side, int r) {
  constexpr int D = 32 * DB;
  constexpr int NW = kStApplyWaves, NT = NW * kWave;
  constexpr int VEC = Vec16<bf16_t>::N;
  constexpr int LDM = D + 8, LDX = D + 8;  // (16-byte operand reads want rows 4 banks apart)
  constexpr int NL = 32 * D / (kWave * VEC);
  extern __shared__ __align__(16) char ap_smem[];
  uint16_t* mt_s = reinterpret_cast<uint16_t*>(ap_smem);                                 // [3][32 AT][LDM]
  const int tid = threadIdx.x, lane = lane_id(), wave = gd_wave();
  uint16_t* x_s = mt_s + 3 * 32 * AT * LDM + wave * 32 * LDX;                            // this wave's rows of X
  const int col = lane & 31, half = lane >> 5;
  // (unit workgroups, chunk): a chunk has eight (head of x, split) pairs side by side, then the same eight for the next head
  // that shares x
  const bool turns = first_side.chunks == second_side.chunks;
  const bool second = turns ? blockIdx.y & 1 : (int)blockIdx.y >= first_side.chunks;
  const StApply<OUT>& g = second ? second_side : first_side;
  const int chunk = turns ? blockIdx.y >> 1 : (int)blockIdx.y - (second ? first_side.chunks : 0);
  const int nh = g.nh, S = g.S;
  const int pair = nh == 1 ? chunk * (int)gridDim.x + (int)blockIdx.x : chunk * 8 + (int)(blockIdx.x & 7);
  if (pair >= g.pairs) return;
  const int xhead = (int)((uint32_t)pair / (uint32_t)S), s = pair - xhead * S;
  const int h = nh == 1 ? xhead : xhead * nh + (int)(blockIdx.x >> 3);
  const int64_t l = g.l;
  const float* __restrict__ Mt = g.mt;
  const bf16_t* __restrict__ Xh = g.x + (int64_t)xhead * g.x_stride;
  OUT* __restrict__ Ah = g.a + (int64_t)h * g.a_stride;
  for (int e = tid; e < 32 * AT * D; e += NT) {
    const int n = e / D, k = e % D;
    const float v = n < r ? Mt[((int64_t)h * r + n) * D + k] : 0.0f;
    uint32_t p0, p1, p2;
    gd_split3(v, p0, p1, p2);
    mt_s[(0 * 32 * AT + n) * LDM + k] = (uint16_t)(p0 >> 16);
    mt_s[(1 * 32 * AT + n) * LDM + k] = (uint16_t)(p1 >> 16);
    mt_s[(2 * 32 * AT + n) * LDM + k] = (uint16_t)(p2 >> 16);
  }
  gd_u32x4 pre[NL];
  auto issue = [&](int64_t t0) {
    const int last = (int)min((int64_t)32, l - t0) - 1;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = (i * kWave + lane) * VEC;
      pre[i] = gd_at<gd_u32x4>(Xh + t0 * D, (uint32_t)(min(e / D, last) * D + e % D) * 2u);
    }
  };
  const int64_t stride = (int64_t)S * NW * 32;
  const int64_t first = ((int64_t)s * NW + wave) * 32;
  if (first < l) issue(first);
  __syncthreads();  // M staged
  for (int64_t t0 = first; t0 < l; t0 += stride) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = (i * kWave + lane) * VEC;
      *reinterpret_cast<gd_u32x4*>(&x_s[(e / D) * LDX + e % D]) = pre[i];  // (rows beyond l are never stored from)
    }
    st_wave_sync();
    if (t0 + stride < l) issue(t0 + stride);
    gd_floatx16 c[AT];
#pragma unroll
    for (int at = 0; at < AT; ++at)
#pragma unroll
      for (int v = 0; v < 16; ++v) c[at][v] = 0.0f;
#pragma unroll
    for (int kb = 0; kb < D / 16; ++kb) {
      const gd_bf16x8 xa = *reinterpret_cast<const gd_bf16x8*>(&x_s[col * LDX + 16 * kb + 8 * half]);
#pragma unroll
      for (int at = 0; at < AT; ++at) {
        gd_bf16x8 m[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          m[p] = *reinterpret_cast<const gd_bf16x8*>(&mt_s[(p * 32 * AT + 32 * at + col) * LDM + 16 * kb + 8 * half]);
#pragma unroll
        for (int p = 2; p >= 0; --p) c[at] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa, m[p], c[at], 0, 0, 0);
      }
    }
#pragma unroll
    for (int at = 0; at < AT; ++at)
      gd_store_tile(Ah + t0 * r, c[at], (int)min((int64_t)32, l - t0), 32 * at + col, half, r);
    st_wave_sync();  // this wave's reads of the tile precede its next staging writes
  }
}

// fp32 factors (heads l rows apart) to the output's type and place
template <typename OUT>
__global__ __launch_bounds__(256) void pf_store_factors_kernel(const float* __restrict__ src, int64_t src_stride,
                                                               OUT* __restrict__ dst, int64_t dst_stride, int64_t n) {
  const float* s = src + (int64_t)blockIdx.y * src_stride;
  OUT* d = dst + (int64_t)blockIdx.y * dst_stride;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) gd_store(d, i, s[i]);
}

template <typename OUT>
int prefill_store(const float* src, int64_t src_stride, OUT* dst, int64_t dst_stride, int64_t n, int heads, hipStream_t st) {
  if (n <= 0 || (const void*)src == (const void*)dst) return LRQK_OK;
  const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 1023) / 1024, 4096 / heads + 1));
  hipLaunchKernelGGL((pf_store_factors_kernel<OUT>), dim3(blocks, (unsigned)heads), dim3(256), 0, st, src, src_stride, dst,
                     dst_stride, n);
  LRQK_HIP_CHECK(hipGetLastError());
  return LRQK_OK;
}
template int prefill_store<float>(const float*, int64_t, float*, int64_t, int64_t, int, hipStream_t);
template int prefill_store<bf16_t>(const float*, int64_t, bf16_t*, int64_t, int64_t, int, hipStream_t);

template <int AT, int DB>
static int sums_impl(const StSums& g, int b, hipStream_t st) {
  const int bkv = b * g.hkv;
  if (DB == 2 && g.hkv == g.hq && g.S == g.Sxk)
    hipLaunchKernelGGL((pf_stream_sums_kernel<AT, DB, DB == 2, DB == 2>), dim3((unsigned)(2 * g.given)), dim3(kStThreads), 0,
                       st, g);
  else
    hipLaunchKernelGGL((pf_stream_sums_kernel<AT, DB, DB == 2, false>),
                       dim3((unsigned)((DB == 2 ? 2 : 3) * g.given + bkv * g.Sxk)), dim3(kStThreads), 0, st, g);
  LRQK_HIP_CHECK(hipGetLastError());
  return LRQK_OK;
}

// Sums of both sides: over the given factors ([b * hq] heads, S splits), Q^T Q ([b * hq] heads, S splits) and K^T K
// ([b * hkv] heads, Sxk splits).
int prefill_stream_sums(const bf16_t* q, const bf16_t* k, int hq, int hkv, int b, int64_t l, int r, int d, const float* a_q,
                        const float* a_k, float* part_q, float* part_k, int S, float* xq_part, float* xk_part, int Sxk,
                        hipStream_t st) {
  const StSums g{q, k, a_q, a_k, part_q, part_k, xq_part, xk_part, l, hq, hkv, r, S, Sxk, b * hq * S};
  if (d == 64) return r <= 32 ? sums_impl<1, 2>(g, b, st) : sums_impl<2, 2>(g, b, st);
  return r <= 32 ? sums_impl<1, 4>(g, b, st) : sums_impl<2, 4>(g, b, st);
}

template <int AT, int DB, typename OUT>
static int apply_impl(StApply<OUT> g0, StApply<OUT> g1, int bh, int r, hipStream_t st) {
  constexpr int D = 32 * DB, NW = kStApplyWaves;
  constexpr size_t smem = (size_t)(3 * 32 * AT + NW * 32) * (D + 8) * sizeof(bf16_t);
  static_assert(smem <= 160 * 1024, "LDS");
  auto kern = pf_stream_apply_kernel<AT, DB, OUT>;
  static std::atomic<bool> attr_dev[kMaxDeviceSlots];
  std::atomic<bool>& attr = attr_dev[per_device_slot()];
  if (!attr) {
    LRQK_HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    attr = true;
  }
  // every workgroup stages M (52 KB in, up to 104 KB of fp32 read): enough of them to fill the GPU once, no more
  const int per_cu = std::max(1, (int)(160 * 1024 / smem));
  const int unit = 8 * std::max(g0.nh, g1.nh);
  for (StApply<OUT>* g : {&g0, &g1}) {
    g->S = (int)std::max<int64_t>(1, std::min<int64_t>(std::max(1, 256 * per_cu / bh), (g->l + 32 * NW - 1) / (32 * NW)));
    g->pairs = bh / g->nh * g->S;
    g->chunks = g->nh == 1 ? (g->pairs + unit - 1) / unit : (g->pairs + 7) / 8;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)unit, (unsigned)(g0.chunks + g1.chunks)), dim3(NW * kWave), smem, st, g0, g1, r);
  LRQK_HIP_CHECK(hipGetLastError());
  return LRQK_OK;
}

// A_K = K Mk (l rows) and A_Q = Q Mq (q_rows rows) for all b * hq query heads.  q: the first of
// those rows, heads q_stride elements apart.
template <typename OUT>
int prefill_stream_apply(const bf16_t* k, int hkv, int64_t l, const float* mt_k, OUT* a_k, int64_t a_k_stride,
                         const bf16_t* q, int64_t q_rows, int64_t q_stride, const float* mt_q, OUT* a_q, int hq, int b, int r,
                         int d, hipStream_t st) {
  const StApply<OUT> gk{k, 0, l, l * d, mt_k, a_k, a_k_stride, hq / hkv, 0, 0};
  const StApply<OUT> gq{q, 0, q_rows, q_stride, mt_q, a_q, q_rows * r, 1, 0, 0};
  if (d == 64) return r <= 32 ? apply_impl<1, 2>(gk, gq, b * hq, r, st) : apply_impl<2, 2>(gk, gq, b * hq, r, st);
  return r <= 32 ? apply_impl<1, 4>(gk, gq, b * hq, r, st) : apply_impl<2, 4>(gk, gq, b * hq, r, st);
}
template int prefill_stream_apply<float>(const bf16_t*, int, int64_t, const float*, float*, int64_t, const bf16_t*, int64_t,
                                         int64_t, const float*, float*, int, int, int, int, hipStream_t);
template int prefill_stream_apply<bf16_t>(const bf16_t*, int, int64_t, const float*, bf16_t*, int64_t, const bf16_t*, int64_t,
                                          int64_t, const float*, bf16_t*, int, int, int, int, hipStream_t);

}  // namespace lrqk
