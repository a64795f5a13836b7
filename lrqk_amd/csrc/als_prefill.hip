// Prefill factorisation: joint rank-r alternating least squares for Q ~ A_Q B_Q, K ~ A_K B_K
// with the coupling term Q K^T ~ A_Q A_K^T (all weights 1).
//
// Per iteration the long axis is streamed twice (once over Q, once over K):
//   apply(X, Mt, A): A <- X Mt^T row by row, and in the same pass accumulate the new
//                    A^T A, A^T X and the squared change of A.
// The r x r / r x d systems between the passes are solved per head by `small` kernels.
// The stopping test (a batch-wide mean squared change) is evaluated on the device; once
// it fires the remaining launches of the loop return immediately, so the host never
// waits inside the loop.
//
// Implementations of each kernel: fp32 MFMA (32x32x2) tiles for r <= 32 and head dimensions that are a
// multiple of the 16-byte vector, fp32 MFMA (16x16x4) tiles for r = 33 .. 64 and fp32 rows of 64 or 128, and a
// generic VALU version for every other shape.  All write the same partial-sum layout.
#include <algorithm>
#include <stdlib.h>
#include <string.h>
#include <type_traits>

#include "common.hpp"
#include "ctx.hpp"
#include "prefill_pieces.hpp"
#include "small_inverse.hpp"

namespace lrqk {

constexpr int kPfThreads = 256;
constexpr int kPfTile = 32;
constexpr int kPfMaxPer = 48;  // accumulators per thread: r*(r+d) <= 256*48 (r = 64 with rows of 128 elements)

// Sums of a tile: out[j][c] += sum_rows a_s[row][j] * (c < r ? a_s[row][c] : x_s[row][c-r]),  0 <= j < r,
// 0 <= c < r + d.  The 256 threads form a 16 x 16 grid; thread (tj, tc) owns rows j = tj + 16 i (i < I) and columns
// c = tc + 16 k (k < 48 / I) and keeps them in acc[i * K + k]: I values of A and K of [A | X] per tile row feed
// I * K products (a sixth of the LDS reads of one output at a time).  I = ceil(r / 16), which the limit
// r (r + d) <= 12288 makes enough: 16 K >= r + d.
template <int I>
__device__ __forceinline__ void accumulate_gram_tile(const float* a_s, int lda, const float* x_s, int ldx, int rows, int r,
                                                     int d, float* acc) {
  constexpr int K = kPfMaxPer / I;
  const int tj = threadIdx.x >> 4, tc = threadIdx.x & 15;
  const float* cp[K];  // column c of a row: in the A tile or in the X tile
  int cs[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = min(tc + 16 * k, r + d - 1);
    cp[k] = c < r ? a_s + c : x_s + (c - r);
    cs[k] = c < r ? lda : ldx;
  }
  for (int row = 0; row < rows; ++row) {
    float av[I], cv[K];
#pragma unroll
    for (int i = 0; i < I; ++i) av[i] = a_s[row * lda + min(tj + 16 * i, r - 1)];
#pragma unroll
    for (int k = 0; k < K; ++k) cv[k] = cp[k][row * cs[k]];
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int k = 0; k < K; ++k) acc[i * K + k] = fmaf(av[i], cv[k], acc[i * K + k]);
  }
}
__device__ __forceinline__ void accumulate_gram(const float* a_s, int lda, const float* x_s, int ldx, int rows, int r,
                                                int d, float* acc) {
  if (r <= 16)
    accumulate_gram_tile<1>(a_s, lda, x_s, ldx, rows, r, d, acc);
  else if (r <= 32)
    accumulate_gram_tile<2>(a_s, lda, x_s, ldx, rows, r, d, acc);
  else if (r <= 48)
    accumulate_gram_tile<3>(a_s, lda, x_s, ldx, rows, r, d, acc);
  else
    accumulate_gram_tile<4>(a_s, lda, x_s, ldx, rows, r, d, acc);
}
// The sums of accumulate_gram to `out` (packed [r][r + d]).
__device__ __forceinline__ void store_gram(const float* acc, int r, int d, float* __restrict__ out) {
  const int I = r <= 16 ? 1 : r <= 32 ? 2 : r <= 48 ? 3 : 4;
  const int K = kPfMaxPer / I;
  const int tj = threadIdx.x >> 4, tc = threadIdx.x & 15;
#pragma unroll
  for (int e = 0; e < kPfMaxPer; ++e) {
    const int i = e / K, k = e % K;
    const int j = tj + 16 * i, c = tc + 16 * k;
    if (i < I && j < r && c < r + d) out[j * (r + d) + c] = acc[e];
  }
}

// X: [b][xh][l][d] storage dtype; head h of the factors reads X head (h % hq) / (hq / xh).
template <typename T>
__global__ __launch_bounds__(kPfThreads) void pf_pass_generic_kernel(const T* __restrict__ X, int xh, int hq, int64_t l, int r,
                                                             int d, const float* __restrict__ Mt, float* __restrict__ A,
                                                             float* __restrict__ part, float* __restrict__ delta_part,
                                                             const int* __restrict__ done_flag, int S) {
  if (done_flag && *done_flag) return;
  extern __shared__ __align__(16) float sm[];
  const int ldx = d + 1, lda = r + 1;
  float* x_s = sm;                       // [tile][d+1]
  float* a_s = x_s + kPfTile * ldx;      // [tile][r+1]
  float* m_s = a_s + kPfTile * lda;      // [r][d+1]   (apply only)
  __shared__ float red[kPfThreads / kWave];
  const int tid = threadIdx.x;
  const int h = blockIdx.y, s = blockIdx.x;
  const int b = h / hq, head = h % hq;
  const int64_t xhead = (int64_t)b * xh + head / (hq / xh);
  const T* Xh = X + xhead * l * d;
  float* Ah = A + (int64_t)h * l * r;
  const bool apply = Mt != nullptr;
  if (apply) {
    for (int e = tid; e < r * d; e += kPfThreads) m_s[(e / d) * ldx + e % d] = Mt[(int64_t)h * r * d + e];
  }
  const int64_t rows_per_split = (l + S - 1) / S;
  const int64_t r0 = (int64_t)s * rows_per_split;
  const int64_t r1 = min(l, r0 + rows_per_split);
  float acc[kPfMaxPer];
#pragma unroll
  for (int i = 0; i < kPfMaxPer; ++i) acc[i] = 0.0f;
  float dsum = 0.0f;
  __syncthreads();
  for (int64_t t0 = r0; t0 < r1; t0 += kPfTile) {
    const int rows = (int)min((int64_t)kPfTile, r1 - t0);
    for (int e = tid; e < rows * d; e += kPfThreads) x_s[(e / d) * ldx + e % d] = ld_f32<T>(Xh, t0 * d + e);
    if (!apply) {
      for (int e = tid; e < rows * r; e += kPfThreads) a_s[(e / r) * lda + e % r] = Ah[t0 * r + e];
    }
    __syncthreads();
    if (apply) {
      // thread -> (row of the tile, eight columns j = jg + 8 u of the new A): one element of X feeds eight products
      static_assert(kPfTile == 32 && kPfThreads == 256, "32 rows x 8 column groups");
      const int row = tid & (kPfTile - 1), jg = tid >> 5;
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = 0.0f;
      const float* mrow[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) mrow[u] = m_s + min(jg + 8 * u, r - 1) * ldx;
      for (int c = 0; c < d; ++c) {
        const float x = x_s[row * ldx + c];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = fmaf(x, mrow[u][c], v[u]);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int j = jg + 8 * u;
        if (row < rows && j < r) {
          const float old = Ah[(t0 + row) * r + j];
          const float df = old - v[u];
          dsum = fmaf(df, df, dsum);
          Ah[(t0 + row) * r + j] = v[u];
          a_s[row * lda + j] = v[u];
        }
      }
      __syncthreads();
    }
    accumulate_gram(a_s, lda, x_s, ldx, rows, r, d, acc);
    __syncthreads();
  }
  const int ne = r * (r + d);
  store_gram(acc, r, d, part + ((int64_t)h * S + s) * ne);
  if (apply) {
    dsum = wave_sum(dsum);
    if (lane_id() == 0) red[wave_id()] = dsum;
    __syncthreads();
    if (tid == 0) {
      float t = 0.0f;
      for (int w = 0; w < kPfThreads / kWave; ++w) t += red[w];
      delta_part[(int64_t)h * S + s] = t;
    }
  }
}

// Gauss-Jordan, no pivoting, r x r system with nrhs right-hand sides stored as columns
// r .. r+nrhs-1 of Mx (row stride ldm).  Afterwards X[i][c] = Mx[i][r+c] / Mx[i][i].
__device__ __forceinline__ void solve_multi(float* Mx, int ldm, int r, int nrhs) {
  const int tid = threadIdx.x;
  for (int p = 0; p < r; ++p) {
    const float inv = 1.0f / Mx[p * ldm + p];
    const int w = r + nrhs - p - 1;  // columns p+1 .. r+nrhs-1
    for (int e = tid; e < r * w; e += kPfThreads) {
      const int i = e / w, j = p + 1 + e % w;
      if (i != p) Mx[i * ldm + j] = fmaf(-(Mx[i * ldm + p] * inv), Mx[p * ldm + j], Mx[i * ldm + j]);
    }
    __syncthreads();
  }
}

__device__ __forceinline__ void reduce_part(const float* part, int S, int ne, float* dst) {
  for (int e = threadIdx.x; e < ne; e += kPfThreads) {
    // (more than 16 partial sums -- long prompts -- are added in fp64)
    float v = 0.0f;
    double w = 0.0;
    for (int s = 0; s < S; ++s) {
      const float x = part[(int64_t)s * ne + e];
      v += x;
      w += (double)x;
    }
    dst[e] = S > 16 ? (float)w : v;
  }
}

// stage 0: (stopping test) B_Q, B_K from the current Grams, then Mt for the A_Q update
// stage 1: Mt for the A_K update from the new A_Q Grams
// stage 2: final B_Q, B_K
__global__ __launch_bounds__(kPfThreads) void pf_small_generic_kernel(int stage, int it, const float* __restrict__ partQ,
                                                              const float* __restrict__ partK, int S, int bh, int r,
                                                              int d, int64_t l, float tol,
                                                              const float* __restrict__ delta_all, int* __restrict__ flags,
                                                              float* __restrict__ Mt, float* __restrict__ b_q,
                                                              float* __restrict__ b_k) {
  extern __shared__ __align__(16) float sm[];
  const int ldm = r + d + 1;
  const int ne = r * (r + d);
  float* G2 = sm;               // [r][r+d] packed (ne)   the K side's sums (the Q side's go straight into Mx)
  float* Mx = G2 + ne;          // [r][ldm]
  float* Bs = Mx + r * ldm;     // [r][d+1]
  __shared__ int s_done;
  const int tid = threadIdx.x;
  const int h = blockIdx.x;

  if (stage == 0) {
    if (tid == 0) {
      int done = 0;
      if (it > 0) {
        done = flags[it - 1];
        if (!done) {
          const float* dq = delta_all + ((int64_t)(it - 1) * 2 + 0) * bh * S;
          const float* dk = delta_all + ((int64_t)(it - 1) * 2 + 1) * bh * S;
          float sq = 0.0f, sk = 0.0f;
          for (int i = 0; i < bh * S; ++i) {
            sq += dq[i];
            sk += dk[i];
          }
          const float n = (float)bh * (float)l * (float)r;
          done = fmaxf(sq / n, sk / n) < tol;
        }
      }
      s_done = done;
    }
    __syncthreads();
    // every head computes the same decision; all must have read flags[it-1] and the deltas
    // before anything of this iteration is overwritten, which the launch order guarantees
    if (h == 0 && tid == 0) flags[it] = s_done;
    if (s_done) return;
  } else if (stage == 1) {
    if (flags[it]) return;
  }

  const float* pq = partQ + (int64_t)h * S * ne;
  const float* pk = partK + (int64_t)h * S * ne;
  // sum over the splits of element e of a head's packed [G | C] block, in split order
  auto summed = [&](const float* part, int e) {
    float v = 0.0f;
    double w = 0.0;
    for (int s = 0; s < S; ++s) {
      const float x = part[(int64_t)s * ne + e];
      v += x;
      w += (double)x;
    }
    return S > 16 ? (float)w : v;
  };
  if (stage == 0 || stage == 2) {
    reduce_part(pk, S, ne, G2);
    // B_Q = (A_Q^T A_Q)^-1 A_Q^T Q
    for (int e = tid; e < ne; e += kPfThreads) Mx[(e / (r + d)) * ldm + e % (r + d)] = summed(pq, e);
    __syncthreads();
    solve_multi(Mx, ldm, r, d);
    for (int e = tid; e < r * d; e += kPfThreads) {
      const int i = e / d, c = e % d;
      const float v = Mx[i * ldm + r + c] / Mx[i * ldm + i];
      Bs[i * (d + 1) + c] = v;
      b_q[(int64_t)h * r * d + e] = v;
    }
    __syncthreads();
    // B_K
    for (int e = tid; e < ne; e += kPfThreads) Mx[(e / (r + d)) * ldm + e % (r + d)] = G2[e];
    __syncthreads();
    solve_multi(Mx, ldm, r, d);
    for (int e = tid; e < r * d; e += kPfThreads) {
      const int i = e / d, c = e % d;
      b_k[(int64_t)h * r * d + e] = Mx[i * ldm + r + c] / Mx[i * ldm + i];
    }
    __syncthreads();
    if (stage == 2) return;
    // Mt_Q = (A_K^T A_K + B_Q B_Q^T)^-1 (A_K^T K + B_Q)
    for (int e = tid; e < ne; e += kPfThreads) {
      const int i = e / (r + d), c = e % (r + d);
      float v = G2[e];
      if (c < r) {
        float g = 0.0f;
        for (int x = 0; x < d; ++x) g = fmaf(Bs[i * (d + 1) + x], Bs[c * (d + 1) + x], g);
        v += g;
      } else {
        v += Bs[i * (d + 1) + c - r];
      }
      Mx[i * ldm + c] = v;
    }
  } else {
    // stage 1: Mt_K = (A_Q^T A_Q + B_K B_K^T)^-1 (A_Q^T Q + B_K)
    for (int e = tid; e < r * d; e += kPfThreads) Bs[(e / d) * (d + 1) + e % d] = b_k[(int64_t)h * r * d + e];
    __syncthreads();
    for (int e = tid; e < ne; e += kPfThreads) {
      const int i = e / (r + d), c = e % (r + d);
      float v = summed(pq, e);
      if (c < r) {
        float g = 0.0f;
        for (int x = 0; x < d; ++x) g = fmaf(Bs[i * (d + 1) + x], Bs[c * (d + 1) + x], g);
        v += g;
      } else {
        v += Bs[i * (d + 1) + c - r];
      }
      Mx[i * ldm + c] = v;
    }
  }
  __syncthreads();
  solve_multi(Mx, ldm, r, d);
  for (int e = tid; e < r * d; e += kPfThreads) {
    const int i = e / d, c = e % d;
    Mt[(int64_t)h * r * d + e] = Mx[i * ldm + r + c] / Mx[i * ldm + i];
  }
}


// ============================================================================ MFMA path
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kPfSmallThreads = 512;

// C tile of mfma_f32_32x32x2f32: lane l, element v -> row (the column is l & 31)
__device__ __forceinline__ int pf_mfma_row(int lane, int v) { return ((v >> 2) << 3) + ((lane >> 5) << 2) + (v & 3); }

// One wave owns 32 rows of X at a time (staged as fp32 in its private LDS tile, row stride
// 32*NB+4, zero beyond d and beyond the last row).
//   apply:  C[32 x 32] = X[32 x d] Mt^T          (A operand from LDS, B operand = Mt)
//   gram:   G_AA += C^T C, G_AX += C^T X          (the C registers are the A operand as they are:
//           element v of lane l is row pf_mfma_row(l, v), and a sum over rows may visit them in any order)
// The k index of the apply and the column index of G_AX are permuted so that every lane reads
// consecutive floats of its LDS row with 16-byte loads: MFMA step kk multiplies columns kk and
// kk + 16*NB; tile nb of G_AX holds the columns n*NB + nb.
// NB = number of 32-column blocks of X.  NW waves per workgroup; the tiles are wave-private, so
// the waves only meet at the start and in the final reduction and otherwise drift apart (one
// wave's staging overlaps another's MFMAs on the same SIMD).  MT_LDS: Mt is kept in LDS (shared
// by the waves) instead of registers, which leaves room for two waves per SIMD.

// orders this wave's LDS writes before its later LDS reads (the tile is exchanged between lanes)
__device__ __forceinline__ void pf_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T, int NB, int NW, bool MT_LDS>
__global__ __launch_bounds__(NW * kWave) void pf_pass_mfma_kernel(const T* __restrict__ X, int xh, int hq, int64_t l,
                                                                  int r, int d, const float* __restrict__ Mt,
                                                                  float* __restrict__ A, float* __restrict__ part,
                                                                  float* __restrict__ delta_part,
                                                                  const int* __restrict__ done_flag, int S) {
  if (done_flag && *done_flag) return;
  constexpr int LDX = 32 * NB + 4;
  constexpr int KH = 16 * NB;
  constexpr int VEC = Vec16<T>::N;
  constexpr int NL = 32 * 32 * NB / (kWave * VEC);
  constexpr int NT = NW * kWave;
  extern __shared__ __align__(16) float sm[];
  __shared__ float red[NW];
  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  const int col = lane & 31, half = lane >> 5;
  float* x_s = sm + wave * 32 * LDX;
  float* mt_s = sm + NW * 32 * LDX;  // [32][LDX], MT_LDS only
  const int h = blockIdx.y, s = blockIdx.x;
  const int b = h / hq, head = h % hq;
  const int64_t xhead = (int64_t)b * xh + head / (hq / xh);
  const T* Xh = X + xhead * l * d;
  float* Ah = A + (int64_t)h * l * r;
  const bool apply = Mt != nullptr;
  const bool full_rows = d == 32 * NB;  // row / column of a flat element index by shifts

  float mt[MT_LDS ? 1 : KH];
  if (apply) {
    const float* Mh = Mt + (int64_t)h * r * d;
    if constexpr (MT_LDS) {
      for (int e = tid; e < 32 * 32 * NB; e += NT) {
        const int n = e / (32 * NB), k = e % (32 * NB);
        const float v = Mh[min(n, r - 1) * d + min(k, d - 1)];
        mt_s[n * LDX + k] = (n < r && k < d) ? v : 0.0f;
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < KH; ++kk) {
        const int k = kk + half * KH;
        const float v = Mh[min(col, r - 1) * d + min(k, d - 1)];
        mt[kk] = (col < r && k < d) ? v : 0.0f;
      }
    }
  }
  for (int e = lane; e < 32 * LDX; e += kWave) x_s[e] = 0.0f;

  const int64_t rows_per_split = (((l + S - 1) / S) + 31) / 32 * 32;
  const int64_t r0 = (int64_t)s * rows_per_split;
  const int64_t r1 = min(l, r0 + rows_per_split);

  floatx16 gAA;
  floatx16 gAX[NB];
#pragma unroll
  for (int v = 0; v < 16; ++v) gAA[v] = 0.0f;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int v = 0; v < 16; ++v) gAX[nb][v] = 0.0f;
  float dsum = 0.0f;

  Vec16<T> pre[NL];
  auto issue = [&](int64_t t0) {
    const int nvalid = t0 < r1 ? (int)min((int64_t)32, r1 - t0) * d : 0;
    const int64_t base = (t0 < r1 ? t0 : r0) * d;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = (i * kWave + lane) * VEC;
      pre[i].load(Xh + base + (e < nvalid ? e : 0));
    }
  };
  if (r0 + (int64_t)wave * 32 < r1) issue(r0 + (int64_t)wave * 32);
  __syncthreads();  // Mt staged, tiles cleared

  for (int64_t t0 = r0 + (int64_t)wave * 32; t0 < r1; t0 += 32 * NW) {
    const int rows = (int)min((int64_t)32, r1 - t0);
    // stage this wave's rows
    {
      const int nvalid = rows * d;
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int e = (i * kWave + lane) * VEC;
        if (e < 32 * d) {
          float f[VEC];
          pre[i].unpack(f);
          const int row = full_rows ? e / (32 * NB) : e / d;
          const int c0 = full_rows ? e % (32 * NB) : e - row * d;
          const bool ok = e < nvalid;
#pragma unroll
          for (int u = 0; u < VEC; u += 4)
            *reinterpret_cast<float4*>(&x_s[row * LDX + c0 + u]) =
                make_float4(ok ? f[u] : 0.0f, ok ? f[u + 1] : 0.0f, ok ? f[u + 2] : 0.0f, ok ? f[u + 3] : 0.0f);
        }
      }
    }
    pf_wave_sync();
    if (t0 + 32 * NW < r1) issue(t0 + 32 * NW);

    floatx16 c;
    float old[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      // unconditional (clamped) load, masked below
      const int64_t rr = min(t0 + pf_mfma_row(lane, v), l - 1);
      old[v] = Ah[rr * r + min(col, r - 1)];
    }
    if (apply) {
#pragma unroll
      for (int v = 0; v < 16; ++v) c[v] = 0.0f;
      // operands of group g4 + 1 are fetched from LDS while the MFMAs of group g4 run
      auto lds4 = [&](const float* base, int g4) {
        return *reinterpret_cast<const float4*>(&base[col * LDX + half * KH + 4 * g4]);
      };
      float4 xa = lds4(x_s, 0);
      float4 mb;
      if constexpr (MT_LDS) mb = lds4(mt_s, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, MT_LDS ? 2 : 1, 0);  // the first reads have their own slot
#pragma unroll
      for (int g4 = 0; g4 < KH / 4; ++g4) {
        float4 xn = xa, mn = mb;
        if (g4 + 1 < KH / 4) {
          xn = lds4(x_s, g4 + 1);
          if constexpr (MT_LDS) mn = lds4(mt_s, g4 + 1);
        }
        if constexpr (!MT_LDS)
          mb = make_float4(mt[(4 * g4) % (MT_LDS ? 1 : KH)], mt[(4 * g4 + 1) % (MT_LDS ? 1 : KH)],
                           mt[(4 * g4 + 2) % (MT_LDS ? 1 : KH)], mt[(4 * g4 + 3) % (MT_LDS ? 1 : KH)]);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(xa.x, mb.x, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(xa.y, mb.y, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(xa.z, mb.z, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(xa.w, mb.w, c, 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, MT_LDS ? 2 : 1, 0);  // DS reads of the next group
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);               // then this group's MFMAs
        xa = xn;
        if constexpr (MT_LDS) mb = mn;
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = pf_mfma_row(lane, v);
        if (row < rows && col < r) {
          const float df = old[v] - c[v];
          dsum = fmaf(df, df, dsum);
          Ah[(t0 + row) * r + col] = c[v];
        }
      }
    } else {
#pragma unroll
      for (int v = 0; v < 16; ++v) c[v] = (pf_mfma_row(lane, v) < rows && col < r) ? old[v] : 0.0f;
    }
    auto ldsb = [&](int v, float (&xb)[NB]) {
      const int row = pf_mfma_row(lane, v);
      if constexpr (NB == 1) {
        xb[0] = x_s[row * LDX + col];
      } else if constexpr (NB == 2) {
        const float2 t = *reinterpret_cast<const float2*>(&x_s[row * LDX + col * 2]);
        xb[0] = t.x; xb[1] = t.y;
      } else {
#pragma unroll
        for (int q = 0; q < NB / 4; ++q) {
          const float4 t = *reinterpret_cast<const float4*>(&x_s[row * LDX + col * NB + 4 * q]);
          xb[4 * q] = t.x; xb[4 * q + 1] = t.y; xb[4 * q + 2] = t.z; xb[4 * q + 3] = t.w;
        }
      }
    };
    float xb[NB];
    ldsb(0, xb);
    __builtin_amdgcn_sched_group_barrier(0x100, NB == 8 ? 2 : 1, 0);  // the first read has its own slot
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float xn[NB];
      if (v + 1 < 16) ldsb(v + 1, xn);
      gAA = __builtin_amdgcn_mfma_f32_32x32x2f32(c[v], c[v], gAA, 0, 0, 0);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) gAX[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(c[v], xb[nb], gAX[nb], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, NB == 8 ? 2 : 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, NB + 1, 0);
      if (v + 1 < 16) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) xb[nb] = xn[nb];
      }
    }
    pf_wave_sync();  // this wave's reads of the tile precede its next staging writes
  }
  __syncthreads();  // every wave is done with its tile (and with Mt): the LDS is reused below

  // reduce the waves' tiles through LDS, one 32 x 32 block at a time
  const int ne = r * (r + d);
  float* out = part + ((int64_t)h * S + s) * ne;
  for (int blk = 0; blk <= NB; ++blk) {
    float* mine = sm + wave * 1024;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float val = gAA[v];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        if (blk == nb + 1) val = gAX[nb][v];
      mine[pf_mfma_row(lane, v) * 32 + col] = val;
    }
    __syncthreads();
    for (int e = tid; e < 1024; e += NT) {
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += sm[w * 1024 + e];
      const int m = e >> 5, n = e & 31;
      if (blk == 0) {
        if (m < r && n < r) out[m * (r + d) + n] = v;
      } else {
        const int cx = n * NB + (blk - 1);
        if (m < r && cx < d) out[m * (r + d) + r + cx] = v;
      }
    }
    __syncthreads();
  }
  if (apply) {
    dsum = wave_sum(dsum);
    if (lane == 0) red[wave] = dsum;
    __syncthreads();
    if (tid == 0) {
      float t = 0.0f;
      for (int w = 0; w < NW; ++w) t += red[w];
      delta_part[(int64_t)h * S + s] = t;
    }
  }
}

// ---- the same pass for r <= 16 and fp32 rows of exactly D = 64 or 128 elements, on 16x16x4 tiles: a 32-wide tile is half
// zeros at these ranks.  The products of the fp32 matrix cores are chains of fused multiply-adds in the order of their k
// index (32x32x2 and 16x16x4 alike), and every sum here takes its terms in the order of pf_pass_mfma_kernel: the results
// are that kernel's to the bit.
//   apply: k in the order 0, D/2, 1, D/2 + 1, ...   A row of X lies in LDS in four quarters (column c = D/2 hi + 2 s + par
//          in quarter hi + 2 par, place s), so a lane's operands of four products are 16 consecutive bytes.
//   sums:  rows in the order 0 4 1 5 | 2 6 3 7 | 8 12 9 13 | 10 14 11 15 (+ 16).  Row m of an apply tile is row
//          pf16_row(m) of the 16, which leaves C in the layout of the sums' left operand.  Tile n of A^T X holds the
//          columns at places 8 i + n (D = 128), so a lane reads its row's 8 operands as 32 bytes.
// Bound by the matrix cores (4352 of ~6000 cycles per wave and tile, two waves per SIMD) and the ends of the launch; Mt
// stays in registers, the rows of A are requested a tile ahead like those of X, and the waves' sums meet in LDS at once.
// 28 heads of 4096 rows, rank 16: 41 -> 23 us a pass (mean of sums alone and apply).
__device__ __forceinline__ int pf16_row(int m) {  // 0 2 8 10 by m % 4, 0 4 1 5 by m / 4
  return ((m & 2) << 2) + ((m & 1) << 1) + ((m & 4) ? 4 : 0) + ((m & 8) ? 1 : 0);
}
constexpr int kPf16Waves = 8;
template <int D>
struct Pf16Shape {
  static constexpr int LDX = D + 4;        // floats per staged row
  static constexpr int NT = D / 16;        // tiles of A^T X
  static constexpr size_t SMEM = (size_t)kPf16Waves * 32 * LDX * sizeof(float);
  static_assert((NT + 1) * 256 <= 32 * LDX, "a wave's sums fit its tile's LDS");
};
template <int D>
__global__ __launch_bounds__(kPf16Waves * kWave, 2) void pf_pass_mfma16_kernel(
    const float* __restrict__ X, int xh, int hq, int64_t l, int r, int, const float* __restrict__ Mt, float* __restrict__ A,
    float* __restrict__ part, float* __restrict__ delta_part, const int* __restrict__ done_flag, int S) {
  if (done_flag && *done_flag) return;
  using Sh = Pf16Shape<D>;
  constexpr int LDX = Sh::LDX, NT = Sh::NT, HALF = D / 2, QUART = D / 4, NW = kPf16Waves;
  constexpr int NL = 32 * D / (kWave * 4);  // 16-byte loads per lane and tile
  extern __shared__ __align__(16) float sm[];
  __shared__ float red[NW];
  const int tid = threadIdx.x, lane = lane_id(), wave = gd_wave();
  const int li = lane & 15, lk = lane >> 4;
  float* x_s = sm + wave * 32 * LDX;
  const int h = blockIdx.y, s = blockIdx.x;
  const int b = h / hq, head = h % hq;
  const float* Xh = X + ((int64_t)b * xh + head / (hq / xh)) * l * D;
  float* Ah = A + (int64_t)h * l * r;
  const bool apply = Mt != nullptr;
  const int64_t rows_per_split = (((l + S - 1) / S) + 31) / 32 * 32;
  const int64_t r0 = (int64_t)s * rows_per_split;
  const int64_t r1 = min(l, r0 + rows_per_split);

  float4 pre[NL];
  float old_next[8];  // rows of A: element 4 t + v is row 16 t + pf16_row(4 lk + v)
  auto issue = [&](int64_t t0) {
    const int last = (int)min((int64_t)32, r1 - t0) - 1;
    const float* xt = Xh + t0 * D;
    const float* at = Ah + t0 * r;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = (i * kWave + lane) * 4;
      pre[i] = gd_at<float4>(xt, 4u * (uint32_t)(min(e / D, last) * D + e % D));
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      old_next[q] = gd_factor(at, 16 * (q >> 2) + pf16_row(4 * lk + (q & 3)), last, r, min(li, r - 1));
  };
  const int64_t first = r0 + (int64_t)wave * 32;
  if (first < r1) issue(first);
  float mt[QUART];  // this lane's operands of the apply: row li of Mt, its quarter of the columns
  if (apply) {
    const float* Mh = Mt + ((int64_t)h * r + min(li, r - 1)) * D + (lk & 1) * HALF + (lk >> 1);
#pragma unroll
    for (int k = 0; k < QUART; ++k) mt[k] = li < r ? Mh[2 * k] : 0.0f;
  }
  floatx4 gAA = floatx4{0.0f, 0.0f, 0.0f, 0.0f}, gAX[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) gAX[n] = gAA;
  float dsum = 0.0f;

  for (int64_t t0 = first; t0 < r1; t0 += 32 * NW) {
    const int rows = (int)min((int64_t)32, r1 - t0);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = (i * kWave + lane) * 4, row = e / D, c = e % D;
      const float4 x = row < rows ? pre[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      float* at = x_s + row * LDX + (c / HALF) * QUART + (c % HALF) / 2;
      *reinterpret_cast<float2*>(at) = make_float2(x.x, x.z);
      *reinterpret_cast<float2*>(at + 2 * QUART) = make_float2(x.y, x.w);
    }
    float old[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) old[q] = old_next[q];
    pf_wave_sync();
    if (t0 + 32 * NW < r1) issue(t0 + 32 * NW);
    floatx4 c[2];
    if (apply) {
      c[0] = c[1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
      const float* xa = x_s + pf16_row(li) * LDX + lk * QUART;
#pragma unroll
      for (int k = 0; k < QUART; k += 4) {
        const float4 a0 = *reinterpret_cast<const float4*>(xa + k);
        const float4 a1 = *reinterpret_cast<const float4*>(xa + 16 * LDX + k);
        c[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0.x, mt[k], c[0], 0, 0, 0);
        c[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1.x, mt[k], c[1], 0, 0, 0);
        c[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0.y, mt[k + 1], c[0], 0, 0, 0);
        c[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1.y, mt[k + 1], c[1], 0, 0, 0);
        c[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0.z, mt[k + 2], c[0], 0, 0, 0);
        c[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1.z, mt[k + 2], c[1], 0, 0, 0);
        c[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0.w, mt[k + 3], c[0], 0, 0, 0);
        c[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1.w, mt[k + 3], c[1], 0, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int row = 16 * (q >> 2) + pf16_row(4 * lk + (q & 3));
        if (row < rows && li < r) {
          const float v = c[q >> 2][q & 3], df = old[q] - v;
          dsum = fmaf(df, df, dsum);
          Ah[(t0 + row) * r + li] = v;
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q)
        c[q >> 2][q & 3] = 16 * (q >> 2) + pf16_row(4 * lk + (q & 3)) < rows && li < r ? old[q] : 0.0f;
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      float xb[NT];
      const float* xr = x_s + (16 * (q >> 2) + pf16_row(4 * lk + (q & 3))) * LDX + NT * li;
#pragma unroll
      for (int n = 0; n < NT; n += 4) {
        const float4 x4 = *reinterpret_cast<const float4*>(xr + n);
        xb[n] = x4.x; xb[n + 1] = x4.y; xb[n + 2] = x4.z; xb[n + 3] = x4.w;
      }
      const float cv = c[q >> 2][q & 3];
      gAA = __builtin_amdgcn_mfma_f32_16x16x4f32(cv, cv, gAA, 0, 0, 0);
#pragma unroll
      for (int n = 0; n < NT; ++n) gAX[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(cv, xb[n], gAX[n], 0, 0, 0);
    }
    pf_wave_sync();  // this wave's reads of the tile precede its next staging writes
  }
  // the waves' sums side by side in LDS (each in its own tile's place), added in the waves' order
  const auto keep = [&](int t, const floatx4& g) {
#pragma unroll
    for (int v = 0; v < 4; ++v) x_s[t * 256 + (4 * lk + v) * 16 + li] = g[v];
  };
  keep(0, gAA);
#pragma unroll
  for (int n = 0; n < NT; ++n) keep(n + 1, gAX[n]);
  __syncthreads();
  const int ld = r + D;
  float* out = part + ((int64_t)h * S + s) * r * ld;
  for (int e = tid; e < (NT + 1) * 256; e += NW * kWave) {
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += sm[w * 32 * LDX + e];
    const int t = e >> 8, j = (e >> 4) & 15, n = e & 15;
    if (j >= r) continue;
    if (t == 0) {
      if (n < r) out[j * ld + n] = v;
    } else {
      const int at = NT * n + t - 1, q = at / QUART;  // place in the row: quarter q
      out[j * ld + r + (q & 1) * HALF + 2 * (at % QUART) + (q >> 1)] = v;
    }
  }
  if (apply) {
    dsum = wave_sum(dsum);
    if (lane == 0) red[wave] = dsum;
    __syncthreads();
    if (tid == 0) {
      float t = 0.0f;
      for (int w = 0; w < NW; ++w) t += red[w];
      delta_part[(int64_t)h * S + s] = t;
    }
  }
}

// ---- the same pass for bf16 input on the bf16 matrix cores (16 x the fp32 MFMA rate), without giving up
// fp32 accuracy: an fp32 number is the exact sum of three bf16 numbers (8 + 8 + 8 mantissa bits, by
// truncation), a product of two bf16 numbers is exact in fp32, and the MFMA accumulates in fp32.  So
//   apply:  C = X Mt^T            = X (Mt_hi + Mt_mid + Mt_lo)^T            (X is bf16 as it is: 3 products)
//   gram:   G_AX += C^T X         = (C_hi + C_mid + C_lo)^T X                (3 products)
//           G_AA += C^T C         = all piece pairs except lo*lo (8 products, error 2^-32; the pieces of a number
//                                   share its sign, so dropping mid*lo as well would bias the diagonal by ~2^-24,
//                                   which the r x r systems amplify by their condition number)
// with 32x32x16 tiles.  The Gram products sum over the rows of the tile, and C comes out of the apply in
// the accumulator layout (lane l, element v: row pf_mfma_row(l, v), column l % 32), where a lane holds
// rows 4 h .. 4 h + 3 (+ 8, 16, 24) of its column, h = l / 32: taken eight at a time these are the k
// elements of an MFMA operand, in an order that does not matter as long as the other operand uses the
// same one.  X gets into that layout by a product with the identity (2 MFMAs per 32 columns, exact).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// the three bf16 pieces of x (as the upper halves of fp32 bit patterns)
__device__ __forceinline__ void pf_split3(float x, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = __float_as_uint(x) & 0xffff0000u;
  const float r1 = x - __uint_as_float(hi);  // exact
  mid = __float_as_uint(r1) & 0xffff0000u;
  const float r2 = r1 - __uint_as_float(mid);  // exact, at most 8 significant bits
  lo = __float_as_uint(r2) & 0xffff0000u;
}
// two bf16 values (upper halves of a, b) in one word, a first
__device__ __forceinline__ uint32_t pf_pack2(uint32_t a, uint32_t b) { return (a >> 16) | (b & 0xffff0000u); }
__device__ __forceinline__ bf16x8 pf_bf16x8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return __builtin_bit_cast(bf16x8, make_uint4(a, b, c, d));
}

template <int NB, int NW>
__global__ __launch_bounds__(NW * kWave) void pf_pass_bf16_kernel(const bf16_t* __restrict__ X, int xh, int hq,
                                                                  int64_t l, int r, int d,
                                                                  const float* __restrict__ Mt, float* __restrict__ A,
                                                                  float* __restrict__ part,
                                                                  float* __restrict__ delta_part,
                                                                  const int* __restrict__ done_flag, int S) {
  if (done_flag && *done_flag) return;
  constexpr int LDB = 32 * NB + 8;  // row stride of a bf16 tile (elements): 16-byte operand reads want rows 4 banks apart
  constexpr int KB = 2 * NB;        // 16-column blocks of X
  constexpr int VEC = 8;
  constexpr int NL = 32 * 32 * NB / (kWave * VEC);
  constexpr int NT = NW * kWave;
  extern __shared__ __align__(16) float sm[];
  __shared__ float red[NW];
  const int tid = threadIdx.x, lane = lane_id(), wave = gd_wave();
  const int col = lane & 31, half = lane >> 5;
  uint16_t* x_s = reinterpret_cast<uint16_t*>(sm) + wave * 32 * LDB;           // this wave's rows of X
  uint16_t* mt_s = reinterpret_cast<uint16_t*>(sm) + NW * 32 * LDB;            // [3][32][LDB] pieces of Mt
  const int h = blockIdx.y, s = blockIdx.x;
  const int b = h / hq, head = h % hq;
  const int64_t xhead = (int64_t)b * xh + head / (hq / xh);
  const bf16_t* Xh = X + xhead * l * d;
  float* Ah = A + (int64_t)h * l * r;
  const bool apply = Mt != nullptr;
  const bool full_rows = d == 32 * NB;

  if (apply) {
    const float* Mh = Mt + (int64_t)h * r * d;
    for (int e = tid; e < 32 * 32 * NB; e += NT) {
      const int n = e / (32 * NB), k = e % (32 * NB);
      const float v = Mh[min(n, r - 1) * d + min(k, d - 1)];
      uint32_t p0, p1, p2;
      pf_split3((n < r && k < d) ? v : 0.0f, p0, p1, p2);
      mt_s[(0 * 32 + n) * LDB + k] = (uint16_t)(p0 >> 16);
      mt_s[(1 * 32 + n) * LDB + k] = (uint16_t)(p1 >> 16);
      mt_s[(2 * 32 + n) * LDB + k] = (uint16_t)(p2 >> 16);
    }
  }
  for (int e = lane; e < 32 * LDB / 2; e += kWave) reinterpret_cast<uint32_t*>(x_s)[e] = 0u;

  const int64_t rows_per_split = (((l + S - 1) / S) + 31) / 32 * 32;
  const int64_t r0 = (int64_t)s * rows_per_split;
  const int64_t r1 = min(l, r0 + rows_per_split);

  floatx16 gAA;
  floatx16 gAX[NB];
#pragma unroll
  for (int v = 0; v < 16; ++v) gAA[v] = 0.0f;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int v = 0; v < 16; ++v) gAX[nb][v] = 0.0f;
  float dsum = 0.0f;
  // B operand of the identity product for the two 16-column halves of a 32-column block: element j of
  // lane (col, half) is row 16 kb2 + 8 half + j of the identity, column col
  bf16x8 ident[2];
#pragma unroll
  for (int kb2 = 0; kb2 < 2; ++kb2) {
    uint32_t w[4];
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int k0 = 16 * kb2 + 8 * half + 2 * jj;
      w[jj] = (col == k0 ? 0x3f80u : 0u) | (col == k0 + 1 ? 0x3f800000u : 0u);  // bf16 1.0 = 0x3f80
    }
    ident[kb2] = pf_bf16x8(w[0], w[1], w[2], w[3]);
  }

  uint4 pre[NL];
  auto issue = [&](int64_t t0) {
    const int nvalid = t0 < r1 ? (int)min((int64_t)32, r1 - t0) * d : 0;
    const int64_t base = (t0 < r1 ? t0 : r0) * d;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = (((i + wave) % NL) * kWave + lane) * VEC;  // (the waves start at different KB of their tiles)
      pre[i] = gd_at<uint4>(Xh + base, 2u * (uint32_t)(e < nvalid ? e : 0));
    }
  };
  if (r0 + (int64_t)wave * 32 < r1) issue(r0 + (int64_t)wave * 32);
  __syncthreads();  // Mt staged, tiles cleared

  for (int64_t t0 = r0 + (int64_t)wave * 32; t0 < r1; t0 += 32 * NW) {
    const int rows = (int)min((int64_t)32, r1 - t0);
    {
      const int nvalid = rows * d;
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int e = (((i + wave) % NL) * kWave + lane) * VEC;
        if (e < 32 * d) {
          const int row = full_rows ? e / (32 * NB) : e / d;
          const int c0 = full_rows ? e % (32 * NB) : e - row * d;
          *reinterpret_cast<uint4*>(&x_s[row * LDB + c0]) = e < nvalid ? pre[i] : make_uint4(0, 0, 0, 0);
        }
      }
    }
    pf_wave_sync();
    floatx16 c;
    float old[16];
    if (t0 + 32 * NW < r1) issue(t0 + 32 * NW);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t rr = min(t0 + pf_mfma_row(lane, v), l - 1);
      old[v] = Ah[rr * r + min(col, r - 1)];
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) c[v] = 0.0f;
    auto x_op = [&](int kb) {  // rows of X as an A operand: row col, columns 16 kb + 8 half .. + 7
      return *reinterpret_cast<const bf16x8*>(&x_s[col * LDB + kb * 16 + 8 * half]);
    };
    if (apply) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const bf16x8 a = x_op(kb);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          const bf16x8 m = *reinterpret_cast<const bf16x8*>(&mt_s[(p * 32 + col) * LDB + kb * 16 + 8 * half]);
          c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, m, c, 0, 0, 0);
        }
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = pf_mfma_row(lane, v);
        if (row < rows && col < r) {
          const float df = old[v] - c[v];
          dsum = fmaf(df, df, dsum);
          Ah[(t0 + row) * r + col] = c[v];
        }
      }
    } else {
      const int valid = (col < r ? rows : 0) - 4 * half;
#pragma unroll
      for (int v = 0; v < 16; ++v) c[v] = gd_mfma_row0(v) < valid ? old[v] : 0.0f;
    }
    // the three pieces of C, eight rows (one k block) at a time
    bf16x8 cp[3][2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      uint32_t pc[3][8];
#pragma unroll
      for (int j = 0; j < 8; ++j) pf_split3(c[8 * kb + j], pc[0][j], pc[1][j], pc[2][j]);
#pragma unroll
      for (int p = 0; p < 3; ++p)
        cp[p][kb] = pf_bf16x8(pf_pack2(pc[p][0], pc[p][1]), pf_pack2(pc[p][2], pc[p][3]), pf_pack2(pc[p][4], pc[p][5]),
                              pf_pack2(pc[p][6], pc[p][7]));
    }
    // The matrix cores do not round to nearest when they add to their accumulator: over thousands of
    // additions to a growing sum that is a bias (measured: -2e-5 relative on a sum of 16K squares, ten times
    // the fp32 pipe's).  So a tile's products are summed in a fresh accumulator, smallest pieces first, and
    // the tile's sum joins the running total by an ordinary fp32 addition.
    {
      floatx16 t;
#pragma unroll
      for (int v = 0; v < 16; ++v) t[v] = 0.0f;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[1][kb], cp[2][kb], t, 0, 0, 0);
        t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[2][kb], cp[1][kb], t, 0, 0, 0);
        t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[0][kb], cp[2][kb], t, 0, 0, 0);
        t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[2][kb], cp[0][kb], t, 0, 0, 0);
      }
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[1][kb], cp[1][kb], t, 0, 0, 0);
        t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[0][kb], cp[1][kb], t, 0, 0, 0);
        t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[1][kb], cp[0][kb], t, 0, 0, 0);
      }
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[0][kb], cp[0][kb], t, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 16; ++v) gAA[v] += t[v];
    }
    // per 32 columns of X: the block in the accumulator layout (identity product), packed to bf16 --
    // xb[kb] = this lane's eight rows of k block kb, column 32 nb + col -- then its Gram products
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      floatx16 xa;
#pragma unroll
      for (int v = 0; v < 16; ++v) xa[v] = 0.0f;
      xa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x_op(2 * nb), ident[0], xa, 0, 0, 0);
      xa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x_op(2 * nb + 1), ident[1], xa, 0, 0, 0);
      bf16x8 xb[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        xb[kb] = pf_bf16x8(pf_pack2(__float_as_uint(xa[8 * kb + 0]), __float_as_uint(xa[8 * kb + 1])),
                           pf_pack2(__float_as_uint(xa[8 * kb + 2]), __float_as_uint(xa[8 * kb + 3])),
                           pf_pack2(__float_as_uint(xa[8 * kb + 4]), __float_as_uint(xa[8 * kb + 5])),
                           pf_pack2(__float_as_uint(xa[8 * kb + 6]), __float_as_uint(xa[8 * kb + 7])));
      floatx16 t;
#pragma unroll
      for (int v = 0; v < 16; ++v) t[v] = 0.0f;
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[p][kb], xb[kb], t, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 16; ++v) gAX[nb][v] += t[v];
    }
    pf_wave_sync();  // this wave's reads of the tile precede its next staging writes
  }
  __syncthreads();  // every wave is done with its tile (and with Mt): the LDS is reused below

  // reduce the waves' tiles through LDS, one 32 x 32 block at a time (tile nb of G_AX: columns 32 nb + n)
  const int ne = r * (r + d);
  float* out = part + ((int64_t)h * S + s) * ne;
  for (int blk = 0; blk <= NB; ++blk) {
    float* mine = sm + wave * 1024;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float val = gAA[v];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        if (blk == nb + 1) val = gAX[nb][v];
      mine[pf_mfma_row(lane, v) * 32 + col] = val;
    }
    __syncthreads();
    for (int e = tid; e < 1024; e += NT) {
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += sm[w * 1024 + e];
      const int m = e >> 5, n = e & 31;
      if (blk == 0) {
        if (m < r && n < r) out[m * (r + d) + n] = v;
      } else {
        const int cx = 32 * (blk - 1) + n;
        if (m < r && cx < d) out[m * (r + d) + r + cx] = v;
      }
    }
    __syncthreads();
  }
  if (apply) {
    dsum = wave_sum(dsum);
    if (lane == 0) red[wave] = dsum;
    __syncthreads();
    if (tid == 0) {
      float t = 0.0f;
      for (int w = 0; w < NW; ++w) t += red[w];
      delta_part[(int64_t)h * S + s] = t;
    }
  }
}

// ---- small per-head systems, r <= 32: X = G^-1 RHS for a packed block [G (r x r) | RHS (r x d)] in LDS.
// Gauss-Jordan elimination of [G | RHS] as symmetric sweeps on the matrix cores, 64 columns of the
// right-hand side per wave (every wave repeats the sweeps of G itself).  No pivoting: G is a Gram matrix
// (plus B B^T), positive definite.
struct PfSmallShared {
  __align__(16) float scale[kPfSmallThreads / kWave][32];  // row scales of the solve each wave has in flight
};

// X = G^-1 RHS for the packed block G0 = [G (r x r) | RHS (r x d)] in LDS: the waves of the workgroup share
// the 32-column blocks of the right-hand side, two (cb0, cb0 + 1) per solve; emit(i, j, x) for i < r, j < d.
template <int PIVOTS, typename Emit>
__device__ __forceinline__ void pf_solve_blocks(const float* G0, int r, int d, int cb0, float* scale, Emit&& emit) {
  const int ld = r + d;
  solve_sweep_mfma<2, PIVOTS>([&](int i, int j) { return G0[min(i, r - 1) * ld + min(j, r - 1)]; },
                              [&](int b, int i, int col) {
                                const int j = (cb0 + b) * 32 + col;
                                const float x = G0[min(i, r - 1) * ld + r + min(j, d - 1)];
                                return j < d ? x : 0.0f;
                              },
                              r, scale,
                              [&](int b, int i, int col, float x) {
                                const int j = (cb0 + b) * 32 + col;
                                if (j < d) emit(i, j, x);
                              });
}

// dst[side][e] = sum of the S partial [r][r+d] blocks of a side, in their order; up to NB partials of an element (four
// elements at a time where the blocks allow it) are requested before the first is added.
template <typename V, int NV>
__device__ __forceinline__ void pf_reduce_vec(const float* __restrict__ pq, const float* __restrict__ pk, int S, int ne,
                                              int sides, float* dst) {
  constexpr int NB = 16;
  const int nv = ne / NV;
  for (int t = threadIdx.x; t < sides * nv; t += kPfSmallThreads) {
    const int side = t >= nv ? 1 : 0, e = (t - side * nv) * NV;
    const float* src = (side ? pk : pq) + e;
    float v[NV];
    double w[NV];  // (more than 16 partial sums -- long prompts -- are added in fp64)
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      v[q] = 0.0f;
      w[q] = 0.0;
    }
    for (int s0 = 0; s0 < S; s0 += NB) {
      V x[NB];
#pragma unroll
      for (int u = 0; u < NB; ++u)
        if (s0 + u < S) x[u] = *reinterpret_cast<const V*>(src + (int64_t)(s0 + u) * ne);  // (uniform)
#pragma unroll
      for (int u = 0; u < NB; ++u)
        if (s0 + u < S) {
          const float* xf = reinterpret_cast<const float*>(&x[u]);
#pragma unroll
          for (int q = 0; q < NV; ++q) {
            v[q] += xf[q];
            w[q] += (double)xf[q];
          }
        }
    }
#pragma unroll
    for (int q = 0; q < NV; ++q) dst[side * ne + e + q] = S > 16 ? (float)w[q] : v[q];
  }
}
__device__ __forceinline__ void pf_reduce_part(const float* pq, const float* pk, int S, int ne, int sides, float* dst) {
  if (ne % 4 == 0)  // (blocks start at multiples of 16 bytes then)
    pf_reduce_vec<float4, 4>(pq, pk, S, ne, sides, dst);
  else
    pf_reduce_vec<float, 1>(pq, pk, S, ne, sides, dst);
}

// G0[i][c] (packed [r][r+d]) <- G[i][c] + (c < r ? (B B^T)[i][c] : B[i][c-r]),  B in LDS [r][d+4], d % 4 == 0
__device__ __forceinline__ void pf_add_bbt(const float* G, const float* Bs, int r, int d, float* G0) {
  const int ldb = d + 4;
  // right-hand side block
  for (int e = threadIdx.x; e < r * d; e += kPfSmallThreads) {
    const int i = e / d, c = e - i * d;
    G0[i * (r + d) + r + c] = G[i * (r + d) + r + c] + Bs[i * ldb + c];
  }
  // Gram block: lanes run over c (16-byte reads, conflict-free at this row stride), i is wave-uniform
  for (int o = threadIdx.x; o < 32 * r; o += kPfSmallThreads) {
    const int i = o >> 5, c = o & 31;
    if (c < r) {
      const float4* bi = reinterpret_cast<const float4*>(Bs + i * ldb);
      const float4* bc = reinterpret_cast<const float4*>(Bs + c * ldb);
      float g0 = 0.0f, g1 = 0.0f;
      for (int x = 0; x < d / 4; ++x) {
        const float4 a = bi[x], b = bc[x];
        g0 = fmaf(a.x, b.x, g0); g1 = fmaf(a.y, b.y, g1);
        g0 = fmaf(a.z, b.z, g0); g1 = fmaf(a.w, b.w, g1);
      }
      G0[i * (r + d) + c] = G[i * (r + d) + c] + (g0 + g1);
    }
  }
}

// stage 0: (stopping test) B_Q, B_K from the current Grams, then Mt for the A_Q update
// stage 1: Mt for the A_K update from the new A_Q Grams
// stage 2: final B_Q, B_K
// One workgroup per head: latency of the partial sums (3 us) and of two solves in a row.  28 heads, rank 16, 9 splits,
// stages 0, 1, 2: 43, 21, 32 -> 18, 11, 9 us (sums requested at once, pivots without tests and copies, one place for
// all solves instead of three: 88 -> 18 KB of code); same results to the bit.
template <int PIVOTS>
__global__ __launch_bounds__(kPfSmallThreads) void pf_small32_kernel(int stage, int it, const float* __restrict__ partQ,
                                                                     const float* __restrict__ partK, int S, int bh,
                                                                     int r, int d, int64_t l, float tol,
                                                                     const float* __restrict__ delta_all,
                                                                     int* __restrict__ flags, float* __restrict__ Mt,
                                                                     float* __restrict__ b_q, float* __restrict__ b_k) {
  extern __shared__ __align__(16) float sm[];
  const int ne = r * (r + d);
  float* G1 = sm;            // [r][r+d] packed
  float* G2 = G1 + ne;       // [r][r+d] packed
  float* G0 = G2 + ne;       // [r][r+d] packed, system being solved
  float* Bs = sm + ((3 * ne + 3) & ~3);  // [r][d+4], 16-byte aligned
  __shared__ PfSmallShared sh;
  __shared__ int s_done;
  __shared__ float s_red[kPfSmallThreads / kWave][2];
  const int tid = threadIdx.x;
  const int h = blockIdx.x;
  const int wave = wave_id();
  constexpr int kWaves = kPfSmallThreads / kWave;
  const int njob = (d + 63) / 64;  // pairs of 32-column blocks of a right-hand side

  if (stage == 0) {
    int done = 0;
    if (it > 0) {
      done = flags[it - 1];
      if (!done) {
        const float* dq = delta_all + ((int64_t)(it - 1) * 2 + 0) * bh * S;
        const float* dk = delta_all + ((int64_t)(it - 1) * 2 + 1) * bh * S;
        float sq = 0.0f, sk = 0.0f;
        for (int i = tid; i < bh * S; i += kPfSmallThreads) {
          sq += dq[i];
          sk += dk[i];
        }
        sq = wave_sum(sq);
        sk = wave_sum(sk);
        if (lane_id() == 0) {
          s_red[wave_id()][0] = sq;
          s_red[wave_id()][1] = sk;
        }
        __syncthreads();
        if (tid == 0) {
          float tq = 0.0f, tk = 0.0f;
          for (int w = 0; w < kPfSmallThreads / kWave; ++w) {
            tq += s_red[w][0];
            tk += s_red[w][1];
          }
          const float n = (float)bh * (float)l * (float)r;
          s_done = fmaxf(tq / n, tk / n) < tol;
        }
        __syncthreads();
        done = s_done;
      }
    }
    // every head computes the same decision from data that no launch of this iteration overwrites
    if (h == 0 && tid == 0) flags[it] = done;
    if (done) return;
  } else if (stage == 1) {
    if (flags[it]) return;
  }

  const float* pq = partQ + (int64_t)h * S * ne;
  const float* pk = partK + (int64_t)h * S * ne;
  const int64_t hrd = (int64_t)h * r * d;
  pf_reduce_part(pq, pk, S, ne, stage == 1 ? 1 : 2, G1);
  if (stage == 1)
    for (int e = tid; e < r * d; e += kPfSmallThreads) Bs[(e / d) * (d + 4) + e % d] = b_k[hrd + e];
  __syncthreads();
  // Stages 0 and 2: B_Q = (A_Q^T A_Q)^-1 A_Q^T Q and B_K likewise, both systems side by side, two column blocks per wave.
  // Then (stages 0 and 1) G0 and Mt.  (One place for both solves: the sweeps are a lot of code.)
  for (int part = stage == 1 ? 1 : 0; part < (stage == 2 ? 1 : 2); ++part) {
    if (part == 1) {
      // Mt_Q = (A_K^T A_K + B_Q B_Q^T)^-1 (A_K^T K + B_Q),  Mt_K = (A_Q^T A_Q + B_K B_K^T)^-1 (A_Q^T Q + B_K)
      pf_add_bbt(stage == 0 ? G2 : G1, Bs, r, d, G0);
      __syncthreads();
    }
    for (int job = wave; job < (part == 1 ? njob : 2 * njob); job += kWaves) {
      const bool k_side = job >= njob;
      float* out = (part == 1 ? Mt : k_side ? b_k : b_q) + hrd;
      const bool keep = part == 0 && !k_side;
      pf_solve_blocks<PIVOTS>(part == 1 ? G0 : k_side ? G2 : G1, r, d, 2 * (k_side ? job - njob : job), sh.scale[wave],
                              [&](int i, int j, float x) {
                                if (keep) Bs[i * (d + 4) + j] = x;
                                out[i * d + j] = x;
                              });
    }
    __syncthreads();
  }
}

// ============================================================================ ranks 33 .. 64, fp32 rows of 64 or 128
// The products of the fp32 matrix cores are chains of fused multiply-adds in the order of their k index
// (32x32x2 and 16x16x4 alike), so tiles of 16 x 16 that take a sum's terms in the general kernels' order have the
// general kernels' results to the bit: the columns of a row for C = X Mt^T, the rows of a split for A^T [A | X].
constexpr int kPfWideThreads = 512;
// Row strides of 20 floats beyond a multiple of 64: an operand of 16 rows x 4 columns meets every bank once, one of
// 4 rows x 16 columns a few twice.
constexpr int kPfWideLda = 64 + 20;

// One workgroup per split and head, 32 rows at a time.  Apply: wave w has the tile of rows 16 (w % 2), columns 16 (w / 2)
// of C.  Sums: wave w has rank columns 16 (w / 2) and half of the tiles of [A | X].  Bound by the matrix cores (5 K of a
// tile's 8 K cycles) and three barriers a tile.  24 heads of 2091 rows, rank 64: 142 -> 35 us a pass.
template <int D>
__global__ __launch_bounds__(kPfWideThreads, 4) void pf_pass_wide_kernel(const float* __restrict__ X, int xh, int hq,
                                                                         int64_t l, int r, int, const float* __restrict__ Mt,
                                                                         float* __restrict__ A, float* __restrict__ part,
                                                                         float* __restrict__ delta_part,
                                                                         const int* __restrict__ done_flag, int S) {
  if (done_flag && *done_flag) return;
  constexpr int LDX = D + 20, LDA = kPfWideLda, NT = kPfWideThreads;
  constexpr int NX = 32 * D / (NT * 4);        // 16-byte loads of X per thread and tile
  constexpr int NA = 32 * 64 / NT;             // elements of A per thread and tile
  constexpr int NC = (4 + D / 16) / 2;         // tiles of [A | X] per wave
  extern __shared__ __align__(16) float sm[];
  float* x_s = sm;               // [32][LDX]
  float* a_s = x_s + 32 * LDX;   // [32][LDA], zero beyond r and beyond the last row
  float* m_s = a_s + 32 * LDA;   // [64][LDX]  Mt (apply only)
  __shared__ float red[NT / kWave];
  const int tid = threadIdx.x, lane = lane_id(), wave = gd_wave();
  const int li = lane & 15, lk = lane >> 4;
  const int h = blockIdx.y, s = blockIdx.x;
  const int b = h / hq, head = h % hq;
  const float* Xh = X + ((int64_t)b * xh + head / (hq / xh)) * l * D;
  float* Ah = A + (int64_t)h * l * r;
  const bool apply = Mt != nullptr;
  if (apply)
    for (int e = tid; e < 64 * D; e += NT) {
      const int n = e / D, k = e % D;
      m_s[n * LDX + k] = n < r ? Mt[((int64_t)h * r + n) * D + k] : 0.0f;
    }
  const int64_t rows_per_split = (l + S - 1) / S;
  const int64_t r0 = (int64_t)s * rows_per_split;
  const int64_t r1 = min(l, r0 + rows_per_split);
  const int jt = wave >> 1, tr = wave & 1;     // apply: tile (tr, jt) of C; sums: rows jt, tiles tr * NC .. of [A | X]
  float4 pre_x[NX];
  float pre_a[NA];                             // given: rows of A as they go to LDS; apply: the old values of the tile of C
  auto issue = [&](int64_t t0) {
    const int last = (int)min((int64_t)32, r1 - t0) - 1;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int e = (i * NT + tid) * 4;
      pre_x[i] = *reinterpret_cast<const float4*>(Xh + (t0 + min(e / D, last)) * D + e % D);
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int row = apply ? 16 * tr + 4 * lk + i : (i * NT + tid) / 64, j = apply ? 16 * jt + li : tid % 64;
      pre_a[i] = Ah[(t0 + min(row, last)) * r + min(j, r - 1)];
    }
  };
  static_assert(NA == 4, "a lane's four elements of a tile of C");
  floatx4 acc[NC];
#pragma unroll
  for (int n = 0; n < NC; ++n) acc[n] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  float dsum = 0.0f;
  if (r0 < r1) issue(r0);
  for (int64_t t0 = r0; t0 < r1; t0 += 32) {
    const int rows = (int)min((int64_t)32, r1 - t0);
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int e = (i * NT + tid) * 4;
      *reinterpret_cast<float4*>(&x_s[e / D * LDX + e % D]) = e / D < rows ? pre_x[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    float old[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      old[i] = pre_a[i];
      if (!apply) {
        const int row = (i * NT + tid) / 64, j = tid % 64;
        a_s[row * LDA + j] = row < rows && j < r ? old[i] : 0.0f;
      }
    }
    __syncthreads();  // (the first one also covers the staging of Mt)
    if (t0 + 32 < r1) issue(t0 + 32);
    if (apply) {
      floatx4 c = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
      const float* xa = x_s + (16 * tr + li) * LDX + lk;
      const float* mb = m_s + (16 * jt + li) * LDX + lk;
#pragma unroll 8
      for (int k = 0; k < D; k += 4) c = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[k], mb[k], c, 0, 0, 0);
      const int j = 16 * jt + li;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * tr + 4 * lk + v;
        const bool ok = row < rows && j < r;
        if (ok) {
          const float df = old[v] - c[v];
          dsum = fmaf(df, df, dsum);
          Ah[(t0 + row) * r + j] = c[v];
        }
        a_s[row * LDA + j] = ok ? c[v] : 0.0f;
      }
      __syncthreads();
    }
    const float* aa = a_s + lk * LDA + 16 * jt + li;
#pragma unroll
    for (int k = 0; k < 32; k += 4) {
      const float av = aa[k * LDA];
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        const int ct = tr * NC + n;  // (wave-uniform)
        const float bv = ct < 4 ? a_s[(k + lk) * LDA + 16 * ct + li] : x_s[(k + lk) * LDX + 16 * (ct - 4) + li];
        acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv, acc[n], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  const int ld = r + D;
  float* out = part + ((int64_t)h * S + s) * r * ld;
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    const int ct = tr * NC + n, c = 16 * (ct < 4 ? ct : ct - 4) + li;
    if (ct < 4 && c >= r) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = 16 * jt + 4 * lk + v;
      if (j < r) out[j * ld + (ct < 4 ? c : r + c)] = acc[n][v];
    }
  }
  if (apply) {
    dsum = wave_sum(dsum);
    if (lane == 0) red[wave] = dsum;
    __syncthreads();
    if (tid == 0) {
      float t = 0.0f;
      for (int w = 0; w < NT / kWave; ++w) t += red[w];
      delta_part[(int64_t)h * S + s] = t;
    }
  }
}

// The stages of pf_small_generic_kernel for 32 < r <= 64 and d <= 128, with its operations in its order (same results to
// the bit; the sums of the stopping test alone are taken in another order, by all threads instead of one): wave w keeps
// rows 8 w .. 8 w + 7 of [G | RHS] in registers, lane and column lane + 64 k; a pivot row goes round through LDS, one
// barrier per pivot (two slots).  Workgroup (h, 0): B_Q (stages 0 and 2), then Mt; (h, 1): B_K.
// A dependent chain of 0.2 us a pivot: 24 heads, rank 64: 947 -> 104 us a stage (median).
constexpr int kPfWideLdb = 128 + 20;
__global__ __launch_bounds__(kPfWideThreads, 2) void pf_small_wide_kernel(
    int stage, int it, const float* __restrict__ partQ, const float* __restrict__ partK, int S, int bh, int r, int d, int64_t l,
    float tol, const float* __restrict__ delta_all, int* __restrict__ flags, float* __restrict__ Mt, float* __restrict__ b_q,
    float* __restrict__ b_k) {
  constexpr int NT = kPfWideThreads, NW = NT / kWave;
  static_assert(NW * 8 == 64, "64 rows");
  __shared__ __align__(16) float Bs[64][kPfWideLdb];  // B, zero beyond r and d
  __shared__ float GG[64][65];                        // B B^T
  __shared__ float prow[2][192];
  __shared__ float red[2][NW];
  const int tid = threadIdx.x, lane = lane_id(), wave = gd_wave();
  const int li = lane & 15, lk = lane >> 4;
  const int h = blockIdx.x;
  const bool k_side = blockIdx.y != 0;
  if (stage == 1 && k_side) return;
  const int ld = r + d, ne = r * ld;
  const int64_t hrd = (int64_t)h * r * d;
  if (stage == 0) {
    int done = 0;
    if (it > 0) {
      const float* dq = delta_all + ((int64_t)(it - 1) * 2 + 0) * bh * S;
      const float* dk = delta_all + ((int64_t)(it - 1) * 2 + 1) * bh * S;
      done = flags[it - 1];
      float sq = 0.0f, sk = 0.0f;
      for (int i = tid; i < bh * S; i += NT) {
        sq += dq[i];
        sk += dk[i];
      }
      sq = wave_sum(sq);
      sk = wave_sum(sk);
      if (lane == 0) {
        red[0][wave] = sq;
        red[1][wave] = sk;
      }
      __syncthreads();
      sq = sk = 0.0f;
      for (int w = 0; w < NW; ++w) {
        sq += red[0][w];
        sk += red[1][w];
      }
      const float n = (float)bh * (float)l * (float)r;
      done = done || fmaxf(sq / n, sk / n) < tol;
    }
    // (every workgroup computes the same decision; nothing it reads is overwritten by a launch of this iteration)
    if (h == 0 && !k_side && tid == 0) flags[it] = done;
    if (done) return;
  } else if (stage == 1) {
    if (flags[it]) return;
  }

  float M[8][3];  // rows 8 wave + e, columns lane + 64 k of [G | RHS]
  // the sum of a side's partial blocks, in split order (more than 16 of them in fp64)
  auto load_sums = [&](const float* part) {
    const float* src = part + (int64_t)h * S * ne;
    int at[8][3];
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        at[e][k] = min(8 * wave + e, r - 1) * ld + min(lane + 64 * k, ld - 1);
        M[e][k] = 0.0f;
      }
    if (S <= 16) {
#pragma unroll 2
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int k = 0; k < 3; ++k) M[e][k] += src[(int64_t)s * ne + at[e][k]];
    } else {
      double w[8][3];
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int k = 0; k < 3; ++k) w[e][k] = 0.0;
#pragma unroll 2
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int k = 0; k < 3; ++k) w[e][k] += (double)src[(int64_t)s * ne + at[e][k]];
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int k = 0; k < 3; ++k) M[e][k] = (float)w[e][k];
    }
  };
  // Gauss-Jordan without pivoting: columns beyond the pivot's of every row but its own; then X = RHS / diagonal.
  auto solve = [&](float* out, bool keep) {
    for (int pw = 0; 8 * pw < r; ++pw) {
#pragma unroll
      for (int pe = 0; pe < 8; ++pe) {
        const int p = 8 * pw + pe;
        if (p >= r) break;  // (uniform)
        float* row = prow[pe & 1];
        if (wave == pw) {
#pragma unroll
          for (int k = 0; k < 3; ++k) row[lane + 64 * k] = M[pe][k];
        }
        __syncthreads();
        const float x0 = row[lane], x1 = row[lane + 64], x2 = row[lane + 128];
        const float inv = 1.0f / row[p];
        const bool beyond = lane > p;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (e == pe && wave == pw) continue;  // (wave-uniform)
          const float mp = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(M[e][0]), p));
          const float f = -(mp * inv);
          const float m0 = fmaf(f, x0, M[e][0]);
          M[e][0] = beyond ? m0 : M[e][0];
          M[e][1] = fmaf(f, x1, M[e][1]);
          M[e][2] = fmaf(f, x2, M[e][2]);
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i = 8 * wave + e;
      if (i >= r) break;  // (wave-uniform)
      const float diag = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(M[e][0]), i));
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int c = lane + 64 * k - r;
        if (c >= 0 && c < d) {
          const float v = M[e][k] / diag;
          out[hrd + i * d + c] = v;
          if (keep) Bs[i][c] = v;
        }
      }
    }
  };
  // M <- M + [B B^T | B]
  auto add_b = [&] {
    __syncthreads();
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int ti = wave >> 1, tj = 2 * (wave & 1) + n;
      floatx4 g = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
      for (int k = 0; k < 128; k += 4)
        if (k < d)  // (uniform; what lies beyond d is zero)
          g = __builtin_amdgcn_mfma_f32_16x16x4f32(Bs[16 * ti + li][k + lk], Bs[16 * tj + li][k + lk], g, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 4; ++v) GG[16 * ti + 4 * lk + v][16 * tj + li] = g[v];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int i = 8 * wave + e, c = lane + 64 * k;
        if (c < r)
          M[e][k] += GG[i][c];
        else if (c < ld)
          M[e][k] += Bs[i][c - r];
      }
  };

  if (stage != 2 && !k_side)
    for (int e = tid; e < 64 * kPfWideLdb; e += NT) {
      const int i = e / kPfWideLdb, c = e % kPfWideLdb;
      Bs[i][c] = stage == 1 && i < r && c < d ? b_k[hrd + i * d + c] : 0.0f;
    }
  __syncthreads();
  if (stage != 1) {
    load_sums(k_side ? partK : partQ);
    solve(k_side ? b_k : b_q, !k_side && stage == 0);
    if (k_side || stage == 2) return;
  }
  // Mt_Q = (A_K^T A_K + B_Q B_Q^T)^-1 (A_K^T K + B_Q),  Mt_K = (A_Q^T A_Q + B_K B_K^T)^-1 (A_Q^T Q + B_K)
  load_sums(stage == 0 ? partK : partQ);
  add_b();
  solve(Mt, false);
}

__global__ void clear_flags_kernel(int* flags, int n) {  // (a kernel: the launches may be captured into a graph)
  for (int i = threadIdx.x; i < n; i += blockDim.x) flags[i] = 0;
}

template <typename T>
using PfPassFn = void (*)(const T*, int, int, int64_t, int, int, const float*, float*, float*, float*, const int*, int);

template <typename T>
static int prefill_impl(lrqk_ctx* ctx, const void* q, const void* k, float* a_q, float* a_k, const PrefillOut& out, int b,
                        int hq, int hkv, int64_t l, int r, int d, int max_iter, float tol, hipStream_t st) {
  constexpr int VEC = Vec16<T>::N;
  const int bh = b * hq;
  const int ne = r * (r + d);
  const int iters = max_iter > 0 ? max_iter : 0;
  const bool aligned = ((uintptr_t)q % 16 == 0) && ((uintptr_t)k % 16 == 0);
  // Every iteration on d x d Gram matrices in fp64, the rows read twice (sums, result) whatever the iteration count:
  // bf16 rows of 64 or 128 elements.  A prompt of fewer rows than two Gram matrices has is left to the row-by-row
  // formulation (X^T X is then no smaller than X, and with about as many rows as the rank both are ill-posed), except
  // rows of 128 elements at ranks up to 32.
  // fp32 rows stay with the row-by-row formulation.  Its factors are 5e-6 .. 8e-5 off the ones from Gram matrices, and a
  // decode step of an ill-conditioned head makes up to 4e-4 of that (a token at the edge of the active set changes
  // places): more than fp32 results may move, whichever side is the closer one.
  // LRQK_PREFILL_ROWWISE, for comparisons: every prompt row by row; `general`: ranks above 32 by the general kernels
  const char* const rowwise = getenv("LRQK_PREFILL_ROWWISE");
  const bool general = rowwise && !strcmp(rowwise, "general");
  if constexpr (sizeof(T) == 2) {
    const bool gram_domain = aligned && (d == 64 || d == 128) && !rowwise &&
                             ((d == 128 && r <= 32) || l >= 2 * d);
    if (gram_domain)
      return prefill_gram_domain(ctx, (const T*)q, (const T*)k, a_q, a_k, out, b, hq, hkv, l, r, d, iters, tol, st);
  }
  const bool mfma = r <= 32 && d % VEC == 0 && d <= 256 && aligned;
  const bool small32 = r <= 32 && d <= 288 && d % 4 == 0;
  LRQK_REQUIRE(mfma || ne <= kPfThreads * kPfMaxPer, LRQK_ELIMIT, "r*(r+d)=%d exceeds %d", ne, kPfThreads * kPfMaxPer);
  // (the general pass: a 16 x 16 thread grid with ceil(r / 16) rows and 48 / that many columns of the sums per thread)
  LRQK_REQUIRE(mfma || (r <= 64 && 16 * (kPfMaxPer / ((r + 15) / 16)) >= r + d), LRQK_ELIMIT,
               "r=%d with rows of %d elements exceeds the general kernel's tile", r, d);
  // splits of the long axis: about one workgroup per CU (a pass keeps one wave per SIMD busy), but
  // at least 128 rows per split
  int S = std::max(1, std::min(64, 256 / bh));
  // This formulation solves its r x r systems from these sums in fp32, and a split adds its rows up in
  // fp32: at most 2048 rows per split there (the partial sums are added in fp64), however few splits fill the GPU.
  // (At most 64 splits per head: beyond 128K rows a split adds up l / 64 rows.)
  S = (int)std::min<int64_t>(64, std::max<int64_t>(S, (l + 2047) / 2048));
  S = (int)std::max<int64_t>(1, std::min<int64_t>(S, (l + 127) / 128));
  // workspace: partQ, partK, Mt, b_q, b_k, deltas[iters][2][bh][S], flags[iters+1]
  const size_t n_part = (size_t)bh * S * ne;
  const size_t n_mt = (size_t)bh * r * d;
  const size_t n_delta = (size_t)(iters > 0 ? iters : 1) * 2 * bh * S;
  const size_t total = (2 * n_part + 3 * n_mt + n_delta) * sizeof(float) + (size_t)(iters + 1) * sizeof(int);
  int rc = ctx->prefill_ws.ensure(total);
  if (rc) return rc;
  float* partQ = (float*)ctx->prefill_ws.p;
  float* partK = partQ + n_part;
  float* Mt = partK + n_part;
  const bool convert = out.storage && sizeof(T) == 2;
  float* b_q = convert ? Mt + n_mt : (float*)out.b_q;  // (fp32 results where they go; the place in the workspace stays unused)
  float* b_k = convert ? Mt + 2 * n_mt : (float*)out.b_k;
  float* deltas = Mt + 3 * n_mt;
  int* flags = (int*)(deltas + n_delta);

  PfPassFn<T> pass = pf_pass_generic_kernel<T>;
  size_t smem_pass = ((size_t)kPfTile * (d + 1) + (size_t)kPfTile * (r + 1) + (size_t)r * (d + 1)) * sizeof(float);
  int pass_threads = kPfThreads;
  if (mfma) {
    const int nb = d <= 32 ? 1 : d <= 64 ? 2 : d <= 128 ? 4 : 8;
    pass = nb == 1 ? pf_pass_mfma_kernel<T, 1, 8, true> : nb == 2 ? pf_pass_mfma_kernel<T, 2, 8, true>
         : nb == 4 ? pf_pass_mfma_kernel<T, 4, 8, true> : pf_pass_mfma_kernel<T, 8, 4, false>;
    const int nw = nb == 8 ? 4 : 8;
    pass_threads = nw * kWave;
    smem_pass = std::max((size_t)(nw + (nb == 8 ? 0 : 1)) * 32 * (32 * nb + 4), (size_t)nw * 1024) * sizeof(float);
    if constexpr (sizeof(T) == 2) {
      if (nb <= 4) {  // bf16 input: the pass on the bf16 matrix cores (three-piece split, fp32 accuracy)
        pass = nb == 1 ? pf_pass_bf16_kernel<1, 8> : nb == 2 ? pf_pass_bf16_kernel<2, 8> : pf_pass_bf16_kernel<4, 8>;
        smem_pass = std::max((size_t)(8 + 3) * 32 * (32 * nb + 8) * sizeof(uint16_t), (size_t)8 * 1024 * sizeof(float));
      }
    }
  }
  if constexpr (sizeof(T) == 4) {
    if (mfma && r <= 16 && (d == 64 || d == 128)) {
      pass = d == 64 ? pf_pass_mfma16_kernel<64> : pf_pass_mfma16_kernel<128>;
      smem_pass = d == 64 ? Pf16Shape<64>::SMEM : Pf16Shape<128>::SMEM;
    }
  }
  auto small = !small32 ? pf_small_generic_kernel : r <= 16 ? pf_small32_kernel<16> : pf_small32_kernel<32>;
  const bool wide = sizeof(T) == 4 && r > 32 && r <= 64 && (d == 64 || d == 128) && aligned && !general;
  if constexpr (sizeof(T) == 4) {
    if (wide) {
      pass = d == 64 ? pf_pass_wide_kernel<64> : pf_pass_wide_kernel<128>;
      pass_threads = kPfWideThreads;
      smem_pass = (size_t)(32 * (d + 20) + 32 * kPfWideLda + 64 * (d + 20)) * sizeof(float);
    }
  }
  const bool small_wide = r > 32 && r <= 64 && d <= 128 && !general;
  if (small_wide) small = pf_small_wide_kernel;
  const size_t smem_small = small_wide ? 0 : small32 ? ((size_t)3 * ne + 4 + (size_t)r * (d + 4)) * sizeof(float)
                                    : ((size_t)ne + (size_t)r * (r + d + 1) + (size_t)r * (d + 1)) * sizeof(float);
  LRQK_REQUIRE(smem_small <= 160 * 1024 && smem_pass <= 160 * 1024, LRQK_ELIMIT, "r=%d d=%d need too much LDS", r, d);
  if (smem_pass > 48 * 1024)
    LRQK_HIP_CHECK(hipFuncSetAttribute((const void*)pass, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem_pass));
  if (smem_small > 48 * 1024)
    LRQK_HIP_CHECK(hipFuncSetAttribute((const void*)small, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem_small));
  const dim3 grid((unsigned)S, (unsigned)bh), blk((unsigned)pass_threads);
  const dim3 sgrid((unsigned)bh, small_wide ? 2 : 1), sblk(small_wide ? kPfWideThreads : small32 ? kPfSmallThreads : kPfThreads);
  const T* Q = (const T*)q;
  const T* K = (const T*)k;
  hipLaunchKernelGGL(clear_flags_kernel, dim3(1), dim3(64), 0, st, flags, iters + 1);
  // the sums over the given initial factors
  hipLaunchKernelGGL(pass, grid, blk, smem_pass, st, Q, hq, hq, l, r, d, (const float*)nullptr, a_q, partQ, (float*)nullptr,
                     (const int*)nullptr, S);
  hipLaunchKernelGGL(pass, grid, blk, smem_pass, st, K, hkv, hq, l, r, d, (const float*)nullptr, a_k, partK, (float*)nullptr,
                     (const int*)nullptr, S);
  LRQK_HIP_CHECK(hipGetLastError());
  for (int it = 0; it < iters; ++it) {
    float* dq = deltas + ((size_t)it * 2 + 0) * bh * S;
    float* dk = deltas + ((size_t)it * 2 + 1) * bh * S;
    hipLaunchKernelGGL(small, sgrid, sblk, smem_small, st, 0, it, partQ, partK, S, bh, r, d, l, tol,
                       deltas, flags, Mt, b_q, b_k);
    hipLaunchKernelGGL(pass, grid, blk, smem_pass, st, Q, hq, hq, l, r, d, (const float*)Mt, a_q, partQ, dq,
                       (const int*)(flags + it), S);
    hipLaunchKernelGGL(small, sgrid, sblk, smem_small, st, 1, it, partQ, partK, S, bh, r, d, l, tol,
                       deltas, flags, Mt, b_q, b_k);
    hipLaunchKernelGGL(pass, grid, blk, smem_pass, st, K, hkv, hq, l, r, d, (const float*)Mt, a_k, partK, dk,
                       (const int*)(flags + it), S);
    LRQK_HIP_CHECK(hipGetLastError());
  }
  hipLaunchKernelGGL(small, sgrid, sblk, smem_small, st, 2, iters, partQ, partK, S, bh, r, d, l, tol,
                     deltas, flags, Mt, b_q, b_k);
  LRQK_HIP_CHECK(hipGetLastError());
  auto finish = [&](auto* o_q, auto* o_k, auto* ob_q, auto* ob_k) -> int {
    using OUT = std::remove_reference_t<decltype(*o_q)>;
    const int64_t n = out.a_q_rows * r, rd = (int64_t)bh * r * d;
    int rcs;
    if ((rcs = prefill_store<OUT>(a_q + (l - out.a_q_rows) * r, l * r, o_q, n, n, bh, st))) return rcs;
    if ((rcs = prefill_store<OUT>(a_k, l * r, o_k, out.a_k_stride, l * r, bh, st))) return rcs;
    if ((rcs = prefill_store<OUT>(b_q, rd, ob_q, rd, rd, 1, st))) return rcs;
    return prefill_store<OUT>(b_k, rd, ob_k, rd, rd, 1, st);
  };
  if (convert) return finish((T*)out.a_q, (T*)out.a_k, (T*)out.b_q, (T*)out.b_k);
  return finish((float*)out.a_q, (float*)out.a_k, (float*)out.b_q, (float*)out.b_k);
}

}  // namespace lrqk

using namespace lrqk;

static int prefill_checked(lrqk_ctx* ctx, const void* q, const void* k, float* a_q, float* a_k, const PrefillOut& out, int b,
                           int hq, int hkv, int64_t l, int r, int d, int max_iter, float tol, int dtype, void* stream) {
  LRQK_REQUIRE(ctx && q && k && a_q && a_k && out.a_q && out.a_k && out.b_q && out.b_k, LRQK_EINVAL, "null pointer");
  LRQK_REQUIRE(dtype == LRQK_F32 || dtype == LRQK_BF16, LRQK_EINVAL, "dtype=%d", dtype);
  LRQK_REQUIRE(b > 0 && hq > 0 && hkv > 0 && hq % hkv == 0 && (int64_t)b * hq <= 65535, LRQK_EINVAL,
               "bad heads b=%d hq=%d hkv=%d", b, hq, hkv);
  LRQK_REQUIRE(r > 0 && r <= LRQK_MAX_R && d > 0 && l > 0 && l < ((int64_t)1 << 31), LRQK_EINVAL, "bad sizes r=%d d=%d l=%lld",
               r, d, (long long)l);
  LRQK_REQUIRE(max_iter <= 64, LRQK_ELIMIT, "max_iter=%d > 64", max_iter);
  LRQK_REQUIRE((out.a_q_rows == 1 || out.a_q_rows == l) && out.a_k_stride >= l * r, LRQK_EINVAL,
               "a_q_rows=%lld (1 or all %lld), a_k_stride=%lld", (long long)out.a_q_rows, (long long)l, (long long)out.a_k_stride);
  ctx->pool.enter((hipStream_t)stream);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == LRQK_F32) return prefill_impl<float>(ctx, q, k, a_q, a_k, out, b, hq, hkv, l, r, d, max_iter, tol, st);
  return prefill_impl<bf16_t>(ctx, q, k, a_q, a_k, out, b, hq, hkv, l, r, d, max_iter, tol, st);
}

extern "C" int lrqk_als_prefill(lrqk_ctx* ctx, const void* q, const void* k, float* a_q, float* a_k, float* b_q,
                                float* b_k, int b, int hq, int hkv, int64_t l, int r, int d, int max_iter, float tol,
                                int dtype, void* stream) {
  const PrefillOut out{a_q, a_k, b_q, b_k, l, l * r, false};
  return prefill_checked(ctx, q, k, a_q, a_k, out, b, hq, hkv, l, r, d, max_iter, tol, dtype, stream);
}

extern "C" int lrqk_als_prefill_store(lrqk_ctx* ctx, const void* q, const void* k, float* a_q0, float* a_k0, void* a_q,
                                      int64_t a_q_rows, void* a_k, int64_t a_k_stride, void* b_q, void* b_k, int b, int hq,
                                      int hkv, int64_t l, int r, int d, int max_iter, float tol, int dtype, void* stream) {
  const PrefillOut out{a_q, a_k, b_q, b_k, a_q_rows, a_k_stride, true};
  return prefill_checked(ctx, q, k, a_q0, a_k0, out, b, hq, hkv, l, r, d, max_iter, tol, dtype, stream);
}
