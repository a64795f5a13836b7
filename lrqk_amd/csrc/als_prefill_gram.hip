// Prefill factorisation, iterations carried out on Gram matrices (bf16 rows of 64 or 128 elements, r <= 64).
//
// After the first half-step of lrqk_attention.py:359-421 every factor is a linear image of its input,
// A_Q = Q Mq and A_K = K Mk with Mq, Mk of size d x r.  Everything an iteration needs from the long axis
// is then a product with Sq = Q^T Q or Sk = K^T K (d x d):
//     A_Q^T A_Q = Mq^T Sq Mq,   A_Q^T Q = Mq^T Sq,   Q^T A_Q = Sq Mq   (likewise for K),
// and the change mse(A, A') that the stopping test looks at is
//     |A - A'|^2 = tr(A^T A) - 2 tr((A^T X) M') + tr(A'^T A').
// With (G, C) = (A^T A, A^T X) as the state of each side, one iteration is, in the reference's order
// (Gauss-Seidel: the A_K update sees the new A_Q),
//     B_Q = Gq^-1 Cq,  B_K = Gk^-1 Ck
//     Mq'^T = (Gk + B_Q B_Q^T)^-1 (Ck + B_Q)          T = Mq'^T Sq      Gq' = Mq'^T T^T     Cq' = T
//     Mk'^T = (Gq' + B_K B_K^T)^-1 (T + B_K)          U = Mk'^T Sk      Gk' = Mk'^T U^T     Ck' = U
// and this holds from the first iteration on (there G, C come from the given initial factors).  The long
// axis is read for Sq, Sk and the initial (G, C) before the loop and once more at the end, to form
// A_Q = Q Mq and A_K = K Mk, whatever the iteration count; the row-by-row formulation reads it twice per
// iteration and twice more.
//
// Sq and Sk square the condition number of the inputs, so the d x d algebra is done in fp64 (on the matrix cores, one
// workgroup per head: these are 32 independent problems of a few MFLOP each); the sums Sq, Sk themselves are exact
// bf16 x bf16 products added in fp32 tile by tile and across tiles, then across splits in fp64.  Measured
// against the fp64 restatement the results are closer than the same iteration in fp32 LAPACK.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "ctx.hpp"
#include "prefill_pieces.hpp"

namespace lrqk {

// ----------------------------------------------------------------------------- X^T X and the sums over given factors
// Both sides in one launch, one reading of the rows for all sums: a workgroup stages 128 rows of X and of the given
// factors A (fp32, [head][l][r]) per step and its waves form X^T X and (A^T A, A^T X).  Workgroups [0, bh * S): head and
// split of the Q side; behind them the K side, where the query heads of a kv head take their X from it and X^T X of split
// s is left to head s % nh of the group.  Those heads lie 8 workgroups apart, on one XCD, and walk the same rows at the same
// time: K comes from that XCD's L2 after the first of them.
//
// The rows of A are split into three bf16 pieces (8 + 8 + 8 mantissa bits, exact) on their way to LDS, so every number is
// split once; all operands then come out of LDS by the transposing read.  Wave (g, ch) = (w / 2, w % 2) takes the 32-row
// group g of the step, there two of the four column blocks of A^T X, k block ch of A^T A and five of the ten blocks of X^T X
// on and above the diagonal.  Which: block i of a wave is block i of X for ch = 0 and block (2, 0, 3, 1)[i] for ch = 1, and
// both take the columns 0, 3 and the products (0,0) (3,3) (0,1) (1,2) (2,3) of their own numbering -- the path 0-1-2-3 through
// the four blocks and its complement 2-0-3-1, so the code is the same and only LDS addresses differ.
// Products per 32 rows as in the row-by-row pass: all piece pairs of A^T A except lo x lo, three pieces of A times X; every
// 32-row group in a fresh accumulator (the matrix cores do not round to nearest when they add to a large one), which is
// added to the running total in fp32.  They round down, so the small errors of A^T X all have one sign and grow with the rows
// while the sums grow with their root: every second step has A with the other sign and its products are subtracted, which
// costs nothing.  B of the given factors against 64 bits, 32 heads, 1e-7, without -> with: 16K rows 1.7 -> 1.0, 32K 2.3 -> 1.2, 128K
// 4.1 -> 1.2 (three launches, where a wave's sums of the K side were half as long, 1 .. 4 % below the figures without).
//
// A step's rows are requested a step ahead, into registers (fp32 sums leave the accumulators 128 of the 256 a wave has), and
// go to the other half of the LDS tile, one barrier a step.  The sides' workgroups alternate in chunks, so that the Q side's,
// which the HBM bounds, and the K side's, which read a third as much of it, run side by side.  32 heads of 32K rows (8 kv
// heads), rank 32, us: 165 (counters: 615 MB read, 3.7 TB/s; matrix cores busy for 32 % of the cycles, LDS for 23 %, a seventh of
// that in bank conflicts); the same sums in three launches (Q; K and its given factors; K^T K), whose waves formed all 16 blocks
// of X^T X and split every factor twice: 122 + 73 + 20.
// On the way: the sides one after the other 182, a branch on X^T X inside the loop 173, all waves in step 172; with 20
// registers spilled (scratch reloads wait for the requested rows) 215.
constexpr int kXtxWaves = 8, kXtxThreads = kXtxWaves * kWave, kXtxRows = 128, kXtxD = 128;
constexpr int kSumXTile = kXtxRows * kXtxD, kSumATile = kXtxRows * 32;  // elements: rows of X, one piece of the rows of A
constexpr int kSumBuf = kSumXTile + 3 * kSumATile;
constexpr int kSumLdr = 33;                                             // floats per row of a tile on its way out
constexpr int kSumSmem = 2 * kSumBuf * (int)sizeof(uint16_t);
static_assert(kXtxWaves * 3 * 32 * kSumLdr * (int)sizeof(float) <= kSumSmem, "the reduction uses the tiles' LDS");

struct SumsArgs {
  const bf16_t *q, *k;
  const float *a_q, *a_k;
  float *part_q, *part_k;    // [head][S][r][r + d]
  float *xq_part, *xk_part;  // [head of X][S][d][d]
  int64_t l;
  int bh, nh, r, S;
};

// ALIGNED: rows of A of whole 16-byte pieces
template <bool ALIGNED>
__global__ __launch_bounds__(kXtxThreads) void pf_sums_kernel(SumsArgs g) {
  extern __shared__ __align__(16) uint16_t sum_s[];
  const int tid = threadIdx.x, lane = lane_id(), wave = gd_wave();
  const int col = lane & 31, half = lane >> 5, s16 = lane & 15;
  const int wg = wave >> 1, ch = wave & 1;
  const int S = g.S, r = g.r, nh = g.nh;
  const int64_t l = g.l;
  // chunks of 8 nh workgroups, the sides in turn
  const int chunk = (int)blockIdx.x / (8 * nh), at = (int)blockIdx.x % (8 * nh);
  const bool k_side = chunk & 1;
  int h, s;
  if (!k_side) {
    const int w = (chunk >> 1) * 8 * nh + at;
    if (w >= g.bh * S) return;
    h = w / S;
    s = w % S;
  } else {
    // eight (kv head, split) pairs side by side, then the same eight for the group's next head
    const int pair = (chunk >> 1) * 8 + at % 8;
    if (pair >= g.bh / nh * S) return;
    h = pair / S * nh + at / 8;
    s = pair % S;
  }
  const int xh = k_side ? h / nh : h;
  const bool xtx = !k_side || h % nh == s % nh;
  const bf16_t* Xh = (k_side ? g.k : g.q) + (int64_t)xh * l * kXtxD;
  const float* Ah = (k_side ? g.a_k : g.a_q) + (int64_t)h * l * r;

  // ---- rows into registers, registers into LDS
  constexpr int NL = kXtxRows * kXtxD / (kXtxThreads * 8);  // 16-byte pieces of X per thread and step
  const int x_row = tid >> 4, x_piece = tid & 15;           // of the first: the others are 32 rows further each
  const int a_row = tid >> 2, a_col = (tid & 3) * 4;        // this thread's factors: a_col .. + 3 and 16 further
  gd_u32x4 px[NL];
  gd_floatx4 pa[2];
  auto issue = [&](int64_t t0) {
    const bf16_t* xb = Xh + t0 * kXtxD;
    const float* ab = Ah + t0 * r;
    const int last = (int)min((int64_t)kXtxRows, l - t0) - 1;
    if (last == kXtxRows - 1) {
      const uint32_t at = (uint32_t)(x_row * kXtxD + 8 * x_piece) * 2u;
#pragma unroll
      for (int i = 0; i < NL; ++i) px[i] = gd_at<gd_u32x4>(xb + i * 32 * kXtxD, at);
    } else {
#pragma unroll
      for (int i = 0; i < NL; ++i)
        px[i] = gd_at<gd_u32x4>(xb, (uint32_t)(min(x_row + 32 * i, last) * kXtxD + 8 * x_piece) * 2u);
    }
    const uint32_t a_at = __umul24((uint32_t)min(a_row, last), 4u * (uint32_t)r);
    if constexpr (ALIGNED) {
#pragma unroll
      for (int j = 0; j < 2; ++j) pa[j] = gd_at<gd_floatx4>(ab, a_at + 4u * (uint32_t)min(a_col + 16 * j, r - 4));
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) pa[q >> 2][q & 3] = gd_at<float>(ab, a_at + 4u * (uint32_t)min(a_col + 16 * (q >> 2) + (q & 3), r - 1));
    }
  };
  // block nb (64 bytes) of row t of X lies at place nb ^ (t & 3): four successive rows of a block then meet all LDS banks
  auto stage = [&](int64_t t0, char* tile, bool minus) {
    const int rows = (int)min((int64_t)kXtxRows, l - t0);
    char* xp = tile + 2 * (x_row * kXtxD + 8 * (x_piece ^ ((x_row & 3) << 2)));
    char* ap = tile + 2 * (kSumXTile + a_row * 32 + a_col);
    const bool whole = rows == kXtxRows && r == 32;
    if (!whole) {
#pragma unroll
      for (int i = 0; i < NL; ++i)
        if (x_row + 32 * i >= rows) px[i] = gd_u32x4{0, 0, 0, 0};
      const int valid = a_row < rows ? r - a_col : 0;  // columns from a_col on that are there
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (16 * (q >> 2) + (q & 3) >= valid) pa[q >> 2][q & 3] = 0.0f;
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<gd_u32x4*>(xp + i * 32 * kXtxD * 2) = px[i];
    const uint32_t sign = minus ? 0x80000000u : 0u;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      uint32_t pc[3][4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        gd_split3(__uint_as_float(__float_as_uint(pa[j][q]) ^ sign), pc[0][q], pc[1][q], pc[2][q]);
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<uint2*>(ap + 2 * (p * kSumATile + 16 * j)) =
            make_uint2(gd_pack2(pc[p][0], pc[p][1]), gd_pack2(pc[p][2], pc[p][3]));
    }
  };

  // ---- operands: rows 32 wg + 16 kb + 4 half .. + 3 and the same + 8 (the same order on both sides of a product) of 32
  // columns.  Within 16 lanes, lane s points at row s / 4, columns 4 (s % 4) .. + 3, and lane t receives column t of the
  // four rows.
  const int row0 = 32 * wg + 4 * half + (s16 >> 2);
  const int c0 = (col & 16) + 4 * (s16 & 3);
  const uint32_t x_at = 2u * (uint32_t)(row0 * kXtxD + 32 * (s16 >> 2) + c0);  // block nb: x_at ^ 64 nb
  const uint32_t a_at = 2u * (uint32_t)(kSumXTile + row0 * 32 + c0);
  auto read8 = [&](const char* p, int rows8) {  // rows8: bytes from a row to the one 8 further
    const gd_v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gd_lds_v4s)p);
    const gd_v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gd_lds_v4s)(p + rows8));
    return __builtin_bit_cast(gd_bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  const int order = ch ? 0x1302 : 0x3210;  // block i of this wave

  gd_floatx16 gAA, gAX[2], gXX[5];
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    gAA[v] = gAX[0][v] = gAX[1][v] = 0.0f;
#pragma unroll
    for (int i = 0; i < 5; ++i) gXX[i][v] = 0.0f;
  }
  auto multiply = [&](char* tile, auto with_xtx, float sign) {
    const char* ar = tile + a_at;
    gd_bf16x8 x[4][2];
    auto read_x = [&](int i) {
      const char* at = tile + (x_at ^ (uint32_t)(64 * ((order >> (4 * i)) & 3)));
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) x[i][kb] = read8(at + kb * 16 * kXtxD * 2, 8 * kXtxD * 2);
    };
    read_x(0);
    read_x(3);
    if constexpr (decltype(with_xtx)::value) {
      auto block = [&](int i, const gd_bf16x8 (&a)[2], const gd_bf16x8 (&b)[2]) {
        gd_floatx16 t;
#pragma unroll
        for (int v = 0; v < 16; ++v) t[v] = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kb], b[kb], t, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 16; ++v) gXX[i][v] += t[v];
      };
      read_x(1);
      read_x(2);
      block(0, x[0], x[0]);
      block(2, x[0], x[1]);
      block(3, x[1], x[2]);
      block(4, x[2], x[3]);
      block(1, x[3], x[3]);
      __builtin_amdgcn_sched_barrier(0);  // (in this order the operands fit the registers)
    }
    {
      gd_bf16x8 c[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) c[p] = read8(ar + ch * 16 * 32 * 2 + p * kSumATile * 2, 8 * 32 * 2);
      gd_floatx16 t;
#pragma unroll
      for (int v = 0; v < 16; ++v) t[v] = 0.0f;
      // k block ch of A^T A, smallest pieces first
      t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[1], c[2], t, 0, 0, 0);
      t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[2], c[1], t, 0, 0, 0);
      t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[0], c[2], t, 0, 0, 0);
      t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[2], c[0], t, 0, 0, 0);
      t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[1], c[1], t, 0, 0, 0);
      t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[0], c[1], t, 0, 0, 0);
      t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[1], c[0], t, 0, 0, 0);
      t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[0], c[0], t, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 16; ++v) gAA[v] += t[v];
    }
    gd_bf16x8 cp[3][2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int p = 0; p < 3; ++p) cp[p][kb] = read8(ar + (p * kSumATile + kb * 16 * 32) * 2, 8 * 32 * 2);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      gd_floatx16 t;
#pragma unroll
      for (int v = 0; v < 16; ++v) t[v] = 0.0f;
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cp[p][kb], x[3 * j][kb], t, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 16; ++v) gAX[j][v] = fmaf(sign, t[v], gAX[j][v]);  // (exact products: rounded once, like a sum)
    }
  };

  // split s takes the steps s, s + S, ...: the workgroups of a head walk the head's rows side by side
  const int64_t stride = (int64_t)S * kXtxRows;
  const int64_t first = (int64_t)s * kXtxRows;
  // Between two barriers a wave multiplies one step and puts the next one into the other half of the tile.  Of the two waves
  // of a SIMD one does so first and the other last, so that matrix and vector work meet.
  const bool stage_first = wave >= kXtxWaves / 2;
  auto walk = [&](auto with_xtx, auto ahead) {
    constexpr int kTileBytes = kSumBuf * (int)sizeof(uint16_t);
    char* const tiles = (char*)sum_s;
    int buf = 0;
    auto minus = [&](int half_at) { return (half_at != 0) != ((s & 1) != 0); };
    auto fetch = [&](int64_t t0, int half_at) {  // the step from t0 on, requested before, into LDS; the next one requested
      stage(t0, tiles + half_at, minus(half_at));
      if (t0 + stride < l) issue(t0 + stride);
    };
    if (first < l) {
      issue(first);
      if constexpr (decltype(ahead)::value) fetch(first, 0);
    }
    for (int64_t t0 = first; t0 < l; t0 += stride) {
      if constexpr (!decltype(ahead)::value) fetch(t0, buf);
      __syncthreads();
      if constexpr (decltype(ahead)::value)
        if (t0 + stride < l) fetch(t0 + stride, kTileBytes - buf);
      multiply(tiles + buf, with_xtx, minus(buf) ? -1.0f : 1.0f);  // (rows beyond the end are zeros)
      buf = kTileBytes - buf;
    }
  };
  // (a loop each: a branch inside one costs the accumulators copies; all meet the same barriers)
  if (xtx) {
    if (stage_first)
      walk(std::true_type(), std::true_type());
    else
      walk(std::true_type(), std::false_type());
  } else {
    if (stage_first)
      walk(std::false_type(), std::true_type());
    else
      walk(std::false_type(), std::false_type());
  }

  // ---- the waves' sums, up to three tiles at a time: add(tile, waves' step, first wave, row, column)
  float* sm = reinterpret_cast<float*>(sum_s);
  constexpr int kTile = 32 * kSumLdr;
  auto put = [&](int slot, const gd_floatx16& acc) {
#pragma unroll
    for (int v = 0; v < 16; ++v) sm[(slot * kXtxWaves + wave) * kTile + gd_mfma_row(lane, v) * kSumLdr + col] = acc[v];
  };
  auto add4 = [&](int slot, int c, int m, int n) {  // over the waves with ch = c
    const float* p = sm + (slot * kXtxWaves + c) * kTile + m * kSumLdr + n;
    return (p[0] + p[2 * kTile]) + (p[4 * kTile] + p[6 * kTile]);
  };
  const int ld = r + kXtxD;
  float* outp = (k_side ? g.part_k : g.part_q) + ((int64_t)h * S + s) * r * ld;
  __syncthreads();
  put(0, gAA);
  put(1, gAX[0]);
  put(2, gAX[1]);
  __syncthreads();
  for (int e = tid; e < 1024; e += kXtxThreads) {
    const int m = e >> 5, n = e & 31;
    if (m < r && n < r) outp[m * ld + n] = add4(0, 0, m, n) + add4(0, 1, m, n);
  }
  for (int e = tid; e < 32 * kXtxD; e += kXtxThreads) {
    const int m = e / kXtxD, n = e % 32, nb = (e / 32) % 4;
    // column block nb is the first or second one of ch 0: 0, 3, or of ch 1: 2, 1
    if (m < r) outp[m * ld + r + 32 * nb + n] = add4(nb == 0 || nb == 2 ? 1 : 2, nb == 1 || nb == 2, m, n);
  }
  if (!xtx) return;
  float* outx = (k_side ? g.xk_part : g.xq_part) + ((int64_t)xh * S + s) * kXtxD * kXtxD;
  // blocks of X of product i, for ch 0 and 1: rows, columns
  auto write = [&](int slot, int bi, int bj) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int ri = c ? (0x1302 >> (4 * bi)) & 3 : bi, rj = c ? (0x1302 >> (4 * bj)) & 3 : bj;
      for (int e = tid; e < 1024; e += kXtxThreads) {
        const int m = e >> 5, n = e & 31;
        outx[(32 * ri + m) * kXtxD + 32 * rj + n] = add4(slot, c, m, n);
        if (bi != bj) outx[(32 * rj + m) * kXtxD + 32 * ri + n] = add4(slot, c, n, m);
      }
    }
  };
  __syncthreads();
  put(0, gXX[0]);
  put(1, gXX[1]);
  put(2, gXX[2]);
  __syncthreads();
  write(0, 0, 0);
  write(1, 3, 3);
  write(2, 0, 1);
  __syncthreads();
  put(0, gXX[3]);
  put(1, gXX[4]);
  __syncthreads();
  write(0, 1, 2);
  write(1, 2, 3);
}

static int prefill_sums(const SumsArgs& g, hipStream_t st) {
  const bool aligned = g.r % 4 == 0 && (uintptr_t)g.a_q % 16 == 0 && (uintptr_t)g.a_k % 16 == 0;
  const auto kern = aligned ? pf_sums_kernel<true> : pf_sums_kernel<false>;
  LRQK_HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kSumSmem));
  const int pairs = g.bh / g.nh * g.S;
  hipLaunchKernelGGL(kern, dim3((unsigned)((pairs + 7) / 8 * 8 * g.nh * 2)), dim3(kXtxThreads), kSumSmem, st, g);
  LRQK_HIP_CHECK(hipGetLastError());
  return LRQK_OK;
}

// ----------------------------------------------------------------------------- d x d algebra, fp64
// Everything below is templated on RT, the number of 16-row tiles that the rank is padded to (ranks up to 16, 32, 64:
// RT = 1, 2, 4), and on the row width D (64 or 128); RP = 16 RT is the padded rank.  Padding costs the matrix cores'
// time (a solve has RP / 4 dependent steps of 800 to 1450 cycles, see gd_solve), so a rank of 16 does not run as 32.
// One workgroup per head takes ranks up to 16, and heads enough to fill the CUs by themselves; the others go in slices
// (pf_gs_kernel below).  Eight waves, two per SIMD: waves 0 .. 3 hold one system of a pair, waves 4 .. 7 the other (D / 4
// right-hand columns each), so that a wave waiting for its pivot block leaves the matrix cores to the other.  Against four
// waves with both systems (D = 128, 32 heads, elimination without products a step behind): the final pair 18.0 -> 12.4 us at
// RT = 2, 47.6 -> 33.0 at RT = 4; an iteration 28 -> 24 us at RT = 1, 49 -> 42 at RT = 2, 133 -> 109 at RT = 4.
constexpr int kGdThreads = 512;
template <int RT, int D>
struct GdShape {
  static constexpr int RP = 16 * RT;
  static constexpr int CT = D / 64;       // 16-column tiles of a right-hand side per wave
  static constexpr int LD = RP + 2;       // doubles per row of a transposed r x d matrix in LDS ([D][LD], 16-byte rows)
  static constexpr int LG = RP + 1;       // doubles per row of an r x r matrix
  // RT = 4: three D x LD matrices do not fit the LDS, so B shares its block with T / U (each is dead when the other is
  // formed) and the r x r matrices lie in global memory (they stay in the L2)
  static constexpr bool WIDE = RT == 4;
  static constexpr int PIV = (WIDE ? 2 * 2 : kGdThreads / 64) * RP * 4;
  static constexpr size_t SMEM = ((size_t)(WIDE ? 2 : 3) * D * LD + (WIDE ? 0 : 3 * RP * LG) + PIV + 8) * sizeof(double);
};

// ---- two systems [W | RHS] (W RP x RP symmetric positive definite up to rounding, rows/columns beyond r the
// identity; RHS RP x D) solved side by side, one per half of the workgroup, by block Gauss-Jordan elimination on the
// fp64 matrix cores, four pivots per step.  The matrices live in the accumulator layout of 16 x 16 tiles (element v of
// lane l = row 16 rt + l / 16 + 4 v, column 16 u + l % 16 of tile (rt, u)).  Up to RT = 2 each of a system's four waves
// holds W itself (every wave eliminates its own copy: no wave waits for another, the solve has no barrier) and D / 4
// columns of RHS; RT = 4 would need 256 registers for the copies and most of the products for work done four times
// over, so there wave w holds column tile w % 4 of W and the pivot columns go round through LDS, one barrier per step.
// Step m, with P the pivot columns 4 m .. 4 m + 3 (RP x 4) and D its rows 4 m .. 4 m + 3:
//     X <- X - (P D^-1) X[4 m .. 4 m + 3, :] outside the pivot rows,   X[pivot rows] <- D^-1 X[pivot rows]
// (one product: the pivot rows' accumulators are cleared and their left operand is D^-1 itself), which clears the
// pivot columns elsewhere.  The right-hand
// operand, four rows of X, is element m % 4 of the lane's own tile in row tile m / 4: no data moves for it.  The
// left operand needs P by rows: the lanes that hold the pivot columns put them into the LDS slot, and every lane inverts
// the pivot block for itself (by 2 x 2 blocks, no pivoting).  The products on W come first (the next step waits for
// them only).
typedef double gd_v4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void gd_wave_sync() {  // orders one wave's LDS writes and reads
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 1 / x to ~1e-14: the hardware estimate (2^-23) and one Newton step.  The pivot blocks' inverses need no more
// (their error enters the solution once, scaled by the condition number, far below the rounding of the fp32 sums
// the systems are built from), and every operation here is on the solve's dependent chain.
__device__ __forceinline__ double gd_rcp(double x) {
  const double inv = __builtin_amdgcn_rcp(x);
  return fma(fma(-x, inv, 1.0), inv, inv);
}

// D x = e for a 4 x 4 matrix with positive definite symmetric part, by 2 x 2 blocks (no pivoting): with
// D = [[A, B], [C, E]], Y = A^-1 B and S = E - C Y,  x2 = S^-1 (e2 - C A^-1 e1),  x1 = A^-1 e1 - Y x2.
// D is taken as it is, not as symmetric: the Gram sums it comes from are symmetric only up to their rounding, and
// the elimination around it uses both triangles.  (A lane needs one column of the inverse: the whole of it took twice
// the operations, and selecting a column from it 24 more.)
__device__ __forceinline__ void gd_solve4(const double (&D)[4][4], const double (&e)[4], double (&x)[4]) {
  const double ia = gd_rcp(fma(D[0][0], D[1][1], -D[0][1] * D[1][0]));
  const double y00 = fma(D[1][1], D[0][2], -D[0][1] * D[1][2]) * ia, y01 = fma(D[1][1], D[0][3], -D[0][1] * D[1][3]) * ia;
  const double y10 = fma(D[0][0], D[1][2], -D[1][0] * D[0][2]) * ia, y11 = fma(D[0][0], D[1][3], -D[1][0] * D[0][3]) * ia;
  const double w0 = fma(D[1][1], e[0], -D[0][1] * e[1]) * ia, w1 = fma(D[0][0], e[1], -D[1][0] * e[0]) * ia;
  const double s00 = fma(-D[2][1], y10, fma(-D[2][0], y00, D[2][2])), s01 = fma(-D[2][1], y11, fma(-D[2][0], y01, D[2][3]));
  const double s10 = fma(-D[3][1], y10, fma(-D[3][0], y00, D[3][2])), s11 = fma(-D[3][1], y11, fma(-D[3][0], y01, D[3][3]));
  const double is = gd_rcp(fma(s00, s11, -s01 * s10));
  const double g0 = fma(-D[2][1], w1, fma(-D[2][0], w0, e[2])), g1 = fma(-D[3][1], w1, fma(-D[3][0], w0, e[3]));
  x[2] = fma(s11, g0, -s01 * g1) * is;
  x[3] = fma(s00, g1, -s10 * g0) * is;
  x[0] = fma(-y01, x[3], fma(-y00, x[2], w0));
  x[1] = fma(-y11, x[3], fma(-y10, x[2], w1));
}

template <int RT, int CT>
struct GdSys {
  static constexpr int WC = RT == 4 ? 1 : RT;  // column tiles of W that a wave holds (all of them, or tile `wave % 4`)
  gd_v4d w[RT][WC];  // W: [row tile][column tile]
  gd_v4d x[RT][CT];  // this wave's columns of RHS: [row tile][column tile CT (wave % 4) + u]
};
// Solves the two systems of a pair, one per half of the workgroup (s: the system of this wave's half).
// A step waits for the step before it only through the column tile that holds its pivots; the products on the other
// tiles (what is left of W, the right-hand columns) are a step behind, so that they run while the next pivot block is on
// its way through LDS and inverted.  A step in cycles at
// RT = 1, 2, 4, one wave per SIMD: 1080, 1450, 2070 with the products of a step behind its inversion and a lane's column
// picked from the whole inverse; 800, 1000, 1450 now (64 of them a product of 16 x 16 x 4).
template <int RT, int CT>
__device__ __forceinline__ void gd_solve(GdSys<RT, CT>& s, double* __restrict__ piv) {
  constexpr int RP = 16 * RT, STEPS = 4 * RT;
  constexpr bool WIDE = RT == 4;
  const int lane = lane_id(), wave = gd_wave(), wq = wave & 3;
  const int li = lane & 15, lk = lane >> 4;
  const double unit[4] = {lk == 0 ? 1.0 : 0.0, lk == 1 ? 1.0 : 0.0, lk == 2 ? 1.0 : 0.0, lk == 3 ? 1.0 : 0.0};
  double aop[RT];
  // the product of step m on a column of tiles
  auto product = [&](int m, auto& t, int u) {
    const int tp = m >> 2, vp = m & 3;
    const double bop = t[tp][u][vp];
    t[tp][u][vp] = 0.0;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) t[rt][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(aop[rt], bop, t[rt][u], 0, 0, 0);
  };
  // what step m leaves for later: the tiles of W beyond the next pivots' (those before it hold finished columns, which
  // nothing reads again), and the right-hand columns
  auto behind = [&](int m) {
    if constexpr (!WIDE) {
#pragma unroll
      for (int u = 0; u < RT; ++u)
        if (u > (m + 1) >> 2) product(m, s.w, u);
    }
#pragma unroll
    for (int u = 0; u < CT; ++u) product(m, s.x, u);
  };
#pragma unroll
  for (int m = 0; m < STEPS; ++m) {
    const int tp = m >> 2, vp = m & 3;  // the pivots' tile (row tile of the pivot rows, column tile of W) and element
    // P: the wave's own slot, or (WIDE) one of two slots per system that its four waves read
    double* P = piv + (WIDE ? (m & 1) * 2 + (wave >> 2) : wave) * RP * 4;
    {
      const int kk = li - 4 * vp;
      if ((!WIDE || wq == tp) && kk >= 0 && kk < 4) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int v = 0; v < 4; ++v) P[(16 * rt + lk + 4 * v) * 4 + kk] = s.w[rt][WIDE ? 0 : tp][v];
      }
    }
    // (two slots: a wave that passes this barrier has read the slot of step m - 2, which step m wrote over)
    if constexpr (WIDE)
      __syncthreads();
    else
      gd_wave_sync();
    double D[4][4], prow[RT][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double2 lo = *reinterpret_cast<const double2*>(&P[(4 * m + i) * 4]);
      const double2 hi = *reinterpret_cast<const double2*>(&P[(4 * m + i) * 4 + 2]);
      D[i][0] = lo.x; D[i][1] = lo.y; D[i][2] = hi.x; D[i][3] = hi.y;
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const double2 lo = *reinterpret_cast<const double2*>(&P[(16 * rt + li) * 4]);
      const double2 hi = *reinterpret_cast<const double2*>(&P[(16 * rt + li) * 4 + 2]);
      prow[rt][0] = lo.x; prow[rt][1] = lo.y; prow[rt][2] = hi.x; prow[rt][3] = hi.y;
    }
    if (m > 0) behind(m - 1);
    // every lane solves for its column l / 16 of the pivot block's inverse, and keeps that column's element of row l % 4
    double ic[4];
    gd_solve4(D, unit, ic);
    // (by value: a choice between array elements is one between addresses, and puts the array into scratch memory)
    auto pick = [](int i, double e0, double e1, double e2, double e3) {
      const double c01 = i & 1 ? e1 : e0, c23 = i & 1 ? e3 : e2;
      return i & 2 ? c23 : c01;
    };
    const double mine = pick(li, ic[0], ic[1], ic[2], ic[3]);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      // pivot rows: the rows of D^-1 themselves (their accumulators are cleared below, so they come out as
      // D^-1 X and not as X - (I - D^-1) X, which cancels in its leading digits when D is far from unit size:
      // with a diagonal of 1e12 solutions were off by 5e-3 where the conditioning allowed 1e-11)
      const double oth = -fma(prow[rt][0], ic[0], fma(prow[rt][1], ic[1], fma(prow[rt][2], ic[2], prow[rt][3] * ic[3])));
      aop[rt] = ((16 * rt + li) >> 2) == m ? mine : oth;
    }
    if constexpr (!WIDE) gd_wave_sync();  // (the reads of the slot precede the next step's writes)
    // W: the column tile of the next pivots (WIDE: every wave its own tile, unless it holds finished columns)
    if (m + 1 < STEPS) {
      if (!WIDE || wq >= (m + 1) >> 2) product(m, s.w, WIDE ? 0 : (m + 1) >> 2);
    }
  }
  behind(STEPS - 1);
  if constexpr (WIDE) __syncthreads();  // (the next solve starts with slot 0 again)
}

// One system filled from fw(row, column of W) and fx(row, column of RHS) / its solution handed to g(row, column
// of RHS, value).
template <int RT, int CT, typename FW, typename FX>
__device__ __forceinline__ void gd_fill(GdSys<RT, CT>& t, FW&& fw, FX&& fx) {
  const int lane = lane_id(), wave = wave_id() & 3;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = 16 * rt + (lane >> 4) + 4 * v;
#pragma unroll
      for (int u = 0; u < GdSys<RT, CT>::WC; ++u) t.w[rt][u][v] = fw(i, 16 * (RT == 4 ? wave : u) + (lane & 15));
#pragma unroll
      for (int u = 0; u < CT; ++u) t.x[rt][u][v] = fx(i, 16 * (CT * wave + u) + (lane & 15));
    }
}
template <int RT, int CT, typename G>
__device__ __forceinline__ void gd_drain(const gd_v4d (&x)[RT][CT], G&& g) {
  const int lane = lane_id(), wave = wave_id() & 3;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int u = 0; u < CT; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) g(16 * rt + (lane >> 4) + 4 * v, 16 * (CT * wave + u) + (lane & 15), x[rt][u][v]);
}

// f(i, j, sum over c < D of PT[c][i] * RT_[c][j])   (two r x d matrices, stored transposed) on the fp64 matrix
// cores: RT x RT tiles of 16 x 16, D / 4 products of depth 4 in a row each; a wave owns two tiles of a row (RT = 4), one
// of the first four waves a tile (RT = 2), and wave 0 the only tile of RT = 1.  Rows/columns beyond r come out as what
// the zero padding gives.
template <int RT, int D, typename F>
__device__ __forceinline__ void gd_outer(const double* __restrict__ PT, const double* __restrict__ QT, F&& f) {
  constexpr int LD = GdShape<RT, D>::LD;
  constexpr int NC = RT == 4 ? 2 : 1;  // column tiles per wave
  const int lane = lane_id(), wave = wave_id();
  if (wave >= RT * RT / NC) return;
  const int li = lane & 15, lk = lane >> 4;
  const int tr = RT == 1 ? 0 : wave >> 1, tc = RT == 1 ? 0 : NC * (wave & 1);
  const double* pa = PT + lk * LD + 16 * tr + li;
  const double* pb = QT + lk * LD + 16 * tc + li;
  gd_v4d acc[NC];
#pragma unroll
  for (int n = 0; n < NC; ++n) acc[n] = gd_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
  for (int c = 0; c < D; c += 4) {
    const double a = pa[c * LD];
#pragma unroll
    for (int n = 0; n < NC; ++n) acc[n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, pb[c * LD + 16 * n], acc[n], 0, 0, 0);
  }
#pragma unroll
  for (int n = 0; n < NC; ++n)
#pragma unroll
    for (int v = 0; v < 4; ++v) f(16 * tr + lk + 4 * v, 16 * (tc + n) + li, acc[n][v]);
}

// TT[c][i] = sum over k of MT[k][i] * S[k][c]   (the transposed form of Mt S, S symmetric D x D in global
// memory) on the fp64 matrix cores: 16 x 16 x 4 tiles, A operand lane l = Mt[i0 + l % 16][k0 + l / 16] (from the
// LDS copy), B operand lane l = S[k0 + l / 16][c0 + l % 16] (16 independent loads per lane in flight), result
// element v of lane l = row l / 16 + 4 v, column l % 16 of the tile.  Each wave takes a column tile (D = 64: two waves
// share one, half of the row tiles each).
// One barrier.
template <int RT, int D>
__device__ __forceinline__ void gd_times_s(const double* __restrict__ MT, const double* __restrict__ S,
                                           double* __restrict__ TT) {
  constexpr int LD = GdShape<RT, D>::LD;
  constexpr bool HALF = D == 64;
  constexpr int NR = HALF ? (RT + 1) / 2 : RT;  // row tiles per wave
  constexpr int U = 16;
  const int lane = lane_id(), wave = wave_id();
  const int li = lane & 15, lk = lane >> 4;
  const int c0 = 16 * (HALF ? wave & 3 : wave), r0 = HALF ? NR * (wave >> 2) : 0;
  if (r0 < RT) {
    gd_v4d acc[NR];
#pragma unroll
    for (int rt = 0; rt < NR; ++rt) acc[rt] = gd_v4d{0.0, 0.0, 0.0, 0.0};
    for (int kb = 0; kb < D; kb += 4 * U) {
      double bv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) bv[u] = S[(int64_t)(kb + 4 * u + lk) * D + c0 + li];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = kb + 4 * u + lk;
#pragma unroll
        for (int rt = 0; rt < NR; ++rt) {
          const double a = MT[k * LD + 16 * (r0 + rt) + li];
          acc[rt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bv[u], acc[rt], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int rt = 0; rt < NR; ++rt)
#pragma unroll
      for (int v = 0; v < 4; ++v) TT[(c0 + li) * LD + 16 * (r0 + rt) + lk + 4 * v] = acc[rt][v];
  }
  __syncthreads();
}

// sum of v over the workgroup, result in every thread.  red: kGdThreads / 64 doubles.  Two barriers.
__device__ __forceinline__ double gd_block_sum(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  if (lane_id() == 0) red[wave_id()] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kGdThreads / kWave; ++w) t += red[w];
  __syncthreads();
  return t;
}

struct GdArgs {
  // initial (G, C) of the two sides as the first Gram passes left them: S partial sums of [r][r + d] floats per head
  const float* partQ;
  const float* partK;
  int S;                // splits of partQ
  int S_k;              // splits of partK
  const double* Sq;     // [bh][d][d]
  const double* Sk;     // [b * hkv][d][d]
  double* G;            // [2][bh][g_parts][RP][RP]  (side 0: Q, 1: K), padded with the identity
  int g_parts;          // 1, or the column slices whose addends of G stand side by side (the init kernel's state is the first)
  double* C;            // [2][bh][RP][d]   zero rows beyond r
  double* BqT;          // [bh][RP][d]      B_Q of the state (written by an iteration for the next)
  double* B;            // in slices: [2][bh][RP][d]  B_Q, B_K of the state
  double* BB;           // in slices: [2][bh][RP][RP]  B_Q B_Q^T, B_K B_K^T
  double* Gs;           // [bh][2][RP][RP + 1]  RT = 4 only: the r x r matrices of an iteration
  double* delta;        // [iters][2][bh]   squared changes |A - A'|^2 per head (in slices: [..][g_parts] addends)
  int* flags;           // [iters + 1]
  float* Mt_q;          // [bh][r][d]  Mq^T, Mk^T for the final pass over the rows
  float* Mt_k;
  void* b_q;            // [bh][r][d] outputs, bf16 or fp32
  void* b_k;
  int out_bf16;
  int bh, hq, hkv, r;
  int64_t l;
  float tol;
};

// One launch for everything that only adds partial sums up, in fp64:
//   blocks [0, nq)        Sq[x][e] = sum over the Sx splits of xq_part[x][s][e]   (nq = bh * d * d / 256)
//   blocks [nq, nq + nk)  Sk likewise over the bkv distinct K heads
//   the rest              the state (G, C) of both sides from the first Gram passes: S partial sums of [G | C]
//                         packed as [r][r + d] floats per head; G padded with the identity, C with zero rows
//                         (RP (RP + d) / 256 blocks per head and side).
template <int RP, int D>
__global__ __launch_bounds__(256) void pf_gramdom_init_kernel(GdArgs a, const float* __restrict__ xq_part, int Sx,
                                                              const float* __restrict__ xk_part, int Sxk, int bkv,
                                                              double* __restrict__ Sq, double* __restrict__ Sk) {
  constexpr int dd = D * D, per = dd / 256;
  constexpr int kBlocks = RP * (RP + D) / 256;
  static_assert(RP * (RP + D) % 256 == 0 && dd % 256 == 0, "whole blocks");
  int blk = blockIdx.x;
  const int nq = a.bh * per, nk = bkv * per;
  if (blk < nq + nk) {
    const bool k_side = blk >= nq;
    if (k_side) blk -= nq;
    const int x = blk / per, e = (blk % per) * 256 + threadIdx.x;
    const int S = k_side ? Sxk : Sx;
    const float* part = (k_side ? xk_part : xq_part) + (int64_t)x * S * dd + e;
    double v = 0.0;
#pragma unroll 4
    for (int s = 0; s < S; ++s) v += (double)part[(int64_t)s * dd];
    (k_side ? Sk : Sq)[(int64_t)x * dd + e] = v;
    return;
  }
  blk -= nq + nk;
  const int h = blk / (2 * kBlocks), side = (blk / kBlocks) & 1;
  const int r = a.r;
  const int e = (blk % kBlocks) * 256 + threadIdx.x;
  const int ne = r * (r + D);
  const int Sn = side ? a.S_k : a.S;
  const float* part = (side ? a.partK : a.partQ) + (int64_t)h * Sn * ne;
  const int i = e / (RP + D), j = e % (RP + D);
  double v = 0.0;
  if (i < r && (j >= RP || j < r)) {
    const int src = i * (r + D) + (j < RP ? j : r + (j - RP));
#pragma unroll 4
    for (int s = 0; s < Sn; ++s) v += (double)part[(int64_t)s * ne + src];
  } else if (j < RP) {
    v = i == j ? 1.0 : 0.0;
  }
  if (j < RP)
    a.G[((int64_t)side * a.bh + h) * a.g_parts * RP * RP + i * RP + j] = v;
  else
    a.C[((int64_t)side * a.bh + h) * RP * D + i * D + (j - RP)] = v;
}

// What a launch of pf_gramdom_kernel does: a whole iteration `it`; the final B_Q, B_K from the state after `it`
// iterations; or a part of an iteration: the first B_Q, the Q side's step, the K side's step.
// RT = 4 runs in parts: with the systems of a whole iteration in one launch the compiler spills 280 registers, and a
// launch more is 2 us where a step takes 50.
enum GdPart { kGdWhole, kGdFinal, kGdStart, kGdQSide, kGdKSide };
template <int RT, int D, int PART>
__global__ __launch_bounds__(kGdThreads) void pf_gramdom_kernel(int it, GdArgs a) {
  using Sh = GdShape<RT, D>;
  constexpr int RP = Sh::RP, CT = Sh::CT, LD = Sh::LD, LG = Sh::LG, d = D;
  extern __shared__ __align__(16) double gsm[];
  double* MT = gsm;                         // [D][LD]  Mq'^T, later Mk'^T (transposed storage)
  double* TT = MT + D * LD;                 // [D][LD]  T, later U
  double* BT = Sh::WIDE ? TT : TT + D * LD; // [D][LD]  B_Q, later B_K
  double* piv = BT + D * LD;                // the solves' slots
  double* red = piv + Sh::PIV;              // [8]
  const int tid = threadIdx.x;
  const bool first = wave_id() < 4;         // this wave's half of the workgroup: the first system of a pair or the second
  const int h = blockIdx.x;
  const int r = a.r, bh = a.bh;
  double* Gs = Sh::WIDE ? a.Gs + (int64_t)h * 2 * RP * LG : red + 8;  // [2 or 3][RP][LG]
  const int b = h / a.hq, kvh = (h % a.hq) / (a.hq / a.hkv);
  const double* Sq = a.Sq + (int64_t)h * d * d;
  const double* Sk = a.Sk + ((int64_t)b * a.hkv + kvh) * d * d;
  double* Gq = a.G + (int64_t)h * RP * RP;
  double* Gk = a.G + ((int64_t)bh + h) * RP * RP;
  double* Cq = a.C + (int64_t)h * RP * d;
  double* Ck = a.C + ((int64_t)bh + h) * RP * d;

  // ---- what an iteration reads of its state is requested before anything else: the handed-over B_Q and this
  // wave's tiles of Ck and Cq (Cq is rewritten only at the end of the Q side's step, Ck at the end of the iteration).
  // (In parts, C is read where it is used, and B_K goes from the Q side's step to the K side's in the block of the
  // handed-over B_Q: each lane reads back what it wrote.)
  constexpr bool FINAL = PART == kGdFinal, kHold = PART == kGdWhole;
  static_assert(FINAL || kHold != Sh::WIDE, "RT = 4 in parts, the others whole");
  const bool fresh = FINAL || PART == kGdStart || (kHold && it == 0);
  constexpr int kBqPer = RP * D / kGdThreads;
  double bq_pre[kHold ? kBqPer : 1];
  gd_v4d ckt[kHold ? RT : 1][CT], cqt[kHold ? RT : 1][CT];
  if (kHold && !fresh) {
    const double* src = a.BqT + (int64_t)h * RP * d;  // [RP][d]
#pragma unroll
    for (int u = 0; u < (kHold ? kBqPer : 1); ++u) bq_pre[u] = src[tid + u * kGdThreads];
  }
  if constexpr (kHold) {
    const int lane = lane_id(), wave = wave_id() & 3;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int u = 0; u < CT; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int e = (16 * rt + (lane >> 4) + 4 * v) * d + 16 * (CT * wave + u) + (lane & 15);
          ckt[rt][u][v] = Ck[e];
          cqt[rt][u][v] = Cq[e];
        }
  }
  if constexpr (PART == kGdKSide) {
    if (a.flags[it]) return;
  }
  if constexpr (PART == kGdWhole || PART == kGdQSide) {
    // ---- the stopping test of the previous iteration (batch-wide, as the reference takes it)
    int done = 0;
    if (it > 0) {
      done = a.flags[it - 1];
      if (!done) {
        const double* dq = a.delta + ((int64_t)(it - 1) * 2 + 0) * bh;
        const double* dk = a.delta + ((int64_t)(it - 1) * 2 + 1) * bh;
        double sq = 0.0, sk = 0.0;
        for (int i = tid; i < bh; i += kGdThreads) {
          sq += dq[i];
          sk += dk[i];
        }
        sq = gd_block_sum(sq, red);
        sk = gd_block_sum(sk, red);
        const double n = (double)bh * (double)a.l * (double)r;
        done = fmax(sq / n, sk / n) < (double)a.tol;
      }
    }
    if (h == 0 && tid == 0) a.flags[it] = done;
    if (done) return;
  }

  // Of an iteration's r x r systems only two follow each other: B_K = Gk^-1 Ck does not depend on the Q side's
  // step and is solved beside it, and the next iteration's B_Q = Gq'^-1 Cq' is solved beside the K side's step
  // and handed over in `BqT`.  Iteration 0 (and the final stage) start from the state alone: B_Q and B_K side by side.
  GdSys<RT, CT> sy;
  gd_v4d bk[kHold ? RT : 1][CT];  // B_K in the layout of the right-hand sides (second half)
  double* BqT = a.BqT + (int64_t)h * RP * d;  // [RP][d]
  if constexpr (PART != kGdQSide && PART != kGdKSide) {
  if (fresh) {
    if (first)
      gd_fill(sy, [&](int i, int j) { return Gq[i * RP + j]; }, [&](int i, int cc) { return Cq[i * d + cc]; });
    else if (FINAL)
      gd_fill(sy, [&](int i, int j) { return Gk[i * RP + j]; }, [&](int i, int cc) { return Ck[i * d + cc]; });
    else
      gd_fill(sy, [&](int i, int j) { return i == j ? 1.0 : 0.0; }, [&](int, int) { return 0.0; });
    gd_solve(sy, piv);
    if constexpr (FINAL) {
      const int64_t o = (int64_t)h * r * d;
      auto put = [&](void* dst, int i, int cc, double v) {
        if (i >= r) return;
        if (a.out_bf16)
          st_f32<bf16_t>((bf16_t*)dst, o + i * d + cc, (float)v);
        else
          ((float*)dst)[o + i * d + cc] = (float)v;
      };
      void* dst = first ? a.b_q : a.b_k;
      gd_drain(sy.x, [&](int i, int cc, double v) { put(dst, i, cc, v); });
      return;
    }
    if constexpr (PART == kGdStart) {
      if (first) gd_drain(sy.x, [&](int i, int cc, double v) { BqT[i * d + cc] = v; });
      return;
    }
    if (first) gd_drain(sy.x, [&](int i, int cc, double v) { BT[cc * LD + i] = v; });
  } else if constexpr (kHold) {
#pragma unroll
    for (int u = 0; u < kBqPer; ++u) {
      const int e = tid + u * kGdThreads;
      BT[(e % d) * LD + e / d] = bq_pre[u];
    }
  }
  }
  if constexpr (PART == kGdQSide) {
#pragma unroll 8
    for (int e = tid; e < RP * d; e += kGdThreads) BT[(e % d) * LD + e / d] = BqT[e];
  }
  if constexpr (PART == kGdWhole || PART == kGdQSide) {
  __syncthreads();
  // ---- W1 = Gk + B_Q B_Q^T
  gd_outer<RT, D>(BT, BT, [&](int i, int j, double o) { Gs[i * LG + j] = Gk[i * RP + j] + o; });
  __syncthreads();
  // ---- Mq'^T = W1^-1 (Ck + B_Q) beside B_K = Gk^-1 Ck
  if (first)
    gd_fill(sy, [&](int i, int j) { return Gs[i * LG + j]; },
            [&](int i, int cc) { return kHold ? BT[cc * LD + i] : BT[cc * LD + i] + Ck[i * d + cc]; });
  else
    gd_fill(sy, [&](int i, int j) { return Gk[i * RP + j]; }, [&](int i, int cc) { return kHold ? 0.0 : Ck[i * d + cc]; });
  if constexpr (kHold) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int u = 0; u < CT; ++u) sy.x[rt][u] += ckt[rt][u];
  }
  __syncthreads();  // (every read of B_Q precedes the rewriting of the B tile below)
  gd_solve(sy, piv);
  // ---- the B tile now holds B_K; Mq'^T goes to its tile and to the caller, with the sum of Cq (the old one) . Mq'^T
  double part_q = 0.0;
  if (first) {
    float* mt = a.Mt_q + (int64_t)h * r * d;
    gd_drain(sy.x, [&](int i, int cc, double v) {
      MT[cc * LD + i] = v;
      if (i < r) mt[i * d + cc] = (float)v;
      if constexpr (!kHold) part_q = fma(Cq[i * d + cc], v, part_q);
    });
    if constexpr (kHold) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int u = 0; u < CT; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) part_q = fma(cqt[rt][u][v], sy.x[rt][u][v], part_q);
    }
  } else {
    if constexpr (kHold) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int u = 0; u < CT; ++u) bk[rt][u] = sy.x[rt][u];
    } else {
      gd_drain(sy.x, [&](int i, int cc, double v) { BqT[i * d + cc] = v; });
    }
    gd_drain(sy.x, [&](int i, int cc, double v) { BT[cc * LD + i] = v; });
  }
  double tr_old = 0.0;
  if (tid < RP) tr_old = tid < r ? Gq[tid * RP + tid] : 0.0;
  __syncthreads();
  gd_outer<RT, D>(BT, BT, [&](int i, int j, double o) { Gs[RP * LG + i * LG + j] = o; });
  if constexpr (Sh::WIDE) __syncthreads();  // (T is formed in the block that holds B_K)
  // ---- T = Mq'^T Sq, Gq' = Mq'^T T^T
  gd_times_s<RT, D>(MT, Sq, TT);
  {
    double tr_new = 0.0;
    gd_outer<RT, D>(MT, TT, [&](int i, int j, double o) {
      const double v = (i < r && j < r) ? o : (i == j ? 1.0 : 0.0);
      if constexpr (kHold) Gs[2 * RP * LG + i * LG + j] = v;
      Gq[i * RP + j] = v;
      if (i == j && i < r) tr_new += v;
    });
    const double dq = gd_block_sum(tr_old - 2.0 * part_q + tr_new, red);
    if (tid == 0) a.delta[((int64_t)it * 2 + 0) * bh + h] = dq;
  }
  // Cq' = T (rows beyond r stay zero: Mq'^T has zero rows there)
#pragma unroll 8
  for (int e = tid; e < RP * d; e += kGdThreads) Cq[e] = TT[(e % d) * LD + e / d];
  }
  if constexpr (PART == kGdWhole || PART == kGdKSide) {
  // ---- the next B_Q = Gq'^-1 T beside Mk'^T = (Gq' + B_K B_K^T)^-1 (T + B_K)
  {
    const double* Gb = Gs + RP * LG;
    if constexpr (kHold) {
      const double* Gn = Gs + 2 * RP * LG;
      gd_fill(sy, [&](int i, int j) { return first ? Gn[i * LG + j] : Gn[i * LG + j] + Gb[i * LG + j]; },
              [&](int i, int cc) { return TT[cc * LD + i]; });
      if (!first) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int u = 0; u < CT; ++u) sy.x[rt][u] += bk[rt][u];
      }
    } else if (first) {
      gd_fill(sy, [&](int i, int j) { return Gq[i * RP + j]; }, [&](int i, int cc) { return Cq[i * d + cc]; });
    } else {
      gd_fill(sy, [&](int i, int j) { return Gq[i * RP + j] + Gb[i * LG + j]; },
              [&](int i, int cc) { return Cq[i * d + cc] + BqT[i * d + cc]; });
    }
  }
  __syncthreads();  // (also: B_K has been read when the next B_Q takes its block)
  gd_solve(sy, piv);
  double part_k = 0.0;
  if (first) {
    gd_drain(sy.x, [&](int i, int cc, double v) { BqT[i * d + cc] = v; });
  } else {
    float* mt = a.Mt_k + (int64_t)h * r * d;
    gd_drain(sy.x, [&](int i, int cc, double v) {
      MT[cc * LD + i] = v;
      if (i < r) mt[i * d + cc] = (float)v;
      if constexpr (!kHold) part_k = fma(Ck[i * d + cc], v, part_k);
    });
    if constexpr (kHold) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int u = 0; u < CT; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) part_k = fma(ckt[rt][u][v], sy.x[rt][u][v], part_k);
    }
  }
  double trk_old = 0.0;
  if (tid < RP) trk_old = tid < r ? Gk[tid * RP + tid] : 0.0;
  __syncthreads();
  // ---- U = Mk'^T Sk, Gk' = Mk'^T U^T, Ck' = U
  gd_times_s<RT, D>(MT, Sk, TT);
  {
    double tr_new = 0.0;
    gd_outer<RT, D>(MT, TT, [&](int i, int j, double o) {
      const double v = (i < r && j < r) ? o : (i == j ? 1.0 : 0.0);
      Gk[i * RP + j] = v;
      if (i == j && i < r) tr_new += v;
    });
    const double dk = gd_block_sum(trk_old - 2.0 * part_k + tr_new, red);
    if (tid == 0) a.delta[((int64_t)it * 2 + 1) * bh + h] = dk;
  }
#pragma unroll 8
  for (int e = tid; e < RP * d; e += kGdThreads) Ck[e] = TT[(e % d) * LD + e / d];
  }
}

template <int RT, int D>
static int gramdom_run(const GdArgs& a, const float* xq_part, int Sx, const float* xk_part, int Sxk, int bkv, double* Sq,
                       double* Sk, int iters, hipStream_t st) {
  using Sh = GdShape<RT, D>;
  constexpr int RP = Sh::RP;
  constexpr bool WIDE = Sh::WIDE;
  using Fn = void (*)(int, GdArgs);
  const Fn last = pf_gramdom_kernel<RT, D, kGdFinal>;
  const Fn start = WIDE ? pf_gramdom_kernel<RT, D, WIDE ? kGdStart : kGdFinal> : nullptr;
  const Fn steps[2] = {pf_gramdom_kernel<RT, D, WIDE ? kGdQSide : kGdWhole>,
                       WIDE ? pf_gramdom_kernel<RT, D, WIDE ? kGdKSide : kGdWhole> : nullptr};
  static_assert(Sh::SMEM <= 160 * 1024, "LDS");
  static std::atomic<bool> attr_dev[kMaxDeviceSlots];
  std::atomic<bool>& attr = attr_dev[per_device_slot()];
  if (!attr) {
    for (Fn f : {last, start, steps[0], steps[1]})
      if (f)
        LRQK_HIP_CHECK(hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Sh::SMEM));
    attr = true;
  }
  const unsigned init_blocks = (unsigned)(((size_t)a.bh + bkv) * (D * D / 256) + (size_t)2 * a.bh * (RP * (RP + D) / 256));
  hipLaunchKernelGGL((pf_gramdom_init_kernel<RP, D>), dim3(init_blocks), dim3(256), 0, st, a, xq_part, Sx, xk_part, Sxk, bkv,
                     Sq, Sk);
  if (start && iters > 0) hipLaunchKernelGGL(start, dim3((unsigned)a.bh), dim3(kGdThreads), Sh::SMEM, st, 0, a);
  for (int it = 0; it < iters; ++it)
    for (Fn f : steps)
      if (f) hipLaunchKernelGGL(f, dim3((unsigned)a.bh), dim3(kGdThreads), Sh::SMEM, st, it, a);
  hipLaunchKernelGGL(last, dim3((unsigned)a.bh), dim3(kGdThreads), Sh::SMEM, st, iters, a);
  LRQK_HIP_CHECK(hipGetLastError());
  return LRQK_OK;
}

// ---- an iteration in two launches over slices of 32 of the D columns
// One workgroup per head leaves most of the CUs idle: 32 heads use 32 of 256, and a head's algebra (4.4 MFLOP an
// iteration at RT = 2, 14.7 at RT = 4) is 14 and 48 us of one CU's fp64 matrix cores.  Here a side's step is one launch of
// several workgroups per head, four waves each (two waves of a SIMD share its fp64 units: eight waves take 1.7 times as
// long for the same columns):
//   * a slice's workgroup solves for the whole M (a solve is a dependent chain: D / 64 tiles of right-hand columns per wave
//     run beside it) and forms its columns of T = M^T S and its addend of G' = M^T T^T;
//   * one more solves the pair's other system, B = G^-1 C, and forms B B^T.
// What a launch exchanges with the next one is T, B, B B^T and the addends of G', which the consumers add up.
// ([M | T] = W^-1 [Y | Y S] for the slice's columns is 10 % less work, but T is then M^T S only up to the solve's rounding.)
// An iteration at D = 128, 32 heads: 44 -> 30 us at RT = 2, 108 -> 57 at RT = 4.
template <int RT, int D>
struct GsShape {
  static constexpr int RP = 16 * RT, LD = RP + 2, LG = RP + 1;
  static constexpr int NS = D / 32;  // slices
  static constexpr int CT = D / 64;  // column tiles of a solve per wave
  static constexpr int PIV = 4 * RP * 4;
  static constexpr int WB = (RP * LG + 1) & ~1;
  // W, M or B (transposed), T (transposed), slots, sums
  static constexpr size_t SMEM = ((size_t)WB + D * LD + 32 * LD + PIV + 16) * sizeof(double);
};
constexpr int kGsThreads = 256, kGsWaves = kGsThreads / kWave;

// The systems of a launch (`plain`: the last workgroup of a head):
//   kGsStart  (all plain)   B_Q = Gq^-1 Cq
//   kGsQ      Mq'^T = (Gk + B_Q B_Q^T)^-1 (Ck + B_Q)    plain: B_K = Gk^-1 Ck
//   kGsK      Mk'^T = (Gq' + B_K B_K^T)^-1 (Cq' + B_K)  plain: B_Q = Gq'^-1 Cq'
//   kGsFinal  (all plain)   the results  B_Q = Gq^-1 Cq  and  B_K = Gk^-1 Ck
// What is read of the state is requested before the stopping test.
enum GsStage { kGsStart, kGsQ, kGsK, kGsFinal };
template <int RT, int D, int STAGE>
__global__ __launch_bounds__(kGsThreads, 2) void pf_gs_kernel(int it, GdArgs a) {
  using Sh = GsShape<RT, D>;
  constexpr int RP = Sh::RP, LD = Sh::LD, LG = Sh::LG, NS = Sh::NS, CT = Sh::CT, NT = kGsThreads;
  constexpr bool STEP = STAGE == kGsQ || STAGE == kGsK;
  constexpr int PER = RP * RP / NT;
  constexpr int NR = RT / 2;  // row tiles of T per wave
  constexpr bool EARLY = RT == 2 || D == 64;  // S is requested ahead of the solve (else the registers do not go round)
  extern __shared__ __align__(16) double gsm[];
  double* WL = gsm;             // [RP][LG]  W
  double* ML = WL + Sh::WB;     // [D][LD]   M or B, transposed (not in W's block: other waves may still read that)
  double* TT = ML + D * LD;     // [32][LD]  the slice of T, transposed
  double* piv = TT + 32 * LD;   // the solves' slots
  double* red = piv + Sh::PIV;  // [3][4]
  const int tid = threadIdx.x, lane = lane_id(), wave = gd_wave();
  const int li = lane & 15, lk = lane >> 4;
  const int s = blockIdx.y, h = blockIdx.x, r = a.r, bh = a.bh;
  if (h >= bh) return;
  const bool plain = !STEP || s >= NS;
  const int ws = STAGE == kGsQ ? 1 : STAGE == kGsK ? 0 : (STAGE == kGsFinal ? s : 0);  // the side of W and C
  const int os = 1 - ws;                                                               // a step: the side that takes the new M
  const int np = STAGE == kGsStart ? 1 : STAGE == kGsK ? NS : it > 0 ? NS : 1;  // addends of G: one before a side's first step
  const int64_t rows = ((int64_t)ws * bh + h) * RP * D, orows = ((int64_t)os * bh + h) * RP * D;
  const double* G = a.G + ((int64_t)ws * bh + h) * NS * RP * RP;
  double* Go = a.G + (((int64_t)os * bh + h) * NS + s) * RP * RP;  // this slice's addend
  const int c0 = 16 * CT * wave + li;                              // this lane's column of the solve, and + 16 u
  const int tc = 32 * s + 16 * (wave & 1) + li;                    // of the slice of T
  const int tr = 16 * NR * (wave >> 1);                            // first row of the wave's tiles of T
  GdSys<RT, CT> sy;

  double w[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) w[u] = G[tid + u * NT];
  if (np > 1) {
#pragma unroll
    for (int p = 1; p < NS; ++p)
#pragma unroll
      for (int u = 0; u < PER; ++u) w[u] += G[(int64_t)p * RP * RP + tid + u * NT];
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = (tid + u * NT) / RP, j = (tid + u * NT) % RP;
    w[u] = i < r && j < r ? w[u] : (i == j ? 1.0 : 0.0);
  }
  if constexpr (STEP) {
    if (!plain) {
      const double* BB = a.BB + ((int64_t)os * bh + h) * RP * RP;
#pragma unroll
      for (int u = 0; u < PER; ++u) w[u] += BB[tid + u * NT];
    }
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) WL[(tid + u * NT) / RP * LG + (tid + u * NT) % RP] = w[u];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int u = 0; u < CT; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) sy.x[rt][u][v] = a.C[rows + (16 * rt + lk + 4 * v) * D + c0 + 16 * u];
  double sv[STEP ? D / 4 : 1];  // S, the right-hand operand of T: column tile wave % 2 of the slice
  auto s_loads = [&] {
    const double* S;
    if constexpr (STAGE == kGsQ) {
      S = a.Sq + (int64_t)h * D * D;
    } else {
      const int b = h / a.hq, kvh = (h % a.hq) / (a.hq / a.hkv);
      S = a.Sk + ((int64_t)b * a.hkv + kvh) * D * D;
    }
    S += lk * D + tc;
#pragma unroll
    for (int u = 0; u < D / 4; ++u) sv[u] = S[4 * u * D];
  };
  double change = 0.0;
  if constexpr (STEP) {
    if (!plain) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int u = 0; u < CT; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) sy.x[rt][u][v] += a.B[orows + (16 * rt + lk + 4 * v) * D + c0 + 16 * u];
      if constexpr (EARLY) s_loads();
      if ((it > 0 || s == 0) && tid < r) change = Go[tid * (RP + 1)];
    }
  }

  asm volatile("" ::: "memory");  // (the loads stay in front of the test)
  if constexpr (STAGE == kGsK) {
    if (a.flags[it]) return;
  }
  if constexpr (STAGE == kGsQ) {
    // ---- the stopping test of the previous iteration (batch-wide, as the reference takes it)
    int done = 0;
    if (it > 0) {
      const int64_t n_add = (int64_t)bh * NS;
      const double* dq = a.delta + (int64_t)(it - 1) * 2 * n_add;
      double sq = 0.0, sk = 0.0;
      for (int64_t i = tid; i < n_add; i += NT) {
        sq += dq[i];
        sk += dq[n_add + i];
      }
      done = a.flags[it - 1];
      for (int off = 32; off > 0; off >>= 1) {
        sq += __shfl_xor(sq, off, kWave);
        sk += __shfl_xor(sk, off, kWave);
      }
      if (lane == 0) {
        red[wave] = sq;
        red[4 + wave] = sk;
      }
      __syncthreads();
      sq = red[0] + red[1] + red[2] + red[3];
      sk = red[4] + red[5] + red[6] + red[7];
      const double n = (double)bh * (double)a.l * (double)r;
      done = done || fmax(sq / n, sk / n) < (double)a.tol;
    }
    if (h == 0 && s == 0 && tid == 0) a.flags[it] = done;
    if (done) return;
  }

  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int u = 0; u < GdSys<RT, CT>::WC; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) sy.w[rt][u][v] = WL[(16 * rt + lk + 4 * v) * LG + 16 * (RT == 4 ? wave : u) + li];
  gd_solve(sy, piv);

  if constexpr (STAGE == kGsFinal) {
    void* dst = s ? a.b_k : a.b_q;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int u = 0; u < CT; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = 16 * rt + lk + 4 * v;
          if (i >= r) continue;
          const int64_t o = (int64_t)h * r * D + i * D + c0 + 16 * u;
          if (a.out_bf16)
            st_f32<bf16_t>((bf16_t*)dst, o, (float)sy.x[rt][u][v]);
          else
            ((float*)dst)[o] = (float)sy.x[rt][u][v];
        }
    return;
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int u = 0; u < CT; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) ML[(c0 + 16 * u) * LD + 16 * rt + lk + 4 * v] = sy.x[rt][u][v];
  // f(i, j, sum over c < N of PT[c][i] * QT[c][j]): a wave has a tile (RT = 2) or a row of tiles (RT = 4)
  constexpr int NC = RT * RT / kGsWaves;
  const int otr = wave * NC / RT, otc = wave * NC % RT;
  auto outer = [&](const double* PT, const double* QT, auto n, auto&& f) {
    gd_v4d acc[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[k] = gd_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
    for (int c = 0; c < decltype(n)::value; c += 4) {
      const double av = PT[(c + lk) * LD + 16 * otr + li];
#pragma unroll
      for (int k = 0; k < NC; ++k)
        acc[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, QT[(c + lk) * LD + 16 * (otc + k) + li], acc[k], 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) f(16 * otr + lk + 4 * v, 16 * (otc + k) + li, acc[k][v]);
  };
  if (plain) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int u = 0; u < CT; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) a.B[rows + (16 * rt + lk + 4 * v) * D + c0 + 16 * u] = sy.x[rt][u][v];
    __syncthreads();
    double* out = a.BB + ((int64_t)ws * bh + h) * RP * RP;
    outer(ML, ML, std::integral_constant<int, D>{}, [&](int i, int j, double v) { out[i * RP + j] = v; });
    return;
  }
  if constexpr (STEP) {
    if constexpr (!EARLY) s_loads();
    const bool in_slice = CT * wave / 2 == s;  // this wave's columns of M are the slice's
    gd_v4d old[RT][CT];                        // there, the other side's C, for the change of its factor
    if (in_slice) {
      float* mt = (STAGE == kGsQ ? a.Mt_q : a.Mt_k) + (int64_t)h * r * D + c0;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int u = 0; u < CT; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int i = 16 * rt + lk + 4 * v;
            old[rt][u][v] = a.C[orows + i * D + c0 + 16 * u];
            if (i < r) mt[i * D + 16 * u] = (float)sy.x[rt][u][v];
          }
    }
    __syncthreads();
    // ---- T = M^T S: wave w takes column tile w % 2 of the slice and half of the row tiles
    gd_v4d t[NR];
#pragma unroll
    for (int n = 0; n < NR; ++n) t[n] = gd_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < D / 4; ++u)
#pragma unroll
      for (int n = 0; n < NR; ++n)
        t[n] = __builtin_amdgcn_mfma_f64_16x16x4f64(ML[(4 * u + lk) * LD + tr + 16 * n + li], sv[u], t[n], 0, 0, 0);
    if (in_slice) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int u = 0; u < CT; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) change = fma(-2.0 * old[rt][u][v], sy.x[rt][u][v], change);
    }
    __syncthreads();  // (the slice's old C has been read)
#pragma unroll
    for (int n = 0; n < NR; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = tr + 16 * n + lk + 4 * v;
        a.C[orows + i * D + tc] = t[n][v];
        TT[(16 * (wave & 1) + li) * LD + i] = t[n][v];
      }
    __syncthreads();
    outer(ML + 32 * s * LD, TT, std::integral_constant<int, 32>{}, [&](int i, int j, double v) {
      Go[i * RP + j] = v;
      if (i == j && i < r) change += v;
    });
    for (int off = 32; off > 0; off >>= 1) change += __shfl_xor(change, off, kWave);
    if (lane == 0) red[8 + wave] = change;
    __syncthreads();
    if (tid == 0) a.delta[(((int64_t)it * 2 + os) * bh + h) * NS + s] = red[8] + red[9] + red[10] + red[11];
  }
}

template <int RT, int D>
static int gramslice_run(const GdArgs& a, const float* xq_part, int Sx, const float* xk_part, int Sxk, int bkv, double* Sq,
                         double* Sk, int iters, hipStream_t st) {
  using Sh = GsShape<RT, D>;
  constexpr int RP = Sh::RP, NS = Sh::NS;
  using Fn = void (*)(int, GdArgs);
  constexpr Fn start = pf_gs_kernel<RT, D, kGsStart>, q_side = pf_gs_kernel<RT, D, kGsQ>, k_side = pf_gs_kernel<RT, D, kGsK>,
               last = pf_gs_kernel<RT, D, kGsFinal>;
  static_assert(Sh::SMEM <= 160 * 1024, "LDS");
  static std::atomic<bool> attr_dev[kMaxDeviceSlots];
  std::atomic<bool>& attr = attr_dev[per_device_slot()];
  if (!attr) {
    for (Fn f : {start, q_side, k_side, last})
      LRQK_HIP_CHECK(hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Sh::SMEM));
    attr = true;
  }
  const unsigned init_blocks = (unsigned)(((size_t)a.bh + bkv) * (D * D / 256) + (size_t)2 * a.bh * (RP * (RP + D) / 256));
  hipLaunchKernelGGL((pf_gramdom_init_kernel<RP, D>), dim3(init_blocks), dim3(256), 0, st, a, xq_part, Sx, xk_part, Sxk, bkv,
                     Sq, Sk);
  // Workgroups go round the XCDs in the order of their index: with a multiple of 8 heads in a row the workgroups of one
  // head share an XCD, and what they all read comes into its L2 once.
  const unsigned bh = ((unsigned)a.bh + 7) & ~7u;
  const dim3 blk(kGsThreads);
  if (iters > 0) hipLaunchKernelGGL(start, dim3(bh, 1), blk, Sh::SMEM, st, 0, a);
  for (int it = 0; it < iters; ++it) {
    hipLaunchKernelGGL(q_side, dim3(bh, NS + 1), blk, Sh::SMEM, st, it, a);
    hipLaunchKernelGGL(k_side, dim3(bh, NS + 1), blk, Sh::SMEM, st, it, a);
  }
  hipLaunchKernelGGL(last, dim3(bh, 2), blk, Sh::SMEM, st, iters, a);
  LRQK_HIP_CHECK(hipGetLastError());
  return LRQK_OK;
}

// The whole factorisation on Gram matrices: q [b][hq][l][d], k [b][hkv][l][d], 16-byte aligned, d = 64 or 128, r <= 64;
// a_q0, a_k0: the given factors, fp32 [b hq][l][r].
int prefill_gram_domain(lrqk_ctx* ctx, const bf16_t* q, const bf16_t* k, float* a_q0, float* a_k0, const PrefillOut& out,
                        int b, int hq, int hkv, int64_t l, int r, int d, int iters, float tol, hipStream_t st) {
  const int bh = b * hq, bkv = b * hkv;
  // rows of 128 elements and ranks up to 32 have a kernel of their own for the sums
  const bool tuned = d == 128 && r <= 32;
  const int RP = r <= 16 ? 16 : r <= 32 ? 32 : 64;
  const size_t ne = (size_t)r * (r + d), dd = (size_t)d * d;
  // Splits of the long axis: one workgroup per CU and launch (the kernels' registers; no more than 64 of a head for that),
  // at most 4096 rows per split however long the prompt (its fp32 sums; the splits are added in fp64; B of 8M equal
  // rows is 1.7e-5 off with 64 splits, 2.2e-7 with 2048), at least one step of rows each.
  auto splits = [&](int heads) {
    const int64_t v = std::max<int64_t>(std::max(1, std::min(64, 256 / heads)), (l + 4095) / 4096);
    return (int)std::max<int64_t>(1, std::min<int64_t>(v, (l + 127) / 128));
  };
  const int S = splits(bh), Sx = S;
  const int Sxk = tuned || hkv == hq ? S : splits(bkv);
  const size_t n_flags = ((size_t)iters + 2) & ~(size_t)1;
  // In slices while a launch of an iteration has few workgroups per CU; with more, what the slices repeat costs more than
  // idle CUs do (a launch is rounded up to 8 heads).  The fit of 4096 rows with four iterations, whole -> in slices, us:
  // d = 128, ranks to 32: 48 heads 282 -> 231, 64 303 -> 286, 72 321 -> 326, 96 360 -> 371;  above: 48 heads 622 -> 448, 64
  // 664 -> 657, 72 696 -> 722, 96 758 -> 798;  d = 64, ranks to 32: 64 heads 188 -> 163, 112 222 -> 216, 128 238 -> 238, 144
  // 261 -> 281;  above: 80 heads 460 -> 370, 88 497 -> 507, 106 518 -> 543.  Ranks up to 16: an iteration whole takes
  // 16 .. 24 us, two launches as long.
  const bool slices = RP > 16 && bh <= (d == 128 ? 64 : RP == 32 ? 112 : 80);
  const size_t g_parts = slices ? d / 32 : 1;
  const size_t n_state = slices ? (size_t)bh * 2 * (RP * d + RP * RP)
                                : (size_t)bh * RP * d + (RP == 64 ? (size_t)bh * 2 * RP * (RP + 1) : 0);
  const size_t n_delta = (size_t)std::max(iters, 1) * 2 * bh * g_parts;
  const size_t bytes = ((size_t)bh + bkv) * dd * 8 + (size_t)2 * bh * RP * (g_parts * RP + d) * 8 + (n_state + n_delta) * 8 +
                       (size_t)2 * bh * RP * d * 4 + ((size_t)bh * Sx + (size_t)bkv * Sxk) * dd * 4 +
                       (size_t)2 * bh * S * ne * 4 + n_flags * 4;
  int rc = ctx->prefill_gd.ensure(bytes);
  if (rc) return rc;
  char* p = (char*)ctx->prefill_gd.p;
  auto take = [&](size_t n) {
    char* at = p;
    p += n;
    return at;
  };
  GdArgs a{};
  double* Sq = (double*)take((size_t)bh * dd * 8);
  double* Sk = (double*)take((size_t)bkv * dd * 8);
  a.Sq = Sq;
  a.Sk = Sk;
  a.G = (double*)take((size_t)2 * bh * g_parts * RP * RP * 8);
  a.g_parts = (int)g_parts;
  a.C = (double*)take((size_t)2 * bh * RP * d * 8);
  if (slices) {
    a.B = (double*)take((size_t)2 * bh * RP * d * 8);
    a.BB = (double*)take((size_t)2 * bh * RP * RP * 8);
  } else {
    a.BqT = (double*)take((size_t)bh * RP * d * 8);
    if (RP == 64) a.Gs = (double*)take((size_t)bh * 2 * RP * (RP + 1) * 8);
  }
  a.delta = (double*)take(n_delta * 8);
  a.Mt_q = (float*)take((size_t)bh * RP * d * 4);
  a.Mt_k = (float*)take((size_t)bh * RP * d * 4);
  float* xq_part = (float*)take((size_t)bh * Sx * dd * 4);
  float* xk_part = (float*)take((size_t)bkv * Sxk * dd * 4);
  float* partQ = (float*)take((size_t)bh * S * ne * 4);
  float* partK = (float*)take((size_t)bh * S * ne * 4);
  a.flags = (int*)take(n_flags * 4);
  a.partQ = partQ;
  a.partK = partK;
  a.S = a.S_k = S;
  a.b_q = out.b_q;
  a.b_k = out.b_k;
  a.out_bf16 = out.storage;
  a.bh = bh;
  a.hq = hq;
  a.hkv = hkv;
  a.r = r;
  a.l = l;
  a.tol = tol;

  if (tuned) {
    if ((rc = prefill_sums({q, k, a_q0, a_k0, partQ, partK, xq_part, xk_part, l, bh, hq / hkv, r, S}, st))) return rc;
  } else {
    if ((rc = prefill_stream_sums(q, k, hq, hkv, b, l, r, d, a_q0, a_k0, partQ, partK, S, xq_part, xk_part, Sxk, st)))
      return rc;
  }
#define LRQK_GD_RUN(RTV, DV) gramdom_run<RTV, DV>(a, xq_part, Sx, xk_part, Sxk, bkv, Sq, Sk, iters, st)
#define LRQK_GS_RUN(RTV, DV) gramslice_run<RTV, DV>(a, xq_part, Sx, xk_part, Sxk, bkv, Sq, Sk, iters, st)
  if (slices)
    rc = d == 64 ? (RP == 32 ? LRQK_GS_RUN(2, 64) : LRQK_GS_RUN(4, 64)) : (RP == 32 ? LRQK_GS_RUN(2, 128) : LRQK_GS_RUN(4, 128));
  else
    rc = d == 64 ? (RP == 16 ? LRQK_GD_RUN(1, 64) : RP == 32 ? LRQK_GD_RUN(2, 64) : LRQK_GD_RUN(4, 64))
                 : (RP == 16 ? LRQK_GD_RUN(1, 128) : RP == 32 ? LRQK_GD_RUN(2, 128) : LRQK_GD_RUN(4, 128));
#undef LRQK_GD_RUN
#undef LRQK_GS_RUN
  if (rc) return rc;
  auto finish = [&](auto* a_q, auto* a_k) -> int {
    using OUT = std::remove_reference_t<decltype(*a_q)>;
    if (iters == 0) {  // the given factors are the result
      int rcs = prefill_store<OUT>(a_q0 + (l - out.a_q_rows) * r, l * r, a_q, out.a_q_rows * r, out.a_q_rows * r, bh, st);
      return rcs ? rcs : prefill_store<OUT>(a_k0, l * r, a_k, out.a_k_stride, l * r, bh, st);
    }
    const int64_t rows = out.a_q_rows;  // (the last ones)
    return prefill_stream_apply<OUT>(k, hkv, l, a.Mt_k, a_k, out.a_k_stride, q + (l - rows) * d, rows, l * d, a.Mt_q, a_q, hq, b,
                                     r, d, st);
  };
  if (out.storage) return finish((bf16_t*)out.a_q, (bf16_t*)out.a_k);
  return finish((float*)out.a_q, (float*)out.a_k);
}

}  // namespace lrqk
