// Host side of the victim cache: sizing, (re)initialisation, statistics.
#include <algorithm>
#include <vector>

#include "common.hpp"
#include "ctx.hpp"

namespace lrqk {

__global__ __launch_bounds__(256) void victim_init_kernel(int32_t* tok, int64_t n_tok, int16_t* pos, int64_t n_pos,
                                                          int32_t* counters, int n_counters) {
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = i0; i < n_tok; i += stride) tok[i] = -1;
  for (int64_t i = i0; i < n_pos; i += stride) pos[i] = -1;
  for (int64_t i = i0; i < n_counters; i += stride) counters[i] = 0;
}

// Memory of a cache of nv rows per head.  meta: tok i32 [bh][nv] | counters i32 [3][bh] (ptr, base, host_rows) |
// pos i16 [bh][cap]
static int victim_reserve(lrqk_ctx* ctx, int bh, int nv, int64_t cap, int chunks) {
  ctx->vic_dirty = true;  // (a block that grows loses its contents, also where the other one is not to be had)
  const int rc = ctx->vic_rows.ensure((size_t)bh * nv * chunks * sizeof(uint4));
  return rc ? rc : ctx->vic_meta.ensure(((size_t)bh * nv + (size_t)3 * bh) * 4 + (size_t)bh * cap * 2 + 16);
}

int victim_prepare(lrqk_ctx* ctx, int bh, int64_t cap, int chunks, hipStream_t st) {
  if (ctx->vic_req <= 0) {
    ctx->vic.nv = 0;
    return LRQK_OK;
  }
  const int nv = ctx->vic_req;
  const bool same = ctx->vic.nv == nv && ctx->vic_bh == bh && ctx->vic.cap == cap && ctx->vic_chunks == chunks;
  if (same && !ctx->vic_dirty) return LRQK_OK;
  const int rc = victim_reserve(ctx, bh, nv, cap, chunks);
  if (rc) return rc;
  const size_t n_tok = (size_t)bh * nv, n_cnt = (size_t)3 * bh, n_pos = (size_t)bh * cap;
  VictimView v{};
  v.rows = (uint4*)ctx->vic_rows.p;
  v.tok = (int32_t*)ctx->vic_meta.p;
  v.ptr = v.tok + n_tok;
  v.base = v.ptr + bh;
  v.host_rows = v.base + bh;
  v.pos = (int16_t*)(v.host_rows + bh);
  v.nv = nv;
  v.cap = cap;
  hipLaunchKernelGGL(victim_init_kernel, dim3(512), dim3(256), 0, st, v.tok, (int64_t)n_tok, v.pos, (int64_t)n_pos, v.ptr,
                     (int)n_cnt);
  LRQK_HIP_CHECK(hipGetLastError());
  ctx->vic = v;
  ctx->vic_bh = bh;
  ctx->vic_chunks = chunks;
  ctx->vic_dirty = false;
  return LRQK_OK;
}

// FIFO positions 0 .. cnt-1 of an empty cache take the K and V rows of the listed tokens, from a prompt on the device.
// Bound by memory (reads of single rows): 32 heads x 1024 rows of 512 bytes a few us.
__global__ __launch_bounds__(256) void victim_fill_kernel(const uint4* __restrict__ k, const uint4* __restrict__ v, int64_t l,
                                                          const int32_t* __restrict__ ids, const int* __restrict__ cnt,
                                                          int id_cap, VictimView vic, int hq, int hkv, int cpr) {
  const int h = blockIdx.y;
  const int n = max(0, min(cnt[h], min(id_cap, vic.nv)));
  const int64_t src0 = ((int64_t)(h / hq) * hkv + (h % hq) / (hq / hkv)) * l;
  const int chunks = 2 * cpr;  // at most 64
  const int c = threadIdx.x % chunks, tpb = 256 / chunks;
  if (blockIdx.x == 0 && threadIdx.x == 0) vic.ptr[h] = n % vic.nv;
  if ((int)threadIdx.x >= tpb * chunks) return;
  for (int j = blockIdx.x * tpb + threadIdx.x / chunks; j < n; j += gridDim.x * tpb) {
    const int64_t id = ids[(int64_t)h * id_cap + j];
    if (id < 0 || id >= l || id >= vic.cap) continue;  // (the position stays empty)
    vic.rows[((int64_t)h * vic.nv + j) * chunks + c] = c < cpr ? k[(src0 + id) * cpr + c] : v[(src0 + id) * cpr + c - cpr];
    if (c == 0) {
      vic.tok[(int64_t)h * vic.nv + j] = (int32_t)id;
      vic.pos[(int64_t)h * vic.cap + id] = (int16_t)j;
    }
  }
}

}  // namespace lrqk

using namespace lrqk;

extern "C" int lrqk_victim_fill(lrqk_ctx* ctx, const void* k, const void* v, int64_t l, int64_t cap, int b, int hq, int hkv,
                                int d, int dtype, void* stream) {
  LRQK_REQUIRE(ctx && k && v, LRQK_EINVAL, "null pointer");
  ctx->pool.enter((hipStream_t)stream);
  LRQK_REQUIRE(dtype == LRQK_F32 || dtype == LRQK_BF16, LRQK_EINVAL, "dtype=%d", dtype);
  LRQK_REQUIRE(b > 0 && hq > 0 && hkv > 0 && hq % hkv == 0 && (int64_t)b * hq <= 65535, LRQK_EINVAL,
               "bad heads b=%d hq=%d hkv=%d", b, hq, hkv);
  const size_t row = (size_t)d * elem_size(dtype);
  LRQK_REQUIRE(d > 0 && row % 16 == 0 && l > 0 && cap >= l, LRQK_EINVAL, "rows of %zu bytes, l=%lld, cap=%lld", row,
               (long long)l, (long long)cap);
  LRQK_REQUIRE((uintptr_t)k % 16 == 0 && (uintptr_t)v % 16 == 0, LRQK_EINVAL, "pointers must be 16-byte aligned");
  const int cpr = (int)(row / 16), bh = b * hq;
  const bool listed = ctx->next_valid && ctx->next_bh == bh && ctx->vic_req > 0 && ctx->vic_dirty;
  ctx->next_valid = false;
  if (!listed || 2 * cpr > kWave) return LRQK_OK;  // (rows that the step fetches without the cache)
  // The cache changes no result, and the first step makes an empty one where there is none: a prompt does not fail for its
  // memory.  In a capture it is left alone: a replay would fill one that the steps in between have used.
  if (stream_capturing((hipStream_t)stream) || victim_reserve(ctx, bh, ctx->vic_req, cap, 2 * cpr) != LRQK_OK) return LRQK_OK;
  int rc = victim_prepare(ctx, bh, cap, 2 * cpr, (hipStream_t)stream);
  if (rc) return rc;
  const int32_t* ids = (const int32_t*)ctx->next_ids.p;
  const int blocks = std::max(1, std::min(ctx->next_cap / 8, 2048 / bh));
  hipLaunchKernelGGL(victim_fill_kernel, dim3((unsigned)blocks, (unsigned)bh), dim3(256), 0, (hipStream_t)stream,
                     (const uint4*)k, (const uint4*)v, l, ids, ids + (size_t)bh * ctx->next_cap, ctx->next_cap, ctx->vic, hq,
                     hkv, cpr);
  LRQK_HIP_CHECK(hipGetLastError());
  return LRQK_OK;
}

extern "C" int lrqk_ctx_victim_cache(lrqk_ctx* ctx, int rows_per_head) {
  LRQK_REQUIRE(ctx != nullptr, LRQK_EINVAL, "ctx is null");
  LRQK_REQUIRE(rows_per_head >= 0 && rows_per_head <= 32767, LRQK_EINVAL, "rows_per_head=%d not in 0..32767",
               rows_per_head);
  ctx->vic_req = rows_per_head;
  ctx->vic_dirty = true;  // contents are dropped: the next step starts from an empty cache
  ctx->next_valid = false;
  if (rows_per_head == 0) ctx->vic.nv = 0;
  return LRQK_OK;
}

extern "C" int lrqk_victim_stats(lrqk_ctx* ctx, int64_t* host_rows, int reset) {
  LRQK_REQUIRE(ctx && host_rows, LRQK_EINVAL, "null pointer");
  *host_rows = 0;
  if (ctx->vic.nv <= 0 || ctx->vic_dirty || ctx->vic_bh <= 0) return LRQK_OK;
  std::vector<int32_t> v((size_t)ctx->vic_bh);
  LRQK_HIP_CHECK(hipMemcpy(v.data(), ctx->vic.host_rows, v.size() * 4, hipMemcpyDeviceToHost));
  for (int32_t x : v) *host_rows += x;
  if (reset) LRQK_HIP_CHECK(hipMemset(ctx->vic.host_rows, 0, v.size() * 4));
  return LRQK_OK;
}
