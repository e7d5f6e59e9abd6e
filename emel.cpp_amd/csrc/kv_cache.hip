// Page-pool kernels: append (f16 and on-the-fly q8_0), block-table gather and
// batched page copies (copy-on-write tail split, eviction compaction), plus
// the device KV owner object.  All are HBM-bound byte/integer work on 16-byte
// coalesced accesses; the q8_0 gather puts its rows together in LDS.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <new>

#include "device_common.hpp"
#include "emelk.h"
#include "pool_layout.hpp"
#include "q8_device.hpp"

namespace emelk {
namespace {

using namespace emelk::dev;

constexpr int k_threads = 256;

__device__ __forceinline__ bool page_ok(uint32_t page, int32_t max_blocks) {
  return page < static_cast<uint32_t>(max_blocks);
}

// ---- append, f16 --------------------------------------------------------
// One thread per 8 values of one (seq, token, kv_head) row: two 16-byte fp32
// loads, RNE conversion, one 16-byte store into the page.  Matches
// store_fp16_rounded_cache + physical_kv_position
// (text/generator/detail.hpp:2976-2982, 3050-3055).
__global__ __launch_bounds__(k_threads) void append_f16_kernel(
    pool_layout L, uint8_t *__restrict__ k_pool, uint8_t *__restrict__ v_pool, int32_t layer,
    const float *__restrict__ k_rows, const float *__restrict__ v_rows, int32_t n_seq,
    int32_t n_tokens, const int32_t *__restrict__ positions, const uint16_t *__restrict__ tables,
    int32_t table_stride) {
  const int32_t chunks = L.head_dim / 8;
  const uint64_t total = static_cast<uint64_t>(n_seq) * n_tokens * L.n_head_kv * chunks;
  for (uint64_t i = blockIdx.x * static_cast<uint64_t>(k_threads) + threadIdx.x; i < total;
       i += static_cast<uint64_t>(gridDim.x) * k_threads) {
    const int32_t c = static_cast<int32_t>(i % chunks);
    uint64_t r = i / chunks;
    const int32_t kvh = static_cast<int32_t>(r % L.n_head_kv);
    r /= L.n_head_kv;
    const int32_t t = static_cast<int32_t>(r % n_tokens);
    const int32_t s = static_cast<int32_t>(r / n_tokens);
    const int32_t pos = positions[s] + t;
    if (pos < 0) continue;
    const int32_t lb = pos / L.block_tokens;
    if (lb >= table_stride) continue;
    const uint32_t page = tables[static_cast<uint64_t>(s) * table_stride + lb];
    if (!page_ok(page, L.max_blocks)) continue;
    const int32_t off = pos % L.block_tokens;
    const uint64_t src = ((static_cast<uint64_t>(s) * n_tokens + t) * L.n_head_kv + kvh) *
                             static_cast<uint64_t>(L.head_dim) +
                         static_cast<uint64_t>(c) * 8u;
    const uint64_t dst = L.region_offset(layer, static_cast<int32_t>(page), kvh) +
                         (static_cast<uint64_t>(off) * L.head_dim + c * 8u) * 2u;
#pragma unroll
    for (int kv = 0; kv < 2; ++kv) {
      const float *rows = kv == 0 ? k_rows : v_rows;
      uint8_t *pool = kv == 0 ? k_pool : v_pool;
      const float4_t a = *reinterpret_cast<const float4_t *>(rows + src);
      const float4_t b = *reinterpret_cast<const float4_t *>(rows + src + 4);
      uint4_t out;
      out.x = as_u32(pack_half2(a.x, a.y));
      out.y = as_u32(pack_half2(a.z, a.w));
      out.z = as_u32(pack_half2(b.x, b.y));
      out.w = as_u32(pack_half2(b.z, b.w));
      store16(pool + dst, out);
    }
  }
}

// ---- append, q8_0 -------------------------------------------------------
// One thread per 32-value block (quantize_block32, q8_device.hpp).
__global__ __launch_bounds__(k_threads) void append_q8_0_kernel(
    pool_layout L, uint8_t *__restrict__ k_pool, uint8_t *__restrict__ v_pool, int32_t layer,
    const float *__restrict__ k_rows, const float *__restrict__ v_rows, int32_t n_seq,
    int32_t n_tokens, const int32_t *__restrict__ positions, const uint16_t *__restrict__ tables,
    int32_t table_stride) {
  const int32_t blocks = L.head_dim / 32;
  const uint64_t total = static_cast<uint64_t>(n_seq) * n_tokens * L.n_head_kv * blocks * 2u;
  for (uint64_t i = blockIdx.x * static_cast<uint64_t>(k_threads) + threadIdx.x; i < total;
       i += static_cast<uint64_t>(gridDim.x) * k_threads) {
    const int32_t kv = static_cast<int32_t>(i & 1u);
    uint64_t r = i >> 1;
    const int32_t blk = static_cast<int32_t>(r % blocks);
    r /= blocks;
    const int32_t kvh = static_cast<int32_t>(r % L.n_head_kv);
    r /= L.n_head_kv;
    const int32_t t = static_cast<int32_t>(r % n_tokens);
    const int32_t s = static_cast<int32_t>(r / n_tokens);
    const int32_t pos = positions[s] + t;
    if (pos < 0) continue;
    const int32_t lb = pos / L.block_tokens;
    if (lb >= table_stride) continue;
    const uint32_t page = tables[static_cast<uint64_t>(s) * table_stride + lb];
    if (!page_ok(page, L.max_blocks)) continue;
    const int32_t off = pos % L.block_tokens;
    const float *src = (kv == 0 ? k_rows : v_rows) +
                       ((static_cast<uint64_t>(s) * n_tokens + t) * L.n_head_kv + kvh) *
                           static_cast<uint64_t>(L.head_dim) +
                       static_cast<uint64_t>(blk) * 32u;
    uint8_t *region = (kv == 0 ? k_pool : v_pool) + L.region_offset(layer, static_cast<int32_t>(page), kvh);
    int8_t qs[32];
    uint16_t d;
    quantize_block32(src, qs, d);
    uint4_t *dst = reinterpret_cast<uint4_t *>(region + static_cast<uint64_t>(off) * L.head_dim +
                                               static_cast<uint64_t>(blk) * 32u);
    dst[0] = __builtin_bit_cast(uint4_t, *reinterpret_cast<int8_t(*)[16]>(qs));
    dst[1] = __builtin_bit_cast(uint4_t, *reinterpret_cast<int8_t(*)[16]>(qs + 16));
    uint16_t *scales = reinterpret_cast<uint16_t *>(region + L.scale_plane());
    scales[static_cast<uint64_t>(off) * blocks + blk] = d;
  }
}

// ---- gather -------------------------------------------------------------
// Dense head-major copy of logical tokens [0, lengths[s]) through the block
// table; positions at or past the length are written as zeros.  A workgroup
// takes runs of tokens of one (sequence, KV head), so those and the destination
// are uniform and the index work is 32-bit.  The output is as large as what is
// read and goes elsewhere, so its stores carry the non-temporal hint and leave
// the cache to the pool; the loads do not, since gathered tokens are often still
// in the cache.  f16, a layer, one division chain per chunk and plain stores ->
// now: 8 sequences of 4096 tokens, 8 heads of 128 47.8 -> 42.9 us, of 64 27.2 ->
// 18.3; 6 ragged ones of up to 12632, one head of 512, 55.3 -> 49.5; 8 of 700,
// two heads of 256, 6.6 -> 5.5.  Hinted loads with plain stores: 17.5 us where
// both plain take 12.9 (8 of 4096, one head of 256).  Runs of 32 tokens in place
// of one row piece per thread were slower at head_dim 512 (57.3 us, plain
// stores, against 53.7).

// Region base of token tok of the workgroup's sequence (its page, its KV head)
// and the token's row; false where zeros are written.
struct gather_src {
  uint64_t region;
  uint64_t row;
  bool ok;
};
__device__ __forceinline__ gather_src gather_at(const pool_layout &L, uint64_t head_base,
                                                const uint16_t *__restrict__ table,
                                                int32_t table_stride, int32_t len, int32_t tok) {
  gather_src r{0u, 0u, false};
  if (tok < len) {
    const int32_t lb = tok / L.block_tokens;
    if (lb < table_stride) {
      const uint32_t page = table[lb];
      if (page_ok(page, L.max_blocks)) {
        r.region = head_base + static_cast<uint64_t>(page) * L.page_bytes;
        r.row = static_cast<uint64_t>(tok - lb * L.block_tokens);
        r.ok = true;
      }
    }
  }
  return r;
}

template <int D>
__global__ __launch_bounds__(k_threads) void gather_f16_kernel(
    pool_layout L, const uint8_t *__restrict__ k_pool, const uint8_t *__restrict__ v_pool,
    int32_t layer, int32_t n_seq, const int32_t *__restrict__ lengths,
    const uint16_t *__restrict__ tables, int32_t table_stride, uint8_t *__restrict__ k_out,
    uint8_t *__restrict__ v_out, int32_t out_tokens) {
  constexpr int CH = D / 8;                      // 16-byte chunks of a row
  constexpr int T = k_threads / CH;              // tokens of a run
  const uint32_t c = threadIdx.x % CH;
  const uint32_t runs = (out_tokens - 1) / T + 1;
  const uint64_t units = static_cast<uint64_t>(n_seq) * L.n_head_kv * runs;
  for (uint64_t u = blockIdx.x; u < units; u += gridDim.x) {
    const uint32_t sh = static_cast<uint32_t>(u / runs);  // s * n_head_kv + kvh
    const int32_t s = static_cast<int32_t>(sh / L.n_head_kv);
    const int32_t kvh = static_cast<int32_t>(sh % L.n_head_kv);
    const int32_t len = lengths[s];
    const uint16_t *table = tables + static_cast<uint64_t>(s) * table_stride;
    const uint64_t head_base = L.region_offset(layer, 0, kvh);
    const uint64_t out0 = static_cast<uint64_t>(sh) * out_tokens;
    const int32_t tok = static_cast<int32_t>(u - static_cast<uint64_t>(sh) * runs) * T +
                        static_cast<int32_t>(threadIdx.x / CH);
    if (tok >= out_tokens) continue;
    const gather_src g = gather_at(L, head_base, table, table_stride, len, tok);
    uint4_t kval = {0u, 0u, 0u, 0u};
    uint4_t vval = kval;
    if (g.ok) {
      const uint64_t src = g.region + (g.row * D + c * 8u) * 2u;
      kval = load16(k_pool + src);
      vval = load16(v_pool + src);
    }
    const uint64_t dst = (out0 + tok) * (2u * D) + c * 16u;
    store16_stream(k_out + dst, kval);
    store16_stream(v_out + dst, vval);
  }
}

// q8_0 gather emits GGUF block_q8_0 (uint16 d, int8 qs[32]; 34 bytes,
// kernel/detail.hpp:226-229).  A thread's 16 values are 16 bytes of the pool
// but straddle words of the output, so a run's rows (tokens are contiguous in
// the output) are put together in LDS and leave as words: 17 two-byte stores
// per block had cost more than the copy (8 sequences of 4096 tokens, 8 heads of
// 128: 35.9 -> 20 us a layer, 7.1 TB/s; with plain stores 29.1, or 25.4 where
// the loads carry the non-temporal hint instead, which costs 29.3 against 24.0
// where the pool is still in the cache).
template <int D>
__global__ __launch_bounds__(k_threads) void gather_q8_0_kernel(
    pool_layout L, const uint8_t *__restrict__ k_pool, const uint8_t *__restrict__ v_pool,
    int32_t layer, int32_t n_seq, const int32_t *__restrict__ lengths,
    const uint16_t *__restrict__ tables, int32_t table_stride, uint8_t *__restrict__ k_out,
    uint8_t *__restrict__ v_out, int32_t out_tokens) {
  constexpr int T = 4096 / D;                    // tokens of a run
  constexpr int ROW = D / 32 * 34;               // bytes of an output row
  constexpr int CH = D / 16;                     // 16-byte pieces of a row's values
  constexpr int N = T * CH / k_threads;          // pieces per thread, of K and of V
  static_assert(T * CH % k_threads == 0, "whole passes");
  __shared__ __align__(16) uint8_t s_out[2][T * ROW];
  const uint64_t splane = L.scale_plane();
  const uint32_t runs = (out_tokens - 1) / T + 1;
  const uint64_t units = static_cast<uint64_t>(n_seq) * L.n_head_kv * runs;
  for (uint64_t u = blockIdx.x; u < units; u += gridDim.x) {
    const uint32_t sh = static_cast<uint32_t>(u / runs);  // s * n_head_kv + kvh
    const int32_t s = static_cast<int32_t>(sh / L.n_head_kv);
    const int32_t kvh = static_cast<int32_t>(sh % L.n_head_kv);
    const int32_t len = lengths[s];
    const uint16_t *table = tables + static_cast<uint64_t>(s) * table_stride;
    const uint64_t head_base = L.region_offset(layer, 0, kvh);
    const uint64_t out0 = static_cast<uint64_t>(sh) * out_tokens;
    const int32_t first = static_cast<int32_t>(u - static_cast<uint64_t>(sh) * runs) * T;
    uint4_t q[2][N];
    uint32_t d[2][N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t item = threadIdx.x + i * k_threads;
      const uint32_t c = item % CH;
      const gather_src g = gather_at(L, head_base, table, table_stride, len,
                                     first + static_cast<int32_t>(item / CH));
#pragma unroll
      for (int kv = 0; kv < 2; ++kv) {
        q[kv][i] = uint4_t{0u, 0u, 0u, 0u};
        d[kv][i] = 0u;
        if (g.ok) {
          const uint8_t *region = (kv == 0 ? k_pool : v_pool) + g.region;
          q[kv][i] = load16(region + g.row * D + c * 16u);
          d[kv][i] = *reinterpret_cast<const uint16_t *>(region + splane +
                                                         (g.row * (D / 32) + c / 2) * 2u);
        }
      }
    }
    if (u != blockIdx.x) __syncthreads();  // the previous run has left LDS
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t item = threadIdx.x + i * k_threads;
      const uint32_t c = item % CH;
#pragma unroll
      for (int kv = 0; kv < 2; ++kv) {
        // block c / 2 of the row: its scale, then its 32 values, 2-byte aligned
        uint16_t *o = reinterpret_cast<uint16_t *>(&s_out[kv][item / CH * ROW + c / 2 * 34u]);
        if (c % 2 == 0) o[0] = static_cast<uint16_t>(d[kv][i]);
        const uint32_t w[4] = {q[kv][i].x, q[kv][i].y, q[kv][i].z, q[kv][i].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          o[1 + 8 * (c % 2) + 2 * k] = static_cast<uint16_t>(w[k]);
          o[2 + 8 * (c % 2) + 2 * k] = static_cast<uint16_t>(w[k] >> 16);
        }
      }
    }
    __syncthreads();
    // the run's bytes; rows are 68 bytes or a multiple, so words from a
    // 4-byte-aligned output (else two bytes at a time)
    const int32_t bytes = min(T, out_tokens - first) * ROW;
    const uint64_t dst = (out0 + first) * ROW;
#pragma unroll
    for (int kv = 0; kv < 2; ++kv) {
      uint8_t *out = (kv == 0 ? k_out : v_out) + dst;
      if ((reinterpret_cast<uintptr_t>(out) & 3u) == 0) {
        for (int32_t b = threadIdx.x * 4; b < bytes; b += k_threads * 4) {
          store4_stream(out + b, *reinterpret_cast<const uint32_t *>(&s_out[kv][b]));
        }
      } else {
        for (int32_t b = threadIdx.x * 2; b < bytes; b += k_threads * 2) {
          *reinterpret_cast<uint16_t *>(out + b) = *reinterpret_cast<const uint16_t *>(&s_out[kv][b]);
        }
      }
    }
  }
}

template <int D>
void launch_gather(const pool_layout &L, hipStream_t st, const uint8_t *k_pool,
                   const uint8_t *v_pool, int32_t layer, int32_t n_seq, const int32_t *lengths,
                   const uint16_t *tables, int32_t table_stride, uint8_t *k_out, uint8_t *v_out,
                   int32_t out_tokens) {
  const bool f16 = L.kv_type == EMELK_KV_F16;
  const int32_t run = f16 ? k_threads / (D / 8) : 4096 / D;
  const uint64_t units = static_cast<uint64_t>(n_seq) * L.n_head_kv * ((out_tokens - 1) / run + 1);
  constexpr uint64_t cap = 1u << 22;  // workgroups; runs beyond them are taken in turn
  const dim3 grid(static_cast<uint32_t>(units < cap ? units : cap));
  if (f16) {
    hipLaunchKernelGGL((gather_f16_kernel<D>), grid, dim3(k_threads), 0, st, L, k_pool, v_pool,
                       layer, n_seq, lengths, tables, table_stride, k_out, v_out, out_tokens);
  } else {
    hipLaunchKernelGGL((gather_q8_0_kernel<D>), grid, dim3(k_threads), 0, st, L, k_pool, v_pool,
                       layer, n_seq, lengths, tables, table_stride, k_out, v_out, out_tokens);
  }
}

// ---- batched page copy --------------------------------------------------
// One workgroup per (move, layer, K|V): a contiguous page_bytes copy with
// 16-byte accesses.
__global__ __launch_bounds__(k_threads) void copy_blocks_kernel(pool_layout L,
                                                                uint8_t *__restrict__ k_pool,
                                                                uint8_t *__restrict__ v_pool,
                                                                const int32_t *__restrict__ moves) {
  const int32_t m = blockIdx.z;
  const int32_t layer = blockIdx.y;
  uint8_t *pool = blockIdx.x == 0 ? k_pool : v_pool;
  const int32_t src = moves[2 * m];
  const int32_t dst = moves[2 * m + 1];
  if (src < 0 || dst < 0 || src >= L.max_blocks || dst >= L.max_blocks || src == dst) return;
  const uint8_t *s = pool + L.region_offset(layer, src, 0);
  uint8_t *d = pool + L.region_offset(layer, dst, 0);
  const uint64_t n16 = L.page_bytes / 16u;
  // batches of 8 loads issued before their stores keep 8 x 16 B per thread in
  // flight; the source is read once, so its loads carry the non-temporal hint.
  // The hint on the stores instead costs a first pass over pools that other
  // kernels just wrote, which is what a compaction is: 218 moves x 32 layers
  // of 64 KiB pages (1.83 GB) 380 -> 441 us, 40 moves x 32 76 -> 108, 40 x 8
  // 24 -> 32, 218 x 32 of q8_0 pages 196 -> 243; only copies repeated on a pool
  // that fits the cache gain (40 x 8: 17.2 -> 13.4).  No hint at all: 405, 101,
  // 31 and 224 on a first pass.
  constexpr int kB = 8;
  uint64_t i = threadIdx.x;
  for (; i + (kB - 1) * k_threads < n16; i += kB * k_threads) {
    uint4_t v[kB];
#pragma unroll
    for (int b = 0; b < kB; ++b) v[b] = load16_stream(s + (i + b * k_threads) * 16u);
#pragma unroll
    for (int b = 0; b < kB; ++b) store16(d + (i + b * k_threads) * 16u, v[b]);
  }
  for (; i < n16; i += k_threads) store16(d + i * 16u, load16_stream(s + i * 16u));
}

int grid_for(uint64_t work_items) {
  const uint64_t blocks = (work_items + k_threads - 1) / k_threads;
  const uint64_t cap = 256u * 32u;  // 32 workgroups per CU on 256 CUs, grid-stride beyond
  return static_cast<int>(blocks < 1 ? 1 : (blocks > cap ? cap : blocks));
}

emel_error_type launch_status() {
  return hipGetLastError() == hipSuccess ? EMELK_ERR_NONE : EMELK_ERR_BACKEND;
}

}  // namespace
}  // namespace emelk

using emelk::pool_layout;

extern "C" emel_error_type emelk_kv_pool_bytes(const emelk_kv_geometry *g, uint64_t *bytes_out) {
  pool_layout L;
  const emel_error_type e = emelk::make_pool_layout(g, L);
  if (e != EMELK_ERR_NONE || bytes_out == nullptr) return e | (bytes_out ? 0u : EMELK_ERR_INVALID_REQUEST);
  *bytes_out = L.pool_bytes;
  return EMELK_ERR_NONE;
}

extern "C" emel_error_type emelk_kv_append(const emelk_kv_geometry *g, void *k_pool, void *v_pool,
                                           int32_t layer, const float *k_rows,
                                           const float *v_rows, int32_t n_seq, int32_t n_tokens,
                                           const int32_t *positions, const uint16_t *block_tables,
                                           int32_t table_stride, void *stream) {
  pool_layout L;
  if (emelk::make_pool_layout(g, L) != EMELK_ERR_NONE || k_pool == nullptr || v_pool == nullptr ||
      k_rows == nullptr || v_rows == nullptr || positions == nullptr || block_tables == nullptr ||
      layer < 0 || layer >= L.n_layer || n_seq < 0 || n_tokens < 0 || table_stride <= 0) {
    return EMELK_ERR_INVALID_REQUEST;
  }
  if (n_seq == 0 || n_tokens == 0) return EMELK_ERR_NONE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint64_t rows = static_cast<uint64_t>(n_seq) * n_tokens * L.n_head_kv;
  if (L.kv_type == EMELK_KV_F16) {
    hipLaunchKernelGGL(emelk::append_f16_kernel, dim3(emelk::grid_for(rows * (L.head_dim / 8))),
                       dim3(emelk::k_threads), 0, st, L, static_cast<uint8_t *>(k_pool),
                       static_cast<uint8_t *>(v_pool), layer, k_rows, v_rows, n_seq, n_tokens,
                       positions, block_tables, table_stride);
  } else {
    hipLaunchKernelGGL(emelk::append_q8_0_kernel,
                       dim3(emelk::grid_for(rows * (L.head_dim / 32) * 2u)), dim3(emelk::k_threads),
                       0, st, L, static_cast<uint8_t *>(k_pool), static_cast<uint8_t *>(v_pool),
                       layer, k_rows, v_rows, n_seq, n_tokens, positions, block_tables,
                       table_stride);
  }
  return emelk::launch_status();
}

extern "C" emel_error_type emelk_kv_gather(const emelk_kv_geometry *g, const void *k_pool,
                                           const void *v_pool, int32_t layer, int32_t n_seq,
                                           const int32_t *lengths, const uint16_t *block_tables,
                                           int32_t table_stride, void *k_out, void *v_out,
                                           int32_t out_tokens, void *stream) {
  pool_layout L;
  if (emelk::make_pool_layout(g, L) != EMELK_ERR_NONE || k_pool == nullptr || v_pool == nullptr ||
      lengths == nullptr || block_tables == nullptr || k_out == nullptr || v_out == nullptr ||
      layer < 0 || layer >= L.n_layer || n_seq < 0 || out_tokens < 0 || table_stride <= 0) {
    return EMELK_ERR_INVALID_REQUEST;
  }
  if (n_seq == 0 || out_tokens == 0) return EMELK_ERR_NONE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const auto launch = L.head_dim == 64    ? emelk::launch_gather<64>
                      : L.head_dim == 128 ? emelk::launch_gather<128>
                      : L.head_dim == 256 ? emelk::launch_gather<256>
                                          : emelk::launch_gather<512>;
  launch(L, st, static_cast<const uint8_t *>(k_pool), static_cast<const uint8_t *>(v_pool), layer,
         n_seq, lengths, block_tables, table_stride, static_cast<uint8_t *>(k_out),
         static_cast<uint8_t *>(v_out), out_tokens);
  return emelk::launch_status();
}

extern "C" emel_error_type emelk_kv_copy_blocks(const emelk_kv_geometry *g, void *k_pool,
                                                void *v_pool, const int32_t *moves,
                                                int32_t n_moves, void *stream) {
  pool_layout L;
  if (emelk::make_pool_layout(g, L) != EMELK_ERR_NONE || k_pool == nullptr || v_pool == nullptr ||
      n_moves < 0 || (n_moves > 0 && moves == nullptr) || n_moves > 65535) {
    return EMELK_ERR_INVALID_REQUEST;
  }
  if (n_moves == 0) return EMELK_ERR_NONE;
  hipLaunchKernelGGL(emelk::copy_blocks_kernel, dim3(2, L.n_layer, n_moves), dim3(emelk::k_threads),
                     0, static_cast<hipStream_t>(stream), L, static_cast<uint8_t *>(k_pool),
                     static_cast<uint8_t *>(v_pool), moves);
  return emelk::launch_status();
}

// ---- device KV owner ------------------------------------------------------
struct emelk_kv_cache {
  emelk_kv_geometry geometry;
  pool_layout layout;
  void *k_pool = nullptr;
  void *v_pool = nullptr;
  int32_t *move_slot = nullptr;  // device int32[2] for single-page copies
  int32_t *move_host = nullptr;  // pinned staging for move_slot
  hipStream_t stream = nullptr;
  // device view upload: pinned snapshot staging (allocated on first use)
  // and the event that tells when the previous upload has read it
  emelk_view_snapshot *view_host = nullptr;
  hipEvent_t view_read = nullptr;
  bool view_pending = false;
};

extern "C" emel_error_type emelk_kv_cache_create(const emelk_kv_geometry *g, void *stream,
                                                 emelk_kv_cache **cache_out) {
  if (cache_out == nullptr) return EMELK_ERR_INVALID_REQUEST;
  *cache_out = nullptr;
  pool_layout L;
  if (emelk::make_pool_layout(g, L) != EMELK_ERR_NONE) return EMELK_ERR_INVALID_REQUEST;
  auto *c = new (std::nothrow) emelk_kv_cache();
  if (c == nullptr) return EMELK_ERR_OUT_OF_MEMORY;
  c->geometry = *g;
  c->layout = L;
  c->stream = static_cast<hipStream_t>(stream);
  if (hipMalloc(&c->k_pool, L.pool_bytes) != hipSuccess ||
      hipMalloc(&c->v_pool, L.pool_bytes) != hipSuccess ||
      hipMalloc(reinterpret_cast<void **>(&c->move_slot), 2 * sizeof(int32_t)) != hipSuccess ||
      hipHostMalloc(reinterpret_cast<void **>(&c->move_host), 2 * sizeof(int32_t),
                    hipHostMallocDefault) != hipSuccess) {
    emelk_kv_cache_destroy(c);
    return EMELK_ERR_OUT_OF_MEMORY;
  }
  *cache_out = c;
  return EMELK_ERR_NONE;
}

extern "C" void emelk_kv_cache_destroy(emelk_kv_cache *c) {
  if (c == nullptr) return;
  if (c->stream != nullptr) (void)hipStreamSynchronize(c->stream);
  else (void)hipDeviceSynchronize();
  if (c->k_pool) (void)hipFree(c->k_pool);
  if (c->v_pool) (void)hipFree(c->v_pool);
  if (c->move_slot) (void)hipFree(c->move_slot);
  if (c->move_host) (void)hipHostFree(c->move_host);
  if (c->view_host) (void)hipHostFree(c->view_host);
  if (c->view_read) (void)hipEventDestroy(c->view_read);
  delete c;
}

// capture_view (kv/sm.hpp:448-465 -> view::snapshot, memory/view.hpp:59-117)
// delivered to device memory: the actor fills the pinned staging snapshot,
// which is copied on the cache's stream, so the copy is ordered with the
// page copies of earlier allocate_slots calls and before later kernels.
extern "C" emel_error_type emelk_kv_cache_upload_view(emelk_kv_cache *c, emelk_kv_actor *actor,
                                                      emelk_view_snapshot *view_dev) {
  if (c == nullptr || actor == nullptr || view_dev == nullptr) return EMELK_ERR_INVALID_REQUEST;
  if (c->view_host == nullptr) {
    if (hipHostMalloc(reinterpret_cast<void **>(&c->view_host), sizeof(emelk_view_snapshot),
                      hipHostMallocDefault) != hipSuccess) {
      c->view_host = nullptr;
      return EMELK_ERR_OUT_OF_MEMORY;
    }
    if (hipEventCreateWithFlags(&c->view_read, hipEventDisableTiming) != hipSuccess) {
      c->view_read = nullptr;
      return EMELK_ERR_BACKEND;
    }
  }
  if (c->view_pending) {  // the copy engine may still read the staging snapshot
    if (hipEventSynchronize(c->view_read) != hipSuccess) return EMELK_ERR_BACKEND;
    c->view_pending = false;
  }
  int32_t err = EMELK_ERR_NONE;
  emelk_event_capture_view ev{c->view_host, &err};
  if (!emelk_kv_capture_view(actor, &ev)) {
    return err != EMELK_ERR_NONE ? static_cast<emel_error_type>(err) : EMELK_ERR_INTERNAL;
  }
  if (hipMemcpyAsync(view_dev, c->view_host, sizeof(emelk_view_snapshot), hipMemcpyHostToDevice,
                     c->stream) != hipSuccess ||
      hipEventRecord(c->view_read, c->stream) != hipSuccess) {
    return EMELK_ERR_BACKEND;
  }
  c->view_pending = true;
  return EMELK_ERR_NONE;
}

extern "C" void *emelk_kv_cache_k_pool(emelk_kv_cache *c) { return c ? c->k_pool : nullptr; }
extern "C" void *emelk_kv_cache_v_pool(emelk_kv_cache *c) { return c ? c->v_pool : nullptr; }
extern "C" void *emelk_kv_cache_stream(const emelk_kv_cache *c) {
  return c ? static_cast<void *>(c->stream) : nullptr;
}

// allocate_slots::copy_block_fn target (text/generator/context.hpp:36-50 ->
// copy_attention_kv_block, detail.hpp:3334-3417): validates the request like
// the reference (block_tokens must match the pool, ids in range), then
// enqueues one page move.  The staging buffer is reused, so the call waits
// for the previous single-page copy's upload before overwriting it.
extern "C" bool emelk_kv_cache_copy_block(int32_t src_block, int32_t dst_block,
                                          int32_t block_tokens, void *user_data,
                                          int32_t *error_out) {
  auto *c = static_cast<emelk_kv_cache *>(user_data);
  if (error_out) *error_out = EMELK_ERR_NONE;
  if (c == nullptr || block_tokens != c->layout.block_tokens || src_block < 0 || dst_block < 0 ||
      src_block >= c->layout.max_blocks || dst_block >= c->layout.max_blocks) {
    if (error_out) *error_out = EMELK_ERR_INVALID_REQUEST;
    return false;
  }
  if (hipStreamSynchronize(c->stream) != hipSuccess) {
    if (error_out) *error_out = EMELK_ERR_BACKEND;
    return false;
  }
  c->move_host[0] = src_block;
  c->move_host[1] = dst_block;
  if (hipMemcpyAsync(c->move_slot, c->move_host, 2 * sizeof(int32_t), hipMemcpyHostToDevice,
                     c->stream) != hipSuccess ||
      emelk_kv_copy_blocks(&c->geometry, c->k_pool, c->v_pool, c->move_slot, 1, c->stream) !=
          EMELK_ERR_NONE) {
    if (error_out) *error_out = EMELK_ERR_BACKEND;
    return false;
  }
  return true;
}
