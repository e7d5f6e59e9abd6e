// The step executor's device memory when the card has little left, on a host
// allocator that refuses blocks past a limit in the place of the HIP runtime's
// (the rest of the runtime and of the library are stubs).  Built and run by
// tests/test_prefill_scratch.py with the host compiler.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "emelk.h"
#include "prefill_split.hpp"

namespace {
constexpr uint64_t k_decode_need = 3u << 20, k_prefill_most = 64u << 20;
uint64_t limit = ~0ull;
int live = 0;
hipError_t sticky = hipSuccess;
uint64_t prefill_got = 0, decode_got = 0;

hipError_t take(void **p, size_t n) {
  if (n > limit) return sticky = hipErrorOutOfMemory;
  *p = std::malloc(16);
  ++live;
  return hipSuccess;
}
hipError_t give(void *p) {
  std::free(p);
  --live;
  return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return take(p, n); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipHostMalloc(void **p, size_t, unsigned) {
  *p = std::malloc(1 << 16);
  ++live;
  return hipSuccess;
}
hipError_t hipHostFree(void *p) { return give(p); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  return take(reinterpret_cast<void **>(e), 0);
}
hipError_t hipEventDestroy(hipEvent_t e) { return give(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) {
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = sticky;
  sticky = hipSuccess;
  return e;
}

emel_error_type emelk_kv_pool_bytes(const emelk_kv_geometry *, uint64_t *b) {
  *b = 1;
  return EMELK_ERR_NONE;
}
int32_t emelk_rope_table_positions(const emelk_rope_table *) { return 1 << 20; }
void *emelk_kv_cache_stream(const emelk_kv_cache *) { return nullptr; }
emel_error_type emelk_attn_decode_workspace_size(const emelk_kv_geometry *, int32_t, int32_t,
                                                 uint64_t *b) {
  *b = k_decode_need;
  return EMELK_ERR_NONE;
}
int32_t emelk_kv_sequence_length(emelk_kv_actor *, int32_t) { return 100; }
bool emelk_kv_allocate_slots(emelk_kv_actor *, const emelk_event_allocate_slots *) { return true; }
bool emelk_kv_rollback_slots(emelk_kv_actor *, const emelk_event_rollback_slots *) { return true; }
bool emelk_kv_cache_copy_block(int32_t, int32_t, int32_t, void *, int32_t *) { return true; }
emel_error_type emelk_kv_export_block_tables(emelk_kv_actor *, const int32_t *, int32_t,
                                             uint16_t *, int32_t) {
  return EMELK_ERR_NONE;
}
void *emelk_kv_cache_k_pool(emelk_kv_cache *) { return nullptr; }
void *emelk_kv_cache_v_pool(emelk_kv_cache *) { return nullptr; }
emel_error_type emelk_kv_qkv_rope_append(const emelk_kv_geometry *, void *, void *, int32_t,
                                         const float *, float *, const float *, const float *,
                                         int32_t, int32_t, const int32_t *, const uint16_t *,
                                         int32_t, const emelk_rope_table *, const float *,
                                         const float *, int32_t, float, void *) {
  return EMELK_ERR_NONE;
}
emel_error_type emelk_attn_decode(const emelk_kv_geometry *, const void *, const void *, int32_t,
                                  const float *, float *, int32_t, const int32_t *, int32_t,
                                  const uint16_t *, int32_t, float, void *, uint64_t bytes, void *) {
  decode_got = bytes;
  return EMELK_ERR_NONE;
}
}

namespace emelk {
uint64_t prefill_workspace_bound(const emelk_kv_geometry *, int64_t) { return k_prefill_most; }
emel_error_type prefill_chunk(const emelk_kv_geometry *, const void *, const void *, int32_t,
                              const float *, float *, int32_t, int32_t, const int32_t *,
                              const uint16_t *, int32_t, float, int64_t, void *, uint64_t bytes,
                              void *) {
  prefill_got = bytes;
  return EMELK_ERR_NONE;
}
}  // namespace emelk

#define CHECK(c)                                               \
  do {                                                         \
    if (!(c)) {                                                \
      std::printf("CHECK failed line %d: %s\n", __LINE__, #c); \
      return 1;                                                \
    }                                                          \
  } while (0)

int main() {
  emelk_kv_geometry g{};
  g.block_tokens = 16;
  char tag[3];
  auto *actor = reinterpret_cast<emelk_kv_actor *>(&tag[0]);
  auto *cache = reinterpret_cast<emelk_kv_cache *>(&tag[1]);
  auto *rope = reinterpret_cast<emelk_rope_table *>(&tag[2]);
  float q[4];
  const int32_t id = 0;
  const struct {
    uint64_t limit, want;
  } cases[] = {{~0ull, k_prefill_most}, {8u << 20, k_decode_need}, {k_decode_need, k_decode_need}};
  for (const auto &c : cases) {
    limit = c.limit;
    emelk_batch_decoder *d = nullptr;
    CHECK(emelk_batch_decoder_create(&g, actor, cache, rope, 4, 2000, nullptr, &d) == EMELK_ERR_NONE);
    CHECK(d != nullptr && sticky == hipSuccess);  // or the next launch would report it
    CHECK(emelk_batch_decoder_begin_step(d, &id, 1, 5, nullptr) == EMELK_ERR_NONE);
    CHECK(emelk_batch_decoder_layer(d, 0, q, q, q, q, nullptr, nullptr, 0, 1e-6f, 1.0f, q) ==
          EMELK_ERR_NONE);
    CHECK(prefill_got == c.want);
    CHECK(emelk_batch_decoder_begin_step(d, &id, 1, 1, nullptr) == EMELK_ERR_NONE);
    CHECK(emelk_batch_decoder_layer(d, 0, q, q, q, q, nullptr, nullptr, 0, 1e-6f, 1.0f, q) ==
          EMELK_ERR_NONE);
    CHECK(decode_got == c.want);
    emelk_batch_decoder_destroy(d);
    CHECK(live == 0);
  }
  limit = k_decode_need - 1;
  emelk_batch_decoder *d = nullptr;
  CHECK(emelk_batch_decoder_create(&g, actor, cache, rope, 4, 2000, nullptr, &d) ==
        EMELK_ERR_OUT_OF_MEMORY);
  CHECK(d == nullptr && live == 0);
  std::printf("ok\n");
  return 0;
}
