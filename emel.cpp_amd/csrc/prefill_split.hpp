// Chunked prefill with the keys split over workgroups (attn_prefill.hip), for
// the C entry points and the step executor.
#pragma once

#include <stdint.h>

#include "emelk.h"

namespace emelk {

// Enough workspace for every call on this geometry whose sequences hold at
// most max_keys tokens, their chunk included (0: every one runs unsplit).
uint64_t prefill_workspace_bound(const emelk_kv_geometry *g, int64_t max_keys);

// emelk_attn_prefill_chunk_ws with the longest sequence's token count given.
emel_error_type prefill_chunk(const emelk_kv_geometry *g, const void *k_pool, const void *v_pool,
                              int32_t layer, const float *q, float *out, int32_t n_seq,
                              int32_t n_q, const int32_t *q_start, const uint16_t *block_tables,
                              int32_t table_stride, float scale, int64_t max_keys,
                              void *workspace, uint64_t workspace_bytes, void *stream);

}  // namespace emelk
