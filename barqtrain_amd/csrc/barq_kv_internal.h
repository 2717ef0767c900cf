// Between libbarq_kv.so and its torch binding, beside the C ABI of include/barq_kv.h: calls that only a
// caller with the binding's host shadow makes.  Not part of the ABI.

#pragma once

#include <stdint.h>

#include "barq_kv.h"

namespace barq_internal {

// barq_kv_append of key_states[i] to row rows[i] (rows null: row i), i < batch <= 64, for a caller
// that knows the rows' lengths and marks and the free stack's top exactly.  BARQ_KV_ERR_UNSUPPORTED,
// nothing launched, for more rows or states and pools that 16-byte vectors do not fit.
int append_known(const barq_kv_pool* pool, const void* key_states, const void* value_states, int64_t batch,
                 int64_t tokens, int64_t stride_b, int64_t stride_h, int64_t stride_t, const int32_t* rows,
                 const int32_t* seq_lens, const int32_t* high_water, int64_t free_top, void* stream);

// The append of BARQ_KV_QUANT_DIRECT to rows [0, batch) that are all empty (length and mark 0), for a
// caller that knows so and the tops of both free stacks; with key_out / value_out also
// barq_kv_gather_cold of the `tokens` positions.  BARQ_KV_ERR_UNSUPPORTED, nothing launched, for what
// the kernel does not take, stacks that hold too few pages included.
int append_fresh_cold(const barq_kv_pool* pool, const barq_kv_cold* cold, const void* key_states,
                      const void* value_states, int64_t batch, int64_t tokens, int64_t stride_b, int64_t stride_h,
                      int64_t stride_t, void* key_out, void* value_out, int64_t osb, int64_t osh, int64_t oss,
                      int64_t free_top, int64_t cold_top, void* stream);

// barq_kv_compress for the lengths that rows [0, batch) reach after `ahead` more tokens, by a caller that
// knows that the cold stack holds enough pages: a row's blocks are then taken by several workgroups.
int compress_spread(const barq_kv_pool* pool, const barq_kv_cold* cold, int64_t batch, int64_t ahead, void* stream);

// barq_kv_update_cold (no BARQ_KV_SEQ_FROM_DEVICE) for a caller that knows the rows' lengths and marks
// exactly, and the free stack's top after the call's compress; BARQ_KV_ERR_UNSUPPORTED, nothing
// launched, for calls its one-launch update does not take.
int update_cold_known(const barq_kv_pool* pool, const barq_kv_cold* cold, const void* key_states,
                      const void* value_states, int64_t batch, int64_t tokens, int64_t stride_b, int64_t stride_h,
                      int64_t stride_t, void* key_out, void* value_out, int64_t seq_out, int64_t osb, int64_t osh,
                      int64_t oss, int64_t flags, const int32_t* seq_lens, const int32_t* high_water,
                      int64_t free_top, void* stream);

// barq_kv_crop of rows [0, batch) of n pools, whose row lengths are at seq_lens[i].
int crop_layers(int32_t* const* seq_lens, int64_t n, int64_t batch, int64_t max_length, void* stream);

// barq_kv_pool_reset (no page order) of n pools, with colds (one per pool, or null) also
// barq_kv_cold_reset.
int reset_layers(const barq_kv_pool* pools, const barq_kv_cold* colds, int64_t n, void* stream);

}  // namespace barq_internal
