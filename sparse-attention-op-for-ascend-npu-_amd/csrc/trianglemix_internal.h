// Entry points of libtrianglemix.so for the torch adapter and the tests: not
// part of the public C ABI.  Same status codes and error text (tm_last_error) as there.
#ifndef TRIANGLEMIX_INTERNAL_H
#define TRIANGLEMIX_INTERNAL_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

// tm_reshape_and_cache with the slots of logical tokens first_token .. +
// num_tokens - 1 taken from the request's block table (table_cols entries).
int tmi_write_chunk_kv(const void* key, const void* value, void* key_cache, void* value_cache,
                       const int32_t* block_table, int64_t table_cols, int64_t first_token, int64_t num_tokens,
                       int64_t key_stride, int64_t value_stride, int64_t num_pages, void* stream);

// Those slots into slots[0 .. num_tokens - 1].
int tmi_chunk_slots(const int32_t* block_table, int64_t table_cols, int64_t first_token, int64_t num_tokens,
                    int64_t* slots, void* stream);

// Whether the kernel with 64 rows per wave runs this chunk (1 or 0; -1 for a
// call the entry points refuse).  Arguments as tm_chunk_plan.
int tmi_chunk_is_wide(int dense, int64_t query_tokens, int64_t query_start, int64_t seq_len, int64_t prompt_len);

#ifdef __cplusplus
}
#endif

#endif  // TRIANGLEMIX_INTERNAL_H
