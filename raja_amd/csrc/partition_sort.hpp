// Long spans sorted by partition: one or two stable scatters by value range,
// then one block per run of neighbouring buckets (partition_sort.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rsort
{
// Levels a span of n pairs would be partitioned in (1 or 2), 0: not at all.
int partition_levels(int key_bytes, int val_bytes, int64_t n);

// Working memory beside the alternate buffers and the lookback descriptors,
// and the descriptor rows of each of the two arrays.
size_t partition_aux_bytes(int key_bytes, int val_bytes, int64_t n);
int64_t partition_desc_rows(int key_bytes, int val_bytes, int64_t n);

// Sorts the span in place if its keys spread evenly enough over their range;
// else *done is false and the span is as it was.  One wait for the stream's
// work up to the counts, none for the scatters.  `host_ok` is a word of
// pinned host memory, `ready` an event.
int partition_sort(int key_dtype, int val_bytes, int descending, void* keys, void* vals, int64_t n,
                   void* alt_keys, void* alt_vals, char* aux, uint32_t* desc, uint32_t* host_ok,
                   hipEvent_t ready, hipStream_t s, bool* done);

// Lookback waits of the partition's scatters that gave up since the last call.
int take_partition_timeouts(uint32_t* count);
}  // namespace rsort
