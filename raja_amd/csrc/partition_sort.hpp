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

struct PartitionMem
{
  void *alt_keys, *alt_vals;
  char* aux;
  uint32_t* desc;
  uint32_t* hist;          // the digit histograms of an LSD sort of the span
  int64_t lsd_desc_words;  // the descriptors of its first pass, at desc
  uint32_t* host;          // pinned: the decision, the sample's answer, the active digits
  hipEvent_t ready;
};

// Sorts the span in place if its keys spread evenly enough over their range;
// else *done is false and the span is as it was.  One wait for the stream's
// work up to the counts, none for the scatters.  Where the sample refuses the
// span, the digit histograms follow it without a word from the host:
// *digits is then the word of active digits (digit_hist.hpp), mem.hist and the
// first pass's descriptors are ready and an LSD sort starts with its passes; 0
// otherwise.
int partition_sort(int key_dtype, int val_bytes, int descending, void* keys, void* vals, int64_t n,
                   const PartitionMem& mem, hipStream_t s, bool* done, uint32_t* digits);

// Lookback waits of the partition's scatters that gave up since the last call.
int take_partition_timeouts(uint32_t* count);
}  // namespace rsort
