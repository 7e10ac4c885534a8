// Stable sorts of ranges of up to local_sort_max() keys, each by one block or
// wave (local_sort.hip).
#pragma once

#include <algorithm>
#include <vector>

#include "segments.hpp"

namespace rsort
{
constexpr int kLocalClasses = 5;
constexpr int64_t kLocalMax[kLocalClasses] = {64, 512, 2048, 5120, 8192};

// Longest range one block sorts.
constexpr int64_t local_sort_max() { return kLocalMax[kLocalClasses - 1]; }

// Length class of a range of 1 .. local_sort_max() keys.
constexpr int local_class(int64_t n)
{
  int c = 0;
  while (c < kLocalClasses - 1 && n > kLocalMax[c]) ++c;
  return c;
}

// Orders the records by class, the longest first inside a class (blocks
// start in this order, so the last ones to end are short), and gives the
// first record of each class (first[kLocalClasses] = the number of records).
inline void order_by_class(std::vector<rs::SortSeg>& segs, int64_t (&first)[kLocalClasses + 1])
{
  std::sort(segs.begin(), segs.end(), [](const rs::SortSeg& a, const rs::SortSeg& b) {
    const int ca = local_class(a.n), cb = local_class(b.n);
    return ca != cb ? ca < cb : a.n > b.n;
  });
  size_t q = 0;
  for (int c = 0; c < kLocalClasses; ++c)
  {
    first[c] = (int64_t)q;
    while (q < segs.size() && local_class(segs[q].n) == c) ++q;
  }
  first[kLocalClasses] = (int64_t)segs.size();
}

// Sorts every range of a record array ordered by order_by_class (element
// offsets from the given bases); a range may be sorted in place.  `redo` holds
// a byte per record (working memory of this call).
int local_sort_batch(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                     void* out_k, void* out_v, const rs::SortSeg* d_segs,
                     const int64_t (&first)[kLocalClasses + 1], uint8_t* redo, hipStream_t s);

// Longest group of each of the two blocks local_sort_groups has (8 keys per thread).
constexpr int kGroupCaps[2] = {2560, 5120};

// Sorts every group [start[g], start[g + 1]) of a span, g < ngroups, one block
// each (start on the device; none longer than cap, one of kGroupCaps).
// `redo`: a byte per group.
int local_sort_groups(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                      void* out_k, void* out_v, const uint32_t* start, int64_t ngroups, int64_t cap, uint8_t* redo,
                      hipStream_t s);

// Sorts one span of 1 .. local_sort_max() keys.
int local_sort_one(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                   void* out_k, void* out_v, int64_t n, hipStream_t s);
}  // namespace rsort
