// Segment plans: the device segment/tile table behind the batched entry
// points.  A plan is built once from host offsets and reused by every
// segmented reduce/scan/sort call on it (and by graph replays of them).
#pragma once

#include <map>
#include <mutex>
#include <vector>

#include "runtime.hpp"

namespace rs
{

// One tile of one segment.
struct TileRec
{
  int64_t seg_start;  // element offset of the segment in the input
  int64_t seg_len;    // segment length
  uint32_t j;         // tile index inside the segment
  uint32_t seg;       // segment index
  int64_t out_delta;  // output element offset minus input element offset
};

// One short segment sorted by one block: where its keys and values are read
// and written (element offsets from the kernel's base pointers), and its
// length.
struct SortSeg
{
  int64_t in_keys;
  int64_t in_vals;
  int64_t out_keys;
  int64_t out_vals;
  int64_t n;
};

// One tile of one range sorted by the segmented onesweep: element offsets of
// the range's keys and values in the input (ik, iv), output (ok, ov) and
// alternate (ak, av) buffers, each from that buffer's base pointer; the
// range length, the tile's index inside the range and the range's index
// (its digit-histogram row).
struct SortTile
{
  int64_t ik, iv, ok, ov, ak, av;
  int64_t len;
  uint32_t j;
  uint32_t seg;
};

// Tile records of segments given as (input start, length, output start).
inline void append_tiles(std::vector<TileRec>& recs, int64_t start, int64_t len, int64_t out_start,
                         uint32_t seg, int64_t tile)
{
  const int64_t nt = (len + tile - 1) / tile;
  for (int64_t j = 0; j < nt; ++j)
  {
    recs.push_back(TileRec{start, len, (uint32_t)j, seg, out_start - start});
  }
}

// Tile records of one tile size.  A table built with a short-segment limit
// holds the tiles of the longer segments only, and the short ones (1 .. limit
// elements) as a separate list of one record each.
struct TileTable
{
  int64_t tile = 0;
  int64_t ntiles = 0;
  TileRec* d_tiles = nullptr;
  int64_t nshort = 0;
  TileRec* d_short = nullptr;
};

// A plan's segments as the batched reduction takes them, per quad size: one
// record for each short one (empty ones too), quad records of the others, and
// the first quad, quad count and output index of those of several quads.
struct ReduceTable
{
  int64_t nquads = 0, nlong = 0, nshort = 0;
  uint32_t max_count = 0;  // quads of the longest segment
  char* mem = nullptr;  // one allocation holds the arrays
  const TileRec* d_quads = nullptr;
  const TileRec* d_short = nullptr;
  const uint32_t* d_first = nullptr;
  const uint32_t* d_count = nullptr;
  const int64_t* d_out = nullptr;
};

}  // namespace rs

struct raja_cdna4_segments_s
{
  int device = 0;
  int64_t nseg = 0;
  int64_t total = 0;
  std::vector<int64_t> offsets;  // nseg + 1, host copy
  int64_t* d_offsets = nullptr;
  std::map<std::pair<int64_t, int64_t>, rs::TileTable> tables;  // scans: (tile, short limit)
  std::map<int64_t, rs::ReduceTable> reduce_tables;             // quad elements
  // The segments as the batched sort takes them, built at the plan's first
  // sort: records of those one block sorts, by length class (rsort::
  // order_by_class), tile records of the longer ones (segmented onesweep) and
  // the longer ones' indices.
  struct SortTable
  {
    bool built = false;
    rs::SortSeg* d_segs = nullptr;
    int64_t first[6] = {0, 0, 0, 0, 0, 0};
    rs::SortTile* d_tiles = nullptr;
    int64_t ntiles = 0;
    std::vector<int64_t> longer;
  };
  SortTable sorts;
  std::mutex lock;
};

namespace rs
{
// Table for tile size `tile` (built on first use, synchronously); with
// short_max > 0, segments of at most short_max elements go to the short list.
int get_table(raja_cdna4_segments_s* p, int64_t tile, const TileTable** out, int64_t short_max = 0);
}  // namespace rs

// Segmented onesweep (sort.hip): every range of a tile table of SortTile
// records (tile = seg_tile() keys, 4-byte keys, values of 4 bytes or none)
// sorted in one histogram launch and one launch per digit pass, from the
// input through the alternates into the output buffers.  hist holds
// seg_hist_bytes(nranges), desc seg_desc_bytes(ntiles); neither needs
// clearing.
namespace rsort
{
int64_t seg_tile();
size_t seg_desc_bytes(int64_t ntiles);
size_t seg_hist_bytes(int64_t nranges);
int seg_sort_table(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                   void* out_k, void* out_v, void* alt_k, void* alt_v, const rs::SortTile* d_recs,
                   int64_t ntiles, int64_t nranges, uint32_t* hist, uint32_t* desc, hipStream_t s);
}  // namespace rsort

// Launcher implemented in scan.hip for segmented scans (SEG mode of the
// single-pass scan kernel; lookback stops at each segment's first tile).
namespace rscan
{
int launch_segmented_scan(int dtype, int op, bool exclusive, const void* in, void* out,
                          raja_cdna4_segments_s* plan, const void* init, hipStream_t s);
}  // namespace rscan
