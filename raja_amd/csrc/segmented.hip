// Batched (segmented) reduce, scan and sort over a segment plan.
//
// The reference runs one algorithm call per range (one forall / scan /
// sort_pairs per segment, include/RAJA/policy/hip/{reduce,scan,sort}.hpp);
// thousands of small uneven ranges then pay one launch (and for scan/sort,
// rocPRIM's temp-storage query and allocation) each.  Here one plan holds
// the device segment/tile table, and each batched call is one or two
// kernels over all segments:
//   * reduce: one block per quad and one wave per short segment, then one
//     wave folds the quad values of each segment of several -- the same tree as the span reduction (reduce_tree.hpp), so a segment's
//     result is bit-identical alone and in the batch;
//   * scan: the single-pass scan kernel over the tile table; each segment
//     starts from init and its lookback stops at its own first tile.
//     Segments of at most one wave chunk are scanned one per wave by a
//     second kernel on the same stream (no descriptors, same bits);
//   * sort_pairs: one block (or wave) per segment of up to 8192 keys sorts
//     it in LDS (local_sort.hip); the longer segments of 4-byte keys (and 4-byte or no values) are sorted
//     together by the segmented onesweep (one histogram launch, one launch
//     per digit pass over all their tiles); 8-byte keys or values take one
//     onesweep sort per longer segment.
#include <string.h>

#include <algorithm>
#include <utility>
#include <vector>

#include "local_sort.hpp"
#include "reduce_tree.hpp"
#include "segments.hpp"
#include "workspace.hpp"

namespace
{
// A host array's copy on the device.  Freed again unless release() hands it
// over, which a table's builder does once all its copies have succeeded: a
// plan never holds an array whose upload failed (a first call under stream
// capture is one way for it to fail).
class Upload
{
 public:
  Upload() = default;
  Upload(const Upload&) = delete;
  Upload& operator=(const Upload&) = delete;
  ~Upload()
  {
    if (p_) (void)hipFree(p_);
  }
  template<typename T>
  int put(const std::vector<T>& v)
  {
    const size_t bytes = sizeof(T) * v.size();
    hipError_t e = hipMalloc(&p_, bytes ? bytes : 1);
    if (e != hipSuccess)
    {
      p_ = nullptr;
    }
    else if (bytes)
    {
      e = hipMemcpy(p_, v.data(), bytes, hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) return RAJA_CDNA4_SUCCESS;
    (void)hipGetLastError();  // reported here, not by the next call's launch
    return rc::hip_error(e, "segment table upload", __FILE__, __LINE__);
  }
  template<typename T>
  T* release()
  {
    return static_cast<T*>(std::exchange(p_, nullptr));
  }

 private:
  void* p_ = nullptr;
};
}  // namespace

namespace rs
{

int get_table(raja_cdna4_segments_s* p, int64_t tile, const TileTable** out, int64_t short_max)
{
  std::lock_guard<std::mutex> g(p->lock);
  const auto key = std::make_pair(tile, short_max);
  auto it = p->tables.find(key);
  if (it != p->tables.end())
  {
    *out = &it->second;
    return RAJA_CDNA4_SUCCESS;
  }
  TileTable t;
  t.tile = tile;
  std::vector<TileRec> recs, shorts;
  for (int64_t s = 0; s < p->nseg; ++s)
  {
    const int64_t b = p->offsets[(size_t)s], len = p->offsets[(size_t)s + 1] - b;
    if (len > 0 && len <= short_max)
      shorts.push_back(TileRec{b, len, 0u, (uint32_t)s, 0});
    else
      append_tiles(recs, b, len, b, (uint32_t)s, tile);
  }
  t.ntiles = (int64_t)recs.size();
  t.nshort = (int64_t)shorts.size();
  Upload up_recs, up_shorts;
  RC_TRY(up_recs.put(recs));
  RC_TRY(up_shorts.put(shorts));
  t.d_tiles = up_recs.release<TileRec>();
  t.d_short = up_shorts.release<TileRec>();
  auto ins = p->tables.emplace(key, t);
  *out = &ins.first->second;
  return RAJA_CDNA4_SUCCESS;
}

}  // namespace rs

namespace
{
using namespace RAJA::cdna4::dev;

// ---- segmented reduce ----------------------------------------------------------

constexpr int kSegMaxGroups = 64;  // segments of up to 4096 tiles

// Blocks 0 .. nquads-1 compute one quad each (a segment of one quad is done
// there, result and init included); the blocks after them do a short segment
// (short_elems() or fewer) per wave, which fills the tail.
template<typename T, typename Op>
__global__ __launch_bounds__(rt::kBlock) void seg_quads_kernel(
    const T* __restrict__ x, const rs::TileRec* __restrict__ quads, int64_t nquads,
    const rs::TileRec* __restrict__ shorts, int64_t nshort,
    typename Op::acc_t* __restrict__ partials, typename Op::acc_t init, rt::ResultOut<Op> out)
{
  using acc_t = typename Op::acc_t;
  __shared__ acc_t s_w[rt::kBlockWaves];
  if ((int64_t)blockIdx.x < nquads)
  {
    const rs::TileRec r = quads[blockIdx.x];
    const acc_t v = rt::fold_quad<T, Op>(x + r.seg_start, r.seg_len, r.j, s_w);
    if (threadIdx.x != 0) return;
    if (r.seg_len > rt::quad_elems<T, Op>())
    {
      partials[blockIdx.x] = v;
      return;
    }
    const acc_t id = Op::ident();
    out.put(r.seg, Op::with_init(init, rt::fold4<Op>(v, id, id, id)));
    return;
  }
  const int64_t q = ((int64_t)blockIdx.x - nquads) * rt::kBlockWaves +
                    __builtin_amdgcn_readfirstlane(wave_id());
  if (q >= nshort) return;
  const rs::TileRec r = shorts[q];
  const acc_t v = rt::fold_short<T, Op>(x + r.seg_start, r.seg_len);
  if (lane_id() == 0) out.put(r.seg, Op::with_init(init, v));
}

// One tile per block (the server's batches: a quarter of the records to
// build and upload, and enough tiles without the finer cut).
template<typename T, typename Op>
__global__ __launch_bounds__(rt::kBlock) void seg_tiles_kernel(
    const T* __restrict__ x, const rs::TileRec* __restrict__ tiles,
    typename Op::acc_t* __restrict__ partials)
{
  using acc_t = typename Op::acc_t;
  __shared__ acc_t s_w[16];
  const rs::TileRec r = tiles[blockIdx.x];
  const acc_t v = rt::fold_tile<T, Op>(x + r.seg_start, r.seg_len, r.j, s_w);
  if (threadIdx.x == 0) partials[blockIdx.x] = v;
}

// The plan's reduction table for quads of `quad` elements and one wave for
// segments of up to short_max, built and uploaded at its first use.
int get_reduce_table(raja_cdna4_segments_s* p, int64_t quad, int64_t short_max, const rs::ReduceTable** out)
{
  std::lock_guard<std::mutex> g(p->lock);
  auto it = p->reduce_tables.find(quad);
  if (it != p->reduce_tables.end())
  {
    *out = &it->second;
    return RAJA_CDNA4_SUCCESS;
  }
  rs::ReduceTable t;
  std::vector<rs::TileRec> quads, shorts;
  std::vector<uint32_t> first, count;
  std::vector<int64_t> index;
  for (int64_t s = 0; s < p->nseg; ++s)
  {
    const int64_t b = p->offsets[(size_t)s], len = p->offsets[(size_t)s + 1] - b;
    if (len <= short_max)
    {
      shorts.push_back(rs::TileRec{b, len, 0u, (uint32_t)s, 0});
      continue;
    }
    const int64_t nq = rc::ceil_div(len, quad);
    if (nq > 1)
    {
      first.push_back((uint32_t)quads.size());
      count.push_back((uint32_t)nq);
      index.push_back(s);
    }
    t.max_count = std::max(t.max_count, (uint32_t)nq);
    rs::append_tiles(quads, b, len, b, (uint32_t)s, quad);
  }
  t.nquads = (int64_t)quads.size();
  t.nlong = (int64_t)first.size();
  t.nshort = (int64_t)shorts.size();
  // one allocation and one copy for the five arrays (8-byte ones first)
  std::vector<char> image;
  auto place = [&image](const auto& v) {
    const size_t at = image.size();
    const size_t bytes = sizeof(v[0]) * v.size();
    image.resize(at + bytes);
    if (bytes) ::memcpy(image.data() + at, v.data(), bytes);
    return at;
  };
  image.reserve(sizeof(rs::TileRec) * (quads.size() + shorts.size()) + 16 * first.size() + 64);
  const size_t at_quads = place(quads), at_shorts = place(shorts), at_out = place(index),
               at_first = place(first), at_count = place(count);
  Upload up;
  RC_TRY(up.put(image));
  t.mem = up.release<char>();
  t.d_quads = (const rs::TileRec*)(t.mem + at_quads);
  t.d_short = (const rs::TileRec*)(t.mem + at_shorts);
  t.d_out = (const int64_t*)(t.mem + at_out);
  t.d_first = (const uint32_t*)(t.mem + at_first);
  t.d_count = (const uint32_t*)(t.mem + at_count);
  *out = &p->reduce_tables.emplace(quad, t).first->second;
  return RAJA_CDNA4_SUCCESS;
}

template<typename T, typename Op>
int seg_reduce(raja_cdna4_segments_s* p, const T* x, typename Op::acc_t init,
               typename Op::acc_t* out, hipStream_t s)
{
  using acc_t = typename Op::acc_t;
  if (p->nseg == 0) return RAJA_CDNA4_SUCCESS;
  const rs::ReduceTable* tab = nullptr;
  RC_TRY(get_reduce_table(p, rt::quad_elems<T, Op>(), rt::short_elems<T, Op>(), &tab));
  if (tab->max_count > (uint32_t)kSegMaxGroups * 64 * 4)
  {
    return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "segment too long for the batched reduce");
  }
  rc::StreamCtx* c = nullptr;
  RC_TRY(rc::get_ctx(s, &c));
  RC_TRY(rc::ensure_tmp(c, (size_t)(tab->nquads + 1) * sizeof(acc_t)));
  acc_t* partials = (acc_t*)c->tmp;
  rc::TimedScope ts("segmented_reduce", s);
  const int64_t grid = tab->nquads + rc::ceil_div(tab->nshort, rt::kBlockWaves);
  hipLaunchKernelGGL((seg_quads_kernel<T, Op>), dim3((unsigned)grid), dim3(rt::kBlock), 0, s, x,
                     tab->d_quads, tab->nquads, tab->d_short,
                     tab->nshort, partials, init, rt::ResultOut<Op>{out});
  RC_HIP(hipGetLastError());
  if (tab->nlong > 0)
  {
    hipLaunchKernelGGL((rt::final_kernel<Op, 1, kSegMaxGroups, true>), dim3((unsigned)tab->nlong),
                       dim3(64), 0, s, partials, tab->d_first, tab->d_count, (int64_t)0, init,
                       rt::ResultOut<Op>{out}, tab->d_out);
    RC_HIP(hipGetLastError());
  }
  return RAJA_CDNA4_SUCCESS;
}

template<typename T>
int seg_reduce_typed(raja_cdna4_segments_s* p, int op, const void* x, const void* init, void* out,
                     hipStream_t s)
{
  const T iv = *static_cast<const T*>(init);
  switch (op)
  {
    case RAJA_CDNA4_OP_PLUS: return seg_reduce<T, rk::OpPlus<T>>(p, (const T*)x, iv, (T*)out, s);
    case RAJA_CDNA4_OP_MIN: return seg_reduce<T, rk::OpMin<T>>(p, (const T*)x, iv, (T*)out, s);
    case RAJA_CDNA4_OP_MAX: return seg_reduce<T, rk::OpMax<T>>(p, (const T*)x, iv, (T*)out, s);
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "operator %d not supported here", op);
  }
}

// ---- segmented sort: short segments in one block or wave each -----------------------

// The plan's sort records, built and uploaded at its first sort.
int get_sort_table(raja_cdna4_segments_s* p, const raja_cdna4_segments_s::SortTable** out)
{
  std::lock_guard<std::mutex> g(p->lock);
  raja_cdna4_segments_s::SortTable& t = p->sorts;
  *out = &t;
  if (t.built) return RAJA_CDNA4_SUCCESS;
  std::vector<rs::SortSeg> small;
  std::vector<rs::SortTile> recs;
  const int64_t tile = rsort::seg_tile();
  t.longer.clear();
  for (int64_t g = 0; g < p->nseg; ++g)
  {
    const int64_t b = p->offsets[(size_t)g];
    const int64_t len = p->offsets[(size_t)g + 1] - b;
    if (len <= 1) continue;
    if (len <= rsort::local_sort_max())
    {
      small.push_back(rs::SortSeg{b, b, b, b, len});
      continue;
    }
    for (int64_t j = 0; j * tile < len; ++j)
    {
      recs.push_back(rs::SortTile{b, b, b, b, b, b, len, (uint32_t)j, (uint32_t)t.longer.size()});
    }
    t.longer.push_back(g);
  }
  rsort::order_by_class(small, t.first);
  t.ntiles = (int64_t)recs.size();
  Upload up_segs, up_tiles;
  if (!small.empty()) RC_TRY(up_segs.put(small));
  if (!recs.empty()) RC_TRY(up_tiles.put(recs));
  t.d_segs = up_segs.release<rs::SortSeg>();
  t.d_tiles = up_tiles.release<rs::SortTile>();
  t.built = true;
  return RAJA_CDNA4_SUCCESS;
}

template<typename K, typename V, bool HAS_VALS, bool DESC>
int seg_sort(raja_cdna4_segments_s* p, K* keys, V* vals, int key_dtype, int val_bytes,
             hipStream_t s)
{
  const raja_cdna4_segments_s::SortTable* tab = nullptr;
  RC_TRY(get_sort_table(p, &tab));
  if (tab->first[rsort::kLocalClasses] == 0 && tab->longer.empty()) return RAJA_CDNA4_SUCCESS;
  rc::StreamCtx* c = nullptr;
  RC_TRY(rc::get_ctx(s, &c));
  // Scratch of the whole call before its first launch: growing it waits for
  // the stream.
  constexpr bool kOneSweep = sizeof(K) == 4 && (!HAS_VALS || sizeof(V) == 4);
  const int64_t nranges = (int64_t)tab->longer.size();
  const size_t kb = rc::align_up((size_t)p->total * sizeof(K), 256);
  const size_t vb = HAS_VALS ? rc::align_up((size_t)p->total * sizeof(V), 256) : 0;
  if (kOneSweep && nranges > 0)
  {
    RC_TRY(rc::ensure_tmp(c, std::max(kb + vb + rsort::seg_hist_bytes(nranges),
                                      (size_t)tab->first[rsort::kLocalClasses])));
    RC_TRY(rc::ensure_sort_desc(c, rsort::seg_desc_bytes(tab->ntiles)));
  }
  if (tab->first[rsort::kLocalClasses] > 0)
  {
    // The block sorts' marks, a byte per segment: in the stream's fixed slots
    // while they fit (no growth, so a capture needs no call of the same size
    // before it, and a graph keeps a pointer that never moves).  The lock
    // keeps another thread's batch on this stream from coming between the
    // kernel that writes them and the one that reads them.
    std::lock_guard<std::mutex> g(c->small_lock);
    const size_t marks = (size_t)tab->first[rsort::kLocalClasses];
    uint8_t* redo = (uint8_t*)c->small;
    if (marks > rc::small_slot_bytes)
    {
      RC_TRY(rc::ensure_tmp(c, marks));
      redo = (uint8_t*)c->tmp;
    }
    rc::TimedScope ts("segmented_block_sort", s);
    RC_TRY(rsort::local_sort_batch(key_dtype, HAS_VALS ? val_bytes : 0, DESC ? 1 : 0, keys, vals, keys,
                                   vals, tab->d_segs, tab->first, redo, s));
  }
  if (tab->longer.empty()) return RAJA_CDNA4_SUCCESS;
  if constexpr (kOneSweep)
  {
    // Every longer segment in one segmented onesweep: alternates, histograms
    // and descriptors from the stream's scratch.
    char* tmp = (char*)c->tmp;
    return rsort::seg_sort_table(key_dtype, HAS_VALS ? 4 : 0, DESC ? 1 : 0, keys, vals, keys, vals,
                                 tmp, HAS_VALS ? (void*)(tmp + kb) : nullptr, tab->d_tiles,
                                 tab->ntiles, nranges, (uint32_t*)(tmp + kb + vb),
                                 (uint32_t*)c->sort_desc, s);
  }
  else
  {
    // 8-byte keys or values: one onesweep sort per longer segment.
    for (int64_t g : tab->longer)
    {
      const int64_t b = p->offsets[(size_t)g], len = p->offsets[(size_t)g + 1] - b;
      RC_TRY(raja_cdna4_sort_pairs(key_dtype, keys + b, HAS_VALS ? (void*)(vals + b) : nullptr,
                                   val_bytes, len, DESC ? 1 : 0, s));
    }
    return RAJA_CDNA4_SUCCESS;
  }
}

template<typename K>
int seg_sort_key(raja_cdna4_segments_s* p, int kd, void* keys, void* vals, int vb, int desc,
                 hipStream_t s)
{
  if (!vals)
  {
    return desc ? seg_sort<K, uint32_t, false, true>(p, (K*)keys, nullptr, kd, 0, s)
                : seg_sort<K, uint32_t, false, false>(p, (K*)keys, nullptr, kd, 0, s);
  }
  if (vb == 4)
  {
    return desc ? seg_sort<K, uint32_t, true, true>(p, (K*)keys, (uint32_t*)vals, kd, 4, s)
                : seg_sort<K, uint32_t, true, false>(p, (K*)keys, (uint32_t*)vals, kd, 4, s);
  }
  if (vb == 8)
  {
    return desc ? seg_sort<K, uint64_t, true, true>(p, (K*)keys, (uint64_t*)vals, kd, 8, s)
                : seg_sort<K, uint64_t, true, false>(p, (K*)keys, (uint64_t*)vals, kd, 8, s);
  }
  return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "value size %d (4 or 8 supported)", vb);
}

}  // namespace

namespace rws
{
int64_t sum_tile_f64() { return rt::tile_elems<double, rk::OpPlus<double>>(); }

int64_t sum_batch_max() { return (int64_t)kSegMaxGroups * 64 * rt::tile_elems<double, rk::OpPlus<double>>(); }

int table_sum_f64(const double* base, const rs::TileRec* d_tiles, int64_t ntiles,
                  const uint32_t* d_first, const uint32_t* d_count, int64_t nseg,
                  const int64_t* d_out_index, void* ws, hipStream_t s)
{
  using Op = rk::OpPlus<double>;
  if (nseg == 0) return RAJA_CDNA4_SUCCESS;
  double* partials = (double*)ws;
  rc::TimedScope ts("segmented_reduce", s);
  if (ntiles > 0)
  {
    hipLaunchKernelGGL((seg_tiles_kernel<double, Op>), dim3((unsigned)ntiles), dim3(rt::kBlock), 0, s,
                       base, d_tiles, partials);
    RC_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL((rt::final_kernel<Op, 1, kSegMaxGroups, false>), dim3((unsigned)nseg), dim3(64), 0, s,
                     (const double*)partials, d_first, d_count, (int64_t)0, 0.0,
                     rt::ResultOut<Op>{(double*)base}, d_out_index);
  RC_HIP(hipGetLastError());
  return RAJA_CDNA4_SUCCESS;
}

int64_t block_sort_max() { return rsort::local_sort_max(); }

int block_sort_u32_i32(const uint32_t* base, const rs::SortSeg* d_segs,
                       const int64_t (&first)[rsort::kLocalClasses + 1], uint8_t* redo, hipStream_t s)
{
  if (first[rsort::kLocalClasses] == 0) return RAJA_CDNA4_SUCCESS;
  rc::TimedScope ts("segmented_block_sort", s);
  return rsort::local_sort_batch(RAJA_CDNA4_U32, 4, 0, base, base, (void*)base, (void*)base, d_segs,
                                 first, redo, s);
}
}  // namespace rws

extern "C" {

int raja_cdna4_segments_create(const int64_t* offsets, int64_t nseg, raja_cdna4_segments_s** out)
{
  if (!out || nseg < 0 || (nseg > 0 && !offsets))
  {
    return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "bad segment arguments");
  }
  if (nseg > 0x7FFFFFFF) return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "too many segments");
  for (int64_t s = 0; s < nseg; ++s)
  {
    if (offsets[s + 1] < offsets[s] || offsets[0] < 0)
    {
      return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "offsets must be non-decreasing");
    }
  }
  raja_cdna4_segments_s* p = new raja_cdna4_segments_s();
  RC_HIP(hipGetDevice(&p->device));
  p->nseg = nseg;
  p->offsets.assign(offsets, offsets + nseg + 1);
  p->total = p->offsets.back();
  if (hipMalloc(&p->d_offsets, sizeof(int64_t) * (size_t)(nseg + 1)) != hipSuccess ||
      hipMemcpy(p->d_offsets, offsets, sizeof(int64_t) * (size_t)(nseg + 1), hipMemcpyHostToDevice) !=
          hipSuccess)
  {
    (void)hipGetLastError();
    delete p;
    return rc::set_error(RAJA_CDNA4_ERROR_OUT_OF_MEMORY, "segment plan upload failed");
  }
  *out = p;
  return RAJA_CDNA4_SUCCESS;
}

int raja_cdna4_segments_destroy(raja_cdna4_segments_s* p)
{
  if (!p) return RAJA_CDNA4_SUCCESS;
  RC_HIP(hipDeviceSynchronize());
  for (auto& kv : p->tables)
  {
    if (kv.second.d_tiles) RC_HIP(hipFree(kv.second.d_tiles));
    if (kv.second.d_short) RC_HIP(hipFree(kv.second.d_short));
  }
  for (auto& kv : p->reduce_tables) RC_HIP(hipFree(kv.second.mem));
  if (p->sorts.d_segs) RC_HIP(hipFree(p->sorts.d_segs));
  if (p->sorts.d_tiles) RC_HIP(hipFree(p->sorts.d_tiles));
  if (p->d_offsets) RC_HIP(hipFree(p->d_offsets));
  delete p;
  return RAJA_CDNA4_SUCCESS;
}

int raja_cdna4_segmented_reduce(raja_cdna4_segments_s* p, int dtype, int op, const void* x,
                                const void* init, void* out_dev, void* stream)
{
  if (!p || !init || !out_dev || (p->total > 0 && !x))
  {
    return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "NULL argument");
  }
  hipStream_t s = (hipStream_t)stream;
  switch (dtype)
  {
    case RAJA_CDNA4_I32: return seg_reduce_typed<int32_t>(p, op, x, init, out_dev, s);
    case RAJA_CDNA4_I64: return seg_reduce_typed<int64_t>(p, op, x, init, out_dev, s);
    case RAJA_CDNA4_F32: return seg_reduce_typed<float>(p, op, x, init, out_dev, s);
    case RAJA_CDNA4_F64: return seg_reduce_typed<double>(p, op, x, init, out_dev, s);
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "dtype %d not supported", dtype);
  }
}

int raja_cdna4_segmented_exclusive_scan(raja_cdna4_segments_s* p, int dtype, int op, const void* in,
                                        void* out, const void* init, void* stream)
{
  if (!p) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "NULL plan");
  return rscan::launch_segmented_scan(dtype, op, true, in, out, p, init, (hipStream_t)stream);
}

int raja_cdna4_segmented_inclusive_scan(raja_cdna4_segments_s* p, int dtype, int op, const void* in,
                                        void* out, void* stream)
{
  if (!p) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "NULL plan");
  return rscan::launch_segmented_scan(dtype, op, false, in, out, p, nullptr, (hipStream_t)stream);
}

int raja_cdna4_segmented_sort_pairs(raja_cdna4_segments_s* p, int key_dtype, void* keys, void* vals,
                                    int val_bytes, int descending, void* stream)
{
  if (!p || (p->total > 0 && !keys)) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "NULL argument");
  hipStream_t s = (hipStream_t)stream;
  switch (key_dtype)
  {
    case RAJA_CDNA4_U32: return seg_sort_key<uint32_t>(p, key_dtype, keys, vals, val_bytes, descending, s);
    case RAJA_CDNA4_I32: return seg_sort_key<int32_t>(p, key_dtype, keys, vals, val_bytes, descending, s);
    case RAJA_CDNA4_F32: return seg_sort_key<float>(p, key_dtype, keys, vals, val_bytes, descending, s);
    case RAJA_CDNA4_U64: return seg_sort_key<uint64_t>(p, key_dtype, keys, vals, val_bytes, descending, s);
    case RAJA_CDNA4_I64: return seg_sort_key<int64_t>(p, key_dtype, keys, vals, val_bytes, descending, s);
    case RAJA_CDNA4_F64: return seg_sort_key<double>(p, key_dtype, keys, vals, val_bytes, descending, s);
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "key dtype %d", key_dtype);
  }
}

}  // extern "C"
