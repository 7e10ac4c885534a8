// Onesweep LSD radix sort of keys or (key, value) pairs.
//
// Reference: RAJA's HIP backend calls rocprim::radix_sort_keys/pairs over
// all key bits with double buffers and copies back when the result lands in
// the alternate buffer (include/RAJA/policy/hip/sort.hpp:77-495, 653-689);
// the semantics are RAJA's stable sort by operators::less / greater.
//
// Design (8-bit digits, P = 8*sizeof(key)/8 passes):
//   1. one read of all keys builds the P digit histograms (LDS counters per
//      block, wave-uniform digits added once per wave, then global atomics);
//   2. for large inputs a small kernel tells the host which digits differ, and
//      every pass whose digit is the same for all keys is skipped;
//   3. each pass is one kernel: each block owns one tile (16384 keys of 32
//      bits; 32 consecutive tiles of every 256 go to one XCD), loads its keys,
//      ranks them inside each wave by 8 ballots (peer lanes
//      with the same digit) against per-wave LDS digit counters, publishes
//      its per-digit counts, stages the keys in LDS in digit order, loads
//      its values, looks back over predecessor tiles for each digit (one
//      thread per digit, 8 predecessor rows in flight per step), then writes
//      the keys out so equal digits land in contiguous runs and stages and
//      writes the values the same way.  Each pass clears the
//      descriptors of the next one (two alternating arrays), so no clearing
//      launch or device counter is needed.
// Ranking follows input order inside a wave (item j, then lane) and across
// waves and tiles, so the sort is stable.
#include "digit_hist.hpp"
#include "local_sort.hpp"
#include "ops.hpp"
#include "onesweep.hpp"
#include "partition_sort.hpp"
#include "runtime.hpp"
#include "segments.hpp"
#include "tune.hpp"
#include "workspace.hpp"

namespace
{
// Working memory of one sort: alternate key/value buffers, the digit
// histograms and two descriptor arrays.
template<typename K, typename V, bool HAS_VALS>
struct SortWs
{
  using S = SortShape<K, V, HAS_VALS>;
  static constexpr int P = (int)sizeof(K);
  int64_t n, ntiles, desc_words;
  size_t keys_bytes, vals_bytes, hist_bytes, desc_bytes;
  explicit SortWs(int64_t n_, int items = 0) : n(n_)
  {
    ntiles = rc::ceil_div(n, S::tile(items));
    desc_words = ntiles * kRowStride;
    keys_bytes = rc::align_up((size_t)n * sizeof(K), 256);
    vals_bytes = HAS_VALS ? rc::align_up((size_t)n * sizeof(V), 256) : 0;
    hist_bytes = rc::align_up((size_t)P * kRadix * sizeof(uint32_t), 256);
    desc_bytes = 2 * (size_t)desc_words * sizeof(uint32_t);
  }
  size_t tmp_bytes() const { return keys_bytes + vals_bytes + hist_bytes; }
  size_t total() const { return tmp_bytes() + desc_bytes; }
};

// ---- segmented onesweep: the tiles of many ranges, one launch per pass ----------
// Consecutive tile records one histogram block takes at most (a range's
// records are consecutive, so a block adds its counts to the global rows
// once per range it meets instead of once per tile), and the blocks a launch
// keeps at least before it gives a block more than one record: a block of
// 4 records takes about 30 us, so small tables take one record per block.
constexpr int kSegHistTiles = 4;
constexpr int64_t kSegHistMinBlocks = 2048;

// Digit histograms of every range of a tile table: block b takes records
// per_block * b .. + per_block - 1, counts their keys' digits in LDS
// and adds the counts to the range's P rows of 256 counters when the range
// changes or its records end; it clears each record's descriptor row of the
// first pass.  Keys are read as 16-byte vectors at the element's alignment
// (a tile starts at any element), 4 in flight per thread, and counted as in
// hist_kernel (8 side-by-side copies of each bin, a digit uniform over a
// wave's full iteration added once).  The bench's batched serving spent
// 14.2 ms in this kernel with one 4-byte load per thread per step and one
// histogram, 9.0 ms with 8 keys in flight and the side-by-side copies, and
// each of those blocks took one record.
template<typename K, bool DESC, int P>
__global__ __launch_bounds__(256) void seg_hist_kernel(const K* __restrict__ keys,
                                                       const rs::SortTile* __restrict__ recs,
                                                       int64_t ntiles, int per_block,
                                                       int64_t tile_elems,
                                                       uint32_t* __restrict__ hist,
                                                       uint32_t* __restrict__ desc0)
{
  static_assert(sizeof(K) == 4, "the segmented onesweep takes 4-byte keys");
  constexpr int kCopies = 8;
  constexpr int VEC = 4;
  constexpr int U = 4;
  constexpr int kBins = P * kRadix * kCopies;
  typedef K uvec_t __attribute__((ext_vector_type(VEC), aligned(sizeof(K))));
  __shared__ uint32_t s_hist[kBins];
  for (int i = threadIdx.x; i < kBins; i += 256) s_hist[i] = 0u;
  __syncthreads();
  const int lane = lane_id();
  const int64_t t0 = (int64_t)blockIdx.x * per_block;
  const int64_t t1 = (t0 + per_block < ntiles) ? t0 + per_block : ntiles;
  for (int64_t t = t0; t < t1; ++t)
  {
    const rs::SortTile r = recs[t];
    const int64_t first = (int64_t)r.j * tile_elems;
    const int64_t rem = r.len - first;
    const int cnt = (int)(rem < tile_elems ? rem : tile_elems);
    const K* const kp = keys + r.ik + first;
    const int nvec = cnt / VEC;
    // waves step through the tile's vectors in runs of U * 256
    for (int base = 0; base < nvec; base += U * 256)
    {
      K k[U * VEC];
      if (base + U * 256 <= nvec)
      {
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
          const uvec_t x = __builtin_nontemporal_load(
              reinterpret_cast<const uvec_t*>(kp + (int64_t)(base + u * 256 + (int)threadIdx.x) * VEC));
#pragma unroll
          for (int e = 0; e < VEC; ++e) k[u * VEC + e] = x[e];
        }
        count_full_wave<K, DESC, P, U * VEC, kCopies>(k, s_hist, lane);
      }
      else
      {
        uint32_t* const hc = s_hist + lane % kCopies;
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
          const int v = base + u * 256 + (int)threadIdx.x;
          if (v < nvec)
          {
            const uvec_t x = *reinterpret_cast<const uvec_t*>(kp + (int64_t)v * VEC);
#pragma unroll
            for (int e = 0; e < VEC; ++e)
            {
#pragma unroll
              for (int p = 0; p < P; ++p)
              {
                atomicAdd(&hc[(p * kRadix + digit_of<K, DESC>(x[e], 8 * p)) * kCopies], 1u);
              }
            }
          }
        }
      }
    }
    // the last cnt % VEC keys
    if ((int)threadIdx.x < cnt - nvec * VEC)
    {
      const K key = kp[(int64_t)nvec * VEC + threadIdx.x];
      uint32_t* const hc = s_hist + lane % kCopies;
#pragma unroll
      for (int p = 0; p < P; ++p) atomicAdd(&hc[(p * kRadix + digit_of<K, DESC>(key, 8 * p)) * kCopies], 1u);
    }
    for (int i = threadIdx.x; i < kRowStride; i += 256) desc0[t * kRowStride + i] = 0u;
    if (t + 1 == t1 || recs[t + 1].seg != r.seg)
    {
      // add the range's counts to its rows and clear them for the next range
      __syncthreads();
      uint32_t* const h = hist + (int64_t)r.seg * P * kRadix;
      for (int b = threadIdx.x; b < P * kRadix; b += 256)
      {
        uint32_t c = 0;
#pragma unroll
        for (int q = 0; q < kCopies; ++q)
        {
          c += s_hist[b * kCopies + q];
          s_hist[b * kCopies + q] = 0u;
        }
        if (c) atomic_add_agent(&h[b], c);
      }
      __syncthreads();
    }
  }
}

// Sorts every range of a tile table (records built with tile SortShape::TILE)
// from the input into the output buffers, through the alternates; P is even,
// so the last pass lands in the output.  hist holds nranges * P * 256
// counters, desc 2 * ntiles descriptor rows; both need no clearing.
template<typename K, typename V, bool HAS_VALS, bool DESC>
int seg_sort_core(const K* in_k, const V* in_v, K* out_k, V* out_v, K* alt_k, V* alt_v,
                  const rs::SortTile* d_recs, int64_t ntiles, int64_t nranges, uint32_t* hist,
                  uint32_t* desc, hipStream_t s)
{
  using S = SortShape<K, V, HAS_VALS>;
  constexpr int P = (int)sizeof(K);
  static_assert(P % 2 == 0, "an even pass count ends in the output");
  if (ntiles <= 0) return RAJA_CDNA4_SUCCESS;
  if (ntiles > 0x7FFFFFFF) return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "too many tiles");
  rc::LookbackGate gate(s);  // one lookback launch at a time on the device
  RC_TRY(gate.status());
  rc::TimedScope ts("segmented_onesweep", s);
  const int64_t words = nranges * P * kRadix;
  const int64_t cb = rc::ceil_div(words, 256);
  hipLaunchKernelGGL(clear_words_kernel, dim3((unsigned)(cb < 1024 ? cb : 1024)), dim3(256), 0, s,
                     hist, words);
  const int per_block =
      (int)std::max<int64_t>(1, std::min<int64_t>(kSegHistTiles, ntiles / kSegHistMinBlocks));
  hipLaunchKernelGGL((seg_hist_kernel<K, DESC, P>), dim3((unsigned)rc::ceil_div(ntiles, (int64_t)per_block)),
                     dim3(256), 0, s, in_k, d_recs, ntiles, per_block, S::TILE, hist, desc);
  RC_HIP(hipGetLastError());
  uint32_t* const d0 = desc;
  uint32_t* const d1 = desc + ntiles * kRowStride;
  for (int p = 0; p < P; ++p)
  {
    hipLaunchKernelGGL((onesweep_kernel<K, V, RadixDigit<K, DESC>, HAS_VALS, S::BLOCK, S::ITEMS, true>),
                       dim3((unsigned)ntiles), dim3(S::BLOCK), 0, s, in_k, out_k, in_v, out_v,
                       (int64_t)0, RadixDigit<K, DESC>{8 * p}, hist + p * kRadix, (p & 1) ? d1 : d0, (p & 1) ? d0 : d1,
                       d_recs, p, alt_k, alt_v);
    RC_HIP(hipGetLastError());
  }
  return RAJA_CDNA4_SUCCESS;
}

// Sort (in_keys, in_vals) into (keys, vals); in_keys == keys sorts in place.
// tmp holds SortWs::tmp_bytes(), desc_mem SortWs::desc_bytes (its contents
// are ignored: the histogram kernel clears the first array and every pass
// clears the next).  With `pinned` (a word of pinned host memory) the host waits
// for the word of active digits, to skip passes whose digit is the same for
// every key.  `digits` not 0: that word, the histograms and the first pass's
// descriptors being there already.
template<typename K, typename V, bool HAS_VALS, bool DESC>
int sort_core(const K* in_keys, const V* in_vals, K* keys, V* vals, int64_t n, hipStream_t s,
              char* tmp, uint32_t* desc_mem, uint32_t* pinned, int items = 0, uint32_t digits = 0)
{
  using S = SortShape<K, V, HAS_VALS>;
  constexpr int P = (int)sizeof(K);
  if (items != S::kChoices[1] && items != S::kChoices[2]) items = 0;
  const SortWs<K, V, HAS_VALS> w(n, items);
  K* alt_keys = (K*)tmp;
  V* alt_vals = HAS_VALS ? (V*)(tmp + w.keys_bytes) : nullptr;
  uint32_t* hist = (uint32_t*)(tmp + w.keys_bytes + w.vals_bytes);
  uint32_t* desc[2] = {desc_mem, desc_mem + w.desc_words};
  const bool inplace = (const void*)in_keys == (const void*)keys;

  if (digits == 0u)
  {
    rc::TimedScope ts("radix_hist", s);
    hipLaunchKernelGGL(clear_words_kernel, dim3(1), dim3(256), 0, s, hist, (int64_t)P * kRadix);
    hipLaunchKernelGGL((hist_kernel<K>), dim3(hist_blocks(n)), dim3(256), 0, s, in_keys, n, DESC, hist, desc[0],
                       w.desc_words, (const uint32_t*)nullptr);
    RC_HIP(hipGetLastError());
    digits = kDigitsKnown | ((1u << P) - 1u);
    if (pinned && n >= (int64_t)1 << 18)
    {
      *(volatile uint32_t*)pinned = 0u;
      hipLaunchKernelGGL((digits_kernel<K>), dim3(1), dim3(256), 0, s, hist, (uint32_t)n, pinned);
      RC_HIP(hipGetLastError());
      RC_TRY(rc::wait_word(pinned, s, &digits));
    }
  }
  const int npass = __builtin_popcount(digits & ~kDigitsKnown);
  rc::LookbackGate gate(s);  // one lookback launch at a time on the device
  RC_TRY(gate.status());
  // Out of place, an even pass count starts into the alternate buffers and
  // an odd one into the outputs, so the last pass always lands in the
  // outputs.  In place, passes start into the alternates and an odd count
  // ends with one copy back.
  const K* ksrc = in_keys;
  const V* vsrc = in_vals;
  bool to_alt = inplace || (npass % 2 == 0);
  int q = 0;
  for (int p = 0; p < P; ++p)
  {
    if (((digits >> p) & 1u) == 0u) continue;
    K* kdst = to_alt ? alt_keys : keys;
    V* vdst = to_alt ? alt_vals : vals;
    rc::TimedScope ts("onesweep_pass", s);
    if (items != 0 && items == S::kChoices[1])
    {
      hipLaunchKernelGGL((onesweep_kernel<K, V, RadixDigit<K, DESC>, HAS_VALS, S::BLOCK, S::kChoices[1] ? S::kChoices[1] : S::ITEMS>),
                         dim3((unsigned)w.ntiles), dim3(S::BLOCK), 0, s, (K*)ksrc, kdst, (V*)vsrc,
                         vdst, n, RadixDigit<K, DESC>{8 * p}, hist + p * kRadix, desc[q & 1], desc[(q + 1) & 1]);
    }
    else if (items != 0 && items == S::kChoices[2])
    {
      hipLaunchKernelGGL((onesweep_kernel<K, V, RadixDigit<K, DESC>, HAS_VALS, S::BLOCK, S::kChoices[2] ? S::kChoices[2] : S::ITEMS>),
                         dim3((unsigned)w.ntiles), dim3(S::BLOCK), 0, s, (K*)ksrc, kdst, (V*)vsrc,
                         vdst, n, RadixDigit<K, DESC>{8 * p}, hist + p * kRadix, desc[q & 1], desc[(q + 1) & 1]);
    }
    else
    {
      hipLaunchKernelGGL((onesweep_kernel<K, V, RadixDigit<K, DESC>, HAS_VALS, S::BLOCK, S::ITEMS>),
                         dim3((unsigned)w.ntiles), dim3(S::BLOCK), 0, s, (K*)ksrc, kdst, (V*)vsrc,
                         vdst, n, RadixDigit<K, DESC>{8 * p}, hist + p * kRadix, desc[q & 1], desc[(q + 1) & 1]);
    }
    RC_HIP(hipGetLastError());
    ksrc = kdst;
    vsrc = vdst;
    to_alt = !to_alt;
    ++q;
  }
  if (ksrc != keys)
  {
    RC_HIP(hipMemcpyAsync(keys, ksrc, (size_t)n * sizeof(K), hipMemcpyDeviceToDevice, s));
    if (HAS_VALS)
    {
      RC_HIP(hipMemcpyAsync(vals, vsrc, (size_t)n * sizeof(V), hipMemcpyDeviceToDevice, s));
    }
  }
  return RAJA_CDNA4_SUCCESS;
}

// In-place sort with the stream's scratch.  items >= 0: LSD passes in this tile
// (0: the full one), for the tuner.  items < 0: one block, the partition or LSD
// passes, by length and keys, the passes in the tuned tile of their (key type,
// length bucket), else the length's.
template<typename K, typename V, bool HAS_VALS, bool DESC>
int sort_impl(K* keys, V* vals, int64_t n, hipStream_t s, int items = -1)
{
  if (n > kMaxSortN)
  {
    return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "sort length %lld exceeds %lld",
                         (long long)n, (long long)kMaxSortN);
  }
  const bool lsd_only = items >= 0;
  if (!lsd_only && n <= rsort::local_sort_max())
  {
    // One launch of one block (local_sort.hip) instead of a clear, a
    // histogram and a pass per digit over one tile.
    rc::TimedScope ts("block_sort", s);
    return rsort::local_sort_one(rk::dtype_code<K>(), HAS_VALS ? (int)sizeof(V) : 0, DESC ? 1 : 0, keys,
                                 vals, keys, vals, n, s);
  }
  using S = SortShape<K, V, HAS_VALS>;
  if (!lsd_only && !S::wide) RC_TRY(rtune::choice(rtune::kSortPairs, rk::dtype_code<K>(), n, s, &items));
  if (items < 0)
  {
    // Untuned spans: small tiles where the full one leaves CUs idle.  FP32
    // keys ~ N(0, 1), per sort at 16384- / 8192- / 4096-key tiles: n = 10^4 93 /
    // 65 / 53 us, 2^17 87 / 66 / 60, 2^20 153 / 137 / 130, 2^21 139 / 125 / 131, 2^22
    // 162 / 161 / 162.
    items = n <= ((int64_t)5 << 18) ? 8 : (!S::wide && n <= ((int64_t)3 << 20) ? 16 : 0);
  }
  rc::StreamCtx* c = nullptr;
  RC_TRY(rc::get_ctx(s, &c));
  const SortWs<K, V, HAS_VALS> w(n, items);
  // Under stream capture the word of active digits (a host wait) cannot be had:
  // every pass is executed instead, with the same result.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  RC_HIP(hipStreamIsCapturing(s, &cap));
  uint32_t* const pinned = cap == hipStreamCaptureStatusNone ? (uint32_t*)c->pinned : nullptr;
  constexpr int kb = (int)sizeof(K), vb = HAS_VALS ? (int)sizeof(V) : 0;
  const bool part = !lsd_only && pinned && rsort::partition_levels(kb, vb, n) > 0;
  size_t tmp = w.tmp_bytes(), desc = w.desc_bytes;
  uint32_t digits = 0;
  if (part)
  {
    tmp += rsort::partition_aux_bytes(kb, vb, n);
    desc = std::max(desc, 2 * (size_t)rsort::partition_desc_rows(kb, vb, n) * kRowStride * sizeof(uint32_t));
  }
  RC_TRY(rc::ensure_tmp(c, tmp));
  RC_TRY(rc::ensure_sort_desc(c, desc));
  if (part)
  {
    if (!c->ready) RC_HIP(hipEventCreateWithFlags(&c->ready, hipEventDisableTiming));
    char* const t = (char*)c->tmp;
    const rsort::PartitionMem mem{t, t + w.keys_bytes, t + w.tmp_bytes(), (uint32_t*)c->sort_desc,
                                  (uint32_t*)(t + w.keys_bytes + w.vals_bytes), w.desc_words, pinned, c->ready};
    bool done = false;
    RC_TRY(rsort::partition_sort(rk::dtype_code<K>(), vb, DESC ? 1 : 0, keys, vals, n, mem, s, &done, &digits));
    if (done) return RAJA_CDNA4_SUCCESS;
  }
  return sort_core<K, V, HAS_VALS, DESC>(keys, vals, keys, vals, n, s, (char*)c->tmp,
                                         (uint32_t*)c->sort_desc, pinned, items, digits);
}

template<typename K>
int sort_key_type(void* keys, void* vals, int val_bytes, int64_t n, int descending, hipStream_t s)
{
  if (!vals)
  {
    return descending ? sort_impl<K, uint32_t, false, true>((K*)keys, nullptr, n, s)
                      : sort_impl<K, uint32_t, false, false>((K*)keys, nullptr, n, s);
  }
  if (val_bytes == 4)
  {
    return descending ? sort_impl<K, uint32_t, true, true>((K*)keys, (uint32_t*)vals, n, s)
                      : sort_impl<K, uint32_t, true, false>((K*)keys, (uint32_t*)vals, n, s);
  }
  if (val_bytes == 8)
  {
    return descending ? sort_impl<K, uint64_t, true, true>((K*)keys, (uint64_t*)vals, n, s)
                      : sort_impl<K, uint64_t, true, false>((K*)keys, (uint64_t*)vals, n, s);
  }
  return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "value size %d (4 or 8 supported)", val_bytes);
}

}  // namespace

namespace rsort
{
void tile_choices(int key_dtype, int out[3])
{
  const int* c = (key_dtype == RAJA_CDNA4_U32 || key_dtype == RAJA_CDNA4_I32 ||
                  key_dtype == RAJA_CDNA4_F32)
                     ? SortShape<uint32_t, uint32_t, true>::kChoices
                     : SortShape<uint64_t, uint32_t, true>::kChoices;
  for (int i = 0; i < 3; ++i) out[i] = c[i];
}

int tune_sort(int key_dtype, void* keys, void* vals, int64_t n, int items, hipStream_t s)
{
  switch (key_dtype)
  {
    case RAJA_CDNA4_U32: return sort_impl<uint32_t, uint32_t, true, false>((uint32_t*)keys, (uint32_t*)vals, n, s, items);
    case RAJA_CDNA4_I32: return sort_impl<int32_t, uint32_t, true, false>((int32_t*)keys, (uint32_t*)vals, n, s, items);
    case RAJA_CDNA4_F32: return sort_impl<float, uint32_t, true, false>((float*)keys, (uint32_t*)vals, n, s, items);
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "sort shapes are tuned for 4-byte keys");
  }
}

int64_t seg_tile() { return SortShape<uint32_t, uint32_t, true>::TILE; }

size_t seg_desc_bytes(int64_t ntiles)
{
  return 2 * (size_t)ntiles * kRowStride * sizeof(uint32_t);
}

size_t seg_hist_bytes(int64_t nranges)
{
  return (size_t)nranges * 4 * kRadix * sizeof(uint32_t);
}

int seg_sort_table(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                   void* out_k, void* out_v, void* alt_k, void* alt_v, const rs::SortTile* d_recs,
                   int64_t ntiles, int64_t nranges, uint32_t* hist, uint32_t* desc, hipStream_t s)
{
  if (val_bytes != 0 && val_bytes != 4)
  {
    return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "segmented onesweep takes 4-byte values");
  }
#define RSORT_SEG_CASE(CODE, K)                                                                   \
  case CODE:                                                                                      \
    if (val_bytes == 4)                                                                           \
      return descending                                                                           \
                 ? seg_sort_core<K, uint32_t, true, true>(                                        \
                       (const K*)in_k, (const uint32_t*)in_v, (K*)out_k, (uint32_t*)out_v,        \
                       (K*)alt_k, (uint32_t*)alt_v, d_recs, ntiles, nranges, hist, desc, s)        \
                 : seg_sort_core<K, uint32_t, true, false>(                                       \
                       (const K*)in_k, (const uint32_t*)in_v, (K*)out_k, (uint32_t*)out_v,        \
                       (K*)alt_k, (uint32_t*)alt_v, d_recs, ntiles, nranges, hist, desc, s);       \
    return descending                                                                             \
               ? seg_sort_core<K, uint32_t, false, true>((const K*)in_k, nullptr, (K*)out_k,      \
                                                          nullptr, (K*)alt_k, nullptr, d_recs,    \
                                                          ntiles, nranges, hist, desc, s)         \
               : seg_sort_core<K, uint32_t, false, false>((const K*)in_k, nullptr, (K*)out_k,     \
                                                           nullptr, (K*)alt_k, nullptr, d_recs,   \
                                                           ntiles, nranges, hist, desc, s);
  switch (key_dtype)
  {
    RSORT_SEG_CASE(RAJA_CDNA4_U32, uint32_t)
    RSORT_SEG_CASE(RAJA_CDNA4_I32, int32_t)
    RSORT_SEG_CASE(RAJA_CDNA4_F32, float)
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "segmented onesweep takes 4-byte keys");
  }
#undef RSORT_SEG_CASE
}

int take_spin_timeouts(uint32_t* count)
{
  uint32_t v = 0;
  RC_HIP(hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_spin_timeouts), sizeof(v)));
  if (v)
  {
    const uint32_t zero = 0;
    RC_HIP(hipMemcpyToSymbol(HIP_SYMBOL(g_spin_timeouts), &zero, sizeof(zero)));
  }
  uint32_t p = 0;
  RC_TRY(take_partition_timeouts(&p));
  *count = v + p;
  return RAJA_CDNA4_SUCCESS;
}
}  // namespace rsort

namespace rws
{
size_t sort_u32_i32_ws_bytes(int64_t n)
{
  return SortWs<uint32_t, uint32_t, true>(n).total();
}

int sort_pairs_u32_i32(const uint32_t* in_keys, const int32_t* in_vals, uint32_t* out_keys,
                       int32_t* out_vals, int64_t n, void* ws, hipStream_t s)
{
  if (n <= 0) return RAJA_CDNA4_SUCCESS;
  if (n > kMaxSortN) return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "sort too long");
  if (n == 1)
  {
    RC_HIP(hipMemcpyAsync(out_keys, in_keys, 4, hipMemcpyDeviceToDevice, s));
    RC_HIP(hipMemcpyAsync(out_vals, in_vals, 4, hipMemcpyDeviceToDevice, s));
    return RAJA_CDNA4_SUCCESS;
  }
  const SortWs<uint32_t, uint32_t, true> w(n);
  return sort_core<uint32_t, uint32_t, true, false>(in_keys, (const uint32_t*)in_vals, out_keys,
                                                    (uint32_t*)out_vals, n, s, (char*)ws,
                                                    (uint32_t*)((char*)ws + w.tmp_bytes()), nullptr);
}
}  // namespace rws

extern "C" {

int raja_cdna4_sort_pairs(int key_dtype, void* keys, void* vals, int val_bytes, int64_t n,
                          int descending, void* stream)
{
  if (n < 0) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "negative length");
  if (n <= 1) return RAJA_CDNA4_SUCCESS;  // pattern/sort.hpp:74-82
  if (!keys) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "keys is NULL");
  hipStream_t s = (hipStream_t)stream;
  switch (key_dtype)
  {
    case RAJA_CDNA4_U32: return sort_key_type<uint32_t>(keys, vals, val_bytes, n, descending, s);
    case RAJA_CDNA4_I32: return sort_key_type<int32_t>(keys, vals, val_bytes, n, descending, s);
    case RAJA_CDNA4_F32: return sort_key_type<float>(keys, vals, val_bytes, n, descending, s);
    case RAJA_CDNA4_U64: return sort_key_type<uint64_t>(keys, vals, val_bytes, n, descending, s);
    case RAJA_CDNA4_I64: return sort_key_type<int64_t>(keys, vals, val_bytes, n, descending, s);
    case RAJA_CDNA4_F64: return sort_key_type<double>(keys, vals, val_bytes, n, descending, s);
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "key dtype %d", key_dtype);
  }
}

}  // extern "C"
