// Long spans sorted by partition (the hybrid of most-significant-digit
// scatters and block-local sorts: Stehle and Jacobsen, "A Memory
// Bandwidth-Efficient Hybrid Radix Sort on GPUs", 2017).
//
// An LSD sort moves every pair once per 8-bit digit: 4 passes for 32-bit keys,
// 8 for 64-bit ones.  Here a monotone map sends keys to 65536 buckets (a
// linear map of the key, or of the value of floating keys, over the range a
// sample shows); a scatter by the map's high byte and one by its low byte, both
// the stable onesweep pass, leave every bucket contiguous and in order, and
// one block per few thousand neighbouring pairs sorts them in LDS
// (local_sort.hip).  That is 3 moves instead of 4 or 8.  Spans of up to about
// a million pairs need only the high byte: 2 moves.
//
// It takes keys that spread evenly enough that no bucket outgrows a block.
// A sample of 4096 keys (one small kernel) rejects most other key sets; the
// exact bucket counts decide before anything is moved; the first scatter checks
// that decision on the device, so the host launches it without waiting, reads
// the decision while it runs and goes on, or runs the LSD sort instead.  Where
// the sample refuses, the LSD sort's digit counts come next on the device and
// the host is told which digits differ by a word in pinned memory (it used to
// start over: clear, count, copy the histograms back, wait).  Refused spans,
// LSD alone as it was before there was a partition / starting over / now: 16
// distinct u32 keys and 4-byte values 2^20 70 / 83 / 64 us, 2^25 288 / 309 / 296;
// 2^12 distinct 2^25 331 / 350 / 337; FP32 ~ N(0, 1) 2^20 137 / 134 / 109, 2^25 617 /
// 638 / 624; FP64 ~ N(0, 1) and 4-byte values 2^20 199 / 214 / 196, 2^24 892 / 914 /
// 899 us: one level no longer loses by being asked, two levels lose 5 to 8 us,
// the sample.
//
// Per sort of uniform keys, LSD before / now: u32 keys and 4-byte values 2^18 109 /
// 47 us, 2^20 127 / 63, 2^25 607 / 550, 2^28 4.07 / 3.50 ms (counts 0.20, scatters 1.00
// and 1.05, local sorts 1.27 ms); u64 keys and 4-byte values 2^20 203 / 71 us, 2^26
// 3.08 / 1.46 ms.  The scatters run at the onesweep pass's rate; the local sorts
// are bound by vector instructions (138 per 64 pairs).
#include "partition_sort.hpp"

#include "digit_hist.hpp"
#include "key_map.hpp"
#include "local_sort.hpp"
#include "onesweep.hpp"

namespace
{

constexpr int kFine = 65536;     // buckets of the map
constexpr int kSample = 4096;    // sampled keys (16384 cost 23 to 41 us in one block's cache misses)
constexpr int kSampleBins = 256;

// What one block sorts at the end: one bucket where they are large enough for
// it, else the buckets that start in one window of `window` pairs.  The block is
// the small one where the largest bucket leaves every group within its room,
// else the large one (small blocks are faster, their barriers wait for fewer
// waves: 2^26 pairs in ranges of 2048 on 256 threads 0.24 ms, of 4096 on 640
// 0.40 ms).
constexpr int64_t buckets_of(int levels) { return levels == 1 ? kRadix : kFine; }
constexpr int64_t window_of(int64_t n, int levels)
{
  const int64_t mean = n / buckets_of(levels);
  return (levels == 1 || mean > 1100) ? 0 : (mean <= 320 ? 1792 : 1280);
}
constexpr int64_t groups_of(int64_t n, int levels)
{
  const int64_t w = window_of(n, levels);
  return w ? (n + w - 1) / w : buckets_of(levels);
}

// Pairs per tile of the scatters (as SortShape of the LSD sort; one-level
// spans take small tiles, for enough blocks).
constexpr int scatter_items(int key_bytes, int val_bytes, int levels)
{
  return levels == 1 ? 8 : ((key_bytes > 4 || val_bytes > 4) ? 16 : 32);
}

// What the kernels of one sort share.
template<typename K>
struct Plan
{
  bits_of<K> lo, hi;   // ordered bits the map spans; keys outside go to its ends
  uint32_t sample_ok;  // the sample allows the partition
  uint32_t overflow;   // a 16-bit counter wrapped
  uint32_t ok;         // the partition runs: 1 + the index of its groups' block (rsort::kGroupCaps)
  uint32_t ntiles2;    // tiles of the second scatter
};

// The map: a key's bucket, 0 .. 65535.
template<typename K>
struct FineMap
{
  bits_of<K> lo, hi, flip;
  BinMap<K, true> bins;
  __device__ FineMap(const Plan<K>* p, bits_of<K> f) : lo(p->lo), hi(p->hi), flip(f), bins(lo, hi, kFine, f) {}
  __device__ __forceinline__ uint32_t operator()(K k) const
  {
    const bits_of<K> b = ordered<K>(k, flip);
    const uint32_t f = bins(k, b);
    return b <= lo ? 0u : (b >= hi ? kFine - 1u : f);
  }
};

// Digit of a scatter (onesweep_kernel's DIG): the map's high or low byte.
template<typename K, int LEVEL>
struct MapDigit
{
  static constexpr int64_t kHistRow = kRadix;
  const Plan<K>* plan;
  bits_of<K> flip;
  struct Fn
  {
    FineMap<K> fine;
    __device__ __forceinline__ uint32_t operator()(K k) const
    {
      const uint32_t f = fine(k);
      return LEVEL == 1 ? f >> 8 : f & 0xFFu;
    }
  };
  __device__ bool runs(int64_t tile) const
  {
    return plan->ok != 0u && (LEVEL == 1 || tile < (int64_t)plan->ntiles2);
  }
  __device__ Fn map() const { return Fn{FineMap<K>(plan, flip)}; }
};

// ---- the sample -----------------------------------------------------------------------
// One block: range of the sampled keys, a little extended so that keys just
// outside do not pile up in the end buckets, and whether the fullest of 256
// equal parts of the range holds at most `most` samples and the range is at
// least `least` wide.  Few integer values: whether the values that share a bucket
// (of per_bucket of the map's fine ones) fit into `bucket_most` keys if all
// occur as often.  Clears count1 and the LSD sort's digit counters.
template<typename K>
__global__ __launch_bounds__(1024) void sample_kernel(const K* __restrict__ keys, int64_t n,
                                                      bits_of<K> flip, uint32_t most,
                                                      bits_of<K> least, Plan<K>* __restrict__ plan,
                                                      uint32_t* __restrict__ count1,
                                                      uint32_t* __restrict__ lsd_hist, uint32_t per_bucket,
                                                      uint32_t bucket_most,
                                                      uint32_t* host_word)
{
  using bits_t = bits_of<K>;
  constexpr int NW = 16, PER = kSample / 1024;
  __shared__ bits_t s_lo[NW], s_hi[NW];
  __shared__ uint32_t s_bin[kSampleBins];
  const int tid = threadIdx.x;
  const int wave = wave_id();
  const int64_t step = n / kSample;  // >= 1
  K k[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j)
  {
    const uint32_t i = (uint32_t)(j * 1024 + tid);
    // a scrambled place inside the i-th stretch: no stride that a periodic
    // input could share
    k[j] = keys[(int64_t)i * step + (int64_t)((uint64_t)(i * 2654435761u) * (uint64_t)step >> 32)];
  }
  if (tid < kSampleBins) s_bin[tid] = 0u;
  if (tid < kRadix) count1[tid] = 0u;
  for (int i = tid; i < (int)sizeof(K) * kRadix; i += 1024) lsd_hist[i] = 0u;
  bits_t lo = ~(bits_t)0, hi = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j)
  {
    const bits_t b = ordered<K>(k[j], flip);
    lo = b < lo ? b : lo;
    hi = b > hi ? b : hi;
  }
  lo = wave_reduce(lo, rk::OpMin<bits_t>{});
  hi = wave_reduce(hi, rk::OpMax<bits_t>{});
  if (lane_id() == 0)
  {
    s_lo[wave] = lo;
    s_hi[wave] = hi;
  }
  __syncthreads();
  for (int w = 0; w < NW; ++w)
  {
    lo = s_lo[w] < lo ? s_lo[w] : lo;
    hi = s_hi[w] > hi ? s_hi[w] : hi;
  }
  const bits_t spread = hi - lo;
  // 8 sample gaps of a uniform key set on both sides
  bool ok = hi - lo >= least;
  if constexpr (std::is_floating_point_v<K>)
  {
    using M = BinMap<K, true>;
    const bool rev = flip != 0;
    const K a = M::value(rev ? ~hi : lo), b = M::value(rev ? ~lo : hi);
    const K ext = (b - a) * (K)(8.0 / kSample);
    const K a2 = a - ext, b2 = b + ext;
    ok = ok && a2 <= a && b2 >= b;  // false for NaN
    if (ok)
    {
      const bits_t ba = KeyTraits<K>::to_bits(a2), bb = KeyTraits<K>::to_bits(b2);
      lo = rev ? ~bb : ba;
      hi = rev ? ~ba : bb;
    }
  }
  else
  {
    const bits_t ext = (hi - lo) / (kSample / 8) + 1;
    lo = lo > ext ? lo - ext : 0;
    hi = hi < ~(bits_t)0 - ext ? hi + ext : ~(bits_t)0;
  }
  Plan<K> p;
  p.lo = lo;
  p.hi = hi;
  const FineMap<K> fine(&p, flip);
  ok = ok && fine.bins.ok && lo < hi;
  if constexpr (!std::is_floating_point_v<K>)
  {
    if (ok && fine.bins.scale == 0u)  // fewer values than fine buckets
    {
      const uint64_t share = (per_bucket - 1u) / fine.bins.mul + 1u;
      ok = (uint64_t)n * share <= (uint64_t)bucket_most * ((uint64_t)spread + 1u);
    }
  }
  if (ok)
  {
#pragma unroll
    for (int j = 0; j < PER; ++j) atomicAdd(&s_bin[fine(k[j]) / (kFine / kSampleBins)], 1u);
  }
  __syncthreads();
  const bool too_many = __syncthreads_or(tid < kSampleBins && s_bin[tid] > most) != 0;
  // A thin end means a tail that goes on past the sample's extremes: the end
  // bucket takes about one key in kSample.
  const bool tail = s_bin[0] < 2u || s_bin[kSampleBins - 1] < 2u;
  ok = ok && !too_many && !(tail && n / kSample > (int64_t)bucket_most);
  if (tid == 0)
  {
    plan->lo = lo;
    plan->hi = hi;
    plan->sample_ok = ok ? 1u : 0u;
    plan->overflow = 0u;
    plan->ok = 0u;
    plan->ntiles2 = 0u;
    __hip_atomic_store(host_word, ok ? 2u : 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// ---- one level: counts of the high byte --------------------------------------------------
constexpr int kHist1Keys = 256 * 16;  // keys per block and step

// Where the sample has refused the span: the LSD sort's digit counts instead, and
// its descriptors.
template<typename K>
__global__ __launch_bounds__(256) void hist1_kernel(const K* __restrict__ keys, int64_t n,
                                                    bits_of<K> flip, const Plan<K>* __restrict__ plan,
                                                    uint32_t* __restrict__ count1,
                                                    uint32_t* __restrict__ desc0, int64_t desc0_words,
                                                    uint32_t* __restrict__ lsd_hist, int64_t lsd_desc_words)
{
  constexpr int kCopies = kHistCopies;
  constexpr int VEC = 16 / sizeof(K);
  constexpr int U = 16 / VEC;
  typedef K uvec_t __attribute__((ext_vector_type(16 / sizeof(K)), aligned(sizeof(K))));
  __shared__ uint32_t s_hist[kHistWords<K>];
  const int tid = threadIdx.x;
  if (!plan->sample_ok)
  {
    count_digits<K>(keys, n, s_hist);
    add_digits<K>(s_hist, lsd_hist, flip != 0);
    for (int64_t i = (int64_t)blockIdx.x * 256 + tid; i < lsd_desc_words; i += (int64_t)gridDim.x * 256) desc0[i] = 0u;
    return;
  }
  for (int i = tid; i < kRadix * kCopies; i += 256) s_hist[i] = 0u;
  const FineMap<K> fine(plan, flip);
  __syncthreads();
  uint32_t* const h = s_hist + (lane_id() % kCopies);
  for (int64_t base = (int64_t)blockIdx.x * kHist1Keys; base < n; base += (int64_t)gridDim.x * kHist1Keys)
  {
    K k[16];
    if (base + kHist1Keys <= n)
    {
#pragma unroll
      for (int u = 0; u < U; ++u)
      {
        const uvec_t x = *reinterpret_cast<const uvec_t*>(keys + base + (u * 256 + tid) * VEC);
#pragma unroll
        for (int e = 0; e < VEC; ++e) k[u * VEC + e] = x[e];
      }
#pragma unroll
      for (int q = 0; q < 16; ++q) atomicAdd(&h[(fine(k[q]) >> 8) * kCopies], 1u);
    }
    else
    {
      for (int64_t i = base + tid; i < n; i += 256) atomicAdd(&h[(fine(keys[i]) >> 8) * kCopies], 1u);
    }
  }
  __syncthreads();
  uint32_t c = 0;
#pragma unroll
  for (int r = 0; r < kCopies; ++r) c += s_hist[tid * kCopies + r];
  if (c) atomic_add_agent(&count1[tid], c);
  for (int64_t i = (int64_t)blockIdx.x * 256 + tid; i < desc0_words; i += (int64_t)gridDim.x * 256) desc0[i] = 0u;
}

// start[g] of every group g that begins inside (off, off + c]: the first
// bucket boundary at or after g * window.  window 0: a group per bucket, this
// one's number being `bucket`.
__device__ __forceinline__ void mark_groups(uint32_t off, uint32_t c, uint32_t window, uint32_t bucket,
                                            uint32_t* __restrict__ start)
{
  if (window == 0)
  {
    start[bucket] = off;
    return;
  }
  for (uint32_t g = off / window + 1; (uint64_t)g * window <= (uint64_t)off + c; ++g) start[g] = off + c;
}

// Block-wide exclusive scan of one value per thread (256 threads).
__device__ __forceinline__ uint32_t scan256(uint32_t v, uint32_t* s_w)
{
  uint32_t ex, total;
  (void)wave_scan(v, rk::OpPlus<uint32_t>{}, 0u, ex, total);
  if (lane_id() == 0) s_w[wave_id()] = total;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) ex += (w < wave_id()) ? s_w[w] : 0u;
  __syncthreads();
  return ex;
}

template<typename K>
__global__ __launch_bounds__(256) void plan1_kernel(Plan<K>* __restrict__ plan,
                                                    const uint32_t* __restrict__ count1, uint32_t n,
                                                    uint32_t most0, uint32_t most1, uint32_t window, uint32_t ngroups,
                                                    uint32_t* __restrict__ start,
                                                    const uint32_t* __restrict__ lsd_hist, uint32_t* host)
{
  __shared__ uint32_t s_w[4];
  const int t = threadIdx.x;
  if (!plan->sample_ok)
  {
    const uint32_t digits = active_digits<K>(lsd_hist, n);
    if (t == 0)
    {
      host[0] = 0u;
      host[2] = digits;
    }
    return;
  }
  const uint32_t c = count1[t];
  const bool small = __syncthreads_or(c > most0) == 0;
  const bool ok = __syncthreads_or(c > most1) == 0;
  if (t == 0)
  {
    const uint32_t v = ok ? (small ? 1u : 2u) : 0u;
    plan->ok = v;
    host[0] = v;
  }
  if (!ok) return;
  const uint32_t off = scan256(c, s_w);
  if (t == 0) start[0] = 0u;
  mark_groups(off, c, window, t, start);
  if (t == 0) start[ngroups] = n;
}

// ---- two levels: counts of all 65536 buckets -----------------------------------------------
// One 1024-thread block per CU counts its share of the keys in 16-bit LDS
// counters, two per word (128 KiB), one LDS atomic per key against four in
// the LSD sort's histograms.  A counter that wraps makes the block's total
// fall short of its keys (every wrap loses 65535 or 65536), which is checked.
template<typename K>
__global__ __launch_bounds__(1024) void hist2_kernel(const K* __restrict__ keys, int64_t n,
                                                     bits_of<K> flip, Plan<K>* __restrict__ plan,
                                                     uint32_t* __restrict__ partial,
                                                     uint32_t* __restrict__ desc0, int64_t desc0_words)
{
  constexpr int VEC = 16 / sizeof(K);
  constexpr int U = 4;
  constexpr int STEP = 1024 * U * VEC;
  typedef K uvec_t __attribute__((ext_vector_type(16 / sizeof(K)), aligned(sizeof(K))));
  if (!plan->sample_ok) return;
  __shared__ uint32_t s_cnt[kFine / 2];
  __shared__ uint32_t s_sum[16];
  const int tid = threadIdx.x;
  for (int i = tid; i < kFine / 2; i += 1024) s_cnt[i] = 0u;
  const FineMap<K> fine(plan, flip);
  __syncthreads();
  uint32_t mine = 0;
  auto count = [&](K k) {
    const uint32_t f = fine(k);
    atomicAdd(&s_cnt[f >> 1], 1u << (16 * (f & 1u)));
  };
  for (int64_t base = (int64_t)blockIdx.x * STEP; base < n; base += (int64_t)gridDim.x * STEP)
  {
    if (base + STEP <= n)
    {
      uvec_t x[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
      {
        x[u] = __builtin_nontemporal_load(reinterpret_cast<const uvec_t*>(keys + base + (u * 1024 + tid) * VEC));
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
      {
#pragma unroll
        for (int e = 0; e < VEC; ++e) count(x[u][e]);
      }
      mine += U * VEC;
    }
    else
    {
      for (int64_t i = base + tid; i < n; i += 1024)
      {
        count(keys[i]);
        ++mine;
      }
    }
  }
  __syncthreads();
  uint32_t* const out = partial + (int64_t)blockIdx.x * (kFine / 2);
  for (int i = tid; i < kFine / 2; i += 1024)
  {
    const uint32_t w = s_cnt[i];
    mine -= (w & 0xFFFFu) + (w >> 16);
    out[i] = w;
  }
  mine = wave_reduce(mine, rk::OpPlus<uint32_t>{});
  if (lane_id() == 0) s_sum[wave_id()] = mine;
  __syncthreads();
  if (tid == 0)
  {
    uint32_t sum = 0;
    for (int w = 0; w < 16; ++w) sum += s_sum[w];
    if (sum != 0u) plan->overflow = 1u;  // every block that writes it writes 1
  }
  for (int64_t i = (int64_t)blockIdx.x * 1024 + tid; i < desc0_words; i += (int64_t)gridDim.x * 1024) desc0[i] = 0u;
}

// Block d adds up the partial counts of buckets 256 d .. 256 d + 255: their
// row, its total and its largest.
template<typename K>
__global__ __launch_bounds__(1024) void rows_kernel(const Plan<K>* __restrict__ plan,
                                                    const uint32_t* __restrict__ partial, int nblocks,
                                                    uint32_t* __restrict__ rows,
                                                    uint32_t* __restrict__ total,
                                                    uint32_t* __restrict__ largest)
{
  if (!plan->sample_ok) return;
  __shared__ uint32_t s_lo[8][128], s_hi[8][128];
  __shared__ uint32_t s_t[2], s_m[2];
  const int w = threadIdx.x & 127, g = threadIdx.x >> 7;
  const uint32_t* const p = partial + (int64_t)blockIdx.x * 128 + w;
  uint32_t a = 0, b = 0;
#pragma unroll 8
  for (int i = g; i < nblocks; i += 8)
  {
    const uint32_t v = p[(int64_t)i * (kFine / 2)];
    a += v & 0xFFFFu;
    b += v >> 16;
  }
  s_lo[g][w] = a;
  s_hi[g][w] = b;
  __syncthreads();
  if (g == 0)
  {
    for (int i = 1; i < 8; ++i)
    {
      a += s_lo[i][w];
      b += s_hi[i][w];
    }
    rows[(int64_t)blockIdx.x * kRadix + 2 * w] = a;
    rows[(int64_t)blockIdx.x * kRadix + 2 * w + 1] = b;
    const uint32_t t = wave_reduce(a + b, rk::OpPlus<uint32_t>{});
    const uint32_t m = wave_reduce(a > b ? a : b, rk::OpMax<uint32_t>{});
    if (lane_id() == 0)
    {
      s_t[wave_id()] = t;
      s_m[wave_id()] = m;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0)
  {
    total[blockIdx.x] = s_t[0] + s_t[1];
    largest[blockIdx.x] = s_m[0] > s_m[1] ? s_m[0] : s_m[1];
  }
}

// The decision, and the first element and tile of every high-byte range.
template<typename K>
__global__ __launch_bounds__(256) void plan2_kernel(Plan<K>* __restrict__ plan,
                                                    const uint32_t* __restrict__ total,
                                                    const uint32_t* __restrict__ largest, uint32_t most0,
                                                    uint32_t most1, uint32_t tile, uint32_t* __restrict__ base,
                                                    uint32_t* __restrict__ tile0, uint32_t* host_ok)
{
  __shared__ uint32_t s_w[4];
  const int t = threadIdx.x;
  bool ok = plan->sample_ok != 0u && plan->overflow == 0u;
  bool small = false;
  if (ok)  // the same branch in every thread
  {
    small = __syncthreads_or(largest[t] > most0) == 0;
    ok = __syncthreads_or(largest[t] > most1) == 0;
  }
  if (t == 0)
  {
    const uint32_t v = ok ? (small ? 1u : 2u) : 0u;
    plan->ok = v;
    *host_ok = v;
  }
  if (!ok) return;
  const uint32_t c = total[t];
  base[t] = scan256(c, s_w);
  const uint32_t tiles = (c + tile - 1) / tile;
  const uint32_t first = scan256(tiles, s_w);
  tile0[t] = first;
  if (t == kRadix - 1) plan->ntiles2 = first + tiles;
}

// Block d: the second scatter's tile records and cleared descriptor rows of
// range d, and the starts of the groups its buckets open.
template<typename K>
__global__ __launch_bounds__(256) void records_kernel(const Plan<K>* __restrict__ plan,
                                                      const uint32_t* __restrict__ rows,
                                                      const uint32_t* __restrict__ total,
                                                      const uint32_t* __restrict__ base,
                                                      const uint32_t* __restrict__ tile0, uint32_t tile,
                                                      uint32_t n, uint32_t window, uint32_t ngroups,
                                                      rs::SortTile* __restrict__ recs,
                                                      uint32_t* __restrict__ start,
                                                      uint32_t* __restrict__ desc1)
{
  if (!plan->ok) return;
  __shared__ uint32_t s_w[4];
  const uint32_t d = blockIdx.x, t = threadIdx.x;
  const uint32_t len = total[d], first = base[d], t0 = tile0[d];
  const uint32_t tiles = (len + tile - 1) / tile;
  for (uint32_t j = t; j < tiles; j += 256)
  {
    recs[t0 + j] = rs::SortTile{first, first, first, first, first, first, (int64_t)len, j, d};
  }
  for (uint64_t i = t; i < (uint64_t)tiles * kRowStride; i += 256) desc1[(uint64_t)t0 * kRowStride + i] = 0u;
  const uint32_t c = rows[d * kRadix + t];
  const uint32_t off = first + scan256(c, s_w);
  mark_groups(off, c, window, d * kRadix + t, start);
  if (d == 0 && t == 0) start[0] = 0u;
  if (d == 0 && t == 0) start[ngroups] = n;
}

// Parts of the aux memory.
struct Aux
{
  size_t plan = 0, count1, total, largest, base, tile0, rows, start, redo, recs, bytes;
  int64_t ntiles, ngroups, tile;
  int levels;
  Aux(int kb, int vb, int64_t n)
  {
    levels = rsort::partition_levels(kb, vb, n);
    tile = 512 * (int64_t)scatter_items(kb, vb, levels);
    ntiles = rc::ceil_div(n, tile);
    ngroups = groups_of(n, levels);
    size_t o = 256;
    auto place = [&o](size_t b) {
      const size_t at = o;
      o = rc::align_up(o + b, 256);
      return at;
    };
    count1 = place(kRadix * 4);
    total = place(kRadix * 4);
    largest = place(kRadix * 4);
    base = place(kRadix * 4);
    tile0 = place(kRadix * 4);
    rows = levels == 2 ? place((size_t)kFine * 4) : 0;
    start = place((size_t)(ngroups + 1) * 4);
    redo = place((size_t)ngroups);
    recs = levels == 2 ? place((size_t)(ntiles + kRadix) * sizeof(rs::SortTile)) : 0;
    bytes = o;
  }
};

// Largest bucket the partition takes.  With 4-byte keys, of which the LSD sort
// makes 4 passes, two levels gain nothing on uneven keys that need the large
// block (FP32 ~ N(0, 1), 2^24 pairs: 408 us against 325).
int64_t most_of(int kb, int64_t n, int levels)
{
  const bool small = levels == 2 && kb == 4 && n / buckets_of(levels) <= 2200;
  return rsort::kGroupCaps[small ? 0 : 1] - window_of(n, levels);
}

// Samples in one of the 256 parts above which a bucket would outgrow the
// large block: the expected count of a part of buckets at the limit, but not
// below what an even key set reaches by chance (16 and 4.5 standard deviations).
uint32_t sample_limit(int kb, int64_t n, int levels)
{
  const double most = (double)most_of(kb, n, levels);
  const double c = kSample * (buckets_of(levels) / (double)kSampleBins) * most / (double)n;
  return c < 34.0 ? 34u : (c < (double)kSample ? (uint32_t)c : (uint32_t)kSample);
}

template<typename K, typename V, bool HAS_VALS, int ITEMS, int LEVEL>
void launch_scatter(const K* ik, K* ok, const V* iv, V* ov, int64_t n, const Plan<K>* plan,
                    bits_of<K> flip, const uint32_t* hist, uint32_t* d0, uint32_t* d1,
                    const rs::SortTile* recs, int64_t grid, hipStream_t s)
{
  if constexpr (LEVEL == 1)
  {
    hipLaunchKernelGGL((onesweep_kernel<K, V, MapDigit<K, 1>, HAS_VALS, 512, ITEMS>), dim3((unsigned)grid),
                       dim3(512), 0, s, ik, ok, iv, ov, n, (MapDigit<K, 1>{plan, flip}), hist, d0, d1);
  }
  else
  {
    // "pass 1" of the record form: from the alternates into the outputs
    hipLaunchKernelGGL((onesweep_kernel<K, V, MapDigit<K, 2>, HAS_VALS, 512, ITEMS, true>),
                       dim3((unsigned)grid), dim3(512), 0, s, (const K*)nullptr, ok, (const V*)nullptr, ov,
                       (int64_t)0, (MapDigit<K, 2>{plan, flip}), hist, d0, d1, recs, 1, (K*)ik, (V*)iv);
  }
}

template<typename K, typename V, bool HAS_VALS>
int partition_typed(int dtype, int descending, K* keys, V* vals, int64_t n, const rsort::PartitionMem& mem,
                    hipStream_t s, bool* done, uint32_t* digits)
{
  K* const alt_k = (K*)mem.alt_keys;
  V* const alt_v = (V*)mem.alt_vals;
  char* const aux = mem.aux;
  constexpr int kb = (int)sizeof(K), vb = HAS_VALS ? (int)sizeof(V) : 0;
  const bits_of<K> flip = descending ? ~(bits_of<K>)0 : (bits_of<K>)0;
  const Aux a(kb, vb, n);
  const uint32_t window = (uint32_t)window_of(n, a.levels);
  const uint32_t most0 = (uint32_t)rsort::kGroupCaps[0] - window, most1 = (uint32_t)most_of(kb, n, a.levels);
  // Two levels move the pairs three times: integer keys of a range of 3 bytes
  // or less take no more LSD passes than that.
  const bits_of<K> least = (a.levels == 2 && !std::is_floating_point_v<K>) ? (bits_of<K>)1 << 24 : 0;
  Plan<K>* const plan = (Plan<K>*)(aux + a.plan);
  uint32_t* const count1 = (uint32_t*)(aux + a.count1);
  uint32_t* const start = (uint32_t*)(aux + a.start);
  uint32_t* const d0 = mem.desc;
  uint32_t* const d1 = mem.desc + (a.ntiles + kRadix) * kRowStride;
  volatile uint32_t* const host = mem.host;
  host[0] = host[1] = host[2] = 0u;
  {
    rc::TimedScope ts("partition_sample", s);
    hipLaunchKernelGGL((sample_kernel<K>), dim3(1), dim3(1024), 0, s, keys, n, flip,
                       sample_limit(kb, n, a.levels), least, plan, count1, mem.hist,
                       (uint32_t)(kFine / buckets_of(a.levels)), most1, mem.host + 1);
    RC_HIP(hipGetLastError());
  }
  // A span that the sample refuses has its digits counted by the kernel that
  // follows, so it pays for the sample and little else.  One level: the counts'
  // kernel does it, and the host goes on without the answer (a wait here
  // would cost an accepted span as much as the kernels that end at once
  // cost a refused one: 2^20 pairs 63 against 75 us).  Two levels: a kernel of its own,
  // which ends at once where the span is accepted, while the host polls the answer.
  if (a.levels == 2)
  {
    {
      rc::TimedScope ts("radix_hist", s);
      hipLaunchKernelGGL((hist_kernel<K>), dim3(hist_blocks(n)), dim3(256), 0, s, keys, n, descending != 0, mem.hist,
                         mem.desc, mem.lsd_desc_words, &plan->sample_ok);
      RC_HIP(hipGetLastError());
    }
    uint32_t answer = 0;
    RC_TRY(rc::wait_word(host + 1, s, &answer));
    if (answer == 1u)
    {
      rc::TimedScope ts("radix_hist", s);
      hipLaunchKernelGGL((digits_kernel<K>), dim3(1), dim3(256), 0, s, mem.hist, (uint32_t)n, mem.host + 2);
      RC_HIP(hipGetLastError());
      return rc::wait_word(host + 2, s, digits);
    }
  }
  {
    rc::TimedScope ts("partition_hist", s);
    if (a.levels == 1)
    {
      const int64_t want = rc::ceil_div(n, (int64_t)kHist1Keys);
      hipLaunchKernelGGL((hist1_kernel<K>), dim3((unsigned)(want < 512 ? want : 512)), dim3(256), 0, s, keys, n,
                         flip, plan, count1, d0, a.ntiles * kRowStride, mem.hist, mem.lsd_desc_words);
      hipLaunchKernelGGL((plan1_kernel<K>), dim3(1), dim3(256), 0, s, plan, count1, (uint32_t)n, most0, most1, window,
                         (uint32_t)a.ngroups, start, mem.hist, mem.host);
    }
    else
    {
      // the partial counts lie in the alternate keys (2 bytes a key or less)
      const int64_t want = n >> 16;
      const int blocks = (int)(want < 256 ? want : 256);
      uint32_t* const total = (uint32_t*)(aux + a.total);
      uint32_t* const largest = (uint32_t*)(aux + a.largest);
      uint32_t* const base = (uint32_t*)(aux + a.base);
      uint32_t* const tile0 = (uint32_t*)(aux + a.tile0);
      uint32_t* const rows = (uint32_t*)(aux + a.rows);
      hipLaunchKernelGGL((hist2_kernel<K>), dim3((unsigned)blocks), dim3(1024), 0, s, keys, n, flip, plan,
                         (uint32_t*)alt_k, d0, a.ntiles * kRowStride);
      hipLaunchKernelGGL((rows_kernel<K>), dim3(kRadix), dim3(1024), 0, s, plan, (const uint32_t*)alt_k, blocks,
                         rows, total, largest);
      hipLaunchKernelGGL((plan2_kernel<K>), dim3(1), dim3(256), 0, s, plan, total, largest, most0, most1,
                         (uint32_t)a.tile, base, tile0, mem.host);
    }
    RC_HIP(hipGetLastError());
  }
  RC_HIP(hipEventRecord(mem.ready, s));
  // The first scatter is launched before the decision is known here (it checks
  // it on the device), so the wait below passes while it runs.  The gate (one
  // lookback launch at a time on the device) is held for each scatter's
  // launch alone, never across the wait: other threads' scans and sorts
  // must be able to go on, and this stream may be waiting for one of them.
  rs::SortTile* const recs = (rs::SortTile*)(aux + a.recs);
  {
    rc::LookbackGate gate(s);
    RC_TRY(gate.status());
    if (a.levels == 1)
    {
      rc::TimedScope ts("partition_scatter", s);
      launch_scatter<K, V, HAS_VALS, scatter_items(kb, vb, 1), 1>(keys, alt_k, vals, alt_v, n, plan, flip, count1, d0,
                                                                  d1, nullptr, a.ntiles, s);
    }
    else
    {
      hipLaunchKernelGGL((records_kernel<K>), dim3(kRadix), dim3(256), 0, s, plan, (uint32_t*)(aux + a.rows),
                         (uint32_t*)(aux + a.total), (uint32_t*)(aux + a.base), (uint32_t*)(aux + a.tile0),
                         (uint32_t)a.tile, (uint32_t)n, window, (uint32_t)a.ngroups, recs, start, d1);
      rc::TimedScope ts("partition_scatter", s);
      launch_scatter<K, V, HAS_VALS, scatter_items(kb, vb, 2), 1>(keys, alt_k, vals, alt_v, n, plan, flip,
                                                                  (uint32_t*)(aux + a.total), d0, d1, nullptr,
                                                                  a.ntiles, s);
    }
    RC_HIP(hipGetLastError());
  }
  RC_HIP(hipEventSynchronize(mem.ready));
  const uint32_t ok = host[0];
  if (ok == 0u)
  {
    *digits = host[2];
    return RAJA_CDNA4_SUCCESS;
  }
  if (a.levels == 2)
  {
    rc::LookbackGate gate(s);
    RC_TRY(gate.status());
    rc::TimedScope ts("partition_scatter", s);
    launch_scatter<K, V, HAS_VALS, scatter_items(kb, vb, 2), 2>(alt_k, keys, alt_v, vals, n, plan, flip,
                                                                (uint32_t*)(aux + a.rows), d1, d0, recs,
                                                                a.ntiles + kRadix, s);
    RC_HIP(hipGetLastError());
  }
  const bool from_alt = a.levels == 1;
  rc::TimedScope ts("partition_local", s);
  RC_TRY(rsort::local_sort_groups(dtype, vb, descending, from_alt ? alt_k : keys,
                                  from_alt ? (const void*)alt_v : (const void*)vals, keys, vals, start, a.ngroups,
                                  rsort::kGroupCaps[ok - 1], (uint8_t*)(aux + a.redo), s));
  *done = true;
  return RAJA_CDNA4_SUCCESS;
}

template<typename K>
int partition_key(int dtype, int val_bytes, int descending, void* keys, void* vals, int64_t n,
                  const rsort::PartitionMem& mem, hipStream_t s, bool* done, uint32_t* digits)
{
  switch (val_bytes)
  {
    case 0:
      return partition_typed<K, uint32_t, false>(dtype, descending, (K*)keys, nullptr, n, mem, s, done, digits);
    case 4:
      return partition_typed<K, uint32_t, true>(dtype, descending, (K*)keys, (uint32_t*)vals, n, mem, s, done, digits);
    default:
      return partition_typed<K, uint64_t, true>(dtype, descending, (K*)keys, (uint64_t*)vals, n, mem, s, done, digits);
  }
}

}  // namespace

namespace rsort
{

int partition_levels(int kb, int vb, int64_t n)
{
  if (n < ((int64_t)1 << 18)) return 0;
  // while an even split stays below the largest bucket: five standard
  // deviations of a bucket of 4700 are 343
  if (n <= kRadix * (int64_t)4700) return 1;
  if (n > kFine * (int64_t)4700) return 0;
  // Per sort, LSD against partition, uniform keys: u64 keys + 4-byte values 2^22
  // 279 / 162 us, 2^24 877 / 411 us; u32 keys + 4-byte values 2^23 186 / 192 us,
  // 2^24 319 / 295, 2^25 608 / 559, 2^26 1111 / 1002, 2^28 4.07 / 3.50 ms, + 8-byte
  // values 2^23 243 / 213, 2^24 467 / 381 us; u32 keys alone 2^24 262 / 261 us, 2^27
  // 1.44 / 1.63 ms.  Refused spans pay 5 to 8 us: 3 to 4 % of a sort of few distinct
  // 4-byte keys below 2^25 (2^24 150 / 154 us), 1 to 2.5 % there and less above.
  // 4-byte keys start at 2^25: the gain at 2^24 (8 to 18 % of even keys) is left
  // for the key sets that would pay for it.
  if (kb == 8) return n >= ((int64_t)1 << 22) ? 2 : 0;
  return (vb > 0 && n >= ((int64_t)1 << 25)) ? 2 : 0;
}

size_t partition_aux_bytes(int kb, int vb, int64_t n) { return Aux(kb, vb, n).bytes; }

int64_t partition_desc_rows(int kb, int vb, int64_t n) { return Aux(kb, vb, n).ntiles + kRadix; }

int partition_sort(int key_dtype, int val_bytes, int descending, void* keys, void* vals, int64_t n,
                   const PartitionMem& mem, hipStream_t s, bool* done, uint32_t* digits)
{
  *done = false;
  *digits = 0u;
#define RSORT_PART(CODE, K)                                                                               \
  case CODE:                                                                                              \
    return partition_key<K>(key_dtype, val_bytes, descending, keys, vals, n, mem, s, done, digits);
  switch (key_dtype)
  {
    RSORT_PART(RAJA_CDNA4_U32, uint32_t)
    RSORT_PART(RAJA_CDNA4_I32, int32_t)
    RSORT_PART(RAJA_CDNA4_F32, float)
    RSORT_PART(RAJA_CDNA4_U64, uint64_t)
    RSORT_PART(RAJA_CDNA4_I64, int64_t)
    RSORT_PART(RAJA_CDNA4_F64, double)
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "key dtype %d", key_dtype);
  }
#undef RSORT_PART
}

int take_partition_timeouts(uint32_t* count)
{
  uint32_t v = 0;
  RC_HIP(hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_spin_timeouts), sizeof(v)));
  if (v)
  {
    const uint32_t zero = 0;
    RC_HIP(hipMemcpyToSymbol(HIP_SYMBOL(g_spin_timeouts), &zero, sizeof(zero)));
  }
  *count = v;
  return RAJA_CDNA4_SUCCESS;
}
}  // namespace rsort
