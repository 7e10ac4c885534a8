// Stable sorts of short ranges inside one workgroup (or one wave): the
// segments of a batch, small spans and small requests.
//
// The work is split by range length, each class with a block as large as its
// longest range: one wave per range of up to 64 keys, 128 x 4 threads x keys
// up to 512, 256 x 8 up to 2048 and 1024 x 8 up to 8192.  A block holds its
// keys and values in registers, reads and writes memory once and coalesced.
//
// Bounded by LDS work, not by memory, so the keys are placed with one LDS
// atomic each instead of one wave ranking per 8-bit digit:
//   1. the range's smallest and largest key give a monotone map of keys to
//      as many bins as keys (integers by a multiply-high of the distance from
//      the smallest, floating keys by their value, so a bell-shaped set
//      spreads as well as a uniform one);
//   2. an LDS atomic per key counts its bin and gives it a slot, a scan of
//      the counters gives each bin its place;
//   3. a key that shares its bin counts the bin's keys that go before it (by
//      key, then by input position: stable whatever the atomics' order);
//   4. keys and values go to their places in LDS and out in whole lines.
// A range whose bins are uneven (more than kMaxBin keys in one: few distinct
// keys, a spike, infinities or NaN) takes LSD passes of 8-bit digits instead,
// the digits that are the same for all its keys left out.
//
// 16,250 uneven ranges (20,000 segments of log-uniform length in [1, 2^16],
// those of up to 8192 pairs, 1.5e7 pairs of uniform keys): 123 us in four
// launches (80 + 26 + 11 + 6 us), against 1787 us with one 512-thread block of
// 16 items per thread and four ballot-ranked LSD passes for every range.  One
// span of 5000 pairs: 11 us in one launch, against 74 us for the clear, the
// histogram and four one-tile passes of the span sort.
#include "local_sort.hpp"

#include <type_traits>

#include "ops.hpp"
#include "radix.hpp"

namespace
{
using namespace RAJA::cdna4::dev;

// Keys one bin may hold before the range takes the LSD passes.  A bin of c
// keys costs each of them c LDS reads: 32 is about what one 8-bit ballot
// ranking costs a key.
constexpr uint32_t kMaxBin = 32;

template<typename K>
using bits_of = typename KeyTraits<K>::bits_t;

// Unsigned bits whose order is the sort's order.
template<typename K>
__device__ __forceinline__ bits_of<K> ordered(K k, bits_of<K> flip)
{
  return KeyTraits<K>::to_bits(k) ^ flip;
}

// Monotone map of ordered bits in [lo, hi] to bins 0 .. nb-1.
template<typename K>
struct BinMap
{
  using bits_t = bits_of<K>;
  static constexpr bool is_float = std::is_floating_point_v<K>;
  bits_t lo;
  uint32_t nb;
  int shift;        // 64-bit integer keys: right shift that leaves 32 bits
  uint32_t scale;   // integer keys: bins per key value, 32 fraction bits; 0: one bin per value
  K kmin, kinv;     // floating keys: smallest value, bins per unit
  bool reverse;     // descending floating keys
  bool ok;

  // Value of ordered (ascending) bits of a floating key.
  static __device__ K value(bits_t b)
  {
    constexpr bits_t top = (bits_t)1 << (8 * sizeof(bits_t) - 1);
    const bits_t u = (b & top) ? (b ^ top) : ~b;
    K k;
    __builtin_memcpy(&k, &u, sizeof(K));
    return k;
  }

  __device__ BinMap(bits_t lo_, bits_t hi_, uint32_t nb_, bits_t flip) : lo(lo_), nb(nb_)
  {
    // 1 - 2^-20 keeps the largest key below nb whatever the roundings (each
    // below 2^-22 relative).
    constexpr float kSlack = 1.0f - 0x1.0p-20f;
    shift = 0;
    scale = 0;
    kmin = K(0);
    kinv = K(0);
    reverse = false;
    ok = true;
    if constexpr (is_float)
    {
      reverse = flip != 0;
      const K a = value(reverse ? ~hi_ : lo_);
      const K b = value(reverse ? ~lo_ : hi_);
      const K d = b - a;
      kmin = a;
      kinv = (K)nb / d * (K)kSlack;
      // false for NaN and infinite keys, a spread that overflows and one so
      // small that its inverse does
      constexpr K big = sizeof(K) == 4 ? (K)0x1.0p126 : (K)0x1.0p1000;
      ok = d > K(0) && d < big && kinv < big && a > -big && b < big;
    }
    else
    {
      bits_t range = hi_ - lo_;
      if constexpr (sizeof(bits_t) == 8)
      {
        const uint32_t top = (uint32_t)(range >> 32);
        shift = top ? 32 - __builtin_clz(top) : 0;
        range >>= shift;
      }
      const uint32_t r = (uint32_t)range;
      if (r >= nb) scale = (uint32_t)((float)nb / ((float)r + 1.0f) * (4294967296.0f * kSlack));
    }
  }

  __device__ uint32_t operator()(K k, bits_t b) const
  {
    if constexpr (is_float)
    {
      const uint32_t bin = (uint32_t)((k - kmin) * kinv);
      return reverse ? nb - 1u - bin : bin;
    }
    else
    {
      const uint32_t x = (uint32_t)((b - lo) >> shift);
      return scale ? __umulhi(x, scale) : x;
    }
  }
};

// ---- one wave per range of up to 64 keys ------------------------------------------
// Lane i holds key i; its place is the number of keys that go before it,
// counted over the range's keys read lane by lane.
template<typename K, typename V, bool HAS_VALS>
__global__ __launch_bounds__(256) void wave_sort_kernel(const K* in_keys, const V* in_vals,
                                                        K* out_keys, V* out_vals,
                                                        const rs::SortSeg* __restrict__ segs,
                                                        int64_t nseg, bits_of<K> flip)
{
  const int64_t g = (int64_t)blockIdx.x * (256 / wave_size) + __builtin_amdgcn_readfirstlane(wave_id());
  if (g >= nseg) return;  // whole wave; the kernel has no barrier
  const rs::SortSeg sg = segs[g];
  const int n = (int)sg.n;
  const int lane = lane_id();
  const bool valid = lane < n;
  const K k = valid ? in_keys[sg.in_keys + lane] : K(0);
  V v = V(0);
  if (HAS_VALS && valid) v = in_vals[sg.in_vals + lane];
  const bits_of<K> b = ordered<K>(k, flip);
  int r = 0;
  for (int j = 0; j < n; ++j)
  {
    const bits_of<K> bj = read_lane(b, j);
    r += (bj < b || (bj == b && j < lane)) ? 1 : 0;
  }
  if (valid)
  {
    out_keys[sg.out_keys + r] = k;
    if (HAS_VALS) out_vals[sg.out_vals + r] = v;
  }
}

// ---- one block per range ---------------------------------------------------------------
template<typename K, typename V, bool HAS_VALS, int BLOCK, int ITEMS>
struct LocalLds
{
  static constexpr int NW = BLOCK / wave_size;
  static constexpr int CAP = BLOCK * ITEMS;
  static constexpr int SLOT = (HAS_VALS && sizeof(V) > sizeof(K)) ? (int)sizeof(V) : (int)sizeof(K);
  // keys by place (then 8-byte values)
  __attribute__((aligned(16))) unsigned char buf[CAP * SLOT];
  // bin counters, then bin places, two 16-bit ones per word (one more for
  // the end), and each placed key's input position; 4-byte values use both
  // once the places are known; LSD: per-wave digit counters
  union
  {
    struct
    {
      uint32_t cnt[CAP / 2 + 1];
      uint16_t idx[CAP];
    } bin;
    uint32_t vals4[CAP];
    struct
    {
      uint32_t whist[NW * kRadix];
      uint32_t tstart[kRadix];
    } lsd;
  };
  bits_of<K> lo[NW], hi[NW];
  uint32_t scan[NW > 4 ? NW : 4];
};

template<typename K, typename V, bool HAS_VALS, int BLOCK, int ITEMS>
__device__ __forceinline__ void local_sort(const K* in_keys, const V* in_vals, K* out_keys,
                                           V* out_vals, int n, bits_of<K> flip)
{
  using L = LocalLds<K, V, HAS_VALS, BLOCK, ITEMS>;
  using bits_t = bits_of<K>;
  constexpr int NW = L::NW;
  constexpr int P = (int)sizeof(K);
  __shared__ L s;
  K* const s_keys = reinterpret_cast<K*>(s.buf);

  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  // Items per thread of this range: wave w holds elements [w*64*per,
  // (w+1)*64*per), item j of a lane is j*64 + lane in there, so input order
  // is (wave, item, lane) order and every load is one run per wave.
  const int per = __builtin_amdgcn_readfirstlane((n + BLOCK - 1) / BLOCK);
  const int wbase = wave * wave_size * per;

  K k[ITEMS];
  V v[HAS_VALS ? ITEMS : 1];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
  {
    if (j < per)
    {
      const int i = wbase + j * wave_size + lane;
      k[j] = (i < n) ? in_keys[i] : K(0);
      if (HAS_VALS) v[j] = (i < n) ? in_vals[i] : V(0);
    }
  }
  // rows of 64 counter words (128 bins) per wave; as many bins as items
  const int rows = (per + 1) / 2;
  const uint32_t nb = (uint32_t)(rows * 2 * BLOCK);
  for (int q = 0; q < rows; ++q) s.bin.cnt[(wave * rows + q) * wave_size + lane] = 0u;

  bits_t lo = ~(bits_t)0, hi = 0;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
  {
    if (j < per && wbase + j * wave_size + lane < n)
    {
      const bits_t b = ordered<K>(k[j], flip);
      lo = b < lo ? b : lo;
      hi = b > hi ? b : hi;
    }
  }
  lo = wave_reduce(lo, rk::OpMin<bits_t>{});
  hi = wave_reduce(hi, rk::OpMax<bits_t>{});
  if (lane == 0)
  {
    s.lo[wave] = lo;
    s.hi[wave] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w)
  {
    const bits_t a = s.lo[w], b = s.hi[w];
    lo = a < lo ? a : lo;
    hi = b > hi ? b : hi;
  }
  const BinMap<K> bin_of(lo, hi, nb, flip);
  bool fast = bin_of.ok;  // the same in every thread

  uint32_t pos[ITEMS];
  if (fast)
  {
    // bin << 16 | slot inside the bin
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      if (j < per && wbase + j * wave_size + lane < n)
      {
        const uint32_t bin = bin_of(k[j], ordered<K>(k[j], flip));
        const uint32_t sh = (bin & 1u) * 16u;
        const uint32_t c = atomicAdd(&s.bin.cnt[bin >> 1], 1u << sh);
        pos[j] = (bin << 16) | ((c >> sh) & 0xFFFFu);
      }
    }
    __syncthreads();
    // Places of the bins: each wave scans its rows, then the wave totals.
    uint32_t w[(ITEMS + 1) / 2], ex[(ITEMS + 1) / 2];
    uint32_t run = 0, worst = 0;
#pragma unroll
    for (int q = 0; q < (ITEMS + 1) / 2; ++q)
    {
      if (q < rows)
      {
        w[q] = s.bin.cnt[(wave * rows + q) * wave_size + lane];
        const uint32_t c0 = w[q] & 0xFFFFu, c1 = w[q] >> 16;
        worst = c0 > worst ? c0 : worst;
        worst = c1 > worst ? c1 : worst;
        uint32_t total;
        (void)wave_scan(c0 + c1, rk::OpPlus<uint32_t>{}, 0u, ex[q], total);
        ex[q] += run;
        run += total;
      }
    }
    if (lane == 0) s.scan[wave] = run;
    fast = __syncthreads_or(worst > kMaxBin) == 0;
    if (fast)
    {
      uint32_t before = 0;
#pragma unroll
      for (int x = 0; x < NW; ++x) before += (x < wave) ? s.scan[x] : 0u;
#pragma unroll
      for (int q = 0; q < (ITEMS + 1) / 2; ++q)
      {
        if (q < rows)
        {
          const uint32_t p0 = before + ex[q];
          s.bin.cnt[(wave * rows + q) * wave_size + lane] = p0 | ((p0 + (w[q] & 0xFFFFu)) << 16);
        }
      }
      if (tid == 0) s.bin.cnt[nb / 2] = (uint32_t)n;
      __syncthreads();
      const uint16_t* const place = reinterpret_cast<const uint16_t*>(s.bin.cnt);
      uint32_t share = 0;  // bit j: item j shares its bin
#pragma unroll
      for (int j = 0; j < ITEMS; ++j)
      {
        if (j < per && wbase + j * wave_size + lane < n)
        {
          const uint32_t bin = pos[j] >> 16;
          const uint32_t first = place[bin], end = place[bin + 1];
          const uint32_t at = first + (pos[j] & 0xFFFFu);
          s_keys[at] = k[j];
          s.bin.idx[at] = (uint16_t)(wbase + j * wave_size + lane);
          pos[j] = (end << 16) | first;
          share |= (end - first > 1u) ? 1u << j : 0u;
        }
      }
      __syncthreads();
      if (__any((int)share))
      {
#pragma unroll
        for (int j = 0; j < ITEMS; ++j)
        {
          if (j < per && ((share >> j) & 1u))
          {
            const uint32_t first = pos[j] & 0xFFFFu, end = pos[j] >> 16;
            const uint32_t me = (uint32_t)(wbase + j * wave_size + lane);
            const bits_t b = ordered<K>(k[j], flip);
            uint32_t r = 0;
            for (uint32_t q = first; q < end; ++q)
            {
              const bits_t bq = ordered<K>(s_keys[q], flip);
              r += (bq < b || (bq == b && s.bin.idx[q] < me)) ? 1u : 0u;
            }
            pos[j] = first + r;
          }
        }
      }
      __syncthreads();
    }
  }
  if (!fast)
  {
    // LSD passes over the digits that differ.
    bits_t diff = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      if (j < per && wbase + j * wave_size + lane < n) diff |= ordered<K>(k[j], flip) ^ lo;
    }
    diff = wave_reduce(diff, rk::OpBitOr<bits_t>{});
    __syncthreads();  // s.hi is read above
    if (lane == 0) s.hi[wave] = diff;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) diff |= s.hi[w];
    const uint64_t lt_mask = lanemask_lt();
    // The last pass leaves the places in pos; before it, keys and values are
    // moved through LDS.  No digit that differs: input order.
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) pos[j] = (uint32_t)(wbase + j * wave_size + lane);
    bool first_pass = true;
#pragma unroll 1
    for (int p = 0; p < P; ++p)
    {
      if (((uint32_t)(diff >> (8 * p)) & 0xFFu) == 0u) continue;
      if (!first_pass)
      {
        // to the places of the previous pass and back in input order of this one
#pragma unroll
        for (int j = 0; j < ITEMS; ++j)
        {
          if (j < per && wbase + j * wave_size + lane < n) s_keys[pos[j]] = k[j];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; ++j)
        {
          const int i = wbase + j * wave_size + lane;
          if (j < per && i < n) k[j] = s_keys[i];
        }
        __syncthreads();
        if (HAS_VALS)
        {
          V* const s_vals = reinterpret_cast<V*>(s.buf);
#pragma unroll
          for (int j = 0; j < ITEMS; ++j)
          {
            if (j < per && wbase + j * wave_size + lane < n) s_vals[pos[j]] = v[j];
          }
          __syncthreads();
#pragma unroll
          for (int j = 0; j < ITEMS; ++j)
          {
            const int i = wbase + j * wave_size + lane;
            if (j < per && i < n) v[j] = s_vals[i];
          }
          __syncthreads();
        }
      }
      first_pass = false;
      for (int i = tid; i < NW * kRadix; i += BLOCK) s.lsd.whist[i] = 0u;
      __syncthreads();
#pragma unroll
      for (int j = 0; j < ITEMS; ++j)
      {
        if (j < per)
        {
          const bool valid = wbase + j * wave_size + lane < n;
          const uint32_t d = (uint32_t)(ordered<K>(k[j], flip) >> (8 * p)) & (kRadix - 1);
          uint64_t peers = ballot(valid);
#pragma unroll
          for (int b = 0; b < 8; ++b)
          {
            const bool bit = (d >> b) & 1u;
            const uint64_t bal = ballot(bit);
            peers &= bit ? bal : ~bal;
          }
          const uint32_t lower = (uint32_t)__popcll(peers & lt_mask);
          uint32_t c = 0;
          if (valid) c = s.lsd.whist[wave * kRadix + d];
          pos[j] = c + lower;
          if (valid && lower == 0) s.lsd.whist[wave * kRadix + d] = c + (uint32_t)__popcll(peers);
        }
      }
      __syncthreads();
      for (int d0 = 0; d0 < kRadix; d0 += BLOCK)
      {
        const int d = d0 + tid;
        uint32_t ex = 0, total = 0;
        if (d < kRadix)
        {
#pragma unroll
          for (int w = 0; w < NW; ++w)
          {
            const uint32_t c = s.lsd.whist[w * kRadix + d];
            s.lsd.whist[w * kRadix + d] = total;
            total += c;
          }
          uint32_t sum;
          (void)wave_scan(total, rk::OpPlus<uint32_t>{}, 0u, ex, sum);
          s.lsd.tstart[d] = ex;
          if (lane == 0) s.scan[d / wave_size] = sum;
        }
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < ITEMS; ++j)
      {
        if (j < per && wbase + j * wave_size + lane < n)
        {
          const uint32_t d = (uint32_t)(ordered<K>(k[j], flip) >> (8 * p)) & (kRadix - 1);
          uint32_t base = s.lsd.tstart[d] + s.lsd.whist[wave * kRadix + d];
#pragma unroll
          for (int x = 0; x < kRadix / wave_size - 1; ++x) base += (x < (int)(d / wave_size)) ? s.scan[x] : 0u;
          pos[j] += base;
        }
      }
      __syncthreads();
    }
  }
  // Keys (and 4-byte values) to their places, then out in order.
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
  {
    if (j < per && wbase + j * wave_size + lane < n)
    {
      const uint32_t p = pos[j] & 0xFFFFu;
      s_keys[p] = k[j];
      if constexpr (HAS_VALS && sizeof(V) == 4) s.vals4[p] = __builtin_bit_cast(uint32_t, v[j]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
  {
    const int i = j * BLOCK + tid;
    if (j < per && i < n)
    {
      out_keys[i] = s_keys[i];
      if constexpr (HAS_VALS && sizeof(V) == 4) out_vals[i] = __builtin_bit_cast(V, s.vals4[i]);
    }
  }
  if constexpr (HAS_VALS && sizeof(V) == 8)
  {
    V* const s_vals = reinterpret_cast<V*>(s.buf);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      if (j < per && wbase + j * wave_size + lane < n) s_vals[pos[j] & 0xFFFFu] = v[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      const int i = j * BLOCK + tid;
      if (j < per && i < n) out_vals[i] = s_vals[i];
    }
  }
}

// segs: one record per block; nullptr: the one range `one`.  4-byte keys and
// values: at most 64 registers, so two of the 1024-thread blocks share a CU.
template<typename K, typename V, bool HAS_VALS, int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK, (sizeof(K) == 4 && (!HAS_VALS || sizeof(V) == 4)) ? 8 : 4) void local_sort_kernel(const K* in_keys, const V* in_vals,
                                                           K* out_keys, V* out_vals,
                                                           const rs::SortSeg* __restrict__ segs,
                                                           rs::SortSeg one, bits_of<K> flip)
{
  const rs::SortSeg sg = segs ? segs[blockIdx.x] : one;
  local_sort<K, V, HAS_VALS, BLOCK, ITEMS>(in_keys + sg.in_keys,
                                           HAS_VALS ? in_vals + sg.in_vals : nullptr,
                                           out_keys + sg.out_keys,
                                           HAS_VALS ? out_vals + sg.out_vals : nullptr, (int)sg.n, flip);
}

template<typename K, typename V, bool HAS_VALS>
int launch_classes(const K* ik, const V* iv, K* ok, V* ov, bits_of<K> flip,
                   const rs::SortSeg* d_segs, const rs::SortSeg& one, const int64_t* first,
                   hipStream_t s)
{
  // long ranges first: the short ones fill the chip while the last long
  // blocks end
  const int64_t c3 = first[4] - first[3], c2 = first[3] - first[2], c1 = first[2] - first[1],
                c0 = first[1] - first[0];
  auto at = [&](int64_t q) { return d_segs ? d_segs + q : nullptr; };
  if (c3 > 0)
  {
    hipLaunchKernelGGL((local_sort_kernel<K, V, HAS_VALS, 1024, 8>), dim3((unsigned)c3), dim3(1024),
                       0, s, ik, iv, ok, ov, at(first[3]), one, flip);
  }
  if (c2 > 0)
  {
    hipLaunchKernelGGL((local_sort_kernel<K, V, HAS_VALS, 256, 8>), dim3((unsigned)c2), dim3(256), 0,
                       s, ik, iv, ok, ov, at(first[2]), one, flip);
  }
  if (c1 > 0)
  {
    hipLaunchKernelGGL((local_sort_kernel<K, V, HAS_VALS, 128, 4>), dim3((unsigned)c1), dim3(128), 0,
                       s, ik, iv, ok, ov, at(first[1]), one, flip);
  }
  if (c0 > 0)
  {
    hipLaunchKernelGGL((wave_sort_kernel<K, V, HAS_VALS>), dim3((unsigned)rc::ceil_div(c0, 4)),
                       dim3(256), 0, s, ik, iv, ok, ov, at(first[0]), c0, flip);
  }
  RC_HIP(hipGetLastError());
  return RAJA_CDNA4_SUCCESS;
}

template<typename K>
int launch_key(int val_bytes, int descending, const void* ik, const void* iv, void* ok, void* ov,
               const rs::SortSeg* d_segs, const rs::SortSeg& one, const int64_t* first, hipStream_t s)
{
  const bits_of<K> flip = descending ? ~(bits_of<K>)0 : (bits_of<K>)0;
  switch (val_bytes)
  {
    case 0:
      return launch_classes<K, uint32_t, false>((const K*)ik, nullptr, (K*)ok, nullptr, flip, d_segs,
                                                one, first, s);
    case 4:
      return launch_classes<K, uint32_t, true>((const K*)ik, (const uint32_t*)iv, (K*)ok,
                                               (uint32_t*)ov, flip, d_segs, one, first, s);
    case 8:
      return launch_classes<K, uint64_t, true>((const K*)ik, (const uint64_t*)iv, (K*)ok,
                                               (uint64_t*)ov, flip, d_segs, one, first, s);
    default:
      return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "value size %d (4 or 8 supported)", val_bytes);
  }
}

int launch_any(int key_dtype, int val_bytes, int descending, const void* ik, const void* iv, void* ok,
               void* ov, const rs::SortSeg* d_segs, const rs::SortSeg& one, const int64_t* first,
               hipStream_t s)
{
  switch (key_dtype)
  {
    case RAJA_CDNA4_U32: return launch_key<uint32_t>(val_bytes, descending, ik, iv, ok, ov, d_segs, one, first, s);
    case RAJA_CDNA4_I32: return launch_key<int32_t>(val_bytes, descending, ik, iv, ok, ov, d_segs, one, first, s);
    case RAJA_CDNA4_F32: return launch_key<float>(val_bytes, descending, ik, iv, ok, ov, d_segs, one, first, s);
    case RAJA_CDNA4_U64: return launch_key<uint64_t>(val_bytes, descending, ik, iv, ok, ov, d_segs, one, first, s);
    case RAJA_CDNA4_I64: return launch_key<int64_t>(val_bytes, descending, ik, iv, ok, ov, d_segs, one, first, s);
    case RAJA_CDNA4_F64: return launch_key<double>(val_bytes, descending, ik, iv, ok, ov, d_segs, one, first, s);
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "key dtype %d", key_dtype);
  }
}

}  // namespace

namespace rsort
{
int local_sort_batch(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                     void* out_k, void* out_v, const rs::SortSeg* d_segs,
                     const int64_t (&first)[kLocalClasses + 1], hipStream_t s)
{
  return launch_any(key_dtype, val_bytes, descending, in_k, in_v, out_k, out_v, d_segs,
                    rs::SortSeg{}, first, s);
}

int local_sort_one(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                   void* out_k, void* out_v, int64_t n, hipStream_t s)
{
  // a span of up to 64 keys takes the smallest block class: no record array
  const int c = local_class(n) > 1 ? local_class(n) : 1;
  int64_t first[kLocalClasses + 1];
  for (int q = 0; q <= kLocalClasses; ++q) first[q] = q > c ? 1 : 0;
  return launch_any(key_dtype, val_bytes, descending, in_k, in_v, out_k, out_v, nullptr,
                    rs::SortSeg{0, 0, 0, 0, n}, first, s);
}
}  // namespace rsort
