// Stable sorts of short ranges inside one workgroup (or one wave): the
// segments of a batch, small spans and small requests.
//
// The work is split by range length, each class with a block as large as its
// longest range: one wave per range of up to 64 keys, 128 x 4 threads x keys
// up to 512, 256 x 8 up to 2048, 640 x 8 up to 5120 and 1024 x 8 up to 8192
// (small batches: the last for all).  A block holds its keys and values in
// registers, reads and writes memory once and coalesced.
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
// those of up to 8192 pairs, 1.5e7 pairs of uniform keys): 130 us, against 1787
// us with one 512-thread block of 16 items per thread and four ballot-ranked
// LSD passes for every range.  2^26 pairs in ranges of 512, 2048, 4096 and 8192:
// 0.27, 0.24, 0.40 and 0.30 ms.  One span of 5000 pairs: 10 us in one launch,
// against 74 us for the clear, the histogram and four one-tile passes of the
// span sort.
#include "local_sort.hpp"

#include "key_map.hpp"
#include "ops.hpp"
#include "radix.hpp"

namespace
{
using namespace RAJA::cdna4::dev;

// Keys one bin may hold before the range takes the LSD passes.  A bin of c
// keys costs each of them c LDS reads: 32 is about what one 8-bit ballot
// ranking costs a key.
constexpr uint32_t kMaxBin = 32;

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
      __attribute__((aligned(16))) uint32_t cnt[CAP / 2 + 1];
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

// The element at a 32-bit byte offset from a uniform base: one address
// register instead of 64-bit arithmetic per access.
template<typename T>
__device__ __forceinline__ T* at_offset(T* base, uint32_t bytes)
{
  return reinterpret_cast<T*>(reinterpret_cast<uintptr_t>(base) + bytes);
}

__device__ __forceinline__ int64_t uniform(int64_t x)
{
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)x >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Sum over each row of 16 lanes, in every lane of the row.
__device__ __forceinline__ uint32_t row_sum(uint32_t v)
{
  v += dpp_move<dpp_quad_1032>(v, v);
  v += dpp_move<dpp_quad_2301>(v, v);
  v += dpp_move<dpp_row_half_mirror>(v, v);
  v += dpp_move<dpp_row_mirror>(v, v);
  return v;
}

// f(j) for every item j this lane holds (element wbase + 64 j + lane of n):
// without a test per item in waves whose items are all in range (whole, the
// same in the whole wave).
template<int ITEMS, typename F>
__device__ __forceinline__ void each_item(bool whole, int per, int wbase, int lane, int n, F&& f)
{
  if (whole)
  {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      if (j < per) f(j);
    }
  }
  else
  {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      if (j < per && wbase + j * wave_size + lane < n) f(j);
    }
  }
}

// Hides a value from the optimiser: what is computed from a key is computed
// again in each phase instead of being kept in a register per item.
template<typename T>
__device__ __forceinline__ void again(T& x)
{
  asm volatile("" : "+v"(x));
}

// The range's keys (and values), item j of a lane being element wbase + 64 j +
// lane; unguarded loads at 32-bit offsets (past the end: element 0 again).
template<typename T, int ITEMS>
__device__ __forceinline__ void load_items(const T* in, int n, int per, int wbase, int lane, T (&x)[ITEMS])
{
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
  {
    if (j < per)
    {
      const int i = wbase + j * wave_size + lane;
      x[j] = *at_offset(in, (uint32_t)(i < n ? i : 0) * (uint32_t)sizeof(T));
    }
  }
}

// Keys and values to the places pos (low 16 bits) in LDS, then out in order.
template<typename K, typename V, bool HAS_VALS, int BLOCK, int ITEMS>
__device__ __forceinline__ void write_sorted(LocalLds<K, V, HAS_VALS, BLOCK, ITEMS>& s, const K (&k)[ITEMS],
                                             const V (&v)[HAS_VALS ? ITEMS : 1], const uint32_t (&pos)[ITEMS],
                                             K* out_keys, V* out_vals, int n, int per, int wbase)
{
  K* const s_keys = reinterpret_cast<K*>(s.buf);
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const bool whole = wbase + per * wave_size <= n;
  auto each = [&](auto&& f) { each_item<ITEMS>(whole, per, wbase, lane, n, f); };
  each([&](int j) {
    const uint32_t p = pos[j] & 0xFFFFu;
    s_keys[p] = k[j];
    if constexpr (HAS_VALS && sizeof(V) == 4) s.vals4[p] = __builtin_bit_cast(uint32_t, v[j]);
  });
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
  {
    const uint32_t i = (uint32_t)(j * BLOCK + tid);
    if (j < per && i < (uint32_t)n)
    {
      *at_offset(out_keys, i * (uint32_t)sizeof(K)) = s_keys[i];
      if constexpr (HAS_VALS && sizeof(V) == 4)
      {
        *at_offset(out_vals, i * 4u) = __builtin_bit_cast(V, s.vals4[i]);
      }
    }
  }
  if constexpr (HAS_VALS && sizeof(V) == 8)
  {
    V* const s_vals = reinterpret_cast<V*>(s.buf);
    __syncthreads();
    each([&](int j) { s_vals[pos[j] & 0xFFFFu] = v[j]; });
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      const uint32_t i = (uint32_t)(j * BLOCK + tid);
      if (j < per && i < (uint32_t)n) *at_offset(out_vals, i * 8u) = s_vals[i];
    }
  }
}

// Bin placement; false (in every thread) if the bins are too uneven, before
// anything is written.
template<typename K, typename V, bool HAS_VALS, int BLOCK, int ITEMS>
__device__ __forceinline__ bool local_sort_bins(LocalLds<K, V, HAS_VALS, BLOCK, ITEMS>& s, const K* in_keys,
                                                const V* in_vals, K* out_keys, V* out_vals, int n, int per,
                                                int wbase, bits_of<K> flip)
{
  using L = LocalLds<K, V, HAS_VALS, BLOCK, ITEMS>;
  using bits_t = bits_of<K>;
  constexpr int NW = L::NW;
  K* const s_keys = reinterpret_cast<K*>(s.buf);
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  K k[ITEMS];
  V v[HAS_VALS ? ITEMS : 1];
  load_items(in_keys, n, per, wbase, lane, k);
  if constexpr (HAS_VALS) load_items(in_vals, n, per, wbase, lane, v);
  // Counter words per thread (two bins each): twice as many bins as keys where
  // the counters have room for them, else as many.
  constexpr int MAXW = ITEMS >= 8 ? 4 : 2;
  static_assert(MAXW * BLOCK <= L::CAP / 2, "counters fit their LDS");
  const int words = per >= MAXW ? MAXW : (per > 2 ? 4 : (per > 1 ? 2 : 1));
  const uint32_t nb = (uint32_t)(words * 2 * BLOCK);
  for (int q = 0; q < words; ++q) s.bin.cnt[q * BLOCK + tid] = 0u;

  const bool whole = wbase + per * wave_size <= n;
  auto each = [&](auto&& f) { each_item<ITEMS>(whole, per, wbase, lane, n, f); };

  bits_t lo = ~(bits_t)0, hi = 0;
  each([&](int j) {
    const bits_t b = ordered<K>(k[j], flip);
    lo = b < lo ? b : lo;
    hi = b > hi ? b : hi;
  });
  lo = wave_reduce(lo, rk::OpMin<bits_t>{});
  hi = wave_reduce(hi, rk::OpMax<bits_t>{});
  if (lane == 0)
  {
    s.lo[wave] = lo;
    s.hi[wave] = hi;
  }
  __syncthreads();
  {
    // one lane per wave value, folded inside a row of 16
    static_assert(NW <= 16, "wave values fit a row");
    const int w = (lane & 15) < NW ? (lane & 15) : 0;
    lo = s.lo[w];
    hi = s.hi[w];
    lo = wave_reduce(lo, rk::OpMin<bits_t>{});
    hi = wave_reduce(hi, rk::OpMax<bits_t>{});
  }
  // Keys that lie close together: the distance from the smallest and the
  // input position fit one word, which orders keys and ties at once.
  const bits_t range = hi - lo;
  const int ibits = 32 - __builtin_clz((uint32_t)n);  // positions < 2^ibits
  const bool narrow = (range >> (32 - ibits)) == 0;
  const float inv =
      narrow ? (float)nb * __builtin_amdgcn_rcpf((float)(uint32_t)range + 1.0f) * (1.0f - 0x1.0p-20f) : 0.0f;
  const BinMap<K> bin_of(lo, hi, nb, flip);
  if (!narrow && !bin_of.ok) return false;

  uint32_t pos[ITEMS];
  // bin << 16 | slot inside the bin
  auto take_slot = [&](int j, uint32_t bin) {
    const uint32_t sh = (bin & 1u) * 16u;
    const uint32_t c = atomicAdd(&s.bin.cnt[bin >> 1], 1u << sh);
    pos[j] = (bin << 16) | ((c >> sh) & 0xFFFFu);
  };
  if (narrow)
  {
    each([&](int j) {
      again(k[j]);
      take_slot(j, (uint32_t)((float)(uint32_t)(ordered<K>(k[j], flip) - lo) * inv));
    });
  }
  else
  {
    each([&](int j) {
      again(k[j]);
      take_slot(j, bin_of(k[j], ordered<K>(k[j], flip)));
    });
  }
  __syncthreads();
  // Places of the bins: a thread's words in a row, one wave scan of the
  // threads' sums, then the wave totals.
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  uint32_t w[MAXW], ex = 0;
  u16x2 worst2 = {0, 0};
  auto read_words = [&](auto count_c) {
    constexpr int W = decltype(count_c)::value;
    uint32_t sum = 0;
#pragma unroll
    for (int q = 0; q < W; ++q) w[q] = s.bin.cnt[tid * W + q];
#pragma unroll
    for (int q = 0; q < W; ++q)
    {
      sum += (w[q] & 0xFFFFu) + (w[q] >> 16);
      worst2 = __builtin_elementwise_max(worst2, __builtin_bit_cast(u16x2, w[q]));
    }
    uint32_t total;
    (void)wave_scan(sum, rk::OpPlus<uint32_t>{}, 0u, ex, total);
    if (lane == 0) s.scan[wave] = total;
  };
  auto write_words = [&](auto count_c) {
    constexpr int W = decltype(count_c)::value;
    uint32_t before = (lane & 15) < wave ? s.scan[lane & 15] : 0u;
    before = __builtin_amdgcn_readfirstlane(row_sum(before));
    uint32_t p = before + ex;
#pragma unroll
    for (int q = 0; q < W; ++q)
    {
      const uint32_t p1 = p + (w[q] & 0xFFFFu);
      s.bin.cnt[tid * W + q] = p | (p1 << 16);
      p = p1 + (w[q] >> 16);
    }
  };
  auto by_words = [&](auto&& f) {
    if (words == 1)
      f(std::integral_constant<int, 1>{});
    else if (words == 2)
      f(std::integral_constant<int, 2>{});
    else if (MAXW >= 4 && words == 4)
      f(std::integral_constant<int, MAXW >= 4 ? 4 : 2>{});
    else
      f(std::integral_constant<int, MAXW>{});
  };
  by_words(read_words);
  const uint32_t worst = worst2[0] > worst2[1] ? worst2[0] : worst2[1];
  if (__syncthreads_or(worst > kMaxBin) != 0) return false;
  by_words(write_words);
  if (tid == 0) s.bin.cnt[nb / 2] = (uint32_t)n;
  __syncthreads();
  const uint16_t* const place = reinterpret_cast<const uint16_t*>(s.bin.cnt);
  uint32_t share = 0;  // bit j: item j shares its bin
  uint32_t* const s_comp = reinterpret_cast<uint32_t*>(s.buf);
  auto put = [&](int j, auto&& store) {
    const uint32_t bin = pos[j] >> 16;
    const uint32_t first = place[bin], end = place[bin + 1];
    store(first + (pos[j] & 0xFFFFu));
    pos[j] = (end << 16) | first;
    share |= (end - first > 1u) ? 1u << j : 0u;
  };
  auto comp_of = [&](int j) {
    again(k[j]);
    return ((uint32_t)(ordered<K>(k[j], flip) - lo) << ibits) | (uint32_t)(wbase + j * wave_size + lane);
  };
  if (narrow)
  {
    each([&](int j) { put(j, [&](uint32_t at) { s_comp[at] = comp_of(j); }); });
  }
  else
  {
    each([&](int j) {
      put(j, [&](uint32_t at) {
        s_keys[at] = k[j];
        s.bin.idx[at] = (uint16_t)(wbase + j * wave_size + lane);
      });
    });
  }
  __syncthreads();
  if (narrow)
  {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      if (j < per && ((share >> j) & 1u))
      {
        const uint32_t first = pos[j] & 0xFFFFu, end = pos[j] >> 16;
        const uint32_t me = comp_of(j);
        uint32_t r = first;
        for (uint32_t q = first; q < end; ++q) r += s_comp[q] < me ? 1u : 0u;
        pos[j] = r;
      }
    }
  }
  else
  {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      if (j < per && ((share >> j) & 1u))
      {
        const uint32_t first = pos[j] & 0xFFFFu, end = pos[j] >> 16;
        const uint32_t me = (uint32_t)(wbase + j * wave_size + lane);
        again(k[j]);
        const bits_t b = ordered<K>(k[j], flip);
        uint32_t r = first;
        for (uint32_t q = first; q < end; ++q)
        {
          const bits_t bq = ordered<K>(s_keys[q], flip);
          r += (bq < b || (bq == b && s.bin.idx[q] < me)) ? 1u : 0u;
        }
        pos[j] = r;
      }
    }
  }
  __syncthreads();
  write_sorted<K, V, HAS_VALS, BLOCK, ITEMS>(s, k, v, pos, out_keys, out_vals, n, per, wbase);
  return true;
}

// LSD passes of 8-bit digits over the digits that differ.
template<typename K, typename V, bool HAS_VALS, int BLOCK, int ITEMS>
__device__ __forceinline__ void local_sort_lsd(LocalLds<K, V, HAS_VALS, BLOCK, ITEMS>& s, const K* in_keys,
                                               const V* in_vals, K* out_keys, V* out_vals, int n, int per,
                                               int wbase, bits_of<K> flip)
{
  using L = LocalLds<K, V, HAS_VALS, BLOCK, ITEMS>;
  using bits_t = bits_of<K>;
  constexpr int NW = L::NW;
  constexpr int P = (int)sizeof(K);
  K* const s_keys = reinterpret_cast<K*>(s.buf);
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  K k[ITEMS];
  V v[HAS_VALS ? ITEMS : 1];
  uint32_t pos[ITEMS];
  load_items(in_keys, n, per, wbase, lane, k);
  if constexpr (HAS_VALS) load_items(in_vals, n, per, wbase, lane, v);
  const bits_t some = ordered<K>(in_keys[0], flip);
  bits_t diff = 0;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
  {
    if (j < per && wbase + j * wave_size + lane < n) diff |= ordered<K>(k[j], flip) ^ some;
  }
  diff = wave_reduce(diff, rk::OpBitOr<bits_t>{});
  __syncthreads();  // s.hi is read above
  if (lane == 0) s.hi[wave] = diff;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) diff |= s.hi[w];
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
        again(k[j]);
        const uint32_t d = (uint32_t)(ordered<K>(k[j], flip) >> (8 * p)) & (kRadix - 1);
        // peers as in onesweep_kernel: one extract and two v_bitop3 per bit
        const uint64_t vb = ballot(valid);
        uint32_t pl = (uint32_t)vb, ph = (uint32_t)(vb >> 32);
#pragma unroll
        for (int b = 0; b < 8; ++b)
        {
          int32_t sx = __builtin_amdgcn_sbfe((int32_t)d, b, 1);
          asm volatile("" : "+v"(sx));
          const uint64_t bal = ballot(sx != 0);
          pl = __builtin_amdgcn_bitop3_b32(pl, (uint32_t)bal, (uint32_t)sx, 0x90);
          ph = __builtin_amdgcn_bitop3_b32(ph, (uint32_t)(bal >> 32), (uint32_t)sx, 0x90);
        }
        const uint32_t lower = __builtin_amdgcn_mbcnt_hi(ph, __builtin_amdgcn_mbcnt_lo(pl, 0u));
        uint32_t c = 0;
        if (valid) c = s.lsd.whist[wave * kRadix + d];
        pos[j] = c + lower;
        asm volatile("" : "+v"(pos[j]));
        if (valid && lower == 0)
        {
          s.lsd.whist[wave * kRadix + d] = c + (uint32_t)__builtin_popcount(pl) + (uint32_t)__builtin_popcount(ph);
        }
        __builtin_amdgcn_sched_barrier(0);  // one item at a time: few live masks
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
        again(k[j]);
        const uint32_t d = (uint32_t)(ordered<K>(k[j], flip) >> (8 * p)) & (kRadix - 1);
        uint32_t base = s.lsd.tstart[d] + s.lsd.whist[wave * kRadix + d];
#pragma unroll
        for (int x = 0; x < kRadix / wave_size - 1; ++x) base += (x < (int)(d / wave_size)) ? s.scan[x] : 0u;
        pos[j] += base;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
  }
  write_sorted<K, V, HAS_VALS, BLOCK, ITEMS>(s, k, v, pos, out_keys, out_vals, n, per, wbase);
}

// Items per thread of a range of n: wave w holds elements [w*64*per,
// (w+1)*64*per), item j of a lane is j*64 + lane in there, so input order is
// (wave, item, lane) order and every load is one run per wave.
template<int BLOCK>
__device__ __forceinline__ int items_of(int n)
{
  return __builtin_amdgcn_readfirstlane((n + BLOCK - 1) / BLOCK);
}

// The passes and the bin placement are kernels of their own where many ranges
// are sorted: in one kernel the passes' registers make the placement spill
// (2048-key ranges, 2^26 pairs: 0.24 ms apart, 0.99 ms together).  The
// placement leaves a byte per range that says whether it is left to do; one
// launch of lsd_kernel does those.

// One record per block; redo[b] = 1 where the range is left to the passes.
// 4-byte keys and values: at most 64 registers, so two of the 1024-thread
// blocks share a CU.
template<typename K, typename V, bool HAS_VALS, int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK, (sizeof(K) == 4 && (!HAS_VALS || sizeof(V) == 4)) ? 8 : 4)
void local_sort_kernel(const K* in_keys, const V* in_vals, K* out_keys, V* out_vals,
                       const rs::SortSeg* __restrict__ segs, uint8_t* __restrict__ redo, bits_of<K> flip)
{
  __shared__ LocalLds<K, V, HAS_VALS, BLOCK, ITEMS> s;
  rs::SortSeg sg = segs[blockIdx.x];
  sg.in_keys = uniform(sg.in_keys);  // block-wide values in scalar registers
  sg.in_vals = uniform(sg.in_vals);
  sg.out_keys = uniform(sg.out_keys);
  sg.out_vals = uniform(sg.out_vals);
  const int n = (int)uniform(sg.n);
  const int per = items_of<BLOCK>(n);
  const int wbase = __builtin_amdgcn_readfirstlane(wave_id()) * wave_size * per;
  const bool done = local_sort_bins<K, V, HAS_VALS, BLOCK, ITEMS>(
      s, in_keys + sg.in_keys, HAS_VALS ? in_vals + sg.in_vals : nullptr, out_keys + sg.out_keys,
      HAS_VALS ? out_vals + sg.out_vals : nullptr, n, per, wbase, flip);
  if (threadIdx.x == 0) redo[blockIdx.x] = done ? 0 : 1;
}

// Groups of neighbouring buckets of a partitioned span.
template<typename K, typename V, bool HAS_VALS, int BLOCK>
__global__ __launch_bounds__(BLOCK, (sizeof(K) == 4 && (!HAS_VALS || sizeof(V) == 4)) ? 8 : 4)
void local_groups_kernel(const K* in_keys, const V* in_vals, K* out_keys, V* out_vals,
                         const uint32_t* __restrict__ start, uint8_t* __restrict__ redo, bits_of<K> flip)
{
  __shared__ LocalLds<K, V, HAS_VALS, BLOCK, 8> s;
  const int64_t first = uniform((int64_t)start[blockIdx.x]);
  const int n = __builtin_amdgcn_readfirstlane((int)(start[blockIdx.x + 1] - (uint32_t)first));
  bool done = true;
  if (n > 0)
  {
    const int per = items_of<BLOCK>(n);
    const int wbase = __builtin_amdgcn_readfirstlane(wave_id()) * wave_size * per;
    done = local_sort_bins<K, V, HAS_VALS, BLOCK, 8>(
        s, in_keys + first, HAS_VALS ? in_vals + first : nullptr, out_keys + first,
        HAS_VALS ? out_vals + first : nullptr, n, per, wbase, flip);
  }
  if (threadIdx.x == 0) redo[blockIdx.x] = done ? 0 : 1;
}

// The ranges (records `segs`, or groups `start`) that redo marks, a
// block taking every gridDim.x-th of `count`.
template<typename K, typename V, bool HAS_VALS>
__global__ __launch_bounds__(1024) void lsd_kernel(const K* in_keys, const V* in_vals, K* out_keys, V* out_vals,
                                                   const rs::SortSeg* __restrict__ segs,
                                                   const uint32_t* __restrict__ start,
                                                   const uint8_t* __restrict__ redo, int64_t count,
                                                   bits_of<K> flip)
{
  __shared__ LocalLds<K, V, HAS_VALS, 1024, 8> s;
  __shared__ uint32_t s_todo[1024], s_n;
  for (int64_t base = blockIdx.x; base < count; base += (int64_t)gridDim.x * 1024)
  {
    const int64_t mine = base + (int64_t)threadIdx.x * gridDim.x;
    const bool todo = mine < count && redo[mine] != 0;
    if (__syncthreads_or(todo) == 0) continue;
    if (threadIdx.x == 0) s_n = 0u;
    __syncthreads();
    if (todo) s_todo[atomicAdd(&s_n, 1u)] = threadIdx.x;
    __syncthreads();
    const int num = __builtin_amdgcn_readfirstlane((int)s_n);
#pragma unroll 1
    for (int q = 0; q < num; ++q)
    {
      const int64_t r = base + (int64_t)__builtin_amdgcn_readfirstlane((int)s_todo[q]) * gridDim.x;
      rs::SortSeg sg;
      if (segs)
      {
        sg = segs[r];
      }
      else
      {
        sg.in_keys = sg.in_vals = sg.out_keys = sg.out_vals = start[r];
        sg.n = (int64_t)(start[r + 1] - start[r]);
      }
      const int n = (int)uniform(sg.n);
      const int per = items_of<1024>(n);
      local_sort_lsd<K, V, HAS_VALS, 1024, 8>(
          s, in_keys + uniform(sg.in_keys), HAS_VALS ? in_vals + uniform(sg.in_vals) : nullptr,
          out_keys + uniform(sg.out_keys), HAS_VALS ? out_vals + uniform(sg.out_vals) : nullptr, n, per,
          __builtin_amdgcn_readfirstlane(wave_id()) * wave_size * per, flip);
      __syncthreads();  // the next range reuses the LDS
    }
  }
}

// Placement or passes: one span (segs nullptr), or a record per block.
template<typename K, typename V, bool HAS_VALS, int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void span_sort_kernel(const K* in_keys, const V* in_vals, K* out_keys,
                                                          V* out_vals, const rs::SortSeg* __restrict__ segs, int n,
                                                          bits_of<K> flip)
{
  __shared__ LocalLds<K, V, HAS_VALS, BLOCK, ITEMS> s;
  if (segs)
  {
    const rs::SortSeg sg = segs[blockIdx.x];
    in_keys += uniform(sg.in_keys);
    in_vals += uniform(sg.in_vals);
    out_keys += uniform(sg.out_keys);
    out_vals += uniform(sg.out_vals);
    n = (int)uniform(sg.n);
  }
  const int per = items_of<BLOCK>(n);
  const int wbase = __builtin_amdgcn_readfirstlane(wave_id()) * wave_size * per;
  if (local_sort_bins<K, V, HAS_VALS, BLOCK, ITEMS>(s, in_keys, in_vals, out_keys, out_vals, n, per, wbase, flip))
  {
    return;
  }
  __syncthreads();
  local_sort_lsd<K, V, HAS_VALS, BLOCK, ITEMS>(s, in_keys, in_vals, out_keys, out_vals, n, per, wbase, flip);
}

constexpr int64_t kLsdBlocks = 512;

// Batches of up to this many ranges, whatever their lengths, are one launch of
// span_sort_kernel's 1024-thread block (two per CU): by classes they are up to
// six launches in a row, each of which leaves most of the chip idle.
// By classes / in one launch, u32 keys and 4-byte values, lengths 2^10 to 2^13:
// 64 ranges 41.8 / 17.0 us, 512 46.6 / 26.1, 1024 50.3 / 41.6, 2048 69 / 74;
// 2^4 to 2^9: 64 16.2 / 9.0, 512 18.0 / 13.9, 768 18.4 / 18.9, 1024 18.6 / 23.9;
// u64 keys and 8-byte values 2^4 to 2^9: 512 19.0 / 18.0.
constexpr int64_t kOneLaunch = 512;

template<typename K, typename V, bool HAS_VALS>
int launch_groups(int descending, const void* ik, const void* iv, void* ok_, void* ov, const uint32_t* start,
                  int64_t ngroups, int64_t cap, uint8_t* redo, hipStream_t s)
{
  const bits_of<K> flip = descending ? ~(bits_of<K>)0 : (bits_of<K>)0;
  if (cap <= rsort::kGroupCaps[0])
  {
    hipLaunchKernelGGL((local_groups_kernel<K, V, HAS_VALS, rsort::kGroupCaps[0] / 8>), dim3((unsigned)ngroups),
                       dim3(rsort::kGroupCaps[0] / 8), 0, s, (const K*)ik, (const V*)iv, (K*)ok_, (V*)ov, start,
                       redo, flip);
  }
  else
  {
    hipLaunchKernelGGL((local_groups_kernel<K, V, HAS_VALS, rsort::kGroupCaps[1] / 8>), dim3((unsigned)ngroups),
                       dim3(rsort::kGroupCaps[1] / 8), 0, s, (const K*)ik, (const V*)iv, (K*)ok_, (V*)ov, start,
                       redo, flip);
  }
  hipLaunchKernelGGL((lsd_kernel<K, V, HAS_VALS>), dim3((unsigned)(ngroups < kLsdBlocks ? ngroups : kLsdBlocks)),
                     dim3(1024), 0, s, (const K*)ik, (const V*)iv, (K*)ok_, (V*)ov,
                     (const rs::SortSeg*)nullptr, start, redo, ngroups, flip);
  RC_HIP(hipGetLastError());
  return RAJA_CDNA4_SUCCESS;
}

// One span (d_segs nullptr) or the records of a batch.
template<typename K, typename V, bool HAS_VALS>
int launch_classes(const K* ik, const V* iv, K* ok, V* ov, bits_of<K> flip, const rs::SortSeg* d_segs,
                   int64_t span, const int64_t* first, uint8_t* redo, hipStream_t s)
{
  if (!d_segs)
  {
    const int n = (int)span;
    if (n > rsort::kLocalMax[2])  // 1024 threads: the one block has the chip to itself
      hipLaunchKernelGGL((span_sort_kernel<K, V, HAS_VALS, 1024, 8>), dim3(1), dim3(1024), 0, s, ik, iv,
                         ok, ov, d_segs, n, flip);
    else if (n > rsort::kLocalMax[1])
      hipLaunchKernelGGL((span_sort_kernel<K, V, HAS_VALS, 256, 8>), dim3(1), dim3(256), 0, s, ik, iv,
                         ok, ov, d_segs, n, flip);
    else
      hipLaunchKernelGGL((span_sort_kernel<K, V, HAS_VALS, 128, 4>), dim3(1), dim3(128), 0, s, ik, iv,
                         ok, ov, d_segs, n, flip);
    RC_HIP(hipGetLastError());
    return RAJA_CDNA4_SUCCESS;
  }
  if (first[rsort::kLocalClasses] <= kOneLaunch)
  {
    hipLaunchKernelGGL((span_sort_kernel<K, V, HAS_VALS, 1024, 8>), dim3((unsigned)first[rsort::kLocalClasses]),
                       dim3(1024), 0, s, ik, iv, ok, ov, d_segs, 0, flip);
    RC_HIP(hipGetLastError());
    return RAJA_CDNA4_SUCCESS;
  }
  // long ranges first: the short ones fill the chip while the last long
  // blocks end
  const int64_t c4 = first[5] - first[4], c3 = first[4] - first[3], c2 = first[3] - first[2], c1 = first[2] - first[1],
                c0 = first[1] - first[0];
  if (c4 > 0)
  {
    hipLaunchKernelGGL((local_sort_kernel<K, V, HAS_VALS, 1024, 8>), dim3((unsigned)c4), dim3(1024), 0, s, ik, iv,
                       ok, ov, d_segs + first[4], redo + first[4], flip);
  }
  if (c3 > 0)
  {
    hipLaunchKernelGGL((local_sort_kernel<K, V, HAS_VALS, 640, 8>), dim3((unsigned)c3), dim3(640), 0, s, ik, iv,
                       ok, ov, d_segs + first[3], redo + first[3], flip);
  }
  if (c2 > 0)
  {
    hipLaunchKernelGGL((local_sort_kernel<K, V, HAS_VALS, 256, 8>), dim3((unsigned)c2), dim3(256), 0, s, ik, iv, ok,
                       ov, d_segs + first[2], redo + first[2], flip);
  }
  if (c1 > 0)
  {
    hipLaunchKernelGGL((local_sort_kernel<K, V, HAS_VALS, 128, 4>), dim3((unsigned)c1), dim3(128), 0, s, ik, iv, ok,
                       ov, d_segs + first[1], redo + first[1], flip);
  }
  if (c0 > 0)
  {
    hipLaunchKernelGGL((wave_sort_kernel<K, V, HAS_VALS>), dim3((unsigned)rc::ceil_div(c0, 4)), dim3(256), 0, s,
                       ik, iv, ok, ov, d_segs + first[0], c0, flip);
  }
  const int64_t blocks = first[5] - first[1];
  if (blocks > 0)
  {
    hipLaunchKernelGGL((lsd_kernel<K, V, HAS_VALS>), dim3((unsigned)(blocks < kLsdBlocks ? blocks : kLsdBlocks)),
                       dim3(1024), 0, s, ik, iv, ok, ov, d_segs + first[1], (const uint32_t*)nullptr,
                       redo + first[1], blocks, flip);
  }
  RC_HIP(hipGetLastError());
  return RAJA_CDNA4_SUCCESS;
}

template<typename K>
int launch_key(int val_bytes, int descending, const void* ik, const void* iv, void* ok, void* ov,
               const rs::SortSeg* d_segs, int64_t span, const int64_t* first, uint8_t* redo, hipStream_t s)
{
  const bits_of<K> flip = descending ? ~(bits_of<K>)0 : (bits_of<K>)0;
  switch (val_bytes)
  {
    case 0:
      return launch_classes<K, uint32_t, false>((const K*)ik, nullptr, (K*)ok, nullptr, flip, d_segs,
                                                span, first, redo, s);
    case 4:
      return launch_classes<K, uint32_t, true>((const K*)ik, (const uint32_t*)iv, (K*)ok,
                                               (uint32_t*)ov, flip, d_segs, span, first, redo, s);
    case 8:
      return launch_classes<K, uint64_t, true>((const K*)ik, (const uint64_t*)iv, (K*)ok,
                                               (uint64_t*)ov, flip, d_segs, span, first, redo, s);
    default:
      return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "value size %d (4 or 8 supported)", val_bytes);
  }
}

int launch_any(int key_dtype, int val_bytes, int descending, const void* ik, const void* iv, void* ok,
               void* ov, const rs::SortSeg* d_segs, int64_t span, const int64_t* first, uint8_t* redo,
               hipStream_t s)
{
  switch (key_dtype)
  {
    case RAJA_CDNA4_U32: return launch_key<uint32_t>(val_bytes, descending, ik, iv, ok, ov, d_segs, span, first, redo, s);
    case RAJA_CDNA4_I32: return launch_key<int32_t>(val_bytes, descending, ik, iv, ok, ov, d_segs, span, first, redo, s);
    case RAJA_CDNA4_F32: return launch_key<float>(val_bytes, descending, ik, iv, ok, ov, d_segs, span, first, redo, s);
    case RAJA_CDNA4_U64: return launch_key<uint64_t>(val_bytes, descending, ik, iv, ok, ov, d_segs, span, first, redo, s);
    case RAJA_CDNA4_I64: return launch_key<int64_t>(val_bytes, descending, ik, iv, ok, ov, d_segs, span, first, redo, s);
    case RAJA_CDNA4_F64: return launch_key<double>(val_bytes, descending, ik, iv, ok, ov, d_segs, span, first, redo, s);
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "key dtype %d", key_dtype);
  }
}

}  // namespace

namespace rsort
{
int local_sort_batch(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                     void* out_k, void* out_v, const rs::SortSeg* d_segs,
                     const int64_t (&first)[kLocalClasses + 1], uint8_t* redo, hipStream_t s)
{
  return launch_any(key_dtype, val_bytes, descending, in_k, in_v, out_k, out_v, d_segs, 0, first, redo, s);
}

int local_sort_groups(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                      void* out_k, void* out_v, const uint32_t* start, int64_t ngroups, int64_t cap, uint8_t* redo,
                      hipStream_t s)
{
#define RSORT_GROUPS(CODE, K)                                                                              \
  case CODE:                                                                                               \
    if (val_bytes == 0)                                                                                    \
      return launch_groups<K, uint32_t, false>(descending, in_k, in_v, out_k, out_v, start, ngroups, cap, redo, s); \
    if (val_bytes == 4)                                                                                    \
      return launch_groups<K, uint32_t, true>(descending, in_k, in_v, out_k, out_v, start, ngroups, cap, redo, s);  \
    return launch_groups<K, uint64_t, true>(descending, in_k, in_v, out_k, out_v, start, ngroups, cap, redo, s);
  switch (key_dtype)
  {
    RSORT_GROUPS(RAJA_CDNA4_U32, uint32_t)
    RSORT_GROUPS(RAJA_CDNA4_I32, int32_t)
    RSORT_GROUPS(RAJA_CDNA4_F32, float)
    RSORT_GROUPS(RAJA_CDNA4_U64, uint64_t)
    RSORT_GROUPS(RAJA_CDNA4_I64, int64_t)
    RSORT_GROUPS(RAJA_CDNA4_F64, double)
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "key dtype %d", key_dtype);
  }
#undef RSORT_GROUPS
}

int local_sort_one(int key_dtype, int val_bytes, int descending, const void* in_k, const void* in_v,
                   void* out_k, void* out_v, int64_t n, hipStream_t s)
{
  return launch_any(key_dtype, val_bytes, descending, in_k, in_v, out_k, out_v, nullptr, n, nullptr, nullptr, s);
}
}  // namespace rsort
