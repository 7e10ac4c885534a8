// Ordered key bits and monotone maps of keys to bins.
#pragma once

#include <type_traits>

#include "radix.hpp"

namespace
{

template<typename K>
using bits_of = typename KeyTraits<K>::bits_t;

// Unsigned bits whose order is the sort's order.
template<typename K>
__device__ __forceinline__ bits_of<K> ordered(K k, bits_of<K> flip)
{
  return KeyTraits<K>::to_bits(k) ^ flip;
}

// Monotone map of keys whose ordered bits lie in [lo, hi] to bins 0 .. nb-1:
// integers by the distance from the smallest, floating keys by value.  SPREAD:
// an integer range of fewer values than bins is spread over them (several
// keys apart) instead of taking the first bins.
template<typename K, bool SPREAD = false>
struct BinMap
{
  using bits_t = bits_of<K>;
  static constexpr bool is_float = std::is_floating_point_v<K>;
  bits_t lo;
  uint32_t nb;
  int shift;        // 64-bit integer keys: right shift that leaves 32 bits
  uint32_t scale;   // integer keys: bins per key value, 32 fraction bits; 0: `mul` bins per value
  uint32_t mul;
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
    mul = 1;
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
      if (SPREAD && r < nb) mul = nb / (r + 1);
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
      return scale ? __umulhi(x, scale) : (SPREAD ? x * mul : x);
    }
  }
};

}  // namespace
