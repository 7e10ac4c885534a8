// Digit histograms of a whole span (the LSD sort's first read of the keys), and
// which digits differ.
#pragma once

#include "ops.hpp"
#include "radix.hpp"
#include "runtime.hpp"

namespace
{
using namespace RAJA::cdna4::dev;

// Counters per bin, side by side (bin b's copy c is word b * kHistCopies + c),
// lane l counting into copy l % kHistCopies: lanes of one atomic instruction that
// meet the same bin use different words in different banks.  2^28 keys: 0.283
// ms with one copy, 0.239 ms with 4 copies as separate histograms, 0.229 /
// 0.212 / 0.27 ms with 4 / 8 / 16 side-by-side copies (copy l / 8 instead of
// l % 8: 0.285 ms).
constexpr int kHistCopies = 8;
// LDS words of a block that counts every digit of K.
template<typename K>
constexpr int kHistWords = kHistCopies * (int)sizeof(K) * kRadix;

// Counts the N keys every lane of the wave holds (all of them valid) into
// s_hist, bin b's copy c at word b * C + c, lane l counting into copy l % C.
// A digit that is the same for all 64 * N keys is added once: the test is
// an OR over the keys of (bits ^ lane 0's first bits), one ballot per digit.
template<typename K, bool DESC, int P, int N, int C>
__device__ __forceinline__ void count_full_wave(const K (&k)[N], uint32_t* s_hist, int lane)
{
  using bits_t = typename KeyTraits<K>::bits_t;
  const bits_t b0 = KeyTraits<K>::to_bits(k[0]);
  bits_t f = 0;
  if constexpr (sizeof(bits_t) == 4)
  {
    f = (bits_t)__builtin_amdgcn_readfirstlane((int)b0);
  }
  else
  {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b0);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b0 >> 32));
    f = ((bits_t)hi << 32) | lo;
  }
  bits_t x = 0;
#pragma unroll
  for (int q = 0; q < N; ++q) x |= KeyTraits<K>::to_bits(k[q]) ^ f;
#pragma unroll
  for (int p = 0; p < P; ++p)
  {
    if (ballot(((x >> (8 * p)) & (bits_t)0xFF) != 0) == 0ull)
    {
      const uint32_t d0 = (uint32_t)((DESC ? ~f : f) >> (8 * p)) & (kRadix - 1);
      if (lane == 0) atomicAdd(&s_hist[(p * kRadix + d0) * C], (uint32_t)(wave_size * N));
    }
    else
    {
      uint32_t* const h = s_hist + p * kRadix * C + (lane % C);
#pragma unroll
      for (int q = 0; q < N; ++q) atomicAdd(&h[digit_of<K, DESC>(k[q], 8 * p) * C], 1u);
    }
  }
}

// Adds the block's share of the span's digit counts (ascending order; every 8-bit
// digit of K) to s_hist, which it clears first: blocks of 256 threads.
// Each wave streams 64 lanes x U x 16-byte vectors per iteration (U vector
// loads in flight per lane) and counts every digit of every key with LDS
// atomics; a digit shared by all keys of a full iteration is added once
// (constant high digits of small keys would otherwise serialise 64 lanes on
// one LDS word).
template<typename K>
__device__ __forceinline__ void count_digits(const K* __restrict__ keys, int64_t n, uint32_t* s_hist)
{
  constexpr int P = (int)sizeof(K);
  constexpr int VEC = 16 / sizeof(K);
  constexpr int U = 4;
  constexpr int PER_WAVE = wave_size * U * VEC;
  typedef K vec_t __attribute__((ext_vector_type(16 / sizeof(K))));
  for (int i = threadIdx.x; i < kHistWords<K>; i += 256) s_hist[i] = 0u;
  __syncthreads();
  const int lane = lane_id();
  const bool aligned = ((uintptr_t)keys % 16) == 0;
  const int64_t nwaves = (int64_t)gridDim.x * (256 / wave_size);
  for (int64_t base = ((int64_t)blockIdx.x * (256 / wave_size) + wave_id()) * PER_WAVE; base < n;
       base += nwaves * PER_WAVE)
  {
    K k[U * VEC];
    const bool full = aligned && base + PER_WAVE <= n;
    if (full)
    {
#pragma unroll
      for (int u = 0; u < U; ++u)
      {
        const vec_t x = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(keys + base + ((int64_t)u * wave_size + lane) * VEC));
#pragma unroll
        for (int e = 0; e < VEC; ++e) k[u * VEC + e] = x[e];
      }
    }
    else
    {
#pragma unroll
      for (int u = 0; u < U; ++u)
      {
#pragma unroll
        for (int e = 0; e < VEC; ++e)
        {
          const int64_t i = base + ((int64_t)u * wave_size + lane) * VEC + e;
          k[u * VEC + e] = (i < n) ? keys[i] : K(0);
        }
      }
    }
    if (full)
    {
      count_full_wave<K, false, P, U * VEC, kHistCopies>(k, s_hist, lane);
      continue;
    }
#pragma unroll
    for (int q = 0; q < U * VEC; ++q)
    {
      const int64_t i = base + ((int64_t)(q / VEC) * wave_size + lane) * VEC + (q % VEC);
      const bool valid = full || i < n;
      // valid lanes of one item form a prefix in lane order
      const uint64_t vmask = ballot(valid);
#pragma unroll
      for (int p = 0; p < P; ++p)
      {
        const uint32_t d = digit_of<K, false>(k[q], 8 * p);
        const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
        const bool uniform = (ballot(d == d0 || !valid) == ~0ull) && (vmask & 1ull);
        if (uniform)
        {
          if (lane == 0) atomicAdd(&s_hist[(p * kRadix + d0) * kHistCopies], (uint32_t)__popcll(vmask));
        }
        else if (valid)
        {
          atomicAdd(&s_hist[(p * kRadix + d) * kHistCopies], 1u);
        }
      }
    }
  }
  __syncthreads();
}

// Adds the block's counts to the P rows of 256 counters in memory; descending
// digits are the ascending ones' complements.
template<typename K>
__device__ __forceinline__ void add_digits(const uint32_t* s_hist, uint32_t* __restrict__ hist, bool descending)
{
  for (int i = threadIdx.x; i < (int)sizeof(K) * kRadix; i += 256)
  {
    uint32_t c = 0;
#pragma unroll
    for (int r = 0; r < kHistCopies; ++r) c += s_hist[i * kHistCopies + r];
    if (c) atomic_add_agent(&hist[descending ? i ^ (kRadix - 1) : i], c);
  }
}

// Histograms of the span, and cleared descriptors for the first pass.  Does
// nothing where *unless is not 0 (a span that the partition takes).
template<typename K>
__global__ __launch_bounds__(256) void hist_kernel(const K* __restrict__ keys, int64_t n, bool descending,
                                                   uint32_t* __restrict__ hist, uint32_t* __restrict__ desc0,
                                                   int64_t desc0_words, const uint32_t* unless)
{
  if (unless && *unless != 0u) return;
  __shared__ uint32_t s_hist[kHistWords<K>];
  count_digits<K>(keys, n, s_hist);
  add_digits<K>(s_hist, hist, descending);
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < desc0_words; i += stride) desc0[i] = 0u;
}

// Blocks of hist_kernel for n keys.
inline unsigned hist_blocks(int64_t n)
{
  const int64_t want = rc::ceil_div(n, (int64_t)256 * 64);
  const int64_t cap = (int64_t)rc::num_cus() * 16;
  return (unsigned)(want < 1 ? 1 : (want < cap ? want : cap));
}

// Set in a word of active digits once it is known; bit p: the keys differ in digit p.
constexpr uint32_t kDigitsKnown = 0x80000000u;

// The word of active digits of a histogram of n keys, in every thread (256 threads).
template<typename K>
__device__ __forceinline__ uint32_t active_digits(const uint32_t* hist, uint32_t n)
{
  uint32_t m = kDigitsKnown;
  for (int p = 0; p < (int)sizeof(K); ++p)
  {
    if (__syncthreads_or(hist[p * kRadix + threadIdx.x] == n) == 0) m |= 1u << p;
  }
  return m;
}

// The word of active digits to pinned host memory: a store by one small kernel and
// a look at it by the host in place of a copy of the histograms and a
// wait for it.
template<typename K>
__global__ __launch_bounds__(256) void digits_kernel(const uint32_t* __restrict__ hist, uint32_t n,
                                                     uint32_t* host_word)
{
  const uint32_t m = active_digits<K>(hist, n);
  if (threadIdx.x == 0) __hip_atomic_store(host_word, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace
