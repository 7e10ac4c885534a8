// The onesweep pass kernel (one stable scatter by 8-bit digits), shared by
// the LSD sort (sort.hip) and the two-level partition (partition_sort.hip).
#pragma once

#include "ops.hpp"
#include "radix.hpp"
#include "runtime.hpp"
#include "segments.hpp"

namespace
{
using namespace RAJA::cdna4::dev;

constexpr uint32_t kAgg = 1u, kInc = 2u;
constexpr uint32_t kCountMask = 0x3FFFFFFFu;
// A descriptor row: 256 digit words, padded to 264 words so rows of
// neighbouring tiles start in different cache-line sets.
constexpr int kRowStride = kRadix + 8;
// Predecessor rows a look-back step reads with all loads in flight.
constexpr int kLookbackRows = 8;
constexpr int64_t kMaxSortN = (int64_t)kCountMask;  // counts live in 30 bits
// Word 3 of a raw buffer resource on gfx9-family GPUs: 32-bit data format,
// the other fields zero (stride 0: offsets and the size are in bytes).
constexpr int kBufferWord3 = 0x00020000;

// Lookback waits that outlived SpinBound's limit (see raja_cdna4_device_status).
static __device__ uint32_t g_spin_timeouts;

__global__ void clear_words_kernel(uint32_t* p, int64_t n)
{
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
  {
    p[i] = 0u;
  }
}

// Digit `shift` .. `shift` + 7 of the ordered key bits (LSD passes).
template<typename K, bool DESC>
struct RadixDigit
{
  static constexpr int64_t kHistRow = (int64_t)sizeof(K) * kRadix;  // counters per range
  int shift;
  __device__ bool runs(int64_t) const { return true; }
  __device__ RadixDigit map() const { return *this; }
  __device__ __forceinline__ uint32_t operator()(K k) const { return digit_of<K, DESC>(k, shift); }
};

// ---- one onesweep pass ---------------------------------------------------------
// Workgroups are dispatched in increasing id order on each XCD and tiles are
// assigned in increasing order per XCD (see the tile mapping below), so every
// tile a block waits for is resident or done.  Keys, then
// values, go through one LDS staging buffer so a 16384-key tile (512
// threads x 32 items; 8192 keys, 16 items, when keys or values are 64-bit)
// fits in ~74 KiB, two blocks per CU, and the output is written in
// digit-contiguous runs.  The per-tile cost (barriers, digit
// scans, look-back) is paid once per 16384 keys: larger tiles measured
// faster than more resident blocks.  The keys are staged and the values
// loaded before the look-back, so both overlap its latency.
// SEG: the tiles of many ranges (one table record per tile, see
// rs::SortTile) sorted in one launch per pass.  keys_in / vals_in /
// keys_out / vals_out are then the bases of the input, output and
// alternate buffers in the order of `bases` below; a range reads the pass's
// source and writes its destination (pass 0: input -> alternate, odd
// passes: alternate -> output, even ones: output -> alternate), takes its
// digit offsets from its own histogram row and looks back only as far as
// its own first tile.
// DIG gives a key's digit and whether the block runs at all.
template<typename K, typename V, typename DIG, bool HAS_VALS, int BLOCK, int ITEMS, bool SEG = false>
__global__ __launch_bounds__(BLOCK) void onesweep_kernel(
    const K* __restrict__ keys_in, K* __restrict__ keys_out, const V* __restrict__ vals_in,
    V* __restrict__ vals_out, int64_t n, DIG dig, const uint32_t* __restrict__ hist,
    uint32_t* __restrict__ desc_cur, uint32_t* __restrict__ desc_next,
    const rs::SortTile* __restrict__ recs = nullptr, int pass = 0,
    K* __restrict__ keys_alt = nullptr, V* __restrict__ vals_alt = nullptr)
{
  static_assert(BLOCK >= kRadix && BLOCK % wave_size == 0, "one thread per digit");
  constexpr int NW = BLOCK / wave_size;
  constexpr int TILE = BLOCK * ITEMS;
  constexpr int WCHUNK = wave_size * ITEMS;
  constexpr int SLOT = (HAS_VALS && sizeof(V) > sizeof(K)) ? sizeof(V) : sizeof(K);
  __shared__ __attribute__((aligned(16))) unsigned char s_buf[TILE * SLOT];
  __shared__ uint32_t s_whist[NW * kRadix];
  __shared__ int32_t s_off[kRadix];
  __shared__ uint32_t s_tstart[kRadix];
  __shared__ uint32_t s_scan[2 * (kRadix / wave_size)];
  K* s_keys = reinterpret_cast<K*>(s_buf);
  V* s_vals = reinterpret_cast<V*>(s_buf);

  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = wave_id();
  // Tile of this block.  Blocks go to the 8 XCDs round-robin (block b to
  // XCD b % 8), and each XCD has its own L2.  Mapping 32 consecutive tiles of
  // every group of 256 to one XCD lets that L2 merge the adjacent digit runs
  // of neighbouring tiles (tile t's run of digit d ends where tile t+1's
  // begins) before they reach HBM: one pass over 2^28 pairs took 1.276 ms
  // with tile = block, 0.997 ms with 8 per group of 64 and 0.985 ms with 32
  // per group of 256.  Each XCD dispatches its blocks in order and receives
  // its tiles in increasing order, so every block before the lowest
  // unfinished tile's block on that XCD is finished and that block is placed
  // as soon as the XCD has room (lookback launches run one at a time per
  // device, rc::LookbackGate); the last, partial group keeps tile = block.
  const int64_t tile = [] {
    constexpr int64_t KX = 32, GX = 8 * KX;
    const int64_t b = blockIdx.x, g = b / GX;
    if ((g + 1) * GX > (int64_t)gridDim.x) return b;
    const int64_t r = b - g * GX;
    return g * GX + (r & 7) * KX + (r >> 3);
  }();
  if (!dig.runs(tile)) return;  // the same for the whole block
  const auto digit = dig.map();
  for (int i = tid; i < NW * kRadix; i += BLOCK) s_whist[i] = 0u;
  int64_t tj = tile;     // tile index inside its range
  int64_t tfirst = 0;    // descriptor row of the range's first tile
  if constexpr (SEG)
  {
    const rs::SortTile r = recs[tile];
    tj = r.j;
    tfirst = tile - r.j;
    n = r.len;
    hist += (int64_t)r.seg * DIG::kHistRow;
    const K* ks = pass == 0 ? keys_in + r.ik : ((pass & 1) ? keys_alt + r.ak : keys_out + r.ok);
    K* kd = (pass & 1) ? keys_out + r.ok : keys_alt + r.ak;
    keys_in = ks;
    keys_out = kd;
    if (HAS_VALS)
    {
      const V* vs = pass == 0 ? vals_in + r.iv : ((pass & 1) ? vals_alt + r.av : vals_out + r.ov);
      V* vd = (pass & 1) ? vals_out + r.ov : vals_alt + r.av;
      vals_in = vs;
      vals_out = vd;
    }
  }
  const int64_t tbase = tj * TILE;
  const int64_t wbase = tbase + (int64_t)wave * WCHUNK;

  // Item j of this lane is element wbase + j*64 + lane; the wave holds
  // wvalid valid elements (32-bit compares below, no 64-bit indices kept).
  const int64_t wrem = n - wbase;
  const int wvalid = wrem <= 0 ? 0 : (wrem >= WCHUNK ? WCHUNK : (int)wrem);

  K k[ITEMS];
  const bool full = tbase + TILE <= n;
  if (full)
  {
    const K* kp = keys_in + wbase;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) k[j] = kp[j * wave_size + lane];
  }
  else
  {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      const int q = j * wave_size + lane;
      k[j] = (q < wvalid) ? keys_in[wbase + q] : K(0);
    }
  }
  for (int i = tid; i < kRowStride; i += BLOCK) desc_next[tile * kRowStride + i] = 0u;  // next pass
  __syncthreads();

  // Wave-local ranks: rank = digit count so far in this wave + lower peers.
  uint32_t rank[ITEMS];
  auto rank_items = [&](auto full_c) {
    constexpr bool FULL = decltype(full_c)::value;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      const bool valid = FULL || j * wave_size + lane < wvalid;
      const uint32_t d = digit(k[j]);
      // Peers: the valid lanes whose digit equals this lane's, bit by bit.
      // sx is 0 or all ones (the bit sign-extended); lane m agrees with this
      // lane on the bit where ~(ballot ^ sx) has bit m set, so
      // p = p & ~(ballot ^ sx), one v_bitop3 per half, keeps the lanes that
      // agree on every bit.  A full tile starts from all lanes, a partial
      // one from the valid lanes.
      uint32_t pl = ~0u, ph = ~0u;
      if constexpr (!FULL)
      {
        const uint64_t vb = ballot(valid);
        pl = (uint32_t)vb;
        ph = (uint32_t)(vb >> 32);
      }
#pragma unroll
      for (int b = 0; b < 8; ++b)
      {
        int32_t sx = __builtin_amdgcn_sbfe((int32_t)d, b, 1);
        asm volatile("" : "+v"(sx));  // keep the one-instruction extract
        const uint64_t bal = ballot(sx != 0);
        pl = __builtin_amdgcn_bitop3_b32(pl, (uint32_t)bal, (uint32_t)sx, 0x90);
        ph = __builtin_amdgcn_bitop3_b32(ph, (uint32_t)(bal >> 32), (uint32_t)sx, 0x90);
      }
      // Peers in lower lanes: v_mbcnt counts the mask's bits below this lane.
      const uint32_t lower = __builtin_amdgcn_mbcnt_hi(ph, __builtin_amdgcn_mbcnt_lo(pl, 0u));
      uint32_t cnt = 0;
      if (valid) cnt = s_whist[wave * kRadix + d];
      rank[j] = (cnt + lower) | (d << 16);  // digit kept beside the rank
      asm volatile("" : "+v"(rank[j]));  // one register per item from here on
      if (valid && lower == 0)
      {
        s_whist[wave * kRadix + d] = cnt + (uint32_t)__builtin_popcount(pl) + (uint32_t)__builtin_popcount(ph);
      }
      __builtin_amdgcn_sched_barrier(0);  // rank one item at a time: few live masks
    }
  };
  if (full)
    rank_items(std::true_type{});
  else
    rank_items(std::false_type{});
  __syncthreads();

  // Per digit (thread = digit): wave offsets, tile count, publication and
  // digit scans.
  uint32_t ex_t = 0, ex_g = 0, prefix = 0, total = 0;
  uint32_t* const row = desc_cur + tile * kRowStride;
  if (tid < kRadix)
  {
    const int d = tid;
#pragma unroll
    for (int w = 0; w < NW; ++w)
    {
      const uint32_t c = s_whist[w * kRadix + d];
      s_whist[w * kRadix + d] = total;
      total += c;
    }
    atomic_store_agent(&row[d], ((tj == 0 ? kInc : kAgg) << 30) | total);
    const uint32_t gcount = hist[d];
    uint32_t tot_t, tot_g;
    (void)wave_scan(total, rk::OpPlus<uint32_t>{}, 0u, ex_t, tot_t);
    (void)wave_scan(gcount, rk::OpPlus<uint32_t>{}, 0u, ex_g, tot_g);
    if (lane == 0)
    {
      s_scan[wave] = tot_t;
      s_scan[kRadix / wave_size + wave] = tot_g;
    }
  }
  __syncthreads();
  uint32_t tstart = 0, gstart = 0;
  if (tid < kRadix)
  {
    tstart = ex_t;
    gstart = ex_g;
    for (int w = 0; w < wave; ++w)
    {
      tstart += s_scan[w];
      gstart += s_scan[kRadix / wave_size + w];
    }
    s_tstart[tid] = tstart;
  }
  __syncthreads();

  // Keys: stage in LDS in digit order (tile-local offsets only), before the
  // look-back, so the keys' registers are free while it runs.
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
  {
    if (j * wave_size + lane < wvalid)
    {
      const uint32_t dj = rank[j] >> 16;
      rank[j] = (rank[j] & 0xFFFFu) + s_tstart[dj] + s_whist[wave * kRadix + dj];  // tile position
      s_keys[rank[j]] = k[j];
    }
  }
  // Values are loaded now: their latency overlaps the look-back.
  V v[HAS_VALS ? ITEMS : 1];
  if (HAS_VALS)
  {
    if (full)
    {
      const V* vp = vals_in + wbase;
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) v[j] = vp[j * wave_size + lane];
    }
    else
    {
#pragma unroll
      for (int j = 0; j < ITEMS; ++j)
      {
        const int q = j * wave_size + lane;
        v[j] = (q < wvalid) ? vals_in[wbase + q] : V(0);
      }
    }
  }
  if (tj > 0)
  {
    if (tid < kRadix)
    {
      // Descriptors tile-1, tile-2, ... are read kLookbackRows at a time
      // with all loads in flight; the fold stops at the first inclusive
      // count.  A descriptor not yet published is re-read.
      const int d = tid;
      bool done = false;
      SpinBound bound;
      for (int64_t t0 = tile - 1; !done; t0 -= kLookbackRows)
      {
        uint32_t w[kLookbackRows];
#pragma unroll
        for (int u = 0; u < kLookbackRows; ++u)
        {
          const int64_t t = t0 - u;
          w[u] = (t >= tfirst) ? atomic_load_agent(&desc_cur[t * kRowStride + d]) : (kInc << 30);
        }
#pragma unroll
        for (int u = 0; u < kLookbackRows; ++u)
        {
          if (done) break;
          const int64_t t = t0 - u;
          if (t < tfirst)
          {
            done = true;
            break;
          }
          while ((w[u] >> 30) == 0u)
          {
            __builtin_amdgcn_s_sleep(1);
            w[u] = atomic_load_agent(&desc_cur[t * kRowStride + d]);
            if ((w[u] >> 30) == 0u && bound.expired())
            {
              atomicAdd(&g_spin_timeouts, 1u);
              w[u] = kInc << 30;  // give up on it: the result is reported invalid
            }
          }
          prefix += w[u] & kCountMask;
          if ((w[u] >> 30) == kInc) done = true;
        }
      }
      atomic_store_agent(&row[d], (kInc << 30) | (prefix + total));
    }
  }
  if (tid < kRadix) s_off[tid] = (int32_t)(gstart + prefix) - (int32_t)tstart;
  __syncthreads();
  const int64_t rem = n - tbase;
  const int tile_n = (rem < TILE) ? (int)rem : TILE;
  // Digits of the tile positions this thread writes, four per register: the
  // value pass writes the same positions after the keys' LDS is reused.
  uint32_t dpk[HAS_VALS ? (ITEMS + 3) / 4 : 1];
#pragma unroll
  for (int q = 0; q < (HAS_VALS ? (ITEMS + 3) / 4 : 1); ++q) dpk[q] = 0u;
  // Groups of G positions: the LDS reads of a group are issued together
  // (positions past tile_n read stale LDS inside the buffer and are not
  // written), then the offsets, then the stores.  Full tiles skip the
  // position test.  Destinations are < n < 2^30 for consistent histograms;
  // an inconsistent one must not write out of range: 4-byte elements are
  // stored through a buffer resource of n elements, whose range check drops
  // a store at or past the end (no compare or branch per store), wider ones
  // test the index.
  constexpr int G = 8;
  static_assert(ITEMS % G == 0, "scatter groups");
  const uint32_t n32 = (uint32_t)n;
  const bool full_tile = tile_n == TILE;
  const __amdgpu_buffer_rsrc_t keys_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(keys_out, (short)0, (int)(n32 * 4u), kBufferWord3);
  const __amdgpu_buffer_rsrc_t vals_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(vals_out, (short)0, (int)(n32 * 4u), kBufferWord3);
  auto scatter_keys = [&](auto full_c) {
    constexpr bool FULL = decltype(full_c)::value;
#pragma unroll
    for (int m0 = 0; m0 < ITEMS; m0 += G)
    {
      K key[G];
      uint32_t dg[G];
      int32_t off[G];
#pragma unroll
      for (int g = 0; g < G; ++g) key[g] = s_keys[tid + (m0 + g) * BLOCK];
#pragma unroll
      for (int g = 0; g < G; ++g)
      {
        dg[g] = digit(key[g]);
        off[g] = s_off[dg[g]];
      }
#pragma unroll
      for (int g = 0; g < G; ++g)
      {
        const int m = m0 + g;
        const int i = tid + m * BLOCK;
        const uint32_t d = (uint32_t)(off[g] + i);
        if constexpr (sizeof(K) == 4)
        {
          if (FULL || i < tile_n)
          {
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, key[g]), keys_rsrc, (int)(d << 2), 0, 0);
          }
        }
        else if ((FULL || i < tile_n) && d < n32)
        {
          keys_out[d] = key[g];
        }
        if (HAS_VALS) dpk[m >> 2] |= dg[g] << (8 * (m & 3));
      }
      __builtin_amdgcn_sched_barrier(0);  // one group in flight: bounded registers
    }
  };
  if (full_tile)
    scatter_keys(std::true_type{});
  else
    scatter_keys(std::false_type{});
  if (HAS_VALS)
  {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
      if (j * wave_size + lane < wvalid) s_vals[rank[j]] = v[j];
    }
    __syncthreads();
    auto scatter_vals = [&](auto full_c) {
      constexpr bool FULL = decltype(full_c)::value;
#pragma unroll
      for (int m0 = 0; m0 < ITEMS; m0 += G)
      {
        V val[G];
        int32_t off[G];
#pragma unroll
        for (int g = 0; g < G; ++g)
        {
          const int m = m0 + g;
          val[g] = s_vals[tid + m * BLOCK];
          off[g] = s_off[(dpk[m >> 2] >> (8 * (m & 3))) & 0xFFu];
        }
#pragma unroll
        for (int g = 0; g < G; ++g)
        {
          const int i = tid + (m0 + g) * BLOCK;
          const uint32_t d = (uint32_t)(off[g] + i);
          if constexpr (sizeof(V) == 4)
          {
            if (FULL || i < tile_n)
            {
              __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, val[g]), vals_rsrc, (int)(d << 2), 0, 0);
            }
          }
          else if ((FULL || i < tile_n) && d < n32)
          {
            vals_out[d] = val[g];
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (full_tile)
      scatter_vals(std::true_type{});
    else
      scatter_vals(std::false_type{});
  }
}

template<typename K, typename V, bool HAS_VALS>
struct SortShape
{
  static constexpr bool wide = sizeof(K) > 4 || (HAS_VALS && sizeof(V) > 4);
  static constexpr int BLOCK = 512;
  static constexpr int ITEMS = wide ? 16 : 32;  // 8192 / 16384 keys per tile
  static constexpr int64_t TILE = (int64_t)BLOCK * ITEMS;
  // Keys per thread that may be chosen instead (by the tuner for 4-byte keys
  // and values, by length otherwise; 0 is the default): smaller tiles give
  // mid-sized sorts enough blocks to fill the chip.
  static constexpr int kChoices[3] = {0, wide ? 8 : 16, wide ? 0 : 8};
  static int64_t tile(int items) { return (int64_t)BLOCK * (items > 0 ? items : ITEMS); }
};

}  // namespace
