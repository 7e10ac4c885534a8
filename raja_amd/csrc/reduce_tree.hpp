// The canonical reduction tree shared by the span reductions and the
// segmented (batched) reductions.
//
// A range of n elements is cut into tiles from its start, a tile into 4
// quads, a quad into 4 wave tiles of 16 16-byte vectors per lane (16 KiB:
// 2048 FP64 or 4096 4-byte elements).
//   wave tile : wave tile w of a quad is every fourth row of 64 vectors, rows
//               w, w+4, ... (a block that folds a quad reads whole rows of 4
//               KiB; 16 KiB runs per wave measured 4 % slower over 2^28 FP64);
//               lane t folds vector t of each row, row k into accumulator
//               k % 4, the accumulators pairwise, then the DPP wave tree;
//   quad      : (w0, w1), (w2, w3) of its wave tiles;
//   tile      : (q0, q1), (q2, q3) of its quads (wide accumulators: one quad);
//   range     : a 64-ary tree over the tile values -- each level folds
//               groups of 64 consecutive values (identity-padded) with the
//               DPP wave tree -- then op(init, value).
// The tree is a function of n alone: any grid, any number of waves working
// on the tile values, and any batch the range is part of give the same
// bits.  A range reduced by the span entry point and the same range as one
// segment of a batch agree exactly.
//
// The small unit is there so that short and mid-sized ranges fill the chip:
// a long span gives a block a whole tile (256 KiB, no barrier until its end),
// a shorter one a block per quad, a short segment one wave.
#pragma once

#include "ops.hpp"
#include "runtime.hpp"

namespace rt
{
using namespace RAJA::cdna4::dev;

constexpr int kBlock = 256;
constexpr int kBlockWaves = kBlock / wave_size;

// 16-byte loads a thread keeps in flight: fewer for operators whose
// accumulators are wide (8 for MinLoc/MaxLoc, 4 for the fused
// Sum/Min/Max/MinLoc), so the kernel keeps enough waves resident.  Element
// -> accumulator assignment (vector k goes to accumulator k % 4, in
// increasing k) does not depend on it, so neither do the result bits.
template<typename Op>
struct LoadsInFlight
{
  static constexpr int value =
      sizeof(typename Op::acc_t) > 24 ? 4 : (sizeof(typename Op::acc_t) > 8 ? 8 : 16);
};

template<typename T>
struct VecOf
{
  static constexpr int n = 16 / sizeof(T);
  typedef T type __attribute__((ext_vector_type(16 / sizeof(T))));
  // The same 16 bytes at the element's own alignment (a segment starts at
  // any element); 16-byte global accesses need only 4-byte alignment on CDNA.
  typedef T utype __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
};

// Accumulators wider than 8 bytes (value/index pairs, the fused four): a wave
// fold of 48 bytes takes about 0.8 us, so their wave tiles are 4 times as long
// (and a tile is one quad: the same 256 KiB).
template<typename Op>
constexpr bool kWide = sizeof(typename Op::acc_t) > 8;

template<typename Op>
constexpr int kVecPerLane = kWide<Op> ? 64 : 16;  // 16-byte vectors per lane per wave tile

template<typename T, typename Op>
constexpr int64_t wave_tile_elems()
{
  return (int64_t)wave_size * kVecPerLane<Op> * VecOf<T>::n;
}
template<typename T, typename Op>
constexpr int64_t quad_elems()
{
  return 4 * wave_tile_elems<T, Op>();
}
template<typename T, typename Op>
constexpr int64_t tile_elems()
{
  return (kWide<Op> ? 1 : 4) * quad_elems<T, Op>();
}

// acc <- op(acc, lift(x_i, i)); operators whose accumulators are wide give a
// cheaper accumulate() that is exact for elements met in increasing index
// order, which is how each accumulator meets them.
template<typename Op, typename T>
__device__ __forceinline__ auto accumulate_one(typename Op::acc_t& a, T v, int64_t i, int)
    -> decltype(Op::accumulate(a, v, i), void())
{
  Op::accumulate(a, v, i);
}
template<typename Op, typename T>
__device__ __forceinline__ void accumulate_one(typename Op::acc_t& a, T v, int64_t i, long)
{
  a = Op{}(a, Op::lift(v, i));
}

// Row loads of a range whose end lies inside: `nv` whole vectors from `x`, row
// r holding vectors 64r .. 64r+63.  Lanes past the last whole vector load that
// one again (their value is not used), rows past it load nothing, so every
// load is the same unguarded 16-byte one as in the middle of a range (a
// guarded element path for the partial quads cost a batch of 20,000 uneven
// segments 8 %).
template<typename T>
__device__ __forceinline__ typename VecOf<T>::type load_row(const T* __restrict__ x, int nv, int row)
{
  using uvec_t = typename VecOf<T>::utype;
  const int q = row * wave_size + lane_id();
  return __builtin_nontemporal_load(reinterpret_cast<const uvec_t*>(x + (q < nv ? q : nv - 1) * VecOf<T>::n));
}

// This lane's part of wave tile w of the quad that starts at element `base` of
// the range x[0..n) (the identity past its end); the wave tile's value is the
// wave tree over the lanes' parts.  The element -> (lane,
// accumulator) assignment does not depend on the alignment of x: loads are 16
// bytes at the element's alignment, nontemporal as each is read once (2^28
// FP64 sum 0.363 -> 0.316 ms).
template<typename T, typename Op>
__device__ __forceinline__ typename Op::acc_t fold_lane(const T* __restrict__ x, int64_t n,
                                                        int64_t base, int w)
{
  using acc_t = typename Op::acc_t;
  using vec_t = typename VecOf<T>::type;
  using uvec_t = typename VecOf<T>::utype;
  constexpr int VEC = VecOf<T>::n;
  constexpr int kVecPerChunk = LoadsInFlight<Op>::value;
  constexpr int kChunks = kVecPerLane<Op> / kVecPerChunk;
  static_assert(kVecPerChunk % 4 == 0 && kVecPerLane<Op> % kVecPerChunk == 0, "chunking keeps k % 4");
  const Op op{};
  const int t = w * wave_size + lane_id();
  acc_t acc[4] = {Op::ident(), Op::ident(), Op::ident(), Op::ident()};
  if (base + quad_elems<T, Op>() <= n)
  {
#pragma unroll 1
    for (int c = 0; c < kChunks; ++c)
    {
      vec_t v[kVecPerChunk];
#pragma unroll
      for (int j = 0; j < kVecPerChunk; ++j)
      {
        const int k = c * kVecPerChunk + j;
        v[j] = __builtin_nontemporal_load(reinterpret_cast<const uvec_t*>(x + base + ((int64_t)k * kBlock + t) * VEC));
      }
#pragma unroll
      for (int j = 0; j < kVecPerChunk; ++j)
      {
        const int k = c * kVecPerChunk + j;
        const int64_t i0 = base + ((int64_t)k * kBlock + t) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e)
        {
          accumulate_one<Op>(acc[j & 3], v[j][e], i0 + e, 0);
        }
      }
    }
  }
  else if (base < n)
  {
    // Partial quad: the same rows and order up to the last whole vector.
    const int rem = __builtin_amdgcn_readfirstlane((int)(n - base));
    const int nv = rem / VEC;
#pragma unroll 1
    for (int c = 0; c < kChunks; ++c)
    {
      if ((c * kVecPerChunk * kBlockWaves + w) * wave_size >= nv) break;
      vec_t v[kVecPerChunk];
#pragma unroll
      for (int j = 0; j < kVecPerChunk; ++j)
      {
        const int row = (c * kVecPerChunk + j) * kBlockWaves + w;
        if (row * wave_size < nv) v[j] = load_row<T>(x + base, nv, row);
      }
#pragma unroll
      for (int j = 0; j < kVecPerChunk; ++j)
      {
        const int row = (c * kVecPerChunk + j) * kBlockWaves + w;
        if (row * wave_size + lane_id() < nv)
        {
          const int64_t i0 = base + (int64_t)(row * wave_size + lane_id()) * VEC;
#pragma unroll
          for (int e = 0; e < VEC; ++e) accumulate_one<Op>(acc[j & 3], v[j][e], i0 + e, 0);
        }
      }
    }
    // The elements after the last whole vector belong to its successor's
    // lane, which has no later row.
    if (nv % kBlock == t)
    {
      const int k = nv / kBlock;
      for (int e = nv * VEC; e < rem; ++e)
      {
        const T v = x[base + e];
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
          if ((k & 3) == j) accumulate_one<Op>(acc[j], v, base + e, 0);
        }
      }
    }
  }
  return op(op(acc[0], acc[1]), op(acc[2], acc[3]));
}

// Fold of 4 values in the order of quads and tiles.
template<typename Op>
__device__ __forceinline__ typename Op::acc_t fold4(const typename Op::acc_t& a,
                                                    const typename Op::acc_t& b,
                                                    const typename Op::acc_t& c,
                                                    const typename Op::acc_t& d)
{
  const Op op{};
  return op(op(a, b), op(c, d));
}

// Elements of the first 16 rows of a quad.
template<typename T, typename Op>
constexpr int64_t short_elems()
{
  return (int64_t)16 * wave_size * VecOf<T>::n;
}

// Value of a range of at most short_elems() elements, by one wave, in every
// lane: row r is row r/4 of wave tile r % 4, so each accumulator of each wave
// tile meets at most one row, and all loads are in flight at once.
template<typename T, typename Op>
__device__ __forceinline__ typename Op::acc_t fold_short(const T* __restrict__ x, int64_t n)
{
  using acc_t = typename Op::acc_t;
  using vec_t = typename VecOf<T>::type;
  constexpr int VEC = VecOf<T>::n;
  const Op op{};
  const acc_t id = Op::ident();
  const int m = __builtin_amdgcn_readfirstlane((int)n);
  const int nv = m / VEC;
  vec_t v[16];
#pragma unroll
  for (int r = 0; r < 16; ++r)
  {
    if (r * wave_size < nv) v[r] = load_row<T>(x, nv, r);
  }
  // the elements after the last whole vector, by its successor's lane
  T tail[VEC];
#pragma unroll
  for (int e = 0; e < VEC - 1; ++e)
  {
    tail[e] = (nv % wave_size == lane_id() && nv * VEC + e < m) ? x[nv * VEC + e] : T(0);
  }
  acc_t w[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
  {
    acc_t acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
      const int r = 4 * j + q;
      const int i0 = (r * wave_size + lane_id()) * VEC;
      acc[j] = id;
      if (i0 + VEC <= m)
      {
#pragma unroll
        for (int e = 0; e < VEC; ++e) accumulate_one<Op>(acc[j], v[r][e], i0 + e, 0);
      }
      else
      {
#pragma unroll
        for (int e = 0; e < VEC - 1; ++e)
        {
          if (i0 + e < m) accumulate_one<Op>(acc[j], tail[e], i0 + e, 0);
        }
      }
    }
    w[q] = wave_reduce(op(op(acc[0], acc[1]), op(acc[2], acc[3])), op);
  }
  return fold4<Op>(fold4<Op>(w[0], w[1], w[2], w[3]), id, id, id);
}

// Value of quad `quad` of x[0..n) by a block of 4 waves, in every thread.
template<typename T, typename Op>
__device__ __forceinline__ typename Op::acc_t fold_quad(const T* __restrict__ x, int64_t n, int64_t quad,
                                                        typename Op::acc_t* s_w)
{
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const typename Op::acc_t v =
      wave_reduce(fold_lane<T, Op>(x, n, quad * quad_elems<T, Op>(), wave), Op{});
  if (lane_id() == 0) s_w[wave] = v;
  __syncthreads();
  return fold4<Op>(s_w[0], s_w[1], s_w[2], s_w[3]);
}

// Tile value of its 16 wave tile values, by one wave: rows of 16 lanes, whose
// butterfly is the order of quads and tiles.
template<typename Op>
__device__ __forceinline__ typename Op::acc_t fold16(const typename Op::acc_t* s_w)
{
  const Op op{};
  typename Op::acc_t v = s_w[lane_id() & 15];
  v = op(v, dpp_move<dpp_quad_1032>(v, v));
  v = op(v, dpp_move<dpp_quad_2301>(v, v));
  v = op(v, dpp_move<dpp_row_half_mirror>(v, v));
  v = op(v, dpp_move<dpp_row_mirror>(v, v));
  return v;
}

// Value of tile `tile` of x[0..n) by a block of 4 waves, in the first wave.
// A wave folds 4 wave tiles (one per quad) before the block's only barrier.
template<typename T, typename Op>
__device__ __forceinline__ typename Op::acc_t fold_tile(const T* __restrict__ x, int64_t n, int64_t tile,
                                                        typename Op::acc_t* s_w)
{
  using acc_t = typename Op::acc_t;
  const Op op{};
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  acc_t v[4];  // the wave trees run together at the end
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = fold_lane<T, Op>(x, n, (tile * 4 + q) * quad_elems<T, Op>(), wave);
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = wave_reduce(v[q], op);
  if (lane_id() == 0)
  {
#pragma unroll
    for (int q = 0; q < 4; ++q) s_w[q * kBlockWaves + wave] = v[q];
  }
  __syncthreads();
  return wave == 0 ? fold16<Op>(s_w) : Op::ident();
}

// Where a reduction's result goes: slot i of an array, and for value/index
// pairs the caller's separate value and index.
template<typename Op>
struct ResultOut
{
  typename Op::acc_t* p;
  __device__ void put(int64_t i, const typename Op::acc_t& v) const { p[i] = v; }
};
template<typename T>
struct LocOut
{
  T* val;
  int64_t* loc;
  __device__ void put(int64_t, const rk::ValLoc<T>& v) const
  {
    *val = v.val;
    *loc = v.loc;
  }
};
template<typename T>
struct ResultOut<rk::OpMinLoc<T>> : LocOut<T>
{};
template<typename T>
struct ResultOut<rk::OpMaxLoc<T>> : LocOut<T>
{};

// Value of tile i of `nquads` quad values (the identity past their end).
template<typename Op>
__device__ __forceinline__ typename Op::acc_t tile_of_quads(const typename Op::acc_t* quads,
                                                            int64_t nquads, int64_t i)
{
  typename Op::acc_t q[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) q[u] = (4 * i + u < nquads) ? quads[4 * i + u] : Op::ident();
  return fold4<Op>(q[0], q[1], q[2], q[3]);
}

// 64-ary tree over `count` tile values, evaluated by the block's waves
// (blockDim.x = 64 * waves).  QUADS: vals are quad values, each tile's 4
// folded as they are read.  s_a holds >= ceil(tiles/64) values, s_b >=
// ceil(tiles/4096) values.  Returns the range value in every thread.
template<typename Op, bool QUADS>
__device__ __forceinline__ typename Op::acc_t tree_fold(const typename Op::acc_t* vals,
                                                        int64_t count,
                                                        typename Op::acc_t* s_a,
                                                        typename Op::acc_t* s_b)
{
  using acc_t = typename Op::acc_t;
  const Op op{};
  const int lane = lane_id();
  const int wave = wave_id();
  const int nw = (int)(blockDim.x / wave_size);
  if (count <= 0) return Op::ident();
  const acc_t* in = vals;
  acc_t* outs[2] = {s_a, s_b};
  int level = 0;
  const int64_t nquads = count;
  if (QUADS) count = (count + 3) / 4;
  while (count > 1 || (QUADS && level == 0))
  {
    const int64_t groups = (count + wave_size - 1) / wave_size;
    acc_t* out = outs[level & 1];
    for (int64_t g = wave; g < groups; g += nw)
    {
      const int64_t i = g * wave_size + lane;
      acc_t v = Op::ident();
      if (QUADS && level == 0)
      {
        v = tile_of_quads<Op>(in, nquads, i);
      }
      else if (i < count)
      {
        v = in[i];
      }
      const acc_t r = wave_reduce(v, op);
      if (lane == 0) out[g] = r;
    }
    __syncthreads();
    in = out;
    count = groups;
    ++level;
  }
  const acc_t r = in[0];
  __syncthreads();
  return r;
}

// A span of at most one quad (WAVES 4) or tile (WAVES 16) in one launch of
// one block, a wave tile per wave: its value and the init.
template<typename T, typename Op, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void short_kernel(const T* __restrict__ x, int64_t n,
                                                           typename Op::acc_t init, ResultOut<Op> out)
{
  using acc_t = typename Op::acc_t;
  __shared__ acc_t s_w[16];
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const acc_t v =
      wave_reduce(fold_lane<T, Op>(x, n, (wave / 4) * quad_elems<T, Op>(), wave % 4), Op{});
  if (lane_id() == 0) s_w[wave] = v;
  if (WAVES < 16 && threadIdx.x >= (unsigned)WAVES && threadIdx.x < 16) s_w[threadIdx.x] = Op::ident();
  __syncthreads();
  if (wave != 0) return;
  const acc_t r = fold16<Op>(s_w);
  if (threadIdx.x == 0) out.put(0, Op::with_init(init, r));
}

// Kernel 1 of a mid-sized span: quad values, one block each.
template<typename T, typename Op>
__global__ __launch_bounds__(kBlock) void quads_kernel(const T* __restrict__ x, int64_t n,
                                                       typename Op::acc_t* __restrict__ partials)
{
  using acc_t = typename Op::acc_t;
  __shared__ acc_t s_w[kBlockWaves];
  const acc_t v = fold_quad<T, Op>(x, n, blockIdx.x, s_w);
  if (threadIdx.x == 0) partials[blockIdx.x] = v;
}

// Kernel 1 of a long span: tile values, grid-stride.
template<typename T, typename Op>
__global__ __launch_bounds__(kBlock) void tiles_kernel(const T* __restrict__ x, int64_t n,
                                                       int64_t ntiles,
                                                       typename Op::acc_t* __restrict__ partials)
{
  using acc_t = typename Op::acc_t;
  __shared__ acc_t s_w[2][16];
  int buf = 0;  // one barrier per tile: the next tile writes the other buffer
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x)
  {
    const acc_t v = fold_tile<T, Op>(x, n, tile, s_w[buf]);
    if (threadIdx.x == 0) partials[tile] = v;
    buf ^= 1;
  }
}

// First level of the 64-ary tree on its own (one 64-lane block per group of
// 64 tile values): group g's value is the wave fold of values 64g..64g+63,
// exactly as tree_fold's first level computes it, so folding the group
// values with tree_fold gives the bits of folding the tile values.  Used
// for wide accumulators, whose wave fold is too slow to run group after
// group in one block.
template<typename Op>
__global__ __launch_bounds__(64) void group_kernel(const typename Op::acc_t* __restrict__ in,
                                                   int64_t count,
                                                   typename Op::acc_t* __restrict__ out)
{
  const int64_t i = (int64_t)blockIdx.x * wave_size + threadIdx.x;
  const typename Op::acc_t v = (i < count) ? in[i] : Op::ident();
  const typename Op::acc_t r = wave_reduce(v, Op{});
  if (threadIdx.x == 0) out[blockIdx.x] = r;
}

// Kernel 2: the 64-ary tree over the tile (QUADS: quad) values of each
// segment (one block per segment; a span reduction is one segment) and the
// init; segment s's result goes to out[out_index[s]] (out[s] without an index).
template<typename Op, int WAVES, int MAX_GROUPS, bool QUADS>
__global__ __launch_bounds__(WAVES * 64) void final_kernel(
    const typename Op::acc_t* __restrict__ partials, const uint32_t* __restrict__ seg_first,
    const uint32_t* __restrict__ seg_count, int64_t single_count, typename Op::acc_t init,
    ResultOut<Op> out, const int64_t* __restrict__ out_index)
{
  using acc_t = typename Op::acc_t;
  __shared__ acc_t s_a[MAX_GROUPS];
  __shared__ acc_t s_b[(MAX_GROUPS + 63) / 64 + 1];
  const int64_t seg = blockIdx.x;
  const int64_t first = seg_first ? seg_first[seg] : 0;
  const int64_t count = seg_count ? seg_count[seg] : single_count;
  const acc_t r = tree_fold<Op, QUADS>(partials + first, count, s_a, s_b);
  if (threadIdx.x == 0) out.put(out_index ? out_index[seg] : seg, Op::with_init(init, r));
}

}  // namespace rt
