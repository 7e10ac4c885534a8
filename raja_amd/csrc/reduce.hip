// Deterministic span reductions (ReduceSum/Min/Max/BitOr/BitAnd,
// MinLoc/MaxLoc and the fused Sum+Min+Max+MinLoc of one forall).
//
// Reference: the HIP reducers fold per-thread values with a shuffle tree,
// per-block slots and a last-block-done pass, replicated 32 ways and folded
// again on the host (include/RAJA/policy/hip/reduce.hpp:127-208, 960-1161).
// Here a span of at most one tile (256 KiB) is one launch of one block; longer
// ones take two: kernel 1 computes the value of every fixed quad (mid-sized
// spans) or tile (long ones) and kernel 2 folds them with the canonical
// 64-ary tree and applies the caller's init (reduce_tree.hpp).  The combine tree depends only on n
// -- not on the grid, the timing or whatever else shares the GPU -- and no
// floating-point atomics are used.  Two kernels instead of a
// last-block-done pass: on MI355X a release fence at device scope writes
// back the whole L2 of the block's XCD, and a same-address device atomic per
// block serialises across the 8 XCDs; the kernel boundary gives the
// visibility for free.
#include "reduce_tree.hpp"
#include "workspace.hpp"

namespace
{
using namespace RAJA::cdna4::dev;

constexpr int kFinalWaves = 16;
constexpr int kFinalMaxGroups = 1024;  // groups of 64 tiles one final block folds
// Longest span: 65536 units of 256 KiB.
template<typename T>
constexpr int64_t max_span()
{
  return (int64_t)65536 * ((256 << 10) / (int64_t)sizeof(T));
}

// How a span runs, by its length:
//   kShort : at most one tile: one block, one launch;
//   kQuads : a block per quad, the quad values folded by one final block;
//   kGroups: the same with a kernel that folds 64 values per wave in between,
//            for wide accumulators (one block folding 8192 values of the fused
//            Sum/Min/Max/MinLoc, 2^28 FP64, takes 20 us, the two kernels 10);
//   kTiles : a block per 4 quads (a tile), for long spans of narrow ones.
// Times per call, FP64 sum, before (a block per tile always, two launches) and
// now: n = 1000 6.4 -> 3.4 us, 2^15 5.9 -> 3.2, 2^20 6.6 -> 5.8, 2^22 7.6 ->
// 6.7; at 256 tiles (2^23) a block per quad takes 12.4 us against 12.1, at 1024
// (2^25) 43 against 41, so spans from there on run a block per tile as before
// (2^28: 306 us).
enum class Shape
{
  kShort,
  kQuads,
  kGroups,
  kTiles
};
constexpr int64_t kQuadTiles = 128;

template<typename T, typename Op>
Shape shape_of(int64_t n)
{
  if (n <= rt::tile_elems<T, Op>()) return Shape::kShort;
  const int64_t ntiles = rc::ceil_div(n, rt::tile_elems<T, Op>());
  if (rt::kWide<Op>) return ntiles <= kFinalWaves * 64 ? Shape::kQuads : Shape::kGroups;
  return ntiles <= kQuadTiles ? Shape::kQuads : Shape::kTiles;
}

// Values the partials buffer holds.
template<typename T, typename Op>
int64_t partial_slots(int64_t n)
{
  const int64_t ntiles = rc::ceil_div(n, rt::tile_elems<T, Op>());
  switch (shape_of<T, Op>(n))
  {
    case Shape::kShort: return 1;
    case Shape::kQuads: return rc::ceil_div(n, rt::quad_elems<T, Op>());
    case Shape::kGroups: return ntiles + rc::ceil_div(ntiles, (int64_t)64);
    default: return ntiles;
  }
}

template<typename Op, bool QUADS>
void launch_final(const typename Op::acc_t* vals, int64_t count, typename Op::acc_t init,
                  rt::ResultOut<Op> out, hipStream_t s)
{
  const uint32_t* const none = nullptr;
  if (count <= (QUADS ? 4 * 64 : 64))
  {
    hipLaunchKernelGGL((rt::final_kernel<Op, 1, 1, QUADS>), dim3(1), dim3(64), 0, s, vals, none, none,
                       count, init, out, (const int64_t*)nullptr);
  }
  else
  {
    hipLaunchKernelGGL((rt::final_kernel<Op, kFinalWaves, kFinalMaxGroups, QUADS>), dim3(1),
                       dim3(kFinalWaves * 64), 0, s, vals, none, none, count, init, out,
                       (const int64_t*)nullptr);
  }
}

// The kernels over caller-provided partials (partial_slots values).
template<typename T, typename Op>
int launch_reduce_core(const T* x, int64_t n, typename Op::acc_t init, rt::ResultOut<Op> out,
                       typename Op::acc_t* partials, hipStream_t s, const char* name)
{
  rc::TimedScope ts(name, s);
  const Shape shape = shape_of<T, Op>(n);
  const int64_t ntiles = rc::ceil_div(n, rt::tile_elems<T, Op>());
  const int64_t nquads = rc::ceil_div(n, rt::quad_elems<T, Op>());
  if (shape == Shape::kShort)
  {
    if (nquads <= 1)
    {
      hipLaunchKernelGGL((rt::short_kernel<T, Op, 4>), dim3(1), dim3(256), 0, s, x, n, init, out);
    }
    else
    {
      hipLaunchKernelGGL((rt::short_kernel<T, Op, 16>), dim3(1), dim3(1024), 0, s, x, n, init, out);
    }
    RC_HIP(hipGetLastError());
    return RAJA_CDNA4_SUCCESS;
  }
  if (shape == Shape::kTiles)
  {
    const int64_t max_blocks = (int64_t)rc::num_cus() * 8;
    const unsigned grid = (unsigned)(ntiles < max_blocks ? ntiles : max_blocks);
    hipLaunchKernelGGL((rt::tiles_kernel<T, Op>), dim3(grid), dim3(rt::kBlock), 0, s, x, n, ntiles,
                       partials);
    RC_HIP(hipGetLastError());
    launch_final<Op, false>(partials, ntiles, init, out, s);
    RC_HIP(hipGetLastError());
    return RAJA_CDNA4_SUCCESS;
  }
  hipLaunchKernelGGL((rt::quads_kernel<T, Op>), dim3((unsigned)nquads), dim3(rt::kBlock), 0, s, x, n,
                     partials);
  RC_HIP(hipGetLastError());
  if (shape == Shape::kGroups)
  {
    const int64_t groups = rc::ceil_div(ntiles, (int64_t)64);
    hipLaunchKernelGGL((rt::group_kernel<Op>), dim3((unsigned)groups), dim3(64), 0, s, partials, ntiles,
                       partials + ntiles);
    RC_HIP(hipGetLastError());
    launch_final<Op, false>(partials + ntiles, groups, init, out, s);
  }
  else
  {
    launch_final<Op, !rt::kWide<Op>>(partials, nquads, init, out, s);
  }
  RC_HIP(hipGetLastError());
  return RAJA_CDNA4_SUCCESS;
}

template<typename T, typename Op>
int launch_reduce(const T* x, int64_t n, typename Op::acc_t init, rt::ResultOut<Op> out,
                  hipStream_t s, const char* name)
{
  using acc_t = typename Op::acc_t;
  if (n < 0) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "negative length");
  if (n > 0 && !x) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "input is NULL");
  rc::StreamCtx* c = nullptr;
  RC_TRY(rc::get_ctx(s, &c));
  if (n > max_span<T>())
  {
    return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "span too long for one reduction");
  }
  RC_TRY(rc::ensure_tmp(c, (size_t)(n > 0 ? partial_slots<T, Op>(n) : 1) * sizeof(acc_t)));
  return launch_reduce_core<T, Op>(x, n, init, out, (acc_t*)c->tmp, s, name);
}

template<typename T>
int reduce_typed(int op, const void* x, int64_t n, const void* init, void* out, hipStream_t s)
{
  const T iv = *static_cast<const T*>(init);
  switch (op)
  {
    case RAJA_CDNA4_OP_PLUS:
      return launch_reduce<T, rk::OpPlus<T>>((const T*)x, n, iv, {(T*)out}, s, "reduce_sum");
    case RAJA_CDNA4_OP_MIN:
      return launch_reduce<T, rk::OpMin<T>>((const T*)x, n, iv, {(T*)out}, s, "reduce_min");
    case RAJA_CDNA4_OP_MAX:
      return launch_reduce<T, rk::OpMax<T>>((const T*)x, n, iv, {(T*)out}, s, "reduce_max");
    default:
      return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "operator %d not supported here", op);
  }
}

template<typename T>
int reduce_bits(int op, const void* x, int64_t n, const void* init, void* out, hipStream_t s)
{
  const T iv = *static_cast<const T*>(init);
  switch (op)
  {
    case RAJA_CDNA4_OP_BIT_OR:
      return launch_reduce<T, rk::OpBitOr<T>>((const T*)x, n, iv, {(T*)out}, s, "reduce_bitor");
    case RAJA_CDNA4_OP_BIT_AND:
      return launch_reduce<T, rk::OpBitAnd<T>>((const T*)x, n, iv, {(T*)out}, s, "reduce_bitand");
    default:
      return reduce_typed<T>(op, x, n, init, out, s);
  }
}

template<typename T>
int reduce_loc_typed(int is_max, const void* x, int64_t n, const void* init_val, int64_t init_loc,
                     void* out_val, int64_t* out_loc, hipStream_t s)
{
  const rk::ValLoc<T> iv = rk::make_valloc<T>(*static_cast<const T*>(init_val), init_loc);
  if (is_max)
  {
    return launch_reduce<T, rk::OpMaxLoc<T>>((const T*)x, n, iv, {{(T*)out_val, out_loc}}, s, "reduce_maxloc");
  }
  return launch_reduce<T, rk::OpMinLoc<T>>((const T*)x, n, iv, {{(T*)out_val, out_loc}}, s, "reduce_minloc");
}

}  // namespace

namespace rws
{
size_t sum_f64_ws_bytes(int64_t n)
{
  return rc::align_up((size_t)(partial_slots<double, rk::OpPlus<double>>(n) + 1) * sizeof(double), 256);
}

int sum_f64(const double* x, int64_t n, double* out, void* ws, hipStream_t s)
{
  if (n > max_span<double>())
  {
    return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "span too long for one reduction");
  }
  return launch_reduce_core<double, rk::OpPlus<double>>(x, n, 0.0, {out}, (double*)ws, s, "reduce");
}
}  // namespace rws

extern "C" {

int raja_cdna4_reduce(int dtype, int op, const void* x, int64_t n, const void* init,
                      void* out_dev, void* stream)
{
  if (!init) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "init is NULL");
  if (!out_dev) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "output is NULL");
  hipStream_t s = (hipStream_t)stream;
  switch (dtype)
  {
    case RAJA_CDNA4_I32: return reduce_bits<int32_t>(op, x, n, init, out_dev, s);
    case RAJA_CDNA4_I64: return reduce_bits<int64_t>(op, x, n, init, out_dev, s);
    case RAJA_CDNA4_U32: return reduce_bits<uint32_t>(op, x, n, init, out_dev, s);
    case RAJA_CDNA4_U64: return reduce_bits<uint64_t>(op, x, n, init, out_dev, s);
    case RAJA_CDNA4_F32: return reduce_typed<float>(op, x, n, init, out_dev, s);
    case RAJA_CDNA4_F64: return reduce_typed<double>(op, x, n, init, out_dev, s);
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "dtype %d not supported", dtype);
  }
}

int raja_cdna4_reduce_loc(int dtype, int is_max, const void* x, int64_t n, const void* init_val,
                          int64_t init_loc, void* out_val_dev, int64_t* out_loc_dev, void* stream)
{
  if (!init_val || !out_val_dev || !out_loc_dev)
  {
    return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "NULL argument");
  }
  hipStream_t s = (hipStream_t)stream;
  switch (dtype)
  {
    case RAJA_CDNA4_I32: return reduce_loc_typed<int32_t>(is_max, x, n, init_val, init_loc, out_val_dev, out_loc_dev, s);
    case RAJA_CDNA4_I64: return reduce_loc_typed<int64_t>(is_max, x, n, init_val, init_loc, out_val_dev, out_loc_dev, s);
    case RAJA_CDNA4_U32: return reduce_loc_typed<uint32_t>(is_max, x, n, init_val, init_loc, out_val_dev, out_loc_dev, s);
    case RAJA_CDNA4_U64: return reduce_loc_typed<uint64_t>(is_max, x, n, init_val, init_loc, out_val_dev, out_loc_dev, s);
    case RAJA_CDNA4_F32: return reduce_loc_typed<float>(is_max, x, n, init_val, init_loc, out_val_dev, out_loc_dev, s);
    case RAJA_CDNA4_F64: return reduce_loc_typed<double>(is_max, x, n, init_val, init_loc, out_val_dev, out_loc_dev, s);
    default: return rc::set_error(RAJA_CDNA4_ERROR_UNSUPPORTED, "dtype %d not supported", dtype);
  }
}

int raja_cdna4_multi_reduce_f64(const double* x, int64_t n, raja_cdna4_multi_f64* out_dev,
                                void* stream)
{
  static_assert(sizeof(raja_cdna4_multi_f64) == sizeof(rk::Multi), "layout");
  if (!out_dev) return rc::set_error(RAJA_CDNA4_ERROR_INVALID_ARGUMENT, "output is NULL");
  return launch_reduce<double, rk::OpMulti>(x, n, rk::OpMulti::ident(), {(rk::Multi*)out_dev},
                                            (hipStream_t)stream, "reduce_multi_f64");
}

}  // extern "C"
