// Reduce of one operand (no fused cluster): sum, product, maximum, minimum over any axes.
// Precompiled over dtype, vector width and form, with sizes and strides as arguments, so
// compiling a graph costs nothing for them (a kernel generated per shape: ~0.25 s each).
// Bound by HBM; forms and accumulation order: reduce_dev.h, reduce_geometry.  us a call, a
// kernel generated with the sizes as literals / here: bf16 [4096,2048] over the rows 8.0 /
// 7.9, over the columns 5.5 / 5.7; fp32 [8192,8192] over the rows 40.6 / 43.0, over the
// columns 39.1 / 39.3; many short rows pay for the arguments, [65536,64] over the columns
// 6.6 / 9.9 (17.5 a wave per output by the earlier kernel), and axes that do not fold for
// their divisions, [6,40,500] over 0 and 2 7.2 / 15.8 (earlier 28).
// Accumulator: fp32 for fp32 / bf16 / f16, fp64 for fp64, 64-bit integers for integers.
#include "reduce_kernels.h"

namespace ghip {
namespace reduce {
extern template void kernels_of<int8_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
extern template void kernels_of<int16_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
extern template void kernels_of<int32_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
extern template void kernels_of<int64_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
extern template void kernels_of<uint8_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
extern template void kernels_of<uint16_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
extern template void kernels_of<uint32_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
extern template void kernels_of<uint64_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
}  // namespace reduce

int reduce_kernels(int dtype, int op, const ReduceAxes& d, const ReduceGeom& g, bool plan_only, ReduceKernels* k,
                   GHipError* err) {
  const void* main = nullptr;
  const void* finish = nullptr;
  switch (dtype) {
    case GHIP_DTYPE_FLOAT32: reduce::kernels_of<float>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_BFLOAT16: reduce::kernels_of<bf16_t>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_FLOAT16: reduce::kernels_of<_Float16>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_FLOAT64: reduce::kernels_of<double>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_INT8: reduce::kernels_of<int8_t>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_INT16: reduce::kernels_of<int16_t>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_INT32: reduce::kernels_of<int32_t>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_INT64: reduce::kernels_of<int64_t>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_UINT8: reduce::kernels_of<uint8_t>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_UINT16: reduce::kernels_of<uint16_t>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_UINT32: reduce::kernels_of<uint32_t>(op, d, g, &main, &finish); break;
    case GHIP_DTYPE_UINT64: reduce::kernels_of<uint64_t>(op, d, g, &main, &finish); break;
    default: return set_error(err, GHIP_ERR_UNSUPPORTED, "reduce: dtype %d", dtype);
  }
  if (plan_only) return GHIP_OK;
  GHIP_CHECK(hipGetFuncBySymbol(&k->main, main), err);
  if (g.C > 1) GHIP_CHECK(hipGetFuncBySymbol(&k->finish, finish), err);
  return GHIP_OK;
}

int launch_reduce(const ReduceKernels& k, int op, const void* x, void* y, void* ws, const ReduceAxes& d,
                  const ReduceGeom& g, int acc_bytes, hipStream_t s, GHipError* err) {
  if (g.osize == 0) return GHIP_OK;
  // Columns without a kept axis before the block: the one after it is ost[0].
  int64_t s_out = g.form == kReduceColumns && d.orank == 1 ? 0 : d.ost[0], s_red = d.rst[0], s_in = d.ost[d.orank - 1];
  ReduceAxes axes = d;
  ReduceGeom geom = g;
  void* line_args[] = {&x, &y, &s_out, &s_red, &s_in, &ws, &geom};
  void* axes_args[] = {&x, &y, &ws, &axes, &geom, &op};
  const unsigned nt = 1u << g.log_nt, lds = static_cast<unsigned>(reduce_lds(g) * acc_bytes);
  hipError_t h = hipModuleLaunchKernel(k.main, reduce_grid_x(g), reduce_grid_y(g), 1, nt, 1, 1, lds, s,
                                       d.line ? line_args : axes_args, nullptr);
  if (h == hipSuccess && g.C > 1) {
    void* fin_args[] = {&y, &ws, &geom};
    h = hipModuleLaunchKernel(k.finish, static_cast<unsigned>((g.osize + 255) / 256), 1, 1, 256, 1, 1, 0, s, fin_args, nullptr);
  }
  GHIP_CHECK(h, err);
  return GHIP_OK;
}

}  // namespace ghip
