// The integer types' Reduce kernels: their own translation unit, which builds beside
// k_reduce.hip.
#include "reduce_kernels.h"

namespace ghip {
namespace reduce {
template void kernels_of<int8_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
template void kernels_of<int16_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
template void kernels_of<int32_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
template void kernels_of<int64_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
template void kernels_of<uint8_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
template void kernels_of<uint16_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
template void kernels_of<uint32_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
template void kernels_of<uint64_t>(int, const ReduceAxes&, const ReduceGeom&, const void**, const void**);
}  // namespace reduce
}  // namespace ghip
