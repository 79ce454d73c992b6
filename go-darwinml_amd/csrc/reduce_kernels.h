// Kernels of a Reduce of one operand (no fused cluster), precompiled over dtype, vector
// width and form, with sizes and strides as arguments; instantiated for the
// floating-point types in k_reduce.hip, for the integers in k_reduce_int.hip.
#pragma once
#include <limits>

#include "common.h"
#include "graph.h"
#include "reduce_dev.h"

namespace ghip {
namespace reduce {

template <typename T> struct Acc { using type = float; };
template <> struct Acc<double> { using type = double; };
template <> struct Acc<int8_t> { using type = long long; };
template <> struct Acc<int16_t> { using type = long long; };
template <> struct Acc<int32_t> { using type = long long; };
template <> struct Acc<int64_t> { using type = long long; };
template <> struct Acc<uint8_t> { using type = unsigned long long; };
template <> struct Acc<uint16_t> { using type = unsigned long long; };
template <> struct Acc<uint32_t> { using type = unsigned long long; };
template <> struct Acc<uint64_t> { using type = unsigned long long; };

template <typename T> __device__ __forceinline__ typename Acc<T>::type widen(T x) { return x; }
__device__ __forceinline__ float widen(bf16_t x) { return bf16_to_f32(x.bits); }
template <typename T> __device__ __forceinline__ void narrow(T* p, typename Acc<T>::type v) { *p = static_cast<T>(v); }
__device__ __forceinline__ void narrow(bf16_t* p, float v) { p->bits = f32_to_bf16(v); }

template <int OP, typename A>
__device__ __forceinline__ A init_of() {
  if constexpr (OP == GHIP_REDUCE_SUM) return A(0);
  else if constexpr (OP == GHIP_REDUCE_PRODUCT) return A(1);
  else if constexpr (std::is_floating_point<A>::value) return OP == GHIP_REDUCE_MAX ? -A(INFINITY) : A(INFINITY);
  else return OP == GHIP_REDUCE_MAX ? std::numeric_limits<A>::lowest() : std::numeric_limits<A>::max();
}
template <int OP>
struct Combine {
  template <typename A>
  __device__ __forceinline__ A operator()(A a, A b) const {
    if constexpr (OP == GHIP_REDUCE_SUM) return a + b;
    else if constexpr (OP == GHIP_REDUCE_PRODUCT) return a * b;
    else if constexpr (OP == GHIP_REDUCE_MAX) return (a > b || a != a) ? a : b;  // NaN propagates
    else return (a < b || a != a) ? a : b;
  }
};

// V consecutive values from p, UNIT: next to each other (one load at element alignment),
// else `step` elements apart.
template <typename T, int V, bool UNIT>
__device__ __forceinline__ void load_values(const T* p, int64_t step, typename Acc<T>::type (&v)[V]) {
  if constexpr (UNIT) {
    struct __attribute__((packed)) W { T x[V]; };
    const W w = *reinterpret_cast<const W*>(p);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = widen(w.x[e]);
  } else {
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = widen(p[e * step]);
  }
}

// An operand of one reduced axis and one kept axis (columns: one before, one after it)
// whose vectors lie together.
template <typename T, int V>
struct LineOperand {
  const T* x;
  int64_t s_out, s_in, s_red;
  const T* row;
  __device__ __forceinline__ void at(long long o) { row = x + o * s_out; }
  __device__ __forceinline__ void at(long long ou, long long col) { row = x + ou * s_out + col * s_in; }
  __device__ __forceinline__ void get(long long r, typename Acc<T>::type (&v)[V]) const {
    load_values<T, V, true>(row + r * s_red, 1, v);
  }
};

// Any axes.
template <typename T, int V, bool UNIT>
struct AxesOperand {
  const T* x;
  const ReduceAxes& d;
  long long inner;
  const T* row;
  __device__ __forceinline__ static long long offset(long long i, bool wide, int rank, const ReduceDiv* div,
                                                     const int64_t* dims, const int64_t* st) {
    long long off = 0;
#pragma unroll 1
    for (int k = rank - 1; k > 0; --k) {
      const long long q = wide ? i / dims[k] : reduce_quot(static_cast<unsigned>(i), div[k]);
      off += (i - q * dims[k]) * st[k];
      i = q;
    }
    return off + i * st[0];
  }
  __device__ __forceinline__ void at(long long o) { row = x + offset(o, d.o_wide, d.orank, d.odiv, d.odims, d.ost); }
  __device__ __forceinline__ void at(long long ou, long long col) { at(ou * inner + col); }
  __device__ __forceinline__ void get(long long r, typename Acc<T>::type (&v)[V]) const {
    load_values<T, V, UNIT>(row + offset(r, d.r_wide, d.rrank, d.rdiv, d.rdims, d.rst), d.step, v);
  }
};
template <typename T>
struct Result {
  T* y;
  typename Acc<T>::type* ws;
  const ReduceGeom& g;
  __device__ __forceinline__ void put(long long o, typename Acc<T>::type a) const {
    if (g.C > 1) ws[blockIdx.y * g.osize + o] = a;
    else narrow(y + o, a);
  }
  template <int V>
  __device__ __forceinline__ void put(long long o, const typename Acc<T>::type (&a)[V]) const {
    struct __attribute__((packed)) W { T x[V]; } w;
#pragma unroll
    for (int e = 0; e < V; ++e) narrow(&w.x[e], a[e]);
    *reinterpret_cast<W*>(y + o) = w;  // one store at element alignment
  }
};

template <typename T, int V, int FORM, int OP>
__global__ __launch_bounds__(1024) void reduce_kernel(const T* __restrict__ x, T* __restrict__ y, int64_t s_out,
                                                      int64_t s_red, int64_t s_in, typename Acc<T>::type* __restrict__ ws,
                                                      ReduceGeom g) {
  using A = typename Acc<T>::type;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  // The arguments at once: fetched where they are first used they are a chain of waits.
  asm volatile("" ::"s"(g.osize), "s"(g.rsize), "s"(g.inner), "s"(g.gx), "s"(g.chunk), "s"(g.C), "s"(g.log_l), "s"(g.log_nt),
               "s"(g.cblocks.d), "s"(g.cblocks.mul), "s"(g.cblocks.shift), "s"(s_in));
  reduce_body<FORM, V, reduce_unroll(V)>(g, init_of<OP, A>(), Combine<OP>{}, LineOperand<T, V>{x, s_out, s_in, s_red, x},
                       Result<T>{y, ws, g}, reinterpret_cast<A*>(lds));
}
// Any axes: fewer calls, so the operation is an argument.
template <typename T, int V, int FORM>
__global__ __launch_bounds__(1024) void reduce_axes_kernel(const T* __restrict__ x, T* __restrict__ y,
                                                           typename Acc<T>::type* __restrict__ ws, ReduceAxes d, ReduceGeom g,
                                                           int op) {
  using A = typename Acc<T>::type;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const A init = op == GHIP_REDUCE_SUM ? init_of<GHIP_REDUCE_SUM, A>() : op == GHIP_REDUCE_PRODUCT ? init_of<GHIP_REDUCE_PRODUCT, A>()
               : op == GHIP_REDUCE_MAX ? init_of<GHIP_REDUCE_MAX, A>() : init_of<GHIP_REDUCE_MIN, A>();
  auto comb = [op](A a, A b) {
    switch (op) {
      case GHIP_REDUCE_SUM: return Combine<GHIP_REDUCE_SUM>{}(a, b);
      case GHIP_REDUCE_PRODUCT: return Combine<GHIP_REDUCE_PRODUCT>{}(a, b);
      case GHIP_REDUCE_MAX: return Combine<GHIP_REDUCE_MAX>{}(a, b);
      default: return Combine<GHIP_REDUCE_MIN>{}(a, b);
    }
  };
  auto body = [&](auto unit) {
    reduce_body<FORM, V, 2>(g, init, comb, AxesOperand<T, V, decltype(unit)::value>{x, d, g.inner, x}, Result<T>{y, ws, g},
                         reinterpret_cast<A*>(lds));
  };
  if constexpr (V == 1) body(std::true_type{});
  else if (d.step == 1) body(std::true_type{});
  else body(std::false_type{});
}
template <typename T, int OP>
__global__ __launch_bounds__(256) void reduce_finish_kernel(T* __restrict__ y, const typename Acc<T>::type* __restrict__ ws,
                                                            ReduceGeom g) {
  const long long o = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (o < g.osize) narrow(y + o, reduce_ranges(g, ws, o, Combine<OP>{}));
}

// go(form, V) with both as compile-time constants.
template <typename T, typename F>
void with_form(const ReduceGeom& g, F go) {
  constexpr int VMAX = 16 / sizeof(T);
  auto width = [&](auto form) {
    if (g.V == 1) go(form, std::integral_constant<int, 1>{});
    else if (g.V == 2) go(form, std::integral_constant<int, 2>{});
    else if (g.V == 4) { if constexpr (VMAX >= 4) go(form, std::integral_constant<int, 4>{}); }
    else if (g.V == 8) { if constexpr (VMAX >= 8) go(form, std::integral_constant<int, 8>{}); }
    else if constexpr (VMAX >= 16) go(form, std::integral_constant<int, 16>{});
  };
  if (g.form == kReduceRows) width(std::integral_constant<int, kReduceRows>{});
  else if (g.form == kReduceColumns) width(std::integral_constant<int, kReduceColumns>{});
  else width(std::integral_constant<int, kReduceThreads>{});
}

// The kernels of a Reduce: over the operand, and over the ranges' values.
template <typename T, int OP>
void kernels_of(const ReduceAxes& d, const ReduceGeom& g, const void** main, const void** finish) {
  with_form<T>(g, [&](auto form, auto v) {
    constexpr int F = decltype(form)::value, V = decltype(v)::value;
    *main = d.line ? reinterpret_cast<const void*>(&reduce_kernel<T, V, F, OP>)
                   : reinterpret_cast<const void*>(&reduce_axes_kernel<T, V, F>);
  });
  *finish = reinterpret_cast<const void*>(&reduce_finish_kernel<T, OP>);
}
template <typename T>
void kernels_of(int op, const ReduceAxes& d, const ReduceGeom& g, const void** main, const void** finish) {
  switch (op) {
    case GHIP_REDUCE_SUM: return kernels_of<T, GHIP_REDUCE_SUM>(d, g, main, finish);
    case GHIP_REDUCE_PRODUCT: return kernels_of<T, GHIP_REDUCE_PRODUCT>(d, g, main, finish);
    case GHIP_REDUCE_MAX: return kernels_of<T, GHIP_REDUCE_MAX>(d, g, main, finish);
    default: return kernels_of<T, GHIP_REDUCE_MIN>(d, g, main, finish);
  }
}

}  // namespace reduce
}  // namespace ghip
