// Bodies of the Reduce kernels: shared by the precompiled kernels (k_reduce.hip), which
// read one operand through strides, and the generated ones (hipRTC compiles this text in
// front of them), which evaluate the operand's elementwise cluster on the fly.  The
// accumulation order is the geometry's alone, so both give the same bits.
#pragma once

namespace ghip {

// Forms:
//   rows:    a wave (few outputs: a workgroup of 256 or 1024 threads) per output, V
//            consecutive values a lane and load, a butterfly, then LDS.
//   columns: a workgroup takes L vectors of V adjacent columns and strides the reduced
//            index with its other lanes, so every load is coalesced; a butterfly over
//            the lanes of one column, then LDS.
//   threads: a thread per output, or per V adjacent outputs.
enum ReduceForm { kReduceRows = 0, kReduceColumns = 1, kReduceThreads = 2 };

// n / d for n < 2^31 by a multiply: q = (mulhi(n, mul) + n) >> shift.
struct ReduceDiv {
  unsigned d, mul;
  int shift;
};
constexpr ReduceDiv reduce_div(unsigned d) {
  int s = 0;
  while ((1ull << s) < d) ++s;
  return ReduceDiv{d, static_cast<unsigned>(((1ull << 32) * ((1ull << s) - d)) / d + 1), s};
}

// Launch shape, a function of the Reduce's shape, axes and dtype (reduce_geometry).
struct ReduceGeom {
  long long osize, rsize;  // outputs, values reduced into each
  long long inner;         // columns: kept elements after the reduced axes
  long long gx;            // workgroups of one range of the reduced index
  long long chunk;         // reduced values of a range
  int C;                   // ranges
  int form;
  int V;                   // consecutive elements a lane and load
  int log_l;               // rows: lanes per output; columns: vectors side by side
  int log_nt;              // threads per workgroup
  ReduceDiv cblocks;       // columns: workgroups side by side
};
// Workgroups in x: HIP takes fewer than 2^32 work-items per dimension, so a grid of more
// workgroups goes on in y.
constexpr long long kReduceGridX = 1 << 21;
constexpr unsigned reduce_grid_x(const ReduceGeom& g) { return static_cast<unsigned>(g.gx < kReduceGridX ? g.gx : kReduceGridX); }
constexpr unsigned reduce_grid_y(const ReduceGeom& g) {
  return g.C > 1 ? static_cast<unsigned>(g.C) : static_cast<unsigned>((g.gx + kReduceGridX - 1) / kReduceGridX);
}
// Accumulators the combine step keeps in LDS.
constexpr int reduce_lds(const ReduceGeom& g) {
  return g.form == kReduceRows ? 1 << g.log_l >> 6 : g.form == kReduceColumns ? (g.V << g.log_nt >> 6) << g.log_l : 1;
}

#if defined(__HIP__) || defined(__HIPCC_RTC__)
// Loads in flight a lane: eight, of wide vectors four.  Kernels generated for one geometry
// take its own number of loads where that is less.
constexpr int reduce_unroll(int v) { return v <= 2 ? 8 : 4; }
constexpr int reduce_unroll(const ReduceGeom& g) {
  const long long lanes = g.form == kReduceRows ? static_cast<long long>(g.V) << g.log_l
                        : g.form == kReduceColumns ? 1ll << (g.log_nt - g.log_l) : 1;
  const long long n = (g.chunk + lanes - 1) / lanes;
  return n < 1 ? 1 : n < reduce_unroll(g.V) ? static_cast<int>(n) : reduce_unroll(g.V);
}

__device__ __forceinline__ unsigned reduce_quot(unsigned n, const ReduceDiv& d) { return (__umulhi(n, d.mul) + n) >> d.shift; }

// src.at(o) / src.at(ou, col): the kept index (columns: before / after the reduced axes)
// whose values src.get(r, v) then gives, V of them from reduced index r (rows) or column
// col (columns).  dst.put(o, a): output o's value (of one range);
// dst.put(o, acc): outputs o .. o + V - 1.
template <int FORM, int V, int U, class A, class Comb, class Src, class Dst>
__device__ __forceinline__ void reduce_body(const ReduceGeom& g, A init, Comb comb, Src src, Dst dst, A* part) {
  const int t = threadIdx.x;
  const unsigned blk = g.gx <= kReduceGridX ? blockIdx.x : blockIdx.y * static_cast<unsigned>(kReduceGridX) + blockIdx.x;
  if (blk >= g.gx) return;
  A acc[V];
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] = init;
  const long long start = g.C > 1 ? blockIdx.y * g.chunk : 0;
  const long long r_end = g.C > 1 && start + g.chunk < g.rsize ? start + g.chunk : g.rsize;
  // Every 2^log-th reduced index from r, U loads in flight (by hand: the trip count
  // differs between lanes, for which the compiler tests it after every load).
  auto sweep = [&](long long r, int log) {
    long long n = r < r_end ? ((r_end - r - 1) >> log) + 1 : 0;
    for (; n >= U; n -= U, r += static_cast<long long>(U) << log) {
      A v[U][V];
#pragma unroll
      for (int u = 0; u < U; ++u) src.get(r + (static_cast<long long>(u) << log), v[u]);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] = comb(acc[e], v[u][e]);
    }
    constexpr int H = U > 3 ? U / 2 : 1;
    for (; n >= H; n -= H, r += static_cast<long long>(H) << log) {
      A v[H][V];
#pragma unroll
      for (int u = 0; u < H; ++u) src.get(r + (static_cast<long long>(u) << log), v[u]);
#pragma unroll
      for (int u = 0; u < H; ++u)
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] = comb(acc[e], v[u][e]);
    }
    if (n > 1) {  // the rest in flight together, the first one again past the end
      A v[H][V];
#pragma unroll
      for (int u = 0; u < H; ++u) src.get(r + (u < n ? static_cast<long long>(u) << log : 0), v[u]);
#pragma unroll
      for (int u = 0; u < H; ++u)
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] = u < n ? comb(acc[e], v[u][e]) : acc[e];
    } else if (n == 1) {
      A v[V];
      src.get(r, v);
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] = comb(acc[e], v[e]);
    }
  };
  if constexpr (FORM == kReduceRows) {
    const int lane = t & ((1 << g.log_l) - 1);
    const long long o = (static_cast<long long>(blk) << (g.log_nt - g.log_l)) +
                        __builtin_amdgcn_readfirstlane(t >> g.log_l);  // the same for a whole wave
    if (g.log_l == 6 && o >= g.osize) return;  // whole waves; wider groups are one output a workgroup
    src.at(o);
    sweep(start + lane * V, g.log_l + (V == 1 ? 0 : V == 2 ? 1 : V == 4 ? 2 : V == 8 ? 3 : 4));
    A a = acc[0];
#pragma unroll
    for (int e = 1; e < V; ++e) a = comb(a, acc[e]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) a = comb(a, __shfl_xor(a, off, 64));
    if (g.log_l > 6) {
      if (t % 64 == 0) part[t / 64] = a;
      __syncthreads();
      if (t != 0) return;
      for (int w = 1; w < 1 << (g.log_l - 6); ++w) a = comb(a, part[w]);
    } else if (lane != 0) {
      return;
    }
    dst.put(o, a);
  } else if constexpr (FORM == kReduceColumns) {
    const int TX = 1 << g.log_l, tx = t & (TX - 1), ty = t >> g.log_l, W = V << g.log_l;
    const unsigned ou = reduce_quot(blk, g.cblocks);
    const long long col0 = static_cast<long long>(blk - ou * g.cblocks.d) * W;
    const long long col = col0 + tx * V;
    src.at(ou, col < g.inner ? col : 0);
    sweep(start + ty, g.log_nt - g.log_l);
    for (int off = TX; off <= 32; off <<= 1)
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] = comb(acc[e], __shfl_xor(acc[e], off, 64));
    if (t % 64 < TX)
#pragma unroll
      for (int e = 0; e < V; ++e) part[t / 64 * W + tx * V + e] = acc[e];
    __syncthreads();
    for (int c = t; c < W; c += 1 << g.log_nt) {
      if (col0 + c >= g.inner) return;
      A a = part[c];
      for (int w = 1; w < 1 << (g.log_nt - 6); ++w) a = comb(a, part[w * W + c]);
      dst.put(ou * g.inner + col0 + c, a);
    }
  } else {
    const long long o = ((static_cast<long long>(blk) << g.log_nt) + t) * V;
    if (o >= g.osize) return;
    src.at(o);
    sweep(0, 0);
    dst.put(o, acc);
  }
}

// The ranges' values of output o, combined in order.
template <class A, class Comb>
__device__ __forceinline__ A reduce_ranges(const ReduceGeom& g, const A* ws, long long o, Comb comb) {
  A a = ws[o];
#pragma unroll 16
  for (int c = 1; c < g.C; ++c) a = comb(a, ws[o + c * g.osize]);
  return a;
}
#endif

}  // namespace ghip
