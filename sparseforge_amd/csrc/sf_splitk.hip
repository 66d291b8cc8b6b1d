// Split-K reduction: C = epilogue(sum over splits of the f32 partials), the
// splits summed in index order (deterministic), then the same output
// rounding, bias, mask product / decay term and accumulation as the GEMM
// epilogue.  Bound by the partials' traffic (written moments before, so mostly
// from the MALL): four columns per thread with 16-byte accesses where the rows
// allow it, four splits' loads in flight.  Model of two 1.1B layers, 86 reduces
// a pass: 941 us an element and a load at a time (64-bit division each), 706 us;
// [4096, 64] in 16 splits 4.6 and 3.9 us.
#include "sf_mfma.hpp"

namespace sf {
namespace {

// Epilogue of one element whose sum is x.
__device__ __forceinline__ float splitk_out(const GemmArgs& g, int elem_dtype, float x, int64_t o, int64_t col) {
  const bool cbf = g.c_dtype == SF_DTYPE_BF16;
  if (cbf) x = hround(x);
  if (g.bias) {
    const float b = load_elem(g.bias, col, g.bias_dtype);
    x = cbf ? hround(x + b) : x + b;
  }
  if (g.emask) {
    const float em = load_elem(g.emask, o, elem_dtype);
    if (g.dw) {
      if (em < 0.5f) {
        float d = g.decay * load_elem(g.dw, o, elem_dtype);
        if (cbf) d = hround(d);
        x = cbf ? hround(x + d) : x + d;
      }
    } else {
      x = cbf ? hround(x * em) : x * em;
    }
  }
  if (g.accumulate) x = load_elem(g.C, o, g.c_dtype) + x;
  return x;
}

// V columns per thread (4: N % 4 == 0, ldc % 4 == 0, C 16-byte aligned).
template <int V>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(GemmArgs g, int elem_dtype) {
  const int64_t total = g.M * g.N, per_row = g.N / V, items = g.M * per_row;
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < items; i += (int64_t)gridDim.x * 256) {
    // rows and columns in 32 bits when the item count allows it
    int64_t row, c;
    if (items < (1ll << 32)) {
      row = static_cast<uint32_t>(i) / static_cast<uint32_t>(per_row);
      c = (i - row * per_row) * V;
    } else {
      row = i / per_row;
      c = (i - row * per_row) * V;
    }
    float x[V];
#pragma unroll
    for (int q = 0; q < V; ++q) x[q] = 0.0f;
    const float* p = g.partial + row * g.N + c;
    auto add = [&](const float4& v) {
      x[0] += v.x;
      if constexpr (V == 4) {
        x[1] += v.y;
        x[2] += v.z;
        x[3] += v.w;
      }
    };
    auto get = [&](int64_t at) {
      if constexpr (V == 4)
        return *reinterpret_cast<const float4*>(p + at);
      else
        return make_float4(p[at], 0.0f, 0.0f, 0.0f);
    };
    int z = 0;
    for (; z + 4 <= g.splits; z += 4, p += 4 * total) {  // four partials in flight, added in index order
      const float4 v0 = get(0), v1 = get(total), v2 = get(2 * total), v3 = get(3 * total);
      add(v0);
      add(v1);
      add(v2);
      add(v3);
    }
    for (; z < g.splits; ++z, p += total) add(get(0));
    const int64_t o = row * g.ldc + c;
#pragma unroll
    for (int q = 0; q < V; ++q) x[q] = splitk_out(g, elem_dtype, x[q], o + q, c + q);
    if constexpr (V == 4) {
      if (g.c_dtype == SF_DTYPE_BF16)
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(g.C) + o) = make_uint2(pack2(x[0], x[1]), pack2(x[2], x[3]));
      else
        *reinterpret_cast<float4*>(static_cast<float*>(g.C) + o) = make_float4(x[0], x[1], x[2], x[3]);
    } else {
      store_from_f32(g.C, o, g.c_dtype, x[0]);
    }
  }
}

}  // namespace

int launch_splitk_reduce(const GemmArgs& g, int elem_dtype, hipStream_t st, const char* what) {
  // four columns a thread where that still gives every CU two workgroups (the small outputs of the rank-64 products
  // are latency-bound: more threads)
  if (g.N % 4 == 0 && g.ldc % 4 == 0 && g.c_aligned && g.M * (g.N / 4) >= 512 * 256)
    splitk_reduce_kernel<4><<<elementwise_grid(g.M * (g.N / 4), 256), 256, 0, st>>>(g, elem_dtype);
  else
    splitk_reduce_kernel<1><<<elementwise_grid(g.M * g.N, 256), 256, 0, st>>>(g, elem_dtype);
  return launch_status(what);
}

}  // namespace sf
