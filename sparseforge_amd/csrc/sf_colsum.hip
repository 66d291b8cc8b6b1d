// Column sums of a row-major [rows, cols] matrix: the bias gradient db = sum_t dy
// (legacy/sparse_modeling.py:127-130), accumulated in f32.
//
// HBM-bound (each element read once).  A workgroup owns one strip of LPR 16-byte
// chunks of every row; its 16 waves read whole strips of consecutive rows, four
// rows of every thread in flight, so the strip streams at the rate one CU can
// fetch.  A strip is as wide as still gives about one workgroup per CU
// (colsum_lanes): the sum needs no second launch and no workspace.  Per thread a
// running sum over its rows, then a butterfly over the wave's row groups and a
// fixed-order fold of the waves in LDS, so the result does not vary between runs.
// Measured: [8168, 3072] f32 590 us with a workgroup per 64 columns reading one
// element per lane and load (48 workgroups), 22 us here (4.6 TB/s); [8192, 4096]
// bf16 609 and 17.5 us; [4096, 2048] bf16 130 and 8.7 us.  Without the XCD-aware
// strip order those were 33, 41 and 14 us (a line's 32-byte strips fetched by
// four L2s).

#include "sf_common.hpp"

namespace sf {
namespace {

constexpr int kColBlock = 1024;

typedef uint32_t u32x4_cs __attribute__((ext_vector_type(4)));

// The 16 bytes at element e0 of a row as f32 values; VEC: one aligned load, else
// element by element up to `n`.
template <int DT, bool VEC>
__device__ __forceinline__ void col_load(const void* A, int64_t e0, int n, float (&v)[DT == SF_DTYPE_F32 ? 4 : 8]) {
  constexpr int VE = DT == SF_DTYPE_F32 ? 4 : 8;
  if constexpr (VEC) {
    if constexpr (DT == SF_DTYPE_F32) {
      const float4 q = *reinterpret_cast<const float4*>(static_cast<const float*>(A) + e0);
      v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
      const u32x4_cs q = *reinterpret_cast<const u32x4_cs*>(static_cast<const uint16_t*>(A) + e0);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[2 * k] = __uint_as_float(q[k] << 16);
        v[2 * k + 1] = __uint_as_float(q[k] & 0xffff0000u);
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < VE; ++k) v[k] = k < n ? load_as_f32(A, e0 + k, DT) : 0.0f;
  }
}

template <int DT, int LPR, bool VEC>
__global__ void __launch_bounds__(kColBlock) column_sum_kernel(const void* __restrict__ A, int64_t rows, int64_t cols,
                                                               void* __restrict__ out, int out_dtype) {
  constexpr int VE = DT == SF_DTYPE_F32 ? 4 : 8, STRIP = LPR * VE, RP = kColBlock / LPR, WAVES = kColBlock / 64;
  __shared__ float part[WAVES][STRIP];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // workgroups go round-robin over the 8 XCDs: neighbouring strips (which share cache lines when
  // they are narrower than one) run on the same XCD and so share its L2
  int64_t strip = blockIdx.x;
  if (gridDim.x % 8 == 0) strip = (strip % 8) * (gridDim.x / 8) + strip / 8;
  const int64_t c0 = strip * STRIP + (t % LPR) * VE;
  const int n = c0 >= cols ? 0 : (cols - c0 >= VE ? VE : static_cast<int>(cols - c0));
  float s[VE];
#pragma unroll
  for (int k = 0; k < VE; ++k) s[k] = 0.0f;
  if (n > 0) {  // VEC: cols is a multiple of VE, so n is 0 or VE
    int64_t r = t / LPR;
    for (; r + 3 * RP < rows; r += 4 * RP) {
      float v[4][VE];
#pragma unroll
      for (int u = 0; u < 4; ++u) col_load<DT, VEC>(A, (r + u * RP) * cols + c0, n, v[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int k = 0; k < VE; ++k) s[k] += v[u][k];
    }
    for (; r < rows; r += RP) {
      float v[VE];
      col_load<DT, VEC>(A, r * cols + c0, n, v);
#pragma unroll
      for (int k = 0; k < VE; ++k) s[k] += v[k];
    }
  }
#pragma unroll
  for (int k = 0; k < VE; ++k)
    for (int off = LPR; off < 64; off <<= 1) s[k] += __shfl_xor(s[k], off, 64);
  if (lane < LPR)
#pragma unroll
    for (int k = 0; k < VE; ++k) part[wave][lane * VE + k] = s[k];
  __syncthreads();
  const int64_t col = strip * STRIP + t;
  if (t < STRIP && col < cols) {
    float x = part[0][t];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) x += part[w][t];
    store_from_f32(out, col, out_dtype, x);
  }
}

// Chunks per strip: 128-byte strips while they give three quarters of the 256 CUs a
// workgroup (a whole cache line per row), else 64- or 32-byte ones.
int colsum_lanes(int64_t cols, int ve) {
  for (int l = 8; l > 2; l >>= 1)
    if (ceil_div(cols, l * ve) >= 192) return l;
  return 2;
}

template <int DT>
void launch_colsum(const void* A, int64_t rows, int64_t cols, void* out, int out_dtype, hipStream_t st) {
  constexpr int VE = DT == SF_DTYPE_F32 ? 4 : 8;
  const bool vec = cols % VE == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0;
  const int lpr = colsum_lanes(cols, VE);
  const dim3 grid(static_cast<unsigned>(ceil_div(cols, lpr * VE)));
#define SF_COLSUM(L)                                                                      \
  do {                                                                                    \
    if (vec)                                                                              \
      column_sum_kernel<DT, L, true><<<grid, kColBlock, 0, st>>>(A, rows, cols, out, out_dtype);  \
    else                                                                                  \
      column_sum_kernel<DT, L, false><<<grid, kColBlock, 0, st>>>(A, rows, cols, out, out_dtype); \
  } while (0)
  if (lpr == 8)
    SF_COLSUM(8);
  else if (lpr == 4)
    SF_COLSUM(4);
  else
    SF_COLSUM(2);
#undef SF_COLSUM
}

}  // namespace
}  // namespace sf

using namespace sf;

extern "C" int sf_column_sum(const void* A, int a_dtype, int64_t rows, int64_t cols, void* out, int out_dtype,
                             void* stream) {
  SF_CHECK_ARG(rows >= 0 && cols >= 0, "negative shape");
  SF_CHECK_ARG((a_dtype == SF_DTYPE_F32 || a_dtype == SF_DTYPE_BF16) &&
                   (out_dtype == SF_DTYPE_F32 || out_dtype == SF_DTYPE_BF16),
               "bad dtype");
  if (cols == 0) return SF_OK;
  SF_CHECK_ARG(out && (rows == 0 || A), "null tensor");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (a_dtype == SF_DTYPE_F32)
    launch_colsum<SF_DTYPE_F32>(A, rows, cols, out, out_dtype, st);
  else
    launch_colsum<SF_DTYPE_BF16>(A, rows, cols, out, out_dtype, st);
  return launch_status("sf_column_sum");
}
