// Pieces shared by the MFMA kernels: vector types, bf16 packing and raw buffer loads.
#pragma once

#include "sf_common.hpp"

namespace sf {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x16_t __attribute__((ext_vector_type(16)));

// 16-byte vector as 4 dwords
struct V4 {
  uint32_t w[4];
};

__device__ __forceinline__ V4 ld16(const void* p) {
  uint4 v = *reinterpret_cast<const uint4*>(p);
  V4 r;
  r.w[0] = v.x;
  r.w[1] = v.y;
  r.w[2] = v.z;
  r.w[3] = v.w;
  return r;
}
__device__ __forceinline__ V4 zero16() {
  V4 r;
  r.w[0] = r.w[1] = r.w[2] = r.w[3] = 0u;
  return r;
}

// bf16 halves of a dword as f32, and the hardware round-to-nearest-even pack
// (v_cvt_pk_bf16_f32) back to two bf16.
__device__ __forceinline__ float lo_f(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_f(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  bf16x2_t v;
  v[0] = static_cast<__bf16>(lo);
  v[1] = static_cast<__bf16>(hi);
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float hround(float x) { return static_cast<float>(static_cast<__bf16>(x)); }
__device__ __forceinline__ uint16_t hbits(float x) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(x)); }

// Raw buffer loads: an SGPR resource holds the tensor base and its byte
// extent; a lane offset at or past the extent reads zeros without touching
// memory, which is how rows past M/N and k past K are padded.
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr uint32_t kOob = 0x80000000u;  // a lane offset past every operand's extent (extents are < 2^31 bytes)

__device__ __forceinline__ Rsrc make_rsrc(const void* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ V4 bload(Rsrc r, uint32_t voff, uint32_t soff) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0);
  V4 o;
  o.w[0] = x[0];
  o.w[1] = x[1];
  o.w[2] = x[2];
  o.w[3] = x[3];
  return o;
}

// Orders a wave's LDS writes before its own later reads for the compiler (the hardware keeps the order).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float load_elem(const void* p, int64_t i, int dtype) { return load_as_f32(p, i, dtype); }

constexpr int kGroupM = 8;  // M-tiles per L2 band
constexpr int kXcds = 8;

// Tile coordinates of workgroup `pid` (XCD-contiguous ranges, bands of kGroupM M-tiles).
__device__ __forceinline__ void tile_coords(int64_t pid, int64_t tiles_m, int64_t tiles_n, int64_t& tm, int64_t& tn) {
  const int64_t total = tiles_m * tiles_n;
  if (total % kXcds == 0) pid = (pid % kXcds) * (total / kXcds) + pid / kXcds;
  const int64_t band = kGroupM * tiles_n;
  const int64_t first_m = (pid / band) * kGroupM;
  const int64_t gm = tiles_m - first_m < kGroupM ? tiles_m - first_m : kGroupM;
  const int64_t r = pid % band;
  tm = first_m + r % gm;
  tn = r / gm;
}

}  // namespace

// A product of sf_gemm as its kernels take it.
struct GemmArgs {
  int64_t M, N, K1, K2;
  const void* A1;
  int64_t lda1;
  const void* A2;
  int64_t lda2;
  const void* B1;
  int64_t ldb1;
  const void* B2;
  int64_t ldb2;
  const void* bmask;  // effective mask of B1 (element dtype, B1's layout and ld)
  float bscale;       // 1: none
  int has_scale;
  void* C;
  int64_t ldc;
  int c_dtype;
  const void* bias;  // [N], element dtype or f32
  int bias_dtype;
  const void* emask;  // [M, N] row-major with ld = ldc: C *= emask
  const void* dw;     // [M, N]: C += decay * dw * (emask < 0.5)
  float decay;
  int accumulate;  // C += result
  int c_aligned;   // C is 16-byte aligned
  int64_t tiles_m, tiles_n;
  int splits;            // K splits (1: the kernel writes C itself)
  int64_t split_stages;  // segment-1 stages per split
  int64_t run_stages;    // f32 kernels: stages summed in one chain
  float* partial;        // splits > 1 (or a split in several runs): [splits][M][N] f32 partial sums
  // block-sparse-16 B1 (B layouts 2 / 3): B1 is the blocks array, b_map its block map
  const int32_t* b_map;
  int64_t b_map_rows, b_map_cols;
  // block-sparse-16 C: the epilogue writes only the blocks c_map lists, into c_blocks
  void* c_blocks;
  const int32_t* c_map;
  int64_t c_map_rows, c_map_cols;
  int64_t ldbm;      // leading dimension of a K-major byte mask ([N][K1])
  int bmask_kmajor;  // bmask is K-major (input gradient: B = W^T, mask given transposed)
  int dma_mask_ok;   // the byte mask can be copied 16 bytes at a time (bf16 direct kernel)
};

namespace {
// 8 consecutive columns of one row of a product (its f32 sums v): to the K split's partials, to the kept blocks of a
// block-sparse C, or through the epilogue (output rounding, bias, mask product / decay term, accumulation) to C.
// EDT: dtype of emask and dw; MASKED = false: there is no emask (a test outside the caller's loop).
template <int EDT, bool MASKED = true>
__device__ __forceinline__ void store_c8(const GemmArgs& g, int64_t row, int64_t col, int64_t kz, float (&v)[8]) {
  const bool cbf = g.c_dtype == SF_DTYPE_BF16;
  if (g.c_blocks) {
    // block-sparse C (the SDDMM weight gradient): only kept 16 x 16 blocks are written,
    // row (row % 16) of block c_map[row / 16][col / 16], 8 columns at a time
    const int64_t bi = (row / 16 < g.c_map_rows && col / 16 < g.c_map_cols)
                           ? g.c_map[(row / 16) * g.c_map_cols + col / 16] : -1;
    if (bi >= 0) {
      const int64_t o = bi * 256 + (row % 16) * 16 + (col % 16);
      if (g.c_dtype == SF_DTYPE_BF16) {
        *reinterpret_cast<uint4*>(static_cast<uint16_t*>(g.c_blocks) + o) =
            make_uint4(pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7]));
      } else {
        float* cp = static_cast<float*>(g.c_blocks) + o;
        *reinterpret_cast<float4*>(cp) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(cp + 4) = make_float4(v[4], v[5], v[6], v[7]);
      }
    }
    return;
  }
  if (g.splits > 1) {
    // split-K: raw f32 partial sums; sf_gemm's reduce kernel applies the epilogue
    float* pp = g.partial + (kz * g.M + row) * g.N + col;
    if (col + 8 <= g.N && (g.N & 3) == 0) {
      *reinterpret_cast<float4*>(pp) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4*>(pp + 4) = make_float4(v[4], v[5], v[6], v[7]);
    } else {
      for (int q = 0; q < 8 && col + q < g.N; ++q) pp[q] = v[q];
    }
    return;
  }
  const int64_t off = row * g.ldc + col;
  const bool vec = g.c_aligned && col + 8 <= g.N && (off & 7) == 0 &&
                   (!MASKED || !g.emask || (reinterpret_cast<uintptr_t>(g.emask) & 15u) == 0);
  if ((!MASKED || !g.dw) && vec) {
    // result of the matmul in the output dtype, then + bias (rounded again), then + C when
    // accumulating: the per-element sequence below, 8 outputs at a time
    if (g.bias) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float b = load_elem(g.bias, col + q, g.bias_dtype);
        v[q] = cbf ? hround(v[q]) + b : v[q] + b;
      }
    }
    if (MASKED && g.emask) {  // times the effective mask, after the product (+ bias) is rounded
      float em[8];
      if constexpr (EDT == SF_DTYPE_BF16) {
        const uint4 ew = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(g.emask) + off);
        const uint32_t w4[4] = {ew.x, ew.y, ew.z, ew.w};
#pragma unroll
        for (int q = 0; q < 8; ++q) em[q] = (q & 1) ? hi_f(w4[q >> 1]) : lo_f(w4[q >> 1]);
      } else {
        const float4 e0 = *reinterpret_cast<const float4*>(static_cast<const float*>(g.emask) + off);
        const float4 e1 = *reinterpret_cast<const float4*>(static_cast<const float*>(g.emask) + off + 4);
        em[0] = e0.x; em[1] = e0.y; em[2] = e0.z; em[3] = e0.w; em[4] = e1.x; em[5] = e1.y; em[6] = e1.z; em[7] = e1.w;
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = (cbf ? hround(v[q]) : v[q]) * em[q];
    }
    if (g.accumulate) {
      float c[8];
      if (cbf) {
        const uint4 cw = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(g.C) + off);
        const uint32_t w4[4] = {cw.x, cw.y, cw.z, cw.w};
#pragma unroll
        for (int q = 0; q < 8; ++q) c[q] = bf16_to_f32(static_cast<uint16_t>(w4[q >> 1] >> (16 * (q & 1))));
      } else {
        const float4 c0 = *reinterpret_cast<const float4*>(static_cast<const float*>(g.C) + off);
        const float4 c1 = *reinterpret_cast<const float4*>(static_cast<const float*>(g.C) + off + 4);
        c[0] = c0.x; c[1] = c0.y; c[2] = c0.z; c[3] = c0.w;
        c[4] = c1.x; c[5] = c1.y; c[6] = c1.z; c[7] = c1.w;
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float x = cbf ? hround(v[q]) : v[q];  // the product (+ bias) in the output dtype
        v[q] = c[q] + x;
      }
    }
    if (cbf) {
      *reinterpret_cast<uint4*>(static_cast<uint16_t*>(g.C) + off) =
          make_uint4(pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7]));
    } else {
      float* cp = static_cast<float*>(g.C) + off;
      *reinterpret_cast<float4*>(cp) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4*>(cp + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
    return;
  }
  const int edt = EDT;
  for (int q = 0; q < 8; ++q) {
    if (col + q >= g.N) break;
    const int64_t o = off + q;
    float x = cbf ? hround(v[q]) : v[q];
    if (g.bias) {
      const float b = load_elem(g.bias, col + q, g.bias_dtype);
      x = cbf ? hround(x + b) : x + b;
    }
    if (MASKED && g.emask) {
      const float em = load_elem(g.emask, o, edt);
      if (g.dw) {
        if (em < 0.5f) {
          float d = g.decay * load_elem(g.dw, o, edt);
          if (cbf) d = hround(d);
          x = cbf ? hround(x + d) : x + d;
        }
      } else {
        x = cbf ? hround(x * em) : x * em;
      }
    }
    if (g.accumulate) x = load_elem(g.C, o, g.c_dtype) + x;
    if (cbf)
      static_cast<uint16_t*>(g.C)[o] = hbits(x);
    else
      static_cast<float*>(g.C)[o] = x;
  }
}
}  // namespace

// C = epilogue(sum of the K splits' partials) (sf_splitk.hip).
int launch_splitk_reduce(const GemmArgs& g, int elem_dtype, hipStream_t st, const char* what);

// The bf16 product of dense, unmasked operands with a side of C of at most 64 (sf_gemm_skinny.hip): its workspace for
// K-split partials (often none), and the launch.
size_t gemm_skinny_workspace(int64_t M, int64_t N, int64_t K, int a_layout, int b_layout);
int launch_gemm_skinny(GemmArgs g, int a_layout, int b_layout, void* workspace, size_t workspace_bytes, hipStream_t st);

// The bf16 product of dense, unmasked operands on 128 x 128 tiles (sf_gemm_mid.hip): K splits it would take (0: the
// 256 x 256 tiles are the better choice), and its launch.
int gemm_mid_splits(int64_t M, int64_t N, int64_t K, int max_splits, int big_splits);
int launch_gemm_mid(GemmArgs g, int a_layout, int b_layout, int splits, void* workspace, hipStream_t st);

// The f32 product of dense, unmasked operands (sf_gemm_f32.hip): its workspace for K-split partials, and the launch.
size_t gemm_f32_workspace(int64_t M, int64_t N, int64_t K, int a_layout);
int launch_gemm_f32(GemmArgs g, int a_layout, int b_layout, void* workspace, size_t workspace_bytes, hipStream_t st);

// y [N tokens, M out] = x W^T (+ A2/B2 low-rank term, + bias), W packed 2:4.
struct Gemm24Args {
  const void* x;       // [N = tokens, K] bf16, row pitch ldx
  int64_t ldx;
  const void* vals;    // M * K / 2 bf16, fragment order (vals_off)
  const void* idx;     // u32 [M / 32][K / 64][2][32]
  int64_t M, N, K;
  const void* bias;    // [M] or null
  int bias_dtype;
  void* y;             // [N, M], row pitch ldy
  int y_dtype;
  int64_t ldy;
  int64_t tiles_m, tiles_n;
  int y_aligned;
  // optional dense second segment y^T += A2 . B2^T: A2 [M, K2] and B2 [N, K2] bf16, K-contiguous
  const void* A2;
  const void* B2;
  int64_t lda2, ldb2, K2;
};

// The kernels of smaller tiles (sf_gemm24_small.hip): whether a shape takes one of them, and the launch.
bool gemm24_split_takes(const Gemm24Args& g);
int launch_gemm24_split(const Gemm24Args& g, hipStream_t st, const char* what);

}  // namespace sf
