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
  float* partial;        // splits > 1: [splits][M][N] f32 partial sums
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

// C = epilogue(sum of the K splits' partials) (sf_splitk.hip).
int launch_splitk_reduce(const GemmArgs& g, int elem_dtype, hipStream_t st, const char* what);

// The f32 product of dense, unmasked operands (sf_gemm_f32.hip): its workspace for K-split partials, and the launch.
size_t gemm_f32_workspace(int64_t M, int64_t N, int64_t K);
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
