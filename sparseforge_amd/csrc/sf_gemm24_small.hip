// The packed 2:4 product below the sizes that fill the GPU with 256 x 256 tiles: y [N, M] = x [N, K] W^T (+ z S^T, + bias)
// with W in the packed layout of sf_pack_2to4 (decoding and short prompts of a
// finalized model, legacy/eval_wiki_ppl.py:548-651).
//
// With few tokens the product is bound by reading the weight (9/8 byte per
// weight), and 256 x 256 tiles leave most CUs idle (M / 256 workgroups: 16 at
// M = 4096).  Here a workgroup owns RB * 32 outputs x NT * 32 tokens and its
// 8 waves split K: wave w takes the 64-k stages w, w + 8, ..., so the
// workgroup streams contiguous runs of its row blocks' values.  Each wave loads
// the sparse A operand straight into registers (the packed layout is the
// fragment order), its tokens' x through a wave-private LDS tile (whole 128-byte
// lines from memory, no barrier: a wave's LDS accesses are performed in order),
// one stage ahead.  The 8 partial tiles meet in LDS and every thread sums 8
// outputs of a token in wave order, so results do not vary between runs.  The
// low-rank term runs on the dense MFMA, its 16-k steps spread over the waves.
#include <type_traits>

#include "sf_mfma.hpp"

namespace sf {
namespace {

constexpr int kSpWaves = 8;

template <int RB, int NT>
constexpr int sp_pitch() { return 16 * RB * NT + 4; }  // f32 per lane of a partial tile in LDS (padded)

template <int RB, int NT>
constexpr size_t sp_smem() {
  constexpr size_t stage = (size_t)kSpWaves * NT * 4096, red = (size_t)kSpWaves * 64 * sp_pitch<RB, NT>() * 4;
  return stage > red ? stage : red;
}

// The low-rank term A2 . B2^T of a tile of RB * 32 outputs from m0 and NT * 32 tokens from n0 on the dense MFMA:
// 16-k steps first, first + step, ... with both operands straight from memory (a few KiB per tile).
template <int RB, int NT>
__device__ __forceinline__ void low_rank_steps(const Gemm24Args& g, f32x16_t (&acc)[RB][NT], int64_t m0, int64_t n0,
                                               int first, int step) {
  if (g.K2 <= 0) return;
  const int row = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
  const Rsrc rs = make_rsrc(g.A2, g.M * g.lda2 * 2), rz = make_rsrc(g.B2, g.N * g.ldb2 * 2);
  for (int64_t t = first; t * 16 < g.K2; t += step) {
    const int64_t k = t * 16 + 8 * h;  // K2 is a multiple of 8: a lane's 8 k are all in or all out
    bf16x8_t a[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const int64_t m = m0 + i * 32 + row;
      a[i] = __builtin_bit_cast(bf16x8_t, bload(rs, m < g.M && k < g.K2 ? (uint32_t)((m * g.lda2 + k) * 2) : kOob, 0));
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int64_t n = n0 + j * 32 + row;
      const bf16x8_t b =
          __builtin_bit_cast(bf16x8_t, bload(rz, n < g.N && k < g.K2 ? (uint32_t)((n * g.ldb2 + k) * 2) : kOob, 0));
#pragma unroll
      for (int i = 0; i < RB; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b, acc[i][j], 0, 0, 0);
    }
  }
}

// 8 consecutive outputs of one token: bias added to the rounded product, then one (M % 32 == 0: all 8 exist).
__device__ __forceinline__ void store_y8(const Gemm24Args& g, int64_t tok, int64_t col, float (&v)[8]) {
  const bool ybf = g.y_dtype == SF_DTYPE_BF16;
  if (g.bias) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float b = load_elem(g.bias, col + q, g.bias_dtype);
      v[q] = ybf ? hround(hround(v[q]) + b) : v[q] + b;
    }
  }
  const int64_t off = tok * g.ldy + col;
  if (g.y_aligned && (off & 7) == 0) {
    if (ybf) {
      *reinterpret_cast<uint4*>(static_cast<uint16_t*>(g.y) + off) =
          make_uint4(pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7]));
    } else {
      float* yp = static_cast<float*>(g.y) + off;
      *reinterpret_cast<float4*>(yp) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4*>(yp + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if (ybf)
        static_cast<uint16_t*>(g.y)[off + q] = hbits(v[q]);
      else
        static_cast<float*>(g.y)[off + q] = v[q];
    }
  }
}

template <int RB, int NT>
__global__ void __launch_bounds__(64 * kSpWaves) gemm24_split_kernel(Gemm24Args g, int64_t tiles_n) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 31, h = lane >> 5;
  // a row tile's token tiles follow each other on one XCD, so they share the weight in its L2
  int64_t pid = blockIdx.x;
  if (gridDim.x % 8 == 0) pid = (pid % 8) * (gridDim.x / 8) + pid / 8;
  const int64_t tm = pid / tiles_n, n0 = (pid - tm * tiles_n) * (NT * 32);
  const int64_t nk = g.K / 64, mb = g.M / 32;

  const Rsrc rx = make_rsrc(g.x, g.N * g.ldx * 2), rv = make_rsrc(g.vals, g.M * g.K),
             ri = make_rsrc(g.idx, mb * nk * 256);
  uint32_t voff[RB], ioff[RB], xoff[NT * 4], xlds[NT * 4], boff[NT][4];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int64_t rb = tm * RB + i;
    voff[i] = rb < mb ? (uint32_t)((rb * nk * 128 + lane) * 16) : kOob;
    ioff[i] = rb < mb ? (uint32_t)((rb * nk * 64 + lane) * 4) : kOob;
  }
  unsigned char* const xs = smem + wave * (NT * 4096);
#pragma unroll
  for (int q = 0; q < NT * 4; ++q) {  // instruction q copies rows 8 q .. 8 q + 7, 128 bytes each
    const int r = 8 * q + (lane >> 3), c = lane & 7;
    xoff[q] = n0 + r < g.N ? (uint32_t)(((n0 + r) * g.ldx + c * 8) * 2) : kOob;
    xlds[q] = (uint32_t)(r * 128 + ((c ^ ((r ^ (r >> 3)) & 7)) << 4));
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int r = j * 32 + row;
#pragma unroll
    for (int q = 0; q < 4; ++q) boff[j][q] = (uint32_t)(r * 128 + (((2 * q + h) ^ ((r ^ (r >> 3)) & 7)) << 4));
  }

  f32x16_t acc[RB][NT];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x16_t{};

  struct Stage {
    V4 a[RB][2], x[NT * 4];
    uint32_t id[RB];
  };
  auto load = [&](Stage& st, int64_t s) {
#pragma unroll
    for (int i = 0; i < RB; ++i) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) st.a[i][kk] = bload(rv, voff[i], (uint32_t)((s * 2 + kk) * 1024));
      st.id[i] = __builtin_amdgcn_raw_buffer_load_b32(ri, (int)ioff[i], (int)(s * 256), 0);
    }
#pragma unroll
    for (int q = 0; q < NT * 4; ++q) st.x[q] = bload(rx, xoff[q], (uint32_t)(s * 128));
  };
  auto compute = [&](const Stage& st) {
#pragma unroll
    for (int q = 0; q < NT * 4; ++q)
      *reinterpret_cast<uint4*>(xs + xlds[q]) = make_uint4(st.x[q].w[0], st.x[q].w[1], st.x[q].w[2], st.x[q].w[3]);
    wave_lds_fence();
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const bf16x8_t lo = *reinterpret_cast<const bf16x8_t*>(xs + boff[j][2 * kk]);
        const bf16x8_t hi = *reinterpret_cast<const bf16x8_t*>(xs + boff[j][2 * kk + 1]);
        const bf16x16_t b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          const bf16x8_t a = __builtin_bit_cast(bf16x8_t, st.a[i][kk]);
          if (kk == 0)
            acc[i][j] = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a, b, acc[i][j], (int)st.id[i], 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a, b, acc[i][j], (int)st.id[i], 0, 1);
        }
      }
    wave_lds_fence();
  };
  // this wave's stages; loads are unconditional (past its last stage they re-read it), so the waits stay exact
  const int64_t cnt = wave < nk ? (nk - wave + kSpWaves - 1) / kSpWaves : 0;
  if (cnt > 0) {
    const int64_t last = wave + (cnt - 1) * kSpWaves;
    auto at = [&](int64_t i) {
      const int64_t s = wave + i * kSpWaves;
      return s < last ? s : last;
    };
    Stage s0, s1;
    load(s0, at(0));
    int64_t i = 0;
    for (; i + 1 < cnt; i += 2) {
      load(s1, at(i + 1));
      compute(s0);
      load(s0, at(i + 2));
      compute(s1);
    }
    if (i < cnt) compute(s0);
  }
  low_rank_steps<RB, NT>(g, acc, tm * (RB * 32), n0, wave, kSpWaves);

  // The 8 partial tiles through LDS: lane l of wave w holds, per (i, j), out rows
  // 32 i + (e / 4) * 8 + (l / 32) * 4 + e % 4 of token 32 j + l % 32.
  constexpr int P = sp_pitch<RB, NT>();
  float* const red = reinterpret_cast<float*>(smem);
  __syncthreads();  // every wave is done with its x tile
  {
    float* mine = red + (wave * 64 + lane) * P;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 16; e += 4)
          *reinterpret_cast<float4*>(mine + (i * NT + j) * 16 + e) =
              make_float4(acc[i][j][e], acc[i][j][e + 1], acc[i][j][e + 2], acc[i][j][e + 3]);
  }
  __syncthreads();
  constexpr int GRP = 4 * RB;  // groups of 8 outputs of a token
  for (int f = threadIdx.x; f < NT * 32 * GRP; f += 64 * kSpWaves) {
    const int og = f % GRP, n = f / GRP;
    const int64_t tok = n0 + n, col = tm * (RB * 32) + og * 8;
    if (tok >= g.N || col >= g.M) continue;
    const int reg = ((og >> 2) * NT + (n >> 5)) * 16 + (og & 3) * 4, l = n & 31;
    float v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = 0.0f;
#pragma unroll
    for (int w = 0; w < kSpWaves; ++w) {
      const float4 p0 = *reinterpret_cast<const float4*>(red + (w * 64 + l) * P + reg);
      const float4 p1 = *reinterpret_cast<const float4*>(red + (w * 64 + 32 + l) * P + reg);
      v[0] += p0.x; v[1] += p0.y; v[2] += p0.z; v[3] += p0.w;
      v[4] += p1.x; v[5] += p1.y; v[6] += p1.z; v[7] += p1.w;
    }
    store_y8(g, tok, col, v);
  }
}

template <int RB, int NT>
int launch_split(const Gemm24Args& g, hipStream_t st, const char* what) {
  constexpr size_t smem = sp_smem<RB, NT>();
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm24_split_kernel<RB, NT>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     static_cast<int>(smem));
  SF_CHECK_HIP(attr);
  const int64_t tm = ceil_div(g.M, 32 * RB), tn = ceil_div(g.N, 32 * NT);
  SF_CHECK_ARG(tm * tn < (1ll << 31), "grid too large");
  gemm24_split_kernel<RB, NT><<<static_cast<unsigned>(tm * tn), 64 * kSpWaves, smem, st>>>(g, tn);
  return launch_status(what);
}

// ---------------------------------------------------------------------------
// 128 outputs x 128 tokens per workgroup, 2 x 2 waves of 64 x 64: between the
// split-K kernel above and the 256 x 256 tile of gemm24_kernel.  The A operand
// goes straight to registers, x through registers into double-buffered LDS, both
// loaded three stages ahead, one barrier per 64-k stage.  At 236 registers two
// workgroups share a CU, so one's loads and barriers run under the other's MFMAs
// and no hand-made schedule is needed.  Bound by the vector memory path: 40 loads
// of 1 KiB a stage and workgroup are 640 clocks against 256 of MFMA (one stage
// of lead instead of three: 80 against 73 us at K = 11008, one workgroup a CU).
// ---------------------------------------------------------------------------
constexpr int kT24 = 128;
constexpr int kT24Pitch = 68;  // f32 row pitch of the transposed epilogue tile: 64 tokens x 64 outputs per wave
constexpr size_t t24_smem() {
  constexpr size_t ops = 2ull * kT24 * 128, epi = 4ull * 64 * kT24Pitch * 4;
  return ops > epi ? ops : epi;
}

__global__ void __launch_bounds__(256, 2) gemm24_tile_kernel(Gemm24Args g, int64_t tiles_m, int64_t tiles_n) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr uint32_t XBUF = kT24 * 128;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1, row = lane & 31, h = lane >> 5;
  // XCD-contiguous ranges of tiles, in bands of 8 row tiles
  int64_t pid = blockIdx.x;
  if (gridDim.x % 8 == 0) pid = (pid % 8) * (gridDim.x / 8) + pid / 8;
  const int64_t band = 8 * tiles_n, first = pid / band * 8, gm = tiles_m - first < 8 ? tiles_m - first : 8;
  const int64_t in_band = pid % band, m0 = (first + in_band % gm) * kT24, n0 = in_band / gm * kT24;
  const int64_t nk = g.K / 64, mb = g.M / 32;

  const Rsrc rx = make_rsrc(g.x, g.N * g.ldx * 2), rv = make_rsrc(g.vals, g.M * g.K),
             ri = make_rsrc(g.idx, mb * nk * 256);
  uint32_t voff[2], ioff[2], xoff[4], xlds[4], boff[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t rb = m0 / 32 + wm * 2 + i;
    voff[i] = rb < mb ? (uint32_t)((rb * nk * 128 + lane) * 16) : kOob;
    ioff[i] = rb < mb ? (uint32_t)((rb * nk * 64 + lane) * 4) : kOob;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {  // thread t copies 16-byte chunk t % 8 of token rows 32 q + t / 8
    const int r = 32 * q + (threadIdx.x >> 3), c = threadIdx.x & 7;
    xoff[q] = n0 + r < g.N ? (uint32_t)(((n0 + r) * g.ldx + c * 8) * 2) : kOob;
    xlds[q] = (uint32_t)(r * 128 + ((c ^ ((r ^ (r >> 3)) & 7)) << 4));
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = wn * 64 + j * 32 + row;
#pragma unroll
    for (int q = 0; q < 4; ++q) boff[j][q] = (uint32_t)(r * 128 + (((2 * q + h) ^ ((r ^ (r >> 3)) & 7)) << 4));
  }
  f32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16_t{};
  V4 fa[4][2][2], xr[4][4];
  uint32_t fi[4][2];
  auto load = [&](auto set_c, int64_t s) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) fa[set][i][kk] = bload(rv, voff[i], (uint32_t)((s * 2 + kk) * 1024));
      fi[set][i] = __builtin_amdgcn_raw_buffer_load_b32(ri, (int)ioff[i], (int)(s * 256), 0);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) xr[set][q] = bload(rx, xoff[q], (uint32_t)(s * 128));
  };
  auto store_x = [&](auto set_c) {  // x held in set -> LDS buffer set % 2
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<uint4*>(smem + (set & 1) * XBUF + xlds[q]) =
          make_uint4(xr[set][q].w[0], xr[set][q].w[1], xr[set][q].w[2], xr[set][q].w[3]);
  };
  // Stage s in register set s % 4 and LDS buffer s % 2: the loads of stage s + 3 are issued first (past the end
  // they re-read the last stage), then the stage's products, then x of s + 1 goes to the other buffer, whose
  // readers passed the previous barrier.
  auto stage = [&](auto set_c, int64_t s) {
    constexpr int set = decltype(set_c)::value;
    load(std::integral_constant<int, (set + 3) & 3>{}, s + 3 < nk ? s + 3 : nk - 1);
    const unsigned char* xb = smem + (set & 1) * XBUF;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const bf16x8_t lo = *reinterpret_cast<const bf16x8_t*>(xb + boff[j][2 * kk]);
        const bf16x8_t hi = *reinterpret_cast<const bf16x8_t*>(xb + boff[j][2 * kk + 1]);
        const bf16x16_t b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const bf16x8_t a = __builtin_bit_cast(bf16x8_t, fa[set][i][kk]);
          if (kk == 0)
            acc[i][j] = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a, b, acc[i][j], (int)fi[set][i], 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a, b, acc[i][j], (int)fi[set][i], 0, 1);
        }
      }
    }
    store_x(std::integral_constant<int, (set + 1) & 3>{});
    __syncthreads();
  };
  if (nk > 0) {
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using S3 = std::integral_constant<int, 3>;
    load(S0{}, 0);
    load(S1{}, nk > 1 ? 1 : 0);
    load(S2{}, nk > 2 ? 2 : nk - 1);
    store_x(S0{});
    __syncthreads();
    int64_t s = 0;
    for (; s + 3 < nk; s += 4) {
      stage(S0{}, s);
      stage(S1{}, s + 1);
      stage(S2{}, s + 2);
      stage(S3{}, s + 3);
    }
    if (s < nk) stage(S0{}, s);
    if (s + 1 < nk) stage(S1{}, s + 1);
    if (s + 2 < nk) stage(S2{}, s + 2);
  }
  low_rank_steps<2, 2>(g, acc, m0 + wm * 64, n0 + wn * 64, 0, 1);
  // each wave's 64 outputs x 64 tokens transposed through LDS, then 8 outputs of a token per lane
  float* ep = reinterpret_cast<float*>(smem) + wave * (64 * kT24Pitch);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; e += 4)
        *reinterpret_cast<float4*>(ep + (j * 32 + row) * kT24Pitch + i * 32 + (e >> 2) * 8 + h * 4) =
            make_float4(acc[i][j][e], acc[i][j][e + 1], acc[i][j][e + 2], acc[i][j][e + 3]);
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int flat = it * 64 + lane, t = flat >> 3, oc = (flat & 7) * 8;
    const int64_t tok = n0 + wn * 64 + t, col = m0 + wm * 64 + oc;
    if (tok >= g.N || col >= g.M) continue;
    float v[8];
    const float4 p0 = *reinterpret_cast<const float4*>(ep + t * kT24Pitch + oc);
    const float4 p1 = *reinterpret_cast<const float4*>(ep + t * kT24Pitch + oc + 4);
    v[0] = p0.x; v[1] = p0.y; v[2] = p0.z; v[3] = p0.w;
    v[4] = p1.x; v[5] = p1.y; v[6] = p1.z; v[7] = p1.w;
    store_y8(g, tok, col, v);
  }
}

int launch_tile(const Gemm24Args& g, hipStream_t st, const char* what) {
  const int64_t tm = ceil_div(g.M, kT24), tn = ceil_div(g.N, kT24);
  SF_CHECK_ARG(tm * tn < (1ll << 31), "grid too large");
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm24_tile_kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     static_cast<int>(t24_smem()));
  SF_CHECK_HIP(attr);
  gemm24_tile_kernel<<<static_cast<unsigned>(tm * tn), 256, t24_smem(), st>>>(g, tm, tn);
  return launch_status(what);
}

// Which kernel takes a product, from a time estimate (us) of each.  st = K / 64 stages; w = the kernel's
// workgroups.  Fitted on this card to M x K of 4096 x 4096, 11008 x 4096, 4096 x 11008, 2048 x 2048 and
// 512 x 1024 at 4 .. 8192 tokens (estimates within about 20 % of what was measured):
//   32 x 32 split (two workgroups a CU):   2.5 + 0.075 st per 256 workgroups (a first, partial 256 counts whole)
//   64 x 64 split (one a CU):              (2.5 + 0.145 st) per round of 256
//   128 x 128 tile (two a CU):             3 + 0.8 st per 512, a remainder of at most 256: 0.43 st
//   256 x 256 tile (one a CU):             6 + 1.2 st per 256, a remainder of at most 208: 0.97 st
// e.g. 4096 x 4096: 4 tokens 56 us on the 256 x 256 tile, at most 11 (launch-bound) on the 32 x 32 split; 512
// tokens 63 against 25 (64 x 64); 1537 tokens 64 against 48 (128 x 128); 4096 tokens 80 against 100.
// 4096 x 11008: 1537 tokens 148 against 124 us, 64 tokens 140 against 16.
enum Kind24 { kSplit32, kSplit64, kTile128, kTile256 };

Kind24 gemm24_kind(const Gemm24Args& g) {
  const double st = static_cast<double>(g.K / 64);
  auto wgs = [&](int64_t m, int64_t n) { return static_cast<double>(ceil_div(g.M, m) * ceil_div(g.N, n)); };
  auto rounds = [](double w, double per, double lim, double full, double part) {
    const double whole = static_cast<double>(static_cast<int64_t>(w / per)), rem = w - whole * per;
    return whole * full + (rem <= 0 ? 0.0 : (rem <= lim ? part : full));
  };
  const double w32 = wgs(32, 32) / 256, w64 = wgs(64, 64);
  const double t[4] = {2.5 + 0.075 * st * (w32 < 1 ? 1 : w32), rounds(w64, 256, 0, 1, 1) * (2.5 + 0.145 * st),
                       3 + st * rounds(wgs(128, 128), 512, 256, 0.8, 0.43),
                       6 + st * rounds(wgs(256, 256), 256, 208, 1.2, 0.97)};
  int best = kSplit32;
  for (int k = kSplit64; k <= kTile256; ++k)
    if (t[k] < t[best]) best = k;
  return static_cast<Kind24>(best);
}

}  // namespace

bool gemm24_split_takes(const Gemm24Args& g) { return gemm24_kind(g) != kTile256; }

int launch_gemm24_split(const Gemm24Args& g, hipStream_t st, const char* what) {
  switch (gemm24_kind(g)) {
    case kSplit32: return launch_split<1, 1>(g, st, what);
    case kSplit64: return launch_split<2, 2>(g, st, what);
    default: return launch_tile(g, st, what);
  }
}

}  // namespace sf
