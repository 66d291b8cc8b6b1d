// bf16 products on 128 x 128 tiles: the shapes whose 256 x 256 tile grid leaves
// compute units idle (the 1.1B model's linears at 2048 or 4096 tokens: 64 to 200
// tiles for 256 CUs), which used to run half the GPU or split K and pay for f32
// partials.
//
// 4 waves of 64 x 64 (2 x 2 blocks of v_mfma_f32_32x32x16_bf16), stages of 64 k
// copied global -> LDS by direct-to-LDS buffer loads (the layouts of
// gemm_bf16_kernel: K-contiguous rows with XOR-swizzled chunks, M/N-contiguous
// k-rows read back transposed), double-buffered in 64 KiB so that two workgroups
// share a CU: one's copies and barriers run under the other's MFMAs, which the
// 256 x 256 tile with its single wave per SIMD has to schedule by hand.  A stage
// copies 32 KiB for 512 MFMA clocks, so at full rate two workgroups would need 64
// bytes a clock and CU from the L2: that, not the MFMA rate, is the bound, and
// the 256 x 256 tile (half the bytes per flop) stays where its grid fills the GPU.
#include <type_traits>

#include "sf_mfma.hpp"

namespace sf {
namespace {

constexpr int kMid = 128, kMidThreads = 256;
constexpr uint32_t kMidBuf = 16384;            // one operand's stage: 128 rows x 128 B, or 64 k x 256 B
constexpr int kMidEpi = 68;                    // f32 pitch of the epilogue tile (32 rows x 64 columns per wave)
constexpr size_t kMidSmem = 4ull * kMidBuf;

// One 16-byte-per-lane copy global -> LDS (lane l's bytes land at lds + 16 l), untracked by the compiler: the kernel
// waits for its copies itself before the barrier that publishes a buffer.
__device__ __forceinline__ void copy16(Rsrc r, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(r), "s"(soff) : "memory", "m0");
}

// Copies of one operand.  L = 0 (K-contiguous): wave w's instruction i covers rows 32 w + 8 i + l / 8, slot l % 8
// holding chunk (l % 8) ^ f(row), f(row) = (row ^ row / 8) & 7.  L = 1: k-rows 16 w + 4 i + l / 16, slot l % 16
// holding column chunk (l % 16) ^ 4 (row & 3).  Rows, columns and k past the operand read zeros.
template <int L>
struct MidCopy {
  Rsrc rs;
  uint32_t off[4];
  uint32_t step;  // L = 1: bytes of a stage
  int64_t k_end;
  int chunk[4];

  __device__ __forceinline__ void init(const void* base, int64_t ld, int64_t row0, int64_t rows, int64_t K,
                                       int64_t kstart) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    k_end = K;
    if constexpr (L == 0) {
      rs = make_rsrc(base, rows * ld * 2);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t r = row0 + 32 * w + 8 * i + (lane >> 3);
        chunk[i] = (lane & 7) ^ (lane >> 3) ^ ((4 * w + i) & 7);
        off[i] = r < rows ? (uint32_t)((r * ld + chunk[i] * 8) * 2) : kOob;
      }
      step = 0;
    } else {
      rs = make_rsrc(base, K * ld * 2);
      step = (uint32_t)(64 * ld * 2);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * w + 4 * i + (lane >> 4);
        const int64_t col = row0 + 8 * ((lane & 15) ^ (4 * (r & 3)));
        off[i] = col < rows ? (uint32_t)(((kstart + r) * ld + col) * 2) : kOob;
      }
    }
  }
  // The stage at k0 (L = 1: the next one, from kstart on) into `lds`.
  __device__ __forceinline__ void issue(uint32_t lds, int64_t k0) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (L == 0) {
        copy16(rs, lds + w * 4096 + i * 1024, k0 + chunk[i] * 8 < k_end ? off[i] : kOob, (uint32_t)(k0 * 2));
      } else {
        copy16(rs, lds + w * 4096 + i * 1024, off[i], 0);
        off[i] = off[i] >= kOob ? kOob : off[i] + step;
      }
    }
  }
};

// Lane offset of the fragment of operand rows [r0, r0 + 32) at k-step 0, and the fragment at k-step kk.
template <int L>
__device__ __forceinline__ uint32_t mid_base(int r0) {
  const int lane = threadIdx.x & 63;
  if constexpr (L == 0) {
    const int r = r0 + (lane & 31);
    return (uint32_t)(r * 128 + ((((r ^ (r >> 3)) & 7) ^ (lane >> 5)) << 4));
  } else {
    const int grp = lane >> 4, t = lane & 15, q = t >> 2, k = 8 * (grp >> 1) + q;
    const int col = r0 + 16 * (grp & 1) + 4 * (t & 3);
    return (uint32_t)(k * 256 + (((col >> 3) ^ (4 * q)) << 4) + (col & 7) * 2);
  }
}
template <int L>
__device__ __forceinline__ bf16x8_t mid_frag(const unsigned char* tile, uint32_t base, int kk) {
  if constexpr (L == 0) {
    return *reinterpret_cast<const bf16x8_t*>(tile + (base ^ (uint32_t)(kk << 5)));
  } else {
    typedef short v4i16_t __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v4i16_t lds_v4;
    const unsigned char* p = tile + base + kk * 4096;
    const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(p));
    const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(p + 1024));
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
}

template <int AL, int BL>
__global__ void __launch_bounds__(kMidThreads, 2) gemm_mid_kernel(GemmArgs g) {
  extern __shared__ __align__(16) unsigned char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)smem;
  const int64_t tiles = g.tiles_m * g.tiles_n, kz = blockIdx.x / tiles;
  int64_t tm, tn;
  tile_coords(blockIdx.x - kz * tiles, g.tiles_m, g.tiles_n, tm, tn);
  const int64_t m0 = tm * kMid, n0 = tn * kMid;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave >> 1, wn = wave & 1;
  f32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16_t{};
  uint32_t ab[2], bb[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    ab[i] = mid_base<AL>(wm * 64 + i * 32);
    bb[i] = mid_base<BL>(wn * 64 + i * 32);
  }
  MidCopy<AL> ca;
  MidCopy<BL> cb;
  // Stages [s, e) of the segment the copies were set up for: A in the first half of LDS (two buffers), B in the second.
  auto segment = [&](int64_t s, int64_t e) {
    if (s >= e) return;
    __syncthreads();  // every wave is done with what the buffers held
    ca.issue(lds0, s * 64);
    cb.issue(lds0 + 2 * kMidBuf, s * 64);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (int64_t st = s; st < e; ++st) {
      const int buf = static_cast<int>((st - s) & 1);
      if (st + 1 < e) {  // the other buffer's readers passed the previous barrier
        ca.issue(lds0 + (buf ^ 1) * kMidBuf, (st + 1) * 64);
        cb.issue(lds0 + 2 * kMidBuf + (buf ^ 1) * kMidBuf, (st + 1) * 64);
      }
      const unsigned char *at = smem + buf * kMidBuf, *bt = smem + 2 * kMidBuf + buf * kMidBuf;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        bf16x8_t a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a[i] = mid_frag<AL>(at, ab[i], kk);
          b[i] = mid_frag<BL>(bt, bb[i], kk);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      __builtin_amdgcn_s_waitcnt(0);  // this wave's copies of the next stage have landed
      __syncthreads();
    }
  };
  const int64_t nk1 = ceil_div(g.K1, 64), s0 = kz * g.split_stages;
  const int64_t s1 = s0 + g.split_stages < nk1 ? s0 + g.split_stages : nk1;
  ca.init(g.A1, g.lda1, m0, g.M, g.K1, s0 * 64);
  cb.init(g.B1, g.ldb1, n0, g.N, g.K1, s0 * 64);
  segment(s0, s1);
  if (g.A2 && kz == g.splits - 1) {
    ca.init(g.A2, g.lda2, m0, g.M, g.K2, 0);
    cb.init(g.B2, g.ldb2, n0, g.N, g.K2, 0);
    segment(0, ceil_div(g.K2, 64));
  }
  // Epilogue: 32 rows x 64 columns of a wave at a time through LDS, then 8 columns of a row per lane.
  float* ep = reinterpret_cast<float*>(smem) + wave * (32 * kMidEpi);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        ep[((e >> 2) * 8 + (lane >> 5) * 4 + (e & 3)) * kMidEpi + j * 32 + (lane & 31)] = acc[i][j][e];
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int flat = it * 64 + lane, r = flat >> 3, c = (flat & 7) * 8;
      const int64_t row = m0 + wm * 64 + i * 32 + r, col = n0 + wn * 64 + c;
      if (row >= g.M || col >= g.N) continue;
      float v[8];
      const float4 p0 = *reinterpret_cast<const float4*>(ep + r * kMidEpi + c);
      const float4 p1 = *reinterpret_cast<const float4*>(ep + r * kMidEpi + c + 4);
      v[0] = p0.x; v[1] = p0.y; v[2] = p0.z; v[3] = p0.w;
      v[4] = p1.x; v[5] = p1.y; v[6] = p1.z; v[7] = p1.w;
      store_c8<SF_DTYPE_BF16>(g, row, col, kz, v);
    }
  }
}

template <int AL, int BL>
int launch_mid(const GemmArgs& g, hipStream_t st) {
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_mid_kernel<AL, BL>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     static_cast<int>(kMidSmem));
  SF_CHECK_HIP(attr);
  gemm_mid_kernel<AL, BL><<<static_cast<unsigned>(g.tiles_m * g.tiles_n * g.splits), kMidThreads, kMidSmem, st>>>(g);
  return launch_status("sf_gemm (128 x 128)");
}

}  // namespace

// K splits on 128 x 128 tiles, or 0 where the 256 x 256 tiles (in `big_splits` K splits) are estimated faster.  Times
// in us fitted on this card (estimates within about 10 % of what was measured): a stage of 64 k takes 0.85 for one
// 128 x 128 workgroup on its CU and 1.1 for two, 1.7 for a 256 x 256 workgroup; a K split adds a launch and moves
// the f32 partials twice at about 5 TB/s.  Against the 256 x 256 tiles at M, N, K: 4096, 2048, 2048 (128 tiles) 57 ->
// 39 us; 2048, 2048, 2048 (64 tiles in 4 splits) 46 -> 30; 512, 2048, 2048 30 -> 22; kept at 5632, 2048, 2048 (176
// tiles) 57 against 61 and 8192, 4096, 4096.
int gemm_mid_splits(int64_t M, int64_t N, int64_t K, int max_splits, int big_splits) {
  const int64_t stages = ceil_div(K, 64), mid = ceil_div(M, kMid) * ceil_div(N, kMid),
                big = ceil_div(M, 256) * ceil_div(N, 256);
  auto split_cost = [&](int sp) { return sp > 1 ? 4.0 + 2.0 * sp * static_cast<double>(M) * N * 4.0 / 5e6 : 0.0; };
  double best_cost = 5.0 + 1.7 * ceil_div(stages, big_splits) * ceil_div(big * big_splits, 256) + split_cost(big_splits);
  int best = 0;
  for (int sp = 1; sp <= max_splits && (sp == 1 || stages / sp >= 2); ++sp) {
    const int64_t per = ceil_div(stages, sp), n = mid * sp, rem = n % 512;
    if ((sp - 1) * per >= stages && sp > 1) continue;  // an empty last split
    const double rounds = static_cast<double>(n / 512) * 1.1 + (rem == 0 ? 0.0 : (rem <= 256 ? 0.85 : 1.1));
    const double cost = 3.0 + rounds * per + split_cost(sp);
    if (cost < best_cost) {
      best_cost = cost;
      best = sp;
    }
  }
  return best;
}

int launch_gemm_mid(GemmArgs g, int a_layout, int b_layout, int splits, void* workspace, hipStream_t st) {
  g.tiles_m = ceil_div(g.M, kMid);
  g.tiles_n = ceil_div(g.N, kMid);
  g.splits = splits;
  g.split_stages = ceil_div(ceil_div(g.K1, 64), splits);
  g.partial = splits > 1 ? static_cast<float*>(workspace) : nullptr;
  SF_CHECK_ARG(g.tiles_m * g.tiles_n * splits < (1ll << 31), "GEMM grid too large");
  int rc;
  if (a_layout == SF_LAYOUT_K && b_layout == SF_LAYOUT_K)
    rc = launch_mid<0, 0>(g, st);
  else if (a_layout == SF_LAYOUT_K)
    rc = launch_mid<0, 1>(g, st);
  else
    rc = launch_mid<1, 1>(g, st);
  if (rc || splits == 1) return rc;
  return launch_splitk_reduce(g, SF_DTYPE_BF16, st, "sf_gemm (split-K reduce)");
}

}  // namespace sf
