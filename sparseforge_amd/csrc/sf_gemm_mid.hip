// bf16 products on 128 x 128 tiles: the shapes whose 256 x 256 tile grid leaves
// compute units idle (the 1.1B model's linears at 2048 or 4096 tokens: 64 to 200
// tiles for 256 CUs), which used to run half the GPU or split K and pay for f32
// partials.
//
// 4 waves of 64 x 64 (2 x 2 blocks of v_mfma_f32_32x32x16_bf16), stages of 64 k
// copied global -> LDS by direct-to-LDS buffer loads (the layouts of
// gemm_bf16_kernel: K-contiguous rows with XOR-swizzled chunks, M/N-contiguous
// k-rows read back transposed) into a ring of stage buffers; a stage's fragments
// are read while the one before multiplies.  Grids of more than one workgroup a CU
// have two share it (a ring of 2, 64 KiB each): one's copies and barriers run under
// the other's MFMAs, and what bounds them is the 32 KiB a stage and workgroup from
// the L2, 1.1 us for two.  Up to one a CU a stage is what its copies' latency makes
// of it, so the ring has 4 buffers and three stages are in flight: 0.62 us a stage,
// 0.85 with one in flight.  Stages of 32 k with more buffers in flight were slower
// (4096, 2048, 2048 nt 50 us against 40: half cache lines), and 256 x 128 tiles, one
// workgroup a CU, gained 5 % at 4096 rows and lost 5 to 25 % below.  The 256 x 256
// tile (half the bytes per flop) stays where its grid fills the GPU.
#include <type_traits>

#include "sf_mfma.hpp"

namespace sf {
namespace {

constexpr int kMid = 128, kMidThreads = 256;
constexpr uint32_t kMidBuf = 16384;            // one operand's stage: 128 rows x 128 B, or 64 k x 256 B
constexpr int kMidEpi = 68;                    // f32 pitch of the epilogue tile (32 rows x 64 columns per wave)

// One 16-byte-per-lane copy global -> LDS (lane l's bytes land at lds + 16 l), untracked by the compiler: the kernel
// waits for its copies itself before the barrier that publishes a buffer.
__device__ __forceinline__ void copy16(Rsrc r, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(r), "s"(soff) : "memory", "m0");
}

// Copies of one operand, 4 instructions a wave and stage.  L = 0 (K-contiguous): wave w's instruction i covers rows
// 32 w + 8 i + l / 8, slot l % 8 holding chunk (l % 8) ^ f(row), f(row) = (row ^ row / 8) & 7.  L = 1: k-rows 16 w + 4 i +
// l / 16, slot l % 16 holding column chunk (l % 16) ^ 4 (row & 3).  Rows, columns and k past the operand or the split
// read zeros.
template <int L>
struct MidCopy {
  Rsrc rs;
  uint32_t off[4];
  uint32_t step;  // bytes of a stage
  int64_t K;
  int kl[4];      // the lane's first k within a stage

  __device__ __forceinline__ void init(const void* base, int64_t ld, int64_t row0, int64_t rows, int64_t k_end) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    K = k_end;
    rs = make_rsrc(base, (L == 0 ? rows : k_end) * ld * 2);
    step = L == 0 ? 128u : (uint32_t)(128 * ld);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (L == 0) {
        const int lr = 32 * w + 8 * i + (lane >> 3);
        kl[i] = 8 * ((lane & 7) ^ ((lr ^ (lr >> 3)) & 7));
        off[i] = row0 + lr < rows ? (uint32_t)(((row0 + lr) * ld + kl[i]) * 2) : kOob;
      } else {
        const int k = 16 * w + 4 * i + (lane >> 4);
        const int64_t col = row0 + 8 * ((lane & 15) ^ (4 * (k & 3)));
        off[i] = col < rows ? (uint32_t)((k * ld + col) * 2) : kOob;
        kl[i] = k;
      }
    }
  }
  // Stage st into `lds`; zeros unless `live`.
  __device__ __forceinline__ void issue(uint32_t lds, int64_t st, bool live) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t so = live ? (uint32_t)st * step : 0u;
    const int left = live ? (K - st * 64 < 64 ? static_cast<int>(K - st * 64) : 64) : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) copy16(rs, lds + w * 4096 + i * 1024, kl[i] < left ? off[i] : kOob, so);
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

// NBUF stage buffers of 32 KiB, WGS workgroups a CU.
template <int AL, int BL, int NBUF, int WGS>
__global__ void __launch_bounds__(kMidThreads, WGS) gemm_mid_kernel(GemmArgs g) {
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
  constexpr int KK = 4, PER = 8;  // MFMA k-steps, copies a wave issues, per stage
  MidCopy<AL> ca;
  MidCopy<BL> cb;
  bf16x8_t fa[2][KK][2], fb[2][KK][2];  // fragments of stage k in set k % 2
  auto read = [&](auto set_c, int buf) {
    constexpr int set = decltype(set_c)::value;
    const unsigned char *at = smem + buf * (2 * kMidBuf), *bt = at + kMidBuf;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fa[set][kk][i] = mid_frag<AL>(at, ab[i], kk);
        fb[set][kk][i] = mid_frag<BL>(bt, bb[i], kk);
      }
  };
  auto mma = [&](auto set_c) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[set][kk][i], fb[set][kk][j], acc[i][j], 0, 0, 0);
  };
  // Stages [s, e) of the segment the copies were set up for.  Buffer k % NBUF holds stage s + k: A, then B.  Stage k's
  // fragments are read while stage k - 1 multiplies; the barrier in between says that stage k has landed for every wave
  // (each waits for all but its newest NBUF - 2 stages of copies) and that stage k - 1 was read, so its buffer takes
  // stage k - 1 + NBUF.  Copies past e are issued as zeros: the counts stay exact.
  auto segment = [&](int64_t s, int64_t e) {
    if (s >= e) return;
    __syncthreads();  // every wave is done with what the buffers held
    auto issue = [&](int64_t st, int buf) {
      ca.issue(lds0 + buf * (2 * kMidBuf), st, st < e);
      cb.issue(lds0 + buf * (2 * kMidBuf) + kMidBuf, st, st < e);
    };
#pragma unroll
    for (int i = 0; i < NBUF; ++i) issue(s + i, i);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 1) * PER) : "memory");
    __syncthreads();
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    read(S0{}, 0);
    int buf = 0;
    auto step = [&](auto set_c, int64_t st) {
      constexpr int set = decltype(set_c)::value;
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NBUF - 2) * PER) : "memory");
      __syncthreads();
      issue(st + NBUF, buf);
      buf = buf + 1 == NBUF ? 0 : buf + 1;
      read(std::integral_constant<int, set ^ 1>{}, buf);
      mma(set_c);
    };
    int64_t st = s;
    for (; st + 1 < e; st += 2) {
      step(S0{}, st);
      step(S1{}, st + 1);
    }
    if (st < e) step(S0{}, st);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no copy is left to land in what follows
  };
  const int64_t nk1 = ceil_div(g.K1, 64), s0 = kz * g.split_stages;
  const int64_t s1 = s0 + g.split_stages < nk1 ? s0 + g.split_stages : nk1;
  ca.init(g.A1, g.lda1, m0, g.M, g.K1);
  cb.init(g.B1, g.ldb1, n0, g.N, g.K1);
  segment(s0, s1);
  if (g.A2 && kz == g.splits - 1) {
    ca.init(g.A2, g.lda2, m0, g.M, g.K2);
    cb.init(g.B2, g.ldb2, n0, g.N, g.K2);
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

template <int AL, int BL, int NBUF, int WGS>
int launch_mid_as(const GemmArgs& g, int64_t wgs, hipStream_t st) {
  constexpr size_t smem = NBUF * 2ull * kMidBuf;
  static_assert(smem * WGS <= 160 * 1024 && smem >= 4 * 32 * kMidEpi * 4);
  constexpr auto kern = gemm_mid_kernel<AL, BL, NBUF, WGS>;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     static_cast<int>(smem));
  SF_CHECK_HIP(attr);
  kern<<<static_cast<unsigned>(wgs), kMidThreads, smem, st>>>(g);
  return launch_status("sf_gemm (128 x 128)");
}

// Up to one workgroup a CU, 4 buffers: three stages of copies in flight instead of one (2048, 2048, 2048, 256
// workgroups: 23 us against 27 to 31 on 2 buffers).  Above, 2 buffers and two workgroups a CU (4096, 2048, 2048, 512
// workgroups: 40 us against 46 to 50).
template <int AL, int BL>
int launch_mid(const GemmArgs& g, hipStream_t st) {
  const int64_t wgs = g.tiles_m * g.tiles_n * g.splits;
  return wgs <= 256 ? launch_mid_as<AL, BL, 4, 1>(g, wgs, st) : launch_mid_as<AL, BL, 2, 2>(g, wgs, st);
}

}  // namespace

// K splits on 128 x 128 tiles, or 0 where the 256 x 256 tiles (in `big_splits` K splits) are estimated faster.  Times
// in us fitted on this card (estimates within about 10 % of what was measured): a stage of 64 k takes 0.62 for a
// 128 x 128 workgroup alone on its CU (0.85 in the tail of a larger grid) and 1.1 for two, 1.7 for a 256 x 256 workgroup; a K split adds a launch and moves
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
    const double rounds = static_cast<double>(n / 512) * 1.1 + (rem == 0 ? 0.0 : (rem > 256 ? 1.1 : (n <= 256 ? 0.62 : 0.85)));
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
