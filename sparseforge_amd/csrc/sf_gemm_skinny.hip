// bf16 products with a side of C of at most 64: the SLoRB terms z = x P^T, dz = dy S,
// dP = dz^T x, dS = dy^T z, and a layer's products on up to 64 tokens.
//   C[M, N] = sum_k A(m, k) B(n, k), either operand K-contiguous or row-contiguous
//
// Bound by reading the long operand once; a 64-wide side gives few output tiles, so
// K has to be split, and f32 partials with a second launch cost as much as the
// product (z of the 1.1B model's q projection at 2048 tokens: 8 us and 4 more for
// its reduce).  Here a workgroup owns (32 or 64) x (32 or 64) of C and its 8 waves
// split K among themselves: wave w takes the 64-k stages w, w + 8, ...  Each wave
// stages both operands through its own LDS tile (whole 128-byte lines from memory,
// one stage ahead in registers, no barrier: a wave's LDS accesses are performed in
// order), row-contiguous ones as k-rows read back transposed, and the 8 partial
// tiles meet in LDS, summed in wave order by threads that own 8 consecutive columns
// of a row, so C leaves with its epilogue and results do not vary between runs.  K is
// split over workgroups as well where few tiles meet a long K (skinny_plan).
// Kernel + reduce at rank 64, z / dP, before (128 x 64 tiles, K split over
// workgroups) and here: 2048 tokens 2048 -> 2048 15.5 / 15.8 us and 8.5 / 8.3; 4096
// tokens 15.5 / 16.9 and 9.3 / 13; 8192 tokens 4096 -> 11008 19.5 / 22 and 20 / 21,
// its dS 49 and 37 (what the long operand takes to read).
#include <type_traits>

#include "sf_mfma.hpp"

namespace sf {
namespace {

constexpr int kSkWaves = 8;

// One operand's stage: NB * 32 rows x 64 k.  L = 0: 128-byte rows of 8 k-chunks, chunk XOR f(row) =
// (row ^ row / 8) & 7.  L = 1: 64 k-rows of NB * 4 chunks; with 8 chunks, chunk XOR 4 ((k / 2) & 1), so the four
// rows that a transposed read takes lie in different banks.
template <int L, int NB>
struct SkOperand {
  static constexpr int CPR = L == 0 ? 8 : NB * 4, ROWS = 64 / CPR, N = NB * 4;  // chunks a row, rows an instruction
  Rsrc rs;
  uint32_t off[N], lds[N];
  uint32_t step;  // bytes a stage advances
  int64_t K;
  int kc;         // L = 0: the lane's k within a stage
  V4 v[2][N];

  __device__ __forceinline__ void init(const void* base, int64_t ld, int64_t row0, int64_t rows, int64_t k_end) {
    const int lane = threadIdx.x & 63;
    K = k_end;
    kc = (lane & 7) * 8;
    rs = make_rsrc(base, (L == 0 ? rows : k_end) * ld * 2);
    step = L == 0 ? 128u : (uint32_t)(64 * ld * 2);
#pragma unroll
    for (int q = 0; q < N; ++q) {
      const int r = q * ROWS + lane / CPR, c = lane % CPR;
      if constexpr (L == 0) {
        off[q] = row0 + r < rows ? (uint32_t)(((row0 + r) * ld + c * 8) * 2) : kOob;
        lds[q] = (uint32_t)(r * 128 + ((c ^ ((r ^ (r >> 3)) & 7)) << 4));
      } else {
        const int64_t col = row0 + c * 8;
        off[q] = col < rows ? (uint32_t)((r * ld + col) * 2) : kOob;  // k rows past K lie past the extent
        lds[q] = (uint32_t)(r * (NB * 64) + ((NB == 2 ? c ^ (4 * ((r >> 1) & 1)) : c) << 4));
      }
    }
  }
  template <int SET>
  __device__ __forceinline__ void load(int64_t s) {
    const uint32_t so = (uint32_t)s * step;
    const bool ok = L == 1 || s * 64 + kc < K;  // K is a multiple of 8 where a chunk lies along it
#pragma unroll
    for (int q = 0; q < N; ++q) {
      if constexpr (L == 0)
        v[SET][q] = bload(rs, ok ? off[q] : kOob, so);
      else
        v[SET][q] = bload(rs, off[q] == kOob ? kOob : off[q] + so, 0);
    }
  }
  template <int SET>
  __device__ __forceinline__ void store(unsigned char* t) const {
#pragma unroll
    for (int q = 0; q < N; ++q)
      *reinterpret_cast<uint4*>(t + lds[q]) =
          make_uint4(v[SET][q].w[0], v[SET][q].w[1], v[SET][q].w[2], v[SET][q].w[3]);
  }
  // Fragment of rows [32 b, 32 b + 32) at k-step kk: lane's row lane % 32, k 8 (lane / 32) ..
  static __device__ __forceinline__ bf16x8_t frag(const unsigned char* t, int b, int kk) {
    const int lane = threadIdx.x & 63;
    if constexpr (L == 0) {
      const int r = b * 32 + (lane & 31);
      return *reinterpret_cast<const bf16x8_t*>(t + r * 128 + (((2 * kk + (lane >> 5)) ^ ((r ^ (r >> 3)) & 7)) << 4));
    } else {
      typedef short v4i16_t __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) v4i16_t lds_v4;
      const int grp = lane >> 4, i = lane & 15, k = kk * 16 + 8 * (grp >> 1) + (i >> 2);
      const int col = b * 32 + 16 * (grp & 1) + 4 * (i & 3), c = col >> 3;
      const unsigned char* p = t + k * (NB * 64) + ((NB == 2 ? c ^ (4 * ((k >> 1) & 1)) : c) << 4) + (col & 7) * 2;
      const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(p));
      const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(p + 4 * NB * 64));
      return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  }
};

template <int NY, int NX>
constexpr int sk_pitch() { return 16 * NY * NX + 4; }  // f32 per lane of a partial tile in LDS (padded)
template <int NY, int NX>
constexpr size_t sk_smem() {
  constexpr size_t stage = (size_t)kSkWaves * (NY + NX) * 4096, red = (size_t)kSkWaves * 64 * sk_pitch<NY, NX>() * 4;
  return stage > red ? stage : red;
}

// NY * 32 rows of C (A) x NX * 32 columns (B).  The MFMA's rows are C's columns, so a lane holds four consecutive
// columns of its C row.
template <int AL, int BL, int NY, int NX>
__global__ void __launch_bounds__(64 * kSkWaves) skinny_kernel(GemmArgs g) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t tiles = g.tiles_m * g.tiles_n, kz = blockIdx.x / tiles, pid = blockIdx.x - kz * tiles;
  const int64_t m0 = pid % g.tiles_m * (NY * 32), n0 = pid / g.tiles_m * (NX * 32);
  SkOperand<AL, NY> ya;
  SkOperand<BL, NX> xb;
  ya.init(g.A1, g.lda1, m0, g.M, g.K1);
  xb.init(g.B1, g.ldb1, n0, g.N, g.K1);
  unsigned char* const ty = smem + wave * ((NY + NX) * 4096);
  unsigned char* const tx = ty + NY * 4096;
  f32x16_t acc[NX][NY];
#pragma unroll
  for (int i = 0; i < NX; ++i)
#pragma unroll
    for (int j = 0; j < NY; ++j) acc[i][j] = f32x16_t{};
  auto compute = [&](auto set_c) {
    constexpr int SET = decltype(set_c)::value;
    ya.template store<SET>(ty);
    xb.template store<SET>(tx);
    wave_lds_fence();
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      bf16x8_t y[NY], x[NX];
#pragma unroll
      for (int j = 0; j < NY; ++j) y[j] = ya.frag(ty, j, kk);
#pragma unroll
      for (int i = 0; i < NX; ++i) x[i] = xb.frag(tx, i, kk);
#pragma unroll
      for (int i = 0; i < NX; ++i)
#pragma unroll
        for (int j = 0; j < NY; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[i], y[j], acc[i][j], 0, 0, 0);
    }
    wave_lds_fence();
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  // this wave's stages of the workgroup's K range; loads are unconditional (past its last stage they re-read it)
  const int64_t nk = ceil_div(g.K1, 64), k0 = kz * g.split_stages;
  const int64_t k1 = k0 + g.split_stages < nk ? k0 + g.split_stages : nk;
  const int64_t first = k0 + wave, cnt = first < k1 ? (k1 - first + kSkWaves - 1) / kSkWaves : 0;
  if (cnt > 0) {
    auto at = [&](int64_t i) { return first + (i < cnt ? i : cnt - 1) * kSkWaves; };
    ya.template load<0>(at(0));
    xb.template load<0>(at(0));
    int64_t i = 0;
    for (; i + 1 < cnt; i += 2) {
      ya.template load<1>(at(i + 1));
      xb.template load<1>(at(i + 1));
      compute(S0{});
      ya.template load<0>(at(i + 2));
      xb.template load<0>(at(i + 2));
      compute(S1{});
    }
    if (i < cnt) compute(S0{});
  }
  // partial tiles: lane l of wave w holds, per (i, j), C columns 32 i + (e / 4) * 8 + (l / 32) * 4 + e % 4 of C row
  // 32 j + l % 32
  constexpr int P = sk_pitch<NY, NX>();
  float* const red = reinterpret_cast<float*>(smem);
  __syncthreads();
  {
    float* mine = red + (wave * 64 + lane) * P;
#pragma unroll
    for (int i = 0; i < NX; ++i)
#pragma unroll
      for (int j = 0; j < NY; ++j)
#pragma unroll
        for (int e = 0; e < 16; e += 4)
          *reinterpret_cast<float4*>(mine + (i * NY + j) * 16 + e) =
              make_float4(acc[i][j][e], acc[i][j][e + 1], acc[i][j][e + 2], acc[i][j][e + 3]);
  }
  __syncthreads();
  constexpr int GRP = 4 * NX;  // groups of 8 columns of a row
  for (int f = threadIdx.x; f < NY * 32 * GRP; f += 64 * kSkWaves) {
    const int og = f % GRP, r = f / GRP;
    const int64_t row = m0 + r, col = n0 + og * 8;
    if (row >= g.M || col >= g.N) continue;
    const int reg = ((og >> 2) * NY + (r >> 5)) * 16 + (og & 3) * 4, l = r & 31;
    float v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = 0.0f;
#pragma unroll
    for (int w = 0; w < kSkWaves; ++w) {
      const float4 p0 = *reinterpret_cast<const float4*>(red + (w * 64 + l) * P + reg);
      const float4 p1 = *reinterpret_cast<const float4*>(red + (w * 64 + 32 + l) * P + reg);
      v[0] += p0.x; v[1] += p0.y; v[2] += p0.z; v[3] += p0.w;
      v[4] += p1.x; v[5] += p1.y; v[6] += p1.z; v[7] += p1.w;
    }
    store_c8<SF_DTYPE_BF16>(g, row, col, kz, v);
  }
}

struct SkPlan {
  int ny, nx, splits;
};

// Tile (32 or 64 of the long side) and K splits over workgroups from a time estimate (us), fitted on 8 shapes at
// 4 .. 8192 tokens with every choice measured: a workgroup takes 3.2 and, per stage of a wave (n of them), 1.1 for a
// K-contiguous long operand in 32-row tiles, 1.45 in 64-row ones, 1.75 for a row-contiguous one in 64-wide tiles, 1.5
// or (above 128 workgroups) 1.9 in 32-wide ones, which read half cache lines; the long operand cannot come faster than about 4.8 TB/s; K split over workgroups costs 9
// for the reduce, its launch and the workspace.  E.g. [64, 4096 tokens]^T [4096, 2048] sp 1 17.1 us, sp 4 8.8 + 3.9;
// at 11008 x 8192 tokens 32-wide 72, 64-wide 37.
SkPlan skinny_plan(int64_t M, int64_t N, int64_t K, bool long_rows, int max_splits) {
  const bool short_m = M <= N;
  const int64_t s = short_m ? M : N, l = short_m ? N : M, stages = ceil_div(K, 64);
  const int ns = s <= 32 ? 1 : 2;
  SkPlan best{};
  double best_cost = -1;
  for (int nl = 2; nl >= 1; --nl) {
    const int64_t tiles = ceil_div(l, 32 * nl) * ceil_div(s, 32 * ns);
    const double stage = !long_rows ? (nl == 1 ? 1.1 : 1.45) : (nl == 2 ? 1.75 : (tiles <= 128 ? 1.5 : 1.9));
    for (int sp = 1; sp <= max_splits && (sp == 1 || stages / sp >= kSkWaves); ++sp) {
      const int64_t per = ceil_div(stages, sp);
      if ((sp - 1) * per >= stages && sp > 1) continue;  // an empty last split
      const double lat = ceil_div(tiles * sp, 256) * (3.2 + stage * ceil_div(per, kSkWaves)), read = 2.0 * l * K / 4.8e6;
      const double cost = (lat > read ? lat : read) + 0.1 * lat + (sp > 1 ? 9.0 + 2.0 * sp * M * N * 4.0 / 5e6 : 0.0);
      if (best_cost < 0 || cost < best_cost) {
        best_cost = cost;
        best = {short_m ? ns : nl, short_m ? nl : ns, sp};
      }
    }
  }
  return best;
}
constexpr int kSkMaxSplits = 16;

template <int AL, int BL, int NY, int NX>
int launch_tile(const GemmArgs& g, hipStream_t st) {
  constexpr size_t smem = sk_smem<NY, NX>();
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(skinny_kernel<AL, BL, NY, NX>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     static_cast<int>(smem));
  SF_CHECK_HIP(attr);
  skinny_kernel<AL, BL, NY, NX>
      <<<static_cast<unsigned>(g.tiles_m * g.tiles_n * g.splits), 64 * kSkWaves, smem, st>>>(g);
  return launch_status("sf_gemm (skinny)");
}

template <int AL, int BL>
int launch_tiles(const SkPlan& p, const GemmArgs& g, hipStream_t st) {
  if (p.ny == 1) return p.nx == 1 ? launch_tile<AL, BL, 1, 1>(g, st) : launch_tile<AL, BL, 1, 2>(g, st);
  return p.nx == 1 ? launch_tile<AL, BL, 2, 1>(g, st) : launch_tile<AL, BL, 2, 2>(g, st);
}

}  // namespace

size_t gemm_skinny_workspace(int64_t M, int64_t N, int64_t K, int a_layout, int b_layout) {
  const int sp = skinny_plan(M, N, K, (M <= N ? b_layout : a_layout) == SF_LAYOUT_MN, kSkMaxSplits).splits;
  return sp > 1 ? static_cast<size_t>(sp) * M * N * sizeof(float) : 0;  // K split over the waves alone needs none
}

int launch_gemm_skinny(GemmArgs g, int a_layout, int b_layout, void* workspace, size_t workspace_bytes, hipStream_t st) {
  // as many K splits over workgroups as the workspace holds partials for
  const size_t per = static_cast<size_t>(g.M) * g.N * sizeof(float);
  const bool ws = workspace && (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0;
  const size_t cap = ws ? workspace_bytes / per : 1;
  const SkPlan p = skinny_plan(g.M, g.N, g.K1, (g.M <= g.N ? b_layout : a_layout) == SF_LAYOUT_MN,
                               cap > kSkMaxSplits ? kSkMaxSplits : (cap < 1 ? 1 : static_cast<int>(cap)));
  g.tiles_m = ceil_div(g.M, 32 * p.ny);
  g.tiles_n = ceil_div(g.N, 32 * p.nx);
  g.splits = p.splits;
  g.split_stages = ceil_div(ceil_div(g.K1, 64), p.splits);
  g.partial = p.splits > 1 ? static_cast<float*>(workspace) : nullptr;
  SF_CHECK_ARG(g.tiles_m * g.tiles_n * p.splits < (1ll << 31), "GEMM grid too large");
  int rc;
  if (a_layout == SF_LAYOUT_K && b_layout == SF_LAYOUT_K)
    rc = launch_tiles<0, 0>(p, g, st);
  else if (a_layout == SF_LAYOUT_K)
    rc = launch_tiles<0, 1>(p, g, st);
  else
    rc = launch_tiles<1, 1>(p, g, st);
  if (rc || p.splits == 1) return rc;
  return launch_splitk_reduce(g, SF_DTYPE_BF16, st, "sf_gemm (skinny reduce)");
}

}  // namespace sf
