// The f32 products of a SparseLinear (dense, unmasked operands; the masked
// weight is written by one elementwise pass before them):
//   C[M, N] = sum_k A(m, k) B(n, k)  (+ segment 2: sum_k A2(m, k) B2(n, k))
// on v_mfma_f32_32x32x2_f32 with f32 accumulation.
//
// Bound by the f32 matrix rate (157 TFLOP/s published; 64 clocks per MFMA): a
// 64 x 64 wave tile needs 1 KiB of LDS reads per 256 MFMA clocks, so the tile
// matters little and what costs is an uneven last round of workgroups.  Tiles
// of 128 x 128, 128 x 64, 64 x 64 and, for a side of at most 32, 128 x 32 and
// 32 x 128 (4 waves each), split over K when that fills the GPU more evenly
// (f32_plan).  Stages of 32 k go global -> registers (one stage ahead) -> LDS
// rows of 36 words; a lane reads 4 consecutive k of its row with one 16-byte
// access and feeds them to four MFMAs (half-wave h holds k 4 h .. 4 h + 3 of
// each 8: the contraction may take k in any order, the same for A and B).  M/N-
// contiguous operands are loaded as 4 x 4 blocks per thread, whose transpose is
// a renaming of registers.  The rounding of an f32 chain grows with the square root
// of its length, so where the plan splits K less than f32_pieces the workgroup sums
// its range in runs, kept in the workspace meanwhile: a second set of accumulators
// costs two of the four waves of a SIMD (8168, 768, 3072: 327 us in one chain, 431
// with the accumulators, 341 in three runs).
// The GPT-2-small MLP at 8168 tokens, against the 256 x 256 register-staged tile
// (2-byte-kernel tiling, scalar LDS accesses): forward 399 -> 329 us, input
// gradient 597 -> 341, weight gradient 631 -> 402, the rank-16 products 75-159 ->
// 17-40; 4096^3 1128 -> 1076 us (128 TFLOP/s).
#include "sf_mfma.hpp"

namespace sf {
namespace {

constexpr int kFBk = 32, kFPitch = kFBk + 4;  // k per stage; LDS row pitch in floats (16-byte reads free of conflicts)

// R rows x 32 k of one operand: CH 16-byte chunks per thread.
template <int L, int R>
struct FLoader {
  static constexpr int CH = R * kFBk / 4 / 256;           // K-contiguous: chunks; row-contiguous: k-rows of blocks
  Rsrc rs;
  V4 v[L == 1 ? 4 : CH];
  uint32_t off[L == 0 ? CH : 1];
  uint32_t ldb;     // row-contiguous: bytes per k row
  int kc, k_end;
  bool live;        // row-contiguous: the thread owns a block (R / 4 * 8 of 256 threads do)

  __device__ __forceinline__ void init(const void* base, int64_t ld, int64_t row0, int64_t rows, int64_t K) {
    const int t = threadIdx.x;
    k_end = static_cast<int>(K);
    if constexpr (L == 0) {  // chunk t + 256 i: row / 8-chunk column
      rs = make_rsrc(base, rows * ld * 4);
      kc = (t & 7) * 4;
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int64_t r = row0 + (t >> 3) + 32 * i;
        off[i] = r < rows ? (uint32_t)((r * ld + kc) * 4) : kOob;
      }
      live = true;
    } else {  // block (k-block t % 8, row-block t / 8): rows 4 (t / 8) .., k 4 (t % 8) ..
      rs = make_rsrc(base, K * ld * 4);
      const int64_t r = row0 + (t >> 3) * 4;
      live = (t >> 3) * 4 < R;
      kc = (t & 7) * 4;
      off[0] = live && r < rows ? (uint32_t)(r * 4) : kOob;
      ldb = (uint32_t)(ld * 4);
    }
  }
  __device__ __forceinline__ void load(int k0) {
    if constexpr (L == 0) {
      const bool ok = k0 + kc < k_end;  // K is a multiple of 4: a chunk is in or out
#pragma unroll
      for (int i = 0; i < CH; ++i) v[i] = bload(rs, ok ? off[i] : kOob, (uint32_t)(k0 * 4));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = k0 + kc + j;
        v[j] = bload(rs, off[0] != kOob && k < k_end ? off[0] + (uint32_t)k * ldb : kOob, 0);
      }
    }
  }
  __device__ __forceinline__ void store(float* lds) const {
    const int t = threadIdx.x;
    if constexpr (L == 0) {
#pragma unroll
      for (int i = 0; i < CH; ++i)
        *reinterpret_cast<uint4*>(lds + ((t >> 3) + 32 * i) * kFPitch + kc) =
            make_uint4(v[i].w[0], v[i].w[1], v[i].w[2], v[i].w[3]);
    } else if (live) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<uint4*>(lds + ((t >> 3) * 4 + i) * kFPitch + kc) =
            make_uint4(v[0].w[i], v[1].w[i], v[2].w[i], v[3].w[i]);
    }
  }
};

__device__ __forceinline__ void f32_store(const GemmArgs& g, int64_t row, int64_t col, float x) {
  const int64_t o = row * g.ldc + col;
  const bool cbf = g.c_dtype == SF_DTYPE_BF16;
  if (cbf) x = hround(x);
  if (g.bias) {
    const float b = load_elem(g.bias, col, g.bias_dtype);
    x = cbf ? hround(x + b) : x + b;
  }
  if (g.emask) {
    const float em = static_cast<const float*>(g.emask)[o];
    if (g.dw) {
      if (em < 0.5f) {
        float d = g.decay * static_cast<const float*>(g.dw)[o];
        if (cbf) d = hround(d);
        x = cbf ? hround(x + d) : x + d;
      }
    } else {
      x = cbf ? hround(x * em) : x * em;
    }
  }
  if (g.accumulate) x = load_elem(g.C, o, g.c_dtype) + x;
  store_from_f32(g.C, o, g.c_dtype, x);
}

// TM x TN tile; WGM x WGN waves of FM x FN blocks of 32 x 32.  RUNS: the first segment in runs of g.run_stages, the sum
// of those before in the split's partials.
template <int AL, int BL, int TM, int TN, int WGM, int WGN, bool RUNS>
__global__ void __launch_bounds__(256) gemm_f32_kernel(GemmArgs g) {
  constexpr int FM = TM / 32 / WGM, FN = TN / 32 / WGN;
  __shared__ __align__(16) float As[TM * kFPitch], Bs[TN * kFPitch];
  const int64_t tiles = g.tiles_m * g.tiles_n;
  const int64_t kz = blockIdx.x / tiles;
  int64_t tm, tn;
  tile_coords(blockIdx.x - kz * tiles, g.tiles_m, g.tiles_n, tm, tn);
  const int64_t m0 = tm * TM, n0 = tn * TN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave / WGN, wn = wave % WGN;
  f32x16_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x16_t{};
  const int frag = (lane & 31) * kFPitch + (lane >> 5) * 4;
  const float* ar = As + wm * FM * 32 * kFPitch + frag;
  const float* br = Bs + wn * FN * 32 * kFPitch + frag;

  FLoader<AL, TM> la;
  FLoader<BL, TN> lb;
  // stages of the segment the loaders were set up for; each_stage(s) after the products of stage s, while the loads of
  // the next are in flight
  auto segment = [&](int64_t s_begin, int64_t s_end, auto&& each_stage) {
    if (s_begin >= s_end) return;
    la.load(static_cast<int>(s_begin * kFBk));
    lb.load(static_cast<int>(s_begin * kFBk));
    for (int64_t s = s_begin; s < s_end; ++s) {
      __syncthreads();  // every wave is done with the previous stage
      la.store(As);
      lb.store(Bs);
      __syncthreads();
      if (s + 1 < s_end) {
        la.load(static_cast<int>((s + 1) * kFBk));
        lb.load(static_cast<int>((s + 1) * kFBk));
      }
#pragma unroll
      for (int kk = 0; kk < kFBk; kk += 8) {
        float4 a[FM], b[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) a[i] = *reinterpret_cast<const float4*>(ar + i * 32 * kFPitch + kk);
#pragma unroll
        for (int j = 0; j < FN; ++j) b[j] = *reinterpret_cast<const float4*>(br + j * 32 * kFPitch + kk);
        auto step = [&](auto pick) {
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(pick(a[i]), pick(b[j]), acc[i][j], 0, 0, 0);
        };
        step([](const float4& v) { return v.x; });
        step([](const float4& v) { return v.y; });
        step([](const float4& v) { return v.z; });
        step([](const float4& v) { return v.w; });
      }
      each_stage(s);
    }
  };
  auto nothing = [](int64_t) {};
  const int64_t nk1 = ceil_div(g.K1, kFBk), s0 = kz * g.split_stages;
  const int64_t s1 = s0 + g.split_stages < nk1 ? s0 + g.split_stages : nk1;
  la.init(g.A1, g.lda1, m0, g.M, g.K1);
  lb.init(g.B1, g.ldb1, n0, g.N, g.K1);
  if constexpr (!RUNS) {
    segment(s0, s1, nothing);
  } else {
    const int64_t rows = g.M - m0 < TM ? g.M - m0 : TM;
    const Rsrc rp = make_rsrc(g.partial + (kz * g.M + m0) * g.N, rows * g.N * 4);
    const uint32_t ldp = (uint32_t)g.N * 4u;
    const int64_t col = n0 + wn * FN * 32 + (lane & 31);
    const uint32_t first = (uint32_t)((wm * FM * 32 + (lane >> 5) * 4) * g.N + col) * 4u;
    // f(offset, element) for the thread's accumulators; rows past M lie past the extent
    auto elements = [&](auto&& f) {
      uint32_t at = first;
      asm volatile("" : "+v"(at));  // the offsets are recomputed here, not kept in registers over the stages
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            acc[i][j][e] = f(col + j * 32 < g.N ? at + (uint32_t)(i * 32 + (e >> 2) * 8 + (e & 3)) * ldp + j * 128u : kOob,
                             acc[i][j][e]);
    };
    int64_t run_end = s0 + g.run_stages - 1;  // last stage of the current run
    segment(s0, s1, [&](int64_t s) {
      if (s != run_end && s + 1 < s1) return;
      if (s >= s0 + g.run_stages)
        elements([&](uint32_t at, float x) {
          return x + __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rp, (int)at, 0, 0));
        });
      if (s + 1 < s1)
        elements([&](uint32_t at, float x) {
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), rp, (int)at, 0, 0);
          return 0.0f;
        });
      run_end += g.run_stages;
    });
  }
  if (g.A2 && kz == g.splits - 1) {
    la.init(g.A2, g.lda2, m0, g.M, g.K2);
    lb.init(g.B2, g.ldb2, n0, g.N, g.K2);
    segment(0, ceil_div(g.K2, kFBk), nothing);
  }
  // lane: column lane % 32, rows (e / 4) * 8 + (lane / 32) * 4 + e % 4 of each block: whole 128-byte row pieces
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t row = m0 + (wm * FM + i) * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3);
        const int64_t col = n0 + (wn * FN + j) * 32 + (lane & 31);
        if (row >= g.M || col >= g.N) continue;
        if (g.splits > 1)
          g.partial[(kz * g.M + row) * g.N + col] = acc[i][j][e];
        else
          f32_store(g, row, col, acc[i][j][e]);
      }
}

// Pieces that K is summed in at least: as many as would give each CU a 256 x 256 tile of C, none shorter than 256 k.
// (The products' splits before they had smaller tiles: the error against float64 of 8168, 768, 3072 is 5.7e-7 with
// them and 9.9e-7 in one chain, of 3312, 312, 632 3.2e-7 and 4.5e-7.)
int64_t f32_pieces(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ceil_div(M, 256) * ceil_div(N, 256), stages = ceil_div(K, kFBk);
  if (tiles >= 128 || stages < 16) return 1;
  int64_t p = ceil_div(256, tiles);
  if (p > stages / 8) p = stages / 8;
  return p > 16 ? 16 : p;
}

struct F32Plan {
  int tm, tn, splits;
};

// Tile and K splits from an estimate of the time in clocks.  A stage of a 32 x 32 block is 1024 clocks of one of a
// CU's 4 SIMDs; `eff` is what each tile loses to its loads and registers (128 x 64 at 128 registers is the best:
// 4096^3 1087 us against 1165 with 128 x 128 and 1170 with 64 x 64); a workgroup alone on its CU takes about 2200
// clocks a stage whatever its tile, so a few per CU (`occ` fit) are needed to reach the matrix rate.  1500 clocks a
// workgroup for its first loads and its stores, and for K splits the second launch and the partials' traffic
// (written and read, about 2000 bytes a clock).  Each further run of a split (`pieces` of K in all) costs its sum's way
// to memory and back: about 16000 clocks a round of workgroups and the traffic.  A row-contiguous A (rows_a: the weight
// gradient) costs 1.4 times as much for its transposed stores and registers; three workgroups of 128 x 64 fit a CU then,
// and one or two alone take as long as 1.7 or 2.3 of them (1024, 4096, 4096, workgroups a CU and K splits: 2 in one 382
// us, 4 in two 427, 8 in four 323).
F32Plan f32_plan(int64_t M, int64_t N, int64_t K, bool rows_a, int max_splits, int64_t pieces) {
  struct Tile {
    int tm, tn, occ;
    double eff;
  };
  static const Tile tiles[5] = {{128, 128, 2, 1.1}, {128, 64, 4, 1.0}, {64, 64, 5, 1.15}, {128, 32, 5, 1.15}, {32, 128, 5, 1.15}};
  const int64_t stages = ceil_div(K, kFBk);
  F32Plan best{128, 64, 1};
  double best_cost = -1;
  for (const Tile& t : tiles) {
    const int64_t n = ceil_div(M, t.tm) * ceil_div(N, t.tn);
    for (int sp = 1; sp <= max_splits && sp <= stages; ++sp) {
      if (sp > 1 && stages / sp < 4) break;
      const int64_t per = ceil_div(stages, sp);
      if ((sp - 1) * per >= stages) continue;  // an empty last split
      const int64_t on_cu = ceil_div(n * sp, 256);
      double wgs = static_cast<double>(on_cu);
      if (rows_a && t.tm == 128 && t.tn == 64 && on_cu % 3) wgs += on_cu % 3 == 1 ? 0.7 : 0.3;
      const double blocks = t.tm / 32.0 * (t.tn / 32.0) / 4.0,
                   rate = wgs * per * blocks * 1024.0 * t.eff * (rows_a ? 1.4 : 1.0),
                   latency = ceil_div(on_cu, t.occ) * per * 2200.0;
      double cost = (rate > latency ? rate : latency) + on_cu * 1500.0;
      const double partials = sp * static_cast<double>(M) * N * 4.0 / 2000.0;
      if (sp > 1) cost += 8000.0 + 2.0 * partials;
      cost += (ceil_div(pieces, sp) - 1) * (16000.0 * ceil_div(on_cu, t.occ) + partials);
      if (best_cost < 0 || cost < best_cost) {
        best_cost = cost;
        best = {t.tm, t.tn, sp};
      }
    }
  }
  return best;
}
constexpr int kF32MaxSplits = 48;

template <int AL, int BL>
int launch_f32_tiles(const F32Plan& p, const GemmArgs& g, hipStream_t st) {
  const unsigned grid = static_cast<unsigned>(g.tiles_m * g.tiles_n * g.splits);
#define SF_F32(TM, TN, WM, WN)                                                  \
  do {                                                                          \
    if (g.run_stages < g.split_stages)                                          \
      gemm_f32_kernel<AL, BL, TM, TN, WM, WN, true><<<grid, 256, 0, st>>>(g);   \
    else                                                                        \
      gemm_f32_kernel<AL, BL, TM, TN, WM, WN, false><<<grid, 256, 0, st>>>(g);  \
  } while (0)
  if (p.tm == 128 && p.tn == 128)
    SF_F32(128, 128, 2, 2);
  else if (p.tm == 128 && p.tn == 64)
    SF_F32(128, 64, 2, 2);
  else if (p.tm == 64)
    SF_F32(64, 64, 2, 2);
  else if (p.tm == 128)
    SF_F32(128, 32, 4, 1);
  else
    SF_F32(32, 128, 1, 4);
#undef SF_F32
  return launch_status("sf_gemm (f32)");
}

}  // namespace

size_t gemm_f32_workspace(int64_t M, int64_t N, int64_t K, int a_layout) {
  const int64_t pieces = f32_pieces(M, N, K);
  const int sp = f32_plan(M, N, K, a_layout == SF_LAYOUT_MN, kF32MaxSplits, pieces).splits;
  return sp > 1 || pieces > 1 ? static_cast<size_t>(sp) * M * N * sizeof(float) : 0;
}

int launch_gemm_f32(GemmArgs g, int a_layout, int b_layout, void* workspace, size_t workspace_bytes, hipStream_t st) {
  // as many K splits as the workspace holds partials for
  const size_t per = static_cast<size_t>(g.M) * g.N * sizeof(float);
  const bool ws = workspace && (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0;
  const int64_t cap = ws ? static_cast<int64_t>(workspace_bytes / per) : 0;
  const int64_t pieces = cap > 0 ? f32_pieces(g.M, g.N, g.K1) : 1;
  const F32Plan p = f32_plan(g.M, g.N, g.K1, a_layout == SF_LAYOUT_MN,
                             cap > kF32MaxSplits ? kF32MaxSplits : (cap < 1 ? 1 : static_cast<int>(cap)), pieces);
  g.tiles_m = ceil_div(g.M, p.tm);
  g.tiles_n = ceil_div(g.N, p.tn);
  g.splits = p.splits;
  g.split_stages = ceil_div(ceil_div(g.K1, kFBk), p.splits);
  g.partial = cap > 0 ? static_cast<float*>(workspace) : nullptr;
  g.run_stages = ceil_div(g.split_stages, ceil_div(pieces, p.splits));
  SF_CHECK_ARG(g.tiles_m * g.tiles_n * p.splits < (1ll << 31), "GEMM grid too large");
  int rc;
  if (a_layout == SF_LAYOUT_K && b_layout == SF_LAYOUT_K)
    rc = launch_f32_tiles<0, 0>(p, g, st);
  else if (a_layout == SF_LAYOUT_K)
    rc = launch_f32_tiles<0, 1>(p, g, st);
  else
    rc = launch_f32_tiles<1, 1>(p, g, st);
  if (rc || p.splits == 1) return rc;
  return launch_splitk_reduce(g, SF_DTYPE_F32, st, "sf_gemm (split-K reduce)");
}

}  // namespace sf
