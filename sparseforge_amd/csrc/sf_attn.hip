// Causal attention of the retraining model in bf16, forward and backward, with
// no S x S tensor in memory (HuggingFace's eager attention, which the reference
// retrains with, legacy/model_llama.py:39-55; the Hutchinson double backward
// keeps the materialised products of llama._causal_attention_device).
//
//   forward   o = softmax(scale q k^T, causal) v, and per row its largest score and
//             the base-2 log of the sum of 2^(c (score - largest)), c = scale log2e
//   backward  p = exp2(c s - lse), lse = c largest + log,  ds = p (do v^T - delta),
//             delta = sum_d do o;  dv = p^T do, dk = scale ds^T q, dq = scale ds k
//
// c s - lse as one fused multiply-add leaves what rounding lse to f32 loses, 2^-13
// at kAtBig; beyond that (scores that have run away) the maximum is subtracted from
// the score first, which is exact at any size but costs another instruction per
// element.  The forward and dq decide that per wave; dk / dv, where a test per tile
// cost 11 of 147 us, by one word that the forward sets, with a body for each case.
//
// The scores, the probabilities' sums and every accumulation stay f32 in
// registers; p and ds round to bf16 as operands of the next product, as the
// eager form's do (which also rounds the scores).  Keys and queries are rotated
// once by rotate_kernel (the eager form's roundings); the rotation's adjoint is
// applied to dq and dk in f32 in their epilogues.
//
// Every product is v_mfma_f32_32x32x16_bf16 with the score tile transposed where
// that leaves its rows in registers: a lane holds one query (forward, dq) or one
// key (dk / dv) and the 32 x 32 tile's rows (e / 4) * 8 + (lane / 32) * 4 + e % 4.
// The next product contracts over those rows, and a contraction may take its
// index in any order, so the packed probabilities are the next B operand as they
// stand, and its A operand (V^T, K^T, dO^T, Q^T) is read in the same order by two
// ds_read_b64_tr_b16 per fragment.  No value crosses lanes but the row maxima
// and sums of the two half-waves.
//
// A workgroup is 4 waves of 32 queries (or keys); tiles of 64 keys (or queries)
// are loaded into registers one tile ahead and then into LDS.  Heads of 64: 53 KB of
// LDS, three workgroups a CU (dk / dv two, by its registers), and the softmax's VALU
// work (exp2 at a quarter rate: about 1000 clocks per 32 x 64 tile against 512 of
// MFMA) runs beside the MFMAs and LDS reads of the others.  Heads of 128: 86 KB, one
// workgroup a CU, so nothing but its own four waves covers a tile's latencies.  The
// blocks of one (batch, head) run on one XCD and share its keys and values in that
// L2; long rows go first.
// Measured, causal, us: rotation / forward / delta / dk, dv / dq:
//   2 x 2048 tokens, 32 heads of 64    12 / 77 / 10 / 150 / 107, the call with its
//     gradients 340; the materialised products and softmax passes 1367
//   1 x 2048 tokens, 32 heads of 128   12 / 107 / 9 / 158 / 144
#include <type_traits>

#include "sf_mfma.hpp"

namespace sf {
namespace {

constexpr int kAtRows = 128;  // queries (forward, dq) or keys (dk / dv) of a workgroup: 4 waves of 32
constexpr int kAtTile = 64;   // the other side's tile
constexpr float kAtBig = 4096.0f;  // |c score| from which the row's maximum is subtracted before c is applied
typedef short v4i16_t __attribute__((ext_vector_type(4)));

struct AttnArgs {
  const uint16_t* q;   // rotated [B, S, H, D]
  const uint16_t* k;   // rotated
  const uint16_t* v;
  const uint16_t* go;  // gradient of the output (backward)
  float* o32;          // [B, S, H, D]: the output before it is rounded (forward: null without a backward)
  float* stats;        // [3][B H, S]: lse, largest score, log2 of the sum; then one word, not 0 if a score is past kAtBig
  float* delta;        // [B H, S]
  uint16_t* out;       // forward: o
  uint16_t* dq;
  uint16_t* dk;
  uint16_t* dv;
  const float* cos;    // [S, D]
  const float* sin;
  int64_t S;
  int H, BH;
  float scale;
};

// LDS row pitch in bytes: 20 words past a multiple of 32, so the 16-byte row reads of 8 lanes fall in different
// banks and the transposed reads of 4 rows x 64 bytes overlap in 4 words only.
template <int D>
constexpr int at_pitch() { return D == 64 ? 208 : 336; }
// Workgroups a CU that the registers are limited for (LDS: three with heads of 64, one with heads of 128).
template <int D>
constexpr int at_wgs() { return D == 64 ? 2 : 1; }

__host__ __device__ __forceinline__ float* at_flag(const AttnArgs& a) { return a.stats + 3 * (int64_t)a.BH * a.S; }

// Block order: the row blocks of one (batch, head) on one XCD, `last` first when its rows are the longest.
__device__ __forceinline__ void at_block(const AttnArgs& a, int nb, bool last_first, int& bh, int& blk) {
  const int id = blockIdx.x;
  if (a.BH % 8 == 0) {
    const int r = id / 8;
    bh = (r / nb) * 8 + id % 8;
    blk = r % nb;
  } else {
    bh = id / nb;
    blk = id % nb;
  }
  if (last_first) blk = nb - 1 - blk;
}

// The rows of one (batch, head) of a [B, S, H, D] tensor: rows past S lie past the extent and read zeros.
template <int D>
__device__ __forceinline__ Rsrc at_rows(const uint16_t* t, const AttnArgs& a, int bh) {
  const int64_t b = bh / a.H, h = bh - b * a.H;
  return make_rsrc(t + (b * a.S * a.H + h) * D, ((a.S - 1) * a.H + 1) * (int64_t)(D * 2));
}

// A tile of 64 rows x D on its way to LDS: thread t holds 16-byte chunks t, t + 256, ...
template <int D>
struct AtTile {
  static constexpr int N = 64 * D * 2 / 16 / 256;
  V4 w[N];
  __device__ __forceinline__ void load(Rsrc r, int64_t row0, int H) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = threadIdx.x + 256 * i, row = c / (D / 8), ch = c % (D / 8);
      w[i] = bload(r, (uint32_t)(((row0 + row) * H * D + ch * 8) * 2), 0);
    }
  }
  __device__ __forceinline__ void store(unsigned char* lds) const {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = threadIdx.x + 256 * i, row = c / (D / 8), ch = c % (D / 8);
      *reinterpret_cast<uint4*>(lds + row * at_pitch<D>() + ch * 16) =
          make_uint4(w[i].w[0], w[i].w[1], w[i].w[2], w[i].w[3]);
    }
  }
};

// Fragments of a wave's own 32 rows, k = d contiguous (lane: row lane % 32, d 16 kk + 8 (lane / 32) ..).
template <int D>
__device__ __forceinline__ void own_frags(Rsrc r, int64_t row0, int H, bf16x8_t (&f)[D / 16]) {
  const int lane = threadIdx.x & 63;
  const int64_t row = row0 + (lane & 31);
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk)
    f[kk] = __builtin_bit_cast(bf16x8_t, bload(r, (uint32_t)((row * H * D + kk * 16 + (lane >> 5) * 8) * 2), 0));
}
// Row fragment kk of tile rows [r0, r0 + 32).
template <int D>
__device__ __forceinline__ bf16x8_t row_frag(const unsigned char* lds, int r0, int kk) {
  const int lane = threadIdx.x & 63;
  return *reinterpret_cast<const bf16x8_t*>(lds + (r0 + (lane & 31)) * at_pitch<D>() + kk * 32 + (lane >> 5) * 16);
}
// Transposed fragment: "rows" are the tile's columns [c0, c0 + 32) (lane % 32), k the 16 tile rows from r0 in the
// accumulator's order: half-wave h takes r0 + 4 h .. + 3 and r0 + 8 + 4 h .. + 3.
template <int D>
__device__ __forceinline__ bf16x8_t tr_frag(const unsigned char* lds, int r0, int c0) {
  typedef __attribute__((address_space(3))) v4i16_t lds_v4;
  const int lane = threadIdx.x & 63, L = lane & 15;
  const unsigned char* p = lds + (r0 + 4 * (lane >> 5) + (L >> 2)) * at_pitch<D>() +
                           (c0 + 16 * ((lane >> 4) & 1) + 4 * (L & 3)) * 2;
  const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(p));
  const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(p + 8 * at_pitch<D>()));
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}
// Values 8 i .. 8 i + 7 of an accumulator block as the next product's operand.
__device__ __forceinline__ bf16x8_t pack_half(const f32x16_t& p, int i) {
  const uint4 w = make_uint4(pack2(p[8 * i], p[8 * i + 1]), pack2(p[8 * i + 2], p[8 * i + 3]),
                             pack2(p[8 * i + 4], p[8 * i + 5]), pack2(p[8 * i + 6], p[8 * i + 7]));
  return __builtin_bit_cast(bf16x8_t, w);
}
__device__ __forceinline__ int acc_row(int e) { return (e >> 2) * 8 + ((threadIdx.x >> 5) & 1) * 4 + (e & 3); }

constexpr float kLog2e = 1.4426950408889634f;

// ---------------------------------------------------------------------------
// rot(x) of q and k: x c + x^ ss with the products and their sum rounded to bf16 (torch's op order, sf_heads.hip).
// One thread per 8 dims of the first half and their partners.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void unpack8(const uint4& q, float (&v)[8]) {
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[2 * k] = lo_f(w[k]);
    v[2 * k + 1] = hi_f(w[k]);
  }
}
template <int D>
__global__ void __launch_bounds__(256) rotate_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
                                                     uint16_t* __restrict__ qr, uint16_t* __restrict__ kr,
                                                     const float* __restrict__ cos, const float* __restrict__ sin,
                                                     int64_t S, int H, int64_t work, float* __restrict__ flag) {
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *flag = 0.0f;  // the forward kernel may set it
  constexpr int C = D / 16;  // chunks of 8 in half a head
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i >= work) return;
  const uint16_t* x = blockIdx.y ? k : q;
  uint16_t* y = blockIdx.y ? kr : qr;
  const int64_t head = i / C;  // (b, s, h)
  const int c = static_cast<int>(i - head * C) * 8;
  const int64_t s = head / H % S, at = head * D + c;
  float a[8], b[8];
  unpack8(*reinterpret_cast<const uint4*>(x + at), a);
  unpack8(*reinterpret_cast<const uint4*>(x + at + D / 2), b);
  float lo[8], hi[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float c0 = hround(cos[s * D + c + j]), s0 = hround(sin[s * D + c + j]);
    const float c1 = hround(cos[s * D + c + D / 2 + j]), s1 = hround(sin[s * D + c + D / 2 + j]);
    lo[j] = hround(a[j] * c0) - hround(b[j] * s0);
    hi[j] = hround(b[j] * c1) + hround(a[j] * s1);
  }
  *reinterpret_cast<uint4*>(y + at) = make_uint4(pack2(lo[0], lo[1]), pack2(lo[2], lo[3]), pack2(lo[4], lo[5]), pack2(lo[6], lo[7]));
  *reinterpret_cast<uint4*>(y + at + D / 2) =
      make_uint4(pack2(hi[0], hi[1]), pack2(hi[2], hi[3]), pack2(hi[4], hi[5]), pack2(hi[6], hi[7]));
}

// Rows of a [B, S, H, D] tensor from accumulators held transposed (lane: row row0 + lane % 32; block db: dims
// 32 db + acc_row(e)), times `f`; ROT: through the rotation's adjoint.
template <int D, bool ROT>
__device__ __forceinline__ void store_rows(uint16_t* t, const AttnArgs& a, int bh, int64_t row0,
                                           const f32x16_t (&acc)[D / 32], float f) {
  const int lane = threadIdx.x & 63, h4 = (lane >> 5) * 4;
  const int64_t row = row0 + (lane & 31);
  if (row >= a.S) return;
  const int64_t b = bh / a.H, h = bh - b * a.H;
  uint16_t* dst = t + ((b * a.S + row) * a.H + h) * D;
  if constexpr (!ROT) {
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<uint2*>(dst + db * 32 + g * 8 + h4) =
            make_uint2(pack2(acc[db][4 * g] * f, acc[db][4 * g + 1] * f),
                       pack2(acc[db][4 * g + 2] * f, acc[db][4 * g + 3] * f));
  } else {
    // adjoint: first half g c + g^ s^, second half g c - g^ s^ (c, s rounded to bf16 as the rotation's)
    const float* cs = a.cos + row * D;
    const float* sn = a.sin + row * D;
#pragma unroll
    for (int db = 0; db < D / 64; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d0 = db * 32 + g * 8 + h4, d1 = d0 + D / 2;
        const float4 c0 = *reinterpret_cast<const float4*>(cs + d0), c1 = *reinterpret_cast<const float4*>(cs + d1);
        const float4 s0 = *reinterpret_cast<const float4*>(sn + d0), s1 = *reinterpret_cast<const float4*>(sn + d1);
        const float cc0[4] = {c0.x, c0.y, c0.z, c0.w}, cc1[4] = {c1.x, c1.y, c1.z, c1.w};
        const float ss0[4] = {s0.x, s0.y, s0.z, s0.w}, ss1[4] = {s1.x, s1.y, s1.z, s1.w};
        float lo[4], hi[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = acc[db][4 * g + j] * f, y = acc[db + D / 64][4 * g + j] * f;
          lo[j] = x * hround(cc0[j]) + y * hround(ss1[j]);
          hi[j] = y * hround(cc1[j]) - x * hround(ss0[j]);
        }
        *reinterpret_cast<uint2*>(dst + d0) = make_uint2(pack2(lo[0], lo[1]), pack2(lo[2], lo[3]));
        *reinterpret_cast<uint2*>(dst + d1) = make_uint2(pack2(hi[0], hi[1]), pack2(hi[2], hi[3]));
      }
  }
}

// The same rows in f32, without rotation.
template <int D>
__device__ __forceinline__ void store_rows_f32(float* t, const AttnArgs& a, int bh, int64_t row0,
                                               const f32x16_t (&acc)[D / 32], float f) {
  const int lane = threadIdx.x & 63, h4 = (lane >> 5) * 4;
  const int64_t row = row0 + (lane & 31);
  if (row >= a.S) return;
  const int64_t b = bh / a.H, h = bh - b * a.H;
  float* dst = t + ((b * a.S + row) * a.H + h) * D;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<float4*>(dst + db * 32 + g * 8 + h4) =
          make_float4(acc[db][4 * g] * f, acc[db][4 * g + 1] * f, acc[db][4 * g + 2] * f, acc[db][4 * g + 3] * f);
}

// ---------------------------------------------------------------------------
// Forward: 128 queries of one (batch, head).
// ---------------------------------------------------------------------------
template <int D>
__global__ void __launch_bounds__(256, at_wgs<D>()) attn_fwd_kernel(AttnArgs a, int nb) {
  __shared__ __align__(16) unsigned char ks[2][kAtTile * at_pitch<D>()];
  __shared__ __align__(16) unsigned char vs[2][kAtTile * at_pitch<D>()];
  int bh, blk;
  at_block(a, nb, true, bh, blk);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t q0 = (int64_t)blk * kAtRows + wave * 32, query = q0 + (lane & 31);
  const Rsrc rk = at_rows<D>(a.k, a, bh), rv = at_rows<D>(a.v, a, bh);
  bf16x8_t qf[D / 16];
  own_frags<D>(at_rows<D>(a.q, a, bh), q0, a.H, qf);
  f32x16_t o[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) o[i] = f32x16_t{};
  const float c = a.scale * kLog2e;
  // of this lane's query: the largest score so far, that score (0 while every score is -inf, so that those count 0 and
  // not NaN) and it times c, and the sum over the keys this half-wave holds
  float m = -INFINITY, mz = 0.0f, ms = 0.0f, l = 0.0f;
  float sub = 0.0f;  // ms, or 0 if big
  bool big = false;  // some query of the wave: |ms| > kAtBig; then mz is taken from the scores as they come
  const int64_t end = (int64_t)(blk + 1) * kAtRows < a.S ? (int64_t)(blk + 1) * kAtRows : a.S;
  const int nt = static_cast<int>(ceil_div(end, kAtTile));
  AtTile<D> tk, tv;
  tk.load(rk, 0, a.H);
  tv.load(rv, 0, a.H);
  for (int t = 0; t < nt; ++t) {
    unsigned char *kb = ks[t & 1], *vb = vs[t & 1];
    tk.store(kb);
    tv.store(vb);
    __syncthreads();  // also: every wave is done with the other buffer's previous tile
    const int64_t n0 = (int64_t)t * kAtTile;
    if (t + 1 < nt) {
      tk.load(rk, n0 + kAtTile, a.H);
      tv.load(rv, n0 + kAtTile, a.H);
    }
    if (n0 > q0 + 31) continue;  // the whole tile lies past this wave's queries (wave-uniform; no barrier below)
    f32x16_t s[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      s[b] = f32x16_t{};
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk)
        s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(kb, b * 32, kk), qf[kk], s[b], 0, 0, 0);
    }
    float mx = -INFINITY;
    if (n0 + kAtTile - 1 > q0) {  // the diagonal crosses the tile
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (n0 + b * 32 + acc_row(e) > query) s[b][e] = -INFINITY;
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[b][e]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);
    if (big || __builtin_amdgcn_ballot_w64(mn > m) != 0) {  // some query's maximum rose: rescale what is accumulated
      const float nz = mn == -INFINITY ? 0.0f : mn, ns = nz * c;
      big = __builtin_amdgcn_ballot_w64(fabsf(ns) > kAtBig) != 0;
      const float al = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(big ? (mz - nz) * c : ms - ns);
      l *= al;
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] *= al;
      m = mn;
      mz = nz;
      ms = ns;
      sub = ms;
      if (big) {
        sub = 0.0f;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int e = 0; e < 16; ++e) s[b][e] -= mz;
      }
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[b][e] = __builtin_amdgcn_exp2f(fmaf(s[b][e], c, -sub));
        l += s[b][e];
      }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x8_t p = pack_half(s[b], i);
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag<D>(vb, b * 32 + i * 16, db * 32), p, o[db], 0, 0, 0);
      }
  }
  l += __shfl_xor(l, 32, 64);
  store_rows<D, false>(a.out, a, bh, q0, o, 1.0f / l);
  if (a.o32) store_rows_f32<D>(a.o32, a, bh, q0, o, 1.0f / l);
  if (lane < 32 && query < a.S) {
    const float lg = __builtin_amdgcn_logf(l), lse = m * c + lg;
    float* st = a.stats + bh * a.S + query;
    st[0] = lse;
    st[a.BH * a.S] = m;
    st[2 * a.BH * a.S] = lg;
    if (fabsf(lse) > kAtBig) *at_flag(a) = 1.0f;  // the same value from every such query
  }
}

// delta[bh, s] = sum_d go o: one thread per 8 dims, folded over the row's D / 8 threads.  From the forward's own f32
// output: the one that it returns is rounded, and may have been changed in place since.
template <int D>
__global__ void __launch_bounds__(256) attn_delta_kernel(AttnArgs a, int64_t work) {
  constexpr int C = D / 8;
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  float d = 0.0f;
  if (i < work) {
    float x[8];
    unpack8(*reinterpret_cast<const uint4*>(a.go + i * 8), x);
    const float4 y0 = *reinterpret_cast<const float4*>(a.o32 + i * 8), y1 = *reinterpret_cast<const float4*>(a.o32 + i * 8 + 4);
    const float y[8] = {y0.x, y0.y, y0.z, y0.w, y1.x, y1.y, y1.z, y1.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) d = fmaf(x[j], y[j], d);
  }
#pragma unroll
  for (int off = 1; off < C; off <<= 1) d += __shfl_xor(d, off, 64);
  if (i < work && i % C == 0) {
    const int64_t head = i / C, h = head % a.H, bs = head / a.H, s = bs % a.S, b = bs / a.S;
    a.delta[(b * a.H + h) * a.S + s] = d;
  }
}

// ---------------------------------------------------------------------------
// dq: 128 queries of one (batch, head), tiles of 64 keys.
// ---------------------------------------------------------------------------
template <int D>
__global__ void __launch_bounds__(256, at_wgs<D>()) attn_dq_kernel(AttnArgs a, int nb) {
  __shared__ __align__(16) unsigned char ks[2][kAtTile * at_pitch<D>()];
  __shared__ __align__(16) unsigned char vs[2][kAtTile * at_pitch<D>()];
  int bh, blk;
  at_block(a, nb, true, bh, blk);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t q0 = (int64_t)blk * kAtRows + wave * 32, query = q0 + (lane & 31);
  const Rsrc rk = at_rows<D>(a.k, a, bh), rv = at_rows<D>(a.v, a, bh);
  bf16x8_t qf[D / 16], gf[D / 16];
  own_frags<D>(at_rows<D>(a.q, a, bh), q0, a.H, qf);
  own_frags<D>(at_rows<D>(a.go, a, bh), q0, a.H, gf);
  const float c = a.scale * kLog2e;
  const float* st = a.stats + bh * a.S + query;
  float sub = query < a.S ? st[0] : INFINITY, mz = 0.0f;
  const bool big = __builtin_amdgcn_ballot_w64(query < a.S && fabsf(sub) > kAtBig) != 0;
  if (big && query < a.S) {
    mz = st[a.BH * a.S];
    sub = st[2 * a.BH * a.S];
  }
  const float delta = query < a.S ? a.delta[bh * a.S + query] : 0.0f;
  f32x16_t dq[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) dq[i] = f32x16_t{};
  const int64_t end = (int64_t)(blk + 1) * kAtRows < a.S ? (int64_t)(blk + 1) * kAtRows : a.S;
  const int nt = static_cast<int>(ceil_div(end, kAtTile));
  AtTile<D> tk, tv;
  tk.load(rk, 0, a.H);
  tv.load(rv, 0, a.H);
  for (int t = 0; t < nt; ++t) {
    unsigned char *kb = ks[t & 1], *vb = vs[t & 1];
    tk.store(kb);
    tv.store(vb);
    __syncthreads();
    const int64_t n0 = (int64_t)t * kAtTile;
    if (t + 1 < nt) {
      tk.load(rk, n0 + kAtTile, a.H);
      tv.load(rv, n0 + kAtTile, a.H);
    }
    if (n0 > q0 + 31) continue;
    const bool diag = n0 + kAtTile - 1 > q0;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f32x16_t s = f32x16_t{}, dp = f32x16_t{};
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(kb, b * 32, kk), qf[kk], s, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(vb, b * 32, kk), gf[kk], dp, 0, 0, 0);
      }
      if (__builtin_expect(big, 0)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] -= mz;
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float p = __builtin_amdgcn_exp2f(fmaf(s[e], c, -sub));
        if (diag && n0 + b * 32 + acc_row(e) > query) p = 0.0f;
        s[e] = p * (dp[e] - delta);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x8_t ds = pack_half(s, i);
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
          dq[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag<D>(kb, b * 32 + i * 16, db * 32), ds, dq[db], 0, 0, 0);
      }
    }
  }
  store_rows<D, true>(a.dq, a, bh, q0, dq, a.scale);
}

// ---------------------------------------------------------------------------
// dk, dv: 128 keys of one (batch, head), tiles of 64 queries from the diagonal on.
// ---------------------------------------------------------------------------
template <int D>
struct DkvLds {
  unsigned char q[2][kAtTile * at_pitch<D>()];
  unsigned char g[2][kAtTile * at_pitch<D>()];
  float rows[2][3][kAtTile];  // of the tile's queries: lse (BIG: log2 of the sum), delta, maximum
};
template <int D, bool BIG>
__device__ __forceinline__ void attn_dkv_block(const AttnArgs& a, int nb, DkvLds<D>& sm) {
  int bh, blk;
  at_block(a, nb, false, bh, blk);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h4 = (lane >> 5) * 4;
  const int64_t k0 = (int64_t)blk * kAtRows + wave * 32, key = k0 + (lane & 31);
  const Rsrc rq = at_rows<D>(a.q, a, bh), rg = at_rows<D>(a.go, a, bh);
  bf16x8_t kf[D / 16], vf[D / 16];
  own_frags<D>(at_rows<D>(a.k, a, bh), k0, a.H, kf);
  own_frags<D>(at_rows<D>(a.v, a, bh), k0, a.H, vf);
  f32x16_t dk[D / 32], dv[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) dk[i] = dv[i] = f32x16_t{};
  const float c = a.scale * kLog2e;
  const int t0 = blk * (kAtRows / kAtTile), nt = static_cast<int>(ceil_div(a.S, kAtTile));
  AtTile<D> tq, tg;
  // threads 0..63: lse of the next tile's query (BIG: log2 of its sum, and its maximum), 64..127: its delta
  float row_v = 0.0f, row_m = 0.0f;
  auto load_rows = [&](int t) {
    const int64_t s = (int64_t)t * kAtTile + (threadIdx.x & 63);
    if (threadIdx.x < 64) {
      row_v = s < a.S ? a.stats[((BIG ? 2 * a.BH : 0) + bh) * a.S + s] : INFINITY;  // past the end: p = 0
      if constexpr (BIG) row_m = s < a.S ? a.stats[(a.BH + bh) * a.S + s] : 0.0f;
    } else if (threadIdx.x < 128) {
      row_v = s < a.S ? a.delta[bh * a.S + s] : 0.0f;
    }
  };
  tq.load(rq, (int64_t)t0 * kAtTile, a.H);
  tg.load(rg, (int64_t)t0 * kAtTile, a.H);
  load_rows(t0);
  for (int t = t0; t < nt; ++t) {
    const int buf = (t - t0) & 1;
    unsigned char *qb = sm.q[buf], *gb = sm.g[buf];
    tq.store(qb);
    tg.store(gb);
    if (threadIdx.x < 128) sm.rows[buf][threadIdx.x >> 6][threadIdx.x & 63] = row_v;
    if constexpr (BIG)
      if (threadIdx.x < 64) sm.rows[buf][2][threadIdx.x] = row_m;
    __syncthreads();
    const int64_t n0 = (int64_t)t * kAtTile;
    if (t + 1 < nt) {
      tq.load(rq, n0 + kAtTile, a.H);
      tg.load(rg, n0 + kAtTile, a.H);
      load_rows(t + 1);
    }
    if (n0 + kAtTile - 1 < k0) continue;  // every query of the tile lies before this wave's keys
    const bool diag = n0 < k0 + 31;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f32x16_t s = f32x16_t{}, dp = f32x16_t{};
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(qb, b * 32, kk), kf[kk], s, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag<D>(gb, b * 32, kk), vf[kk], dp, 0, 0, 0);
      }
      if constexpr (BIG) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4 mx = *reinterpret_cast<const float4*>(&sm.rows[buf][2][b * 32 + g * 8 + h4]);
          const float m4[4] = {mx.x, mx.y, mx.z, mx.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) s[4 * g + j] -= m4[j];
        }
      }
      f32x16_t p;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 ls = *reinterpret_cast<const float4*>(&sm.rows[buf][0][b * 32 + g * 8 + h4]);
        const float4 de = *reinterpret_cast<const float4*>(&sm.rows[buf][1][b * 32 + g * 8 + h4]);
        const float l4[4] = {ls.x, ls.y, ls.z, ls.w}, d4[4] = {de.x, de.y, de.z, de.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int e = 4 * g + j;
          p[e] = __builtin_amdgcn_exp2f(fmaf(s[e], c, -l4[j]));
          if (diag && n0 + b * 32 + acc_row(e) < key) p[e] = 0.0f;
          s[e] = p[e] * (dp[e] - d4[j]);
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x8_t pb = pack_half(p, i), ds = pack_half(s, i);
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
          dv[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag<D>(gb, b * 32 + i * 16, db * 32), pb, dv[db], 0, 0, 0);
          dk[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag<D>(qb, b * 32 + i * 16, db * 32), ds, dk[db], 0, 0, 0);
        }
      }
    }
  }
  store_rows<D, false>(a.dv, a, bh, k0, dv, 1.0f);
  store_rows<D, true>(a.dk, a, bh, k0, dk, a.scale);
}

template <int D>
__global__ void __launch_bounds__(256, at_wgs<D>()) attn_dkv_kernel(AttnArgs a, int nb) {
  __shared__ __align__(16) DkvLds<D> sm;
  if (__builtin_expect(*at_flag(a) != 0.0f, 0))
    attn_dkv_block<D, true>(a, nb, sm);
  else
    attn_dkv_block<D, false>(a, nb, sm);
}

bool at_ok(int64_t B, int64_t S, int64_t H, int64_t D) {
  return B > 0 && S > 0 && H > 0 && (D == 64 || D == 128) && S * H * D * 2 < (int64_t(1) << 31) &&
         B * H * ceil_div(S, kAtRows) < (int64_t(1) << 31) && B * S * H * (D / 8) < (int64_t(1) << 31);
}
bool at_al(const void* p) { return p && (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int D>
int attn_forward(AttnArgs a, const uint16_t* q, const uint16_t* k, uint16_t* qr, uint16_t* kr, int64_t B,
                 hipStream_t st) {
  const int64_t work = B * a.S * a.H * (D / 16);
  rotate_kernel<D><<<dim3(static_cast<unsigned>(ceil_div(work, 256)), 2), 256, 0, st>>>(q, k, qr, kr, a.cos, a.sin, a.S,
                                                                                       a.H, work, at_flag(a));
  const int nb = static_cast<int>(ceil_div(a.S, kAtRows));
  attn_fwd_kernel<D><<<a.BH * nb, 256, 0, st>>>(a, nb);
  return launch_status("sf_attention_forward");
}
template <int D>
int attn_backward(AttnArgs a, int64_t B, hipStream_t st) {
  const int64_t work = B * a.S * a.H * (D / 8);
  attn_delta_kernel<D><<<static_cast<unsigned>(ceil_div(work, 256)), 256, 0, st>>>(a, work);
  const int nb = static_cast<int>(ceil_div(a.S, kAtRows));
  attn_dkv_kernel<D><<<a.BH * nb, 256, 0, st>>>(a, nb);
  attn_dq_kernel<D><<<a.BH * nb, 256, 0, st>>>(a, nb);
  return launch_status("sf_attention_backward");
}

}  // namespace
}  // namespace sf

using namespace sf;

extern "C" int sf_attention_forward(const void* q, const void* k, const void* v, int64_t B, int64_t S, int64_t H,
                                    int64_t D, const float* cos, const float* sin, float scale, void* out, float* out_f32,
                                    float* row_stats, void* q_rot, void* k_rot, void* stream) {
  SF_CHECK_ARG(at_ok(B, S, H, D), "attention: unsupported shape B=%lld S=%lld H=%lld D=%lld", (long long)B,
               (long long)S, (long long)H, (long long)D);
  SF_CHECK_ARG(at_al(q) && at_al(k) && at_al(v) && at_al(out) && at_al(q_rot) && at_al(k_rot) && at_al(cos) &&
                   at_al(sin) && row_stats && (!out_f32 || at_al(out_f32)),
               "attention: null or unaligned tensor");
  AttnArgs a = {};
  a.q = static_cast<const uint16_t*>(q_rot);
  a.k = static_cast<const uint16_t*>(k_rot);
  a.v = static_cast<const uint16_t*>(v);
  a.out = static_cast<uint16_t*>(out);
  a.o32 = out_f32;
  a.stats = row_stats;
  a.cos = cos;
  a.sin = sin;
  a.S = S;
  a.H = static_cast<int>(H);
  a.BH = static_cast<int>(B * H);
  a.scale = scale;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t *qi = static_cast<const uint16_t*>(q), *ki = static_cast<const uint16_t*>(k);
  uint16_t *qo = static_cast<uint16_t*>(q_rot), *ko = static_cast<uint16_t*>(k_rot);
  return D == 64 ? attn_forward<64>(a, qi, ki, qo, ko, B, st) : attn_forward<128>(a, qi, ki, qo, ko, B, st);
}

extern "C" int sf_attention_backward(const void* q_rot, const void* k_rot, const void* v, const float* out_f32,
                                     const void* grad_out, const float* row_stats, int64_t B, int64_t S, int64_t H,
                                     int64_t D, const float* cos, const float* sin, float scale, float* delta,
                                     void* dq, void* dk, void* dv, void* stream) {
  SF_CHECK_ARG(at_ok(B, S, H, D), "attention: unsupported shape B=%lld S=%lld H=%lld D=%lld", (long long)B,
               (long long)S, (long long)H, (long long)D);
  SF_CHECK_ARG(at_al(q_rot) && at_al(k_rot) && at_al(v) && at_al(out_f32) && at_al(grad_out) && at_al(dq) && at_al(dk) &&
                   at_al(dv) && at_al(cos) && at_al(sin) && row_stats && delta,
               "attention: null or unaligned tensor");
  AttnArgs a = {};
  a.q = static_cast<const uint16_t*>(q_rot);
  a.k = static_cast<const uint16_t*>(k_rot);
  a.v = static_cast<const uint16_t*>(v);
  a.o32 = const_cast<float*>(out_f32);
  a.go = static_cast<const uint16_t*>(grad_out);
  a.stats = const_cast<float*>(row_stats);
  a.delta = delta;
  a.dq = static_cast<uint16_t*>(dq);
  a.dk = static_cast<uint16_t*>(dk);
  a.dv = static_cast<uint16_t*>(dv);
  a.cos = cos;
  a.sin = sin;
  a.S = S;
  a.H = static_cast<int>(H);
  a.BH = static_cast<int>(B * H);
  a.scale = scale;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return D == 64 ? attn_backward<64>(a, B, st) : attn_backward<128>(a, B, st);
}
