// Multi-token forward (chunked prefill and k-token verify) on bf16 MFMA.
//
// The reference runs its prompt one token at a time (metal_infrence_engine/src/bin/bench.rs:174-176
// calls forward per position); these kernels run a chunk of M tokens through a layer at once, so
// every weight is read once per chunk and the projections become GEMMs on the matrix cores:
//   GEMMs          C[m][n] = sum_k A'[m][k] W[n][k], A' = A or an RMSNorm of its rows, split into
//                  hi + lo bf16 so the products keep ~16 mantissa bits (gemm_dma.h); epilogues store /
//                  residual add / silu(gate)*up / q-k norm + RoPE + K/V append (cpu_inference.rs:225-257):
//                  k_gemm_kslice (<= 64 rows), k_gemm_wide (more: gemm_choice.h); k_mv_rows (few rows, f32 FMA)
//   k_resadd_norm_split  residual add of a split GEMM, then the next norm, split for the next GEMM
//   k_qk_rope      per token and head: q/k RMSNorm + RoPE, K/V append   (cpu_inference.rs:134-141)
//   k_attn_causal_bf  token m attends positions 0..start+m, split bf16 MFMA (cpu_inference.rs:144-162)
//   k_row_argmax_*    greedy token per logit row (main.rs:37-42)
#include "batch.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "device_common.h"
#include "gemm_dma.h"
#include "l2_prefetch.h"

namespace qe {
namespace {

// x[m] += sum_z part[z][m] (in z order; none: x as it is), then out[m] = x[m] / sqrt(mean x[m]^2 +
// eps) x gain as a split row (cpu_inference.rs:189-194); one workgroup per row, float4 per thread
// per pass. The products that read the norm read it split, so it is computed and split once here.
__global__ __launch_bounds__(256) void k_resadd_norm_split(float* __restrict__ x, const float* __restrict__ part,
                                                           uint32_t splits, uint32_t M, uint32_t N, float eps,
                                                           const uint16_t* __restrict__ gain,
                                                           float* __restrict__ out) {
  constexpr int U = 4;  // N <= 4096: a row is at most 4 float4 per thread
  __shared__ float red[4];
  const uint32_t m = blockIdx.x, tid = threadIdx.x, n4 = N / 4;
  float4 v[U];
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < U; u++) {
    const uint32_t c = tid + 256 * u;
    if (c >= n4) break;
    float4* xr = reinterpret_cast<float4*>(x + size_t(m) * N) + c;
    v[u] = *xr;
    if (splits) {
      float4 acc = reinterpret_cast<const float4*>(part + size_t(m) * N)[c];
      for (uint32_t z = 1; z < splits; z++) {
        const float4 w = reinterpret_cast<const float4*>(part + (size_t(z) * M + m) * N)[c];
        acc.x += w.x; acc.y += w.y; acc.z += w.z; acc.w += w.w;
      }
      v[u].x += acc.x; v[u].y += acc.y; v[u].z += acc.z; v[u].w += acc.w;
      *xr = v[u];
    }
    ss += (v[u].x * v[u].x + v[u].y * v[u].y) + (v[u].z * v[u].z + v[u].w * v[u].w);
  }
  if (!gain) return;
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float sc = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / float(N) + eps);
#pragma unroll
  for (int u = 0; u < U; u++) {
    const uint32_t c = tid + 256 * u;
    if (c >= n4) break;
    const uint2 g = reinterpret_cast<const uint2*>(gain)[c];
    store_split4(out + size_t(m) * N, 4 * c, v[u].x * sc * __uint_as_float(g.x << 16),
                 v[u].y * sc * __uint_as_float(g.x & 0xFFFF0000u), v[u].z * sc * __uint_as_float(g.y << 16),
                 v[u].w * sc * __uint_as_float(g.y & 0xFFFF0000u));
  }
}

// ---------------------------------------------------------------------------------------------
// Per token m and row r of [q heads, k heads, v heads]: q/k RMSNorm + RoPE with the table row of
// position start + m; q goes to Q [M][n_heads][128], k and v to the cache slot (f32 or bf16).
// One wave per (token, row); lane l holds dims l and l + 64.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_qk_rope(BatchAttnParams p) {
  const uint32_t item = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const uint32_t rows = p.n_heads + 2 * p.n_kv;
  if (item >= p.M * rows) return;
  const uint32_t m = item / rows, r = item % rows, pos = p.start + m;
  const float* src = p.qkv + size_t(m) * rows * kHeadDim + size_t(r) * kHeadDim;
  float a = src[lane], b = src[lane + 64];
  if (r < p.n_heads + p.n_kv) {
    const uint16_t* gain = r < p.n_heads ? p.q_norm : p.k_norm;
    const float ss = wave_sum(a * a + b * b);
    const float sc = 1.0f / sqrtf(ss / float(kHeadDim) + p.eps);
    a = a * sc * bf16f(gain[lane]);
    b = b * sc * bf16f(gain[lane + 64]);
    const float2 cs = reinterpret_cast<const float2*>(p.rope)[size_t(pos) * (kHeadDim / 2) + lane];
    const float ar = a * cs.x - b * cs.y, br = b * cs.x + a * cs.y;
    a = ar;
    b = br;
  }
  if (r < p.n_heads) {
    float* q = p.q + (size_t(m) * p.n_heads + r) * kHeadDim;
    q[lane] = a;
    q[lane + 64] = b;
  } else {
    const uint32_t kvh = r < p.n_heads + p.n_kv ? r - p.n_heads : r - p.n_heads - p.n_kv;
    void* cache = r < p.n_heads + p.n_kv ? p.k_cache : p.v_cache;
    const size_t slot = (size_t(kvh) * p.max_seq + pos) * kHeadDim;
    if (p.kv_bf16) {
      static_cast<uint16_t*>(cache)[slot + lane] = f32_to_bf16(a);
      static_cast<uint16_t*>(cache)[slot + lane + 64] = f32_to_bf16(b);
    } else {
      static_cast<float*>(cache)[slot + lane] = a;
      static_cast<float*>(cache)[slot + lane + 64] = b;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Causal attention of a chunk on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16) with split
// operands: q, and f32 K / V, are split into hi + lo bf16 (K and V once, when a tile is staged
// in LDS), and each product keeps the hi*hi, hi*lo and lo*hi terms (lo*lo is below 2^-16 of the
// product); a bf16 cache is exact in hi, so its tiles take two terms.
// Workgroup (KV head g, block of TOK = 64 RB / G tokens, key run s) serves 64 RB query rows,
// row r = token mb + r / G of head g G + r % G, with eight waves: wave w owns RB blocks of 16 rows
// (rows 16 (RB (w % 4) + b) .. + 15), lane l the row l % 16 of each, and the keys of half w / 4 of
// every tile; the two halves' sums meet in LDS at the end. Keys come in LDS tiles of 64 positions,
// and every fragment a wave reads from LDS feeds the MFMAs of all its RB row blocks. Per tile a wave
// computes the transposed scores S^T[key][row] of its 32 keys (A = K rows: lane has key 16 j + l %
// 16, dims 32 s + 8 kg .. +7 with kg = l / 16; B = q of row l % 16, same dims). In the 16 x 16 output
// layout a lane then holds keys 16 j + 4 kg + r (j < 2, r < 4) of its own row, so the online softmax
// stays in the lane plus two shuffles across kg, with no LDS round trip for P. Next O^T[d][row] +=
// V^T P^T, with the k index mapped so that lane kg's eight B values are its own probabilities for
// keys 4 kg + r and 16 + 4 kg + r (r < 4); the A side reads those keys from a transposed V tile whose
// key slots are permuted to match (Vt[d][slot], key 32 s + 16 h + 4 kg + r in slot 32 s + 8 kg + 4 h +
// r), so a lane's eight keys are one 16-byte read, and O^T's column is again the lane's row. Rows with
// no visible key in the run keep m = -inf, l = 0. One run: normalized output to att [M][n_heads][128];
// several: (m, l, acc) partials to part [M][n_heads][runs][kPartStride], combined by
// k_attn_merge_rows.
// ROPE (short passes): q, k and v are the raw projections in qkv; the workgroup applies the q/k
// RMSNorm and RoPE to the rows it reads and appends the pass's K/V rows, so that no launch of its own
// has to.
// Bound: per SIMD and tile 96 MFMAs (1536 clocks) a wave beside ~230 VALU instructions (920); with
// both waves of a SIMD in one phase they add up (3.7 us per tile of 128 rows), a phase apart they
// overlap (2.9 us; four waves of all 64 keys, staged between two barriers, took 5). 512 rows at
// position 1536: 46 -> 34 us.
// ---------------------------------------------------------------------------------------------
template <int G, bool KV_BF16, int RB, bool ROPE>
__global__ __launch_bounds__(512) void k_attn_causal_bf(const float* q_in, const void* k_cache, const void* v_cache,
                                                        uint32_t start, uint32_t M, uint32_t max_seq,
                                                        uint32_t key_run, uint32_t runs, uint32_t n_heads,
                                                        uint32_t n_kv, BatchAttnParams p) {
  // what the first loads need comes first, as plain values (in scalar registers when a wave starts)
  if constexpr (ROPE) p.qkv = q_in;
  else p.q = const_cast<float*>(q_in);
  p.k_cache = const_cast<void*>(k_cache), p.v_cache = const_cast<void*>(v_cache);
  p.start = start, p.M = M, p.max_seq = max_seq, p.key_run = key_run, p.n_heads = n_heads, p.n_kv = n_kv;
  constexpr int D = kHeadDim, BK = 64, TOK = 64 * RB / G, KP = D + 8, VP = BK + 8, NL = KV_BF16 ? 1 : 2;
  constexpr int KS = NL * BK * KP, TILE = KS + NL * D * VP;        // u16s: K [hi, lo][key][dim], V [hi, lo][dim][key slot]
  constexpr int MERGE = 4 * RB * (8 * 64 * 8 + 16 * 4);            // ... of the halves' merge
  constexpr int NB = ROPE ? 1 : 2;                                 // LDS tiles
  __shared__ __align__(16) uint16_t smem[NB * TILE > MERGE ? NB * TILE : MERGE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kg = lane >> 4;
  const int rw = wave & 3, kh = wave >> 2;
  const uint32_t g = blockIdx.x, mb = blockIdx.y * TOK, run = blockIdx.z;
  if (run >= runs) {  // a prefetch workgroup (whole workgroup, before any load)
    l2_prefetch_tiles<512>(p.pf.pf, (run - runs) * gridDim.x * gridDim.y + blockIdx.y * gridDim.x + g,
                      reinterpret_cast<uint32_t*>(p.att));
    return;
  }
  uint32_t tok[RB], head[RB], my_pos[RB];
#pragma unroll
  for (int b = 0; b < RB; b++) {
    const uint32_t row = uint32_t(rw * RB + b) * 16 + uint32_t(li);
    tok[b] = mb + row / G;
    head[b] = g * G + row % G;
    my_pos[b] = p.start + min(tok[b], p.M - 1);
  }
  const uint32_t last = p.start + min(mb + TOK - 1, p.M - 1);  // positions 0..last are needed
  const uint32_t k_begin = run * p.key_run;
  const uint32_t k_end = min(last + 1, k_begin + p.key_run);  // this run: positions [k_begin, k_end)
  // scores in base-2 units (q carries the factor): softmax weights are 2^(s - m), the partials' m in
  // the same units
  const float sl2 = p.scale * 1.44269504088896341f;

  const uint32_t heads = ROPE ? p.n_heads + 2 * p.n_kv : p.n_heads;  // heads of a token's row of q
  float4 qv[RB][4][2];
#pragma unroll
  for (int b = 0; b < RB; b++) {
    const float* qp = (ROPE ? p.qkv : p.q) + (size_t(min(tok[b], p.M - 1)) * heads + head[b]) * D + 8 * kg;
#pragma unroll
    for (int st = 0; st < 4; st++) {
      qv[b][st][0] = *reinterpret_cast<const float4*>(qp + 32 * st);
      qv[b][st][1] = *reinterpret_cast<const float4*>(qp + 32 * st + 4);
    }
  }
  float4 q_rope[RB][2][4];  // ROPE: (cos, sin) of dims 32 st + 8 kg .. + 7 and the gains
  uint4 q_gain[4];
  if constexpr (ROPE) {
#pragma unroll
    for (int st = 0; st < 4; st++) q_gain[st] = *reinterpret_cast<const uint4*>(p.q_norm + 32 * st + 8 * kg);
#pragma unroll
    for (int b = 0; b < RB; b++)
#pragma unroll
      for (int st = 0; st < 2; st++)
#pragma unroll
        for (int c = 0; c < 4; c++)
          q_rope[b][st][c] =
              *reinterpret_cast<const float4*>(p.rope + size_t(my_pos[b]) * D + 2 * (32 * st + 8 * kg) + 4 * c);
  }

  // staging: K rows lr + 16 i (i < 4) at dims ld .. ld + 3; V key pair 2 vk, 2 vk + 1 at dims
  // vd + 64 i .. +3 (i < 2), so that Vt gets (key, key + 1) words; 8 lanes on one row
  const size_t hbase = size_t(g) * p.max_seq * D;
  const int lr = tid >> 5, ld = (tid & 31) * 4, vk = (tid >> 3) & 31, vd = 4 * (tid & 7) + 32 * (tid >> 8);
  // Vt slot of keys 2 vk, 2 vk + 1 (adjacent slots): key 32 s + 16 h + 4 c + r -> 32 s + 8 c + 4 h + r
  const int vslot = (2 * vk & 32) | ((2 * vk >> 2) & 3) << 3 | ((2 * vk >> 4) & 1) << 2 | (2 * vk & 3);
  using Pre = typename std::conditional<KV_BF16, uint2, float4>::type;
  Pre kp[4], vp[4];
  auto k_row = [&](int i) __attribute__((always_inline)) { return uint32_t(lr + 16 * i); };
  auto v_row = [&](int i) __attribute__((always_inline)) { return uint32_t(2 * vk + (i & 1)); };
  auto v_dim = [&](int i) __attribute__((always_inline)) { return vd + 64 * (i >> 1); };
  auto load_k = [&](uint32_t t0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const size_t ko = hbase + size_t(min(t0 + k_row(i), k_end - 1)) * D + ld;
      if constexpr (KV_BF16) kp[i] = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p.k_cache) + ko);
      else kp[i] = *reinterpret_cast<const float4*>(static_cast<const float*>(p.k_cache) + ko);
    }
  };
  auto load_v = [&](uint32_t t0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const size_t vo = hbase + size_t(min(t0 + v_row(i), k_end - 1)) * D + v_dim(i);
      if constexpr (KV_BF16) vp[i] = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p.v_cache) + vo);
      else vp[i] = *reinterpret_cast<const float4*>(static_cast<const float*>(p.v_cache) + vo);
    }
  };
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  auto pk = [](float x, float y) __attribute__((always_inline)) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x, y}), bf16x2));
  };
  auto store_k = [&](uint16_t* ks) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uint16_t* at = ks + k_row(i) * KP + ld;
      if constexpr (KV_BF16) {
        *reinterpret_cast<uint2*>(at) = kp[i];
      } else {
        const float4 v = kp[i];
        const uint32_t h0 = pk(v.x, v.y), h1 = pk(v.z, v.w);
        *reinterpret_cast<uint2*>(at) = make_uint2(h0, h1);
        *reinterpret_cast<uint2*>(at + BK * KP) =
            make_uint2(pk(v.x - __uint_as_float(h0 << 16), v.y - __uint_as_float(h0 & 0xFFFF0000u)),
                       pk(v.z - __uint_as_float(h1 << 16), v.w - __uint_as_float(h1 & 0xFFFF0000u)));
      }
    }
  };
  auto store_v = [&](uint16_t* vt) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; i += 2) {  // vp[i]: key 2 vk, vp[i + 1]: key 2 vk + 1
      uint16_t* at = vt + v_dim(i) * VP + vslot;
      if constexpr (KV_BF16) {
        const uint2 x = vp[i], y = vp[i + 1];
        const uint32_t w[4] = {(x.x & 0xFFFFu) | (y.x << 16), (x.x >> 16) | (y.x & 0xFFFF0000u),
                               (x.y & 0xFFFFu) | (y.y << 16), (x.y >> 16) | (y.y & 0xFFFF0000u)};
#pragma unroll
        for (int c = 0; c < 4; c++) *reinterpret_cast<uint32_t*>(at + c * VP) = w[c];
      } else {
        const float x[4] = {vp[i].x, vp[i].y, vp[i].z, vp[i].w};
        const float y[4] = {vp[i + 1].x, vp[i + 1].y, vp[i + 1].z, vp[i + 1].w};
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const uint32_t h = pk(x[c], y[c]);
          *reinterpret_cast<uint32_t*>(at + c * VP) = h;
          *reinterpret_cast<uint32_t*>(at + (D + c) * VP) =
              pk(x[c] - __uint_as_float(h << 16), y[c] - __uint_as_float(h & 0xFFFF0000u));
        }
      }
    }
  };
  // ROPE: the rows of this pass's own tokens come from its raw projections instead of the cache: k
  // normalized and rotated (a row sits in 32 lanes, its dims d and d + 64 in lanes 16 apart), in the
  // cache's type, and appended to the cache by the last token block, which sees all of them. All
  // loads come before the first use: one latency, not one per row.
  const bool append = ROPE && blockIdx.y == gridDim.y - 1;
  auto has_new = [&](uint32_t t0) __attribute__((always_inline)) {
    return ROPE && t0 + BK > p.start && k_end > p.start;
  };
  auto new_pos = [&](uint32_t t) __attribute__((always_inline)) { return max(min(t, k_end - 1), p.start); };
  auto to_cache = [&](float4 x) __attribute__((always_inline)) {
    if constexpr (KV_BF16)
      return make_uint2(f32_to_bf16(x.x) | uint32_t(f32_to_bf16(x.y)) << 16,
                        f32_to_bf16(x.z) | uint32_t(f32_to_bf16(x.w)) << 16);
    else return x;
  };
  auto pick = [](bool c, Pre x, Pre y) __attribute__((always_inline)) {  // component-wise (see k_gemm_wide's end)
    if constexpr (KV_BF16) return make_uint2(c ? x.x : y.x, c ? x.y : y.y);
    else return make_float4(c ? x.x : y.x, c ? x.y : y.y, c ? x.z : y.z, c ? x.w : y.w);
  };
  auto put = [&](void* cache, uint32_t t, int d, Pre x) __attribute__((always_inline)) {
    if (!append || t < p.start || t >= k_end) return;
    const size_t slot = hbase + size_t(t) * D + d;
    if constexpr (KV_BF16) *reinterpret_cast<uint2*>(static_cast<uint16_t*>(cache) + slot) = x;
    else *reinterpret_cast<float4*>(static_cast<float*>(cache) + slot) = x;
  };
  float4 x[4], r0[4], r1[4], y[4];  // k, (cos, sin) of its four dims, v
  uint2 gn;
  auto load_new = [&](uint32_t t0) __attribute__((always_inline)) {
    if (!has_new(t0)) return;
    gn = *reinterpret_cast<const uint2*>(p.k_norm + ld);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t tk = new_pos(t0 + k_row(i)), tv = new_pos(t0 + v_row(i));
      x[i] = *reinterpret_cast<const float4*>(p.qkv + (size_t(tk - p.start) * heads + p.n_heads + g) * D + ld);
      const float4* rp = reinterpret_cast<const float4*>(p.rope + size_t(tk) * D + 2 * (ld & 63));
      r0[i] = rp[0];
      r1[i] = rp[1];
      y[i] = *reinterpret_cast<const float4*>(p.qkv + (size_t(tv - p.start) * heads + p.n_heads + p.n_kv + g) * D +
                                              v_dim(i));
    }
  };
  auto apply_new = [&](uint32_t t0) __attribute__((always_inline)) {
    if (!has_new(t0)) return;
    float ss[4];
#pragma unroll
    for (int i = 0; i < 4; i++) ss[i] = (x[i].x * x[i].x + x[i].y * x[i].y) + (x[i].z * x[i].z + x[i].w * x[i].w);
#pragma unroll
    for (int m = 1; m < 32; m <<= 1)
#pragma unroll
      for (int i = 0; i < 4; i++) ss[i] += __shfl_xor(ss[i], m);
    const float s = ld < 64 ? -1.f : 1.f;  // a cos - b sin, b cos + a sin
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float sc = 1.0f / sqrtf(ss[i] / float(D) + p.eps);
      const float4 v =
          make_float4(x[i].x * sc * __uint_as_float(gn.x << 16), x[i].y * sc * __uint_as_float(gn.x & 0xFFFF0000u),
                      x[i].z * sc * __uint_as_float(gn.y << 16), x[i].w * sc * __uint_as_float(gn.y & 0xFFFF0000u));
      const float4 w = make_float4(s * __shfl_xor(v.x, 16), s * __shfl_xor(v.y, 16), s * __shfl_xor(v.z, 16),
                                   s * __shfl_xor(v.w, 16));
      const Pre nk = to_cache(make_float4(v.x * r0[i].x + w.x * r0[i].y, v.y * r0[i].z + w.y * r0[i].w,
                                          v.z * r1[i].x + w.z * r1[i].y, v.w * r1[i].z + w.w * r1[i].w));
      const Pre nv = to_cache(y[i]);
      // (rows past k_end hold row k_end - 1, which may be a new one: finite either way)
      kp[i] = pick(min(t0 + k_row(i), k_end - 1) >= p.start, nk, kp[i]);
      vp[i] = pick(min(t0 + v_row(i), k_end - 1) >= p.start, nv, vp[i]);
      put(p.k_cache, t0 + k_row(i), ld, nk);
      put(p.v_cache, t0 + v_row(i), v_dim(i), nv);
    }
  };
  // the first tile's K and V are in flight before q is used: a short pass's runs are one tile, and
  // its time is these loads' latency
  if (k_begin < k_end) {
    load_k(k_begin);
    load_v(k_begin);
    load_new(k_begin);
  }
  __builtin_amdgcn_sched_barrier(0);
  bf16x8 qh[RB][4], ql[RB][4];
  f32x4 o[RB][8];
  float m_run[RB], l_run[RB];
#pragma unroll
  for (int b = 0; b < RB; b++) {
#pragma unroll
    for (int i = 0; i < 8; i++) o[b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run[b] = -INFINITY;
    l_run[b] = 0.f;
    float v[4][8];
#pragma unroll
    for (int st = 0; st < 4; st++) {
      const float4 x = qv[b][st][0], y = qv[b][st][1];
      const float u[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
      for (int e = 0; e < 8; e++) v[st][e] = u[e];
    }
    if constexpr (ROPE) {  // q RMSNorm + RoPE (cpu_inference.rs:134-141): dims d, d + 64 in one lane
      float ss = 0.f;
#pragma unroll
      for (int st = 0; st < 4; st++)
#pragma unroll
        for (int e = 0; e < 8; e++) ss += v[st][e] * v[st][e];
      ss += __shfl_xor(ss, 16);
      ss += __shfl_xor(ss, 32);
      const float sc = 1.0f / sqrtf(ss / float(D) + p.eps);
#pragma unroll
      for (int st = 0; st < 2; st++) {
        const uint32_t ga[4] = {q_gain[st].x, q_gain[st].y, q_gain[st].z, q_gain[st].w};
        const uint32_t gb[4] = {q_gain[st + 2].x, q_gain[st + 2].y, q_gain[st + 2].z, q_gain[st + 2].w};
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float a = v[st][e] * sc * __uint_as_float(e & 1 ? ga[e / 2] & 0xFFFF0000u : ga[e / 2] << 16);
          const float c = v[st + 2][e] * sc * __uint_as_float(e & 1 ? gb[e / 2] & 0xFFFF0000u : gb[e / 2] << 16);
          const float4 r = q_rope[b][st][e / 2];
          const float cs = e & 1 ? r.z : r.x, sn = e & 1 ? r.w : r.y;
          v[st][e] = a * cs - c * sn;
          v[st + 2][e] = c * cs + a * sn;
        }
      }
    }
#pragma unroll
    for (int st = 0; st < 4; st++) {
#pragma unroll
      for (int e = 0; e < 8; e++) v[st][e] *= sl2;
      split8(v[st], qh[b][st], ql[b][st]);
    }
  }
  auto load_tile = [&](uint32_t t0) __attribute__((always_inline)) {
    if (t0 >= k_end) return;
    load_k(t0);
    load_v(t0);
  };
  auto store_tile = [&](uint16_t* at) __attribute__((always_inline)) {
    store_k(at);
    store_v(at + KS);
  };
  if (k_begin < k_end) {
    apply_new(k_begin);
    store_tile(smem);
  }
  load_tile(k_begin + BK);
  // Two LDS tiles, one barrier per tile: the next tile waits in registers and goes to the other LDS
  // tile before this one's products in the waves of key half 1, after them in those of key half 0.
  // The two waves of a SIMD are so in different phases: one's MFMAs run beside the other's staging
  // and softmax.
  uint32_t cur = 0;
  for (uint32_t t0 = k_begin; t0 < k_end; t0 += BK) {
    const bool more = t0 + BK < k_end;
    __syncthreads();  // this tile is in LDS; every wave is done with the other one
    auto stage = [&]() __attribute__((always_inline)) {
      load_new(t0 + BK);
      apply_new(t0 + BK);
      store_tile(smem + (NB == 2 ? cur ^ 1 : 0) * TILE);
      load_tile(t0 + 2 * BK);
    };
    if (NB == 2 && kh == 1 && more) stage();
    const uint16_t* ks = smem + cur * TILE + 32 * kh * KP;
    const uint16_t* vt = smem + cur * TILE + KS + 32 * kh;

    f32x4 s[RB][2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
#pragma unroll
      for (int b = 0; b < RB; b++) s[b][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < 4; st++) {
        const uint16_t* at = ks + (16 * j + li) * KP + 32 * st + 8 * kg;
        const bf16x8 hi = *reinterpret_cast<const bf16x8*>(at);
        bf16x8 lo;
        if constexpr (!KV_BF16) lo = *reinterpret_cast<const bf16x8*>(at + BK * KP);
#pragma unroll
        for (int b = 0; b < RB; b++) s[b][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, qh[b][st], s[b][j], 0, 0, 0);
#pragma unroll
        for (int b = 0; b < RB; b++) s[b][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, ql[b][st], s[b][j], 0, 0, 0);
        if constexpr (!KV_BF16) {
#pragma unroll
          for (int b = 0; b < RB; b++)
            s[b][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, qh[b][st], s[b][j], 0, 0, 0);
        }
      }
    }
    // every key of the tile is visible to every row
    const bool all_seen = t0 + BK <= k_end && t0 + BK <= p.start + mb + 1;
    bf16x8 ph[RB], pl[RB];
#pragma unroll
    for (int b = 0; b < RB; b++) {
      if (!all_seen) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const uint32_t t = t0 + uint32_t(32 * kh + 16 * j + 4 * kg + r);
            s[b][j][r] = t <= my_pos[b] && t < k_end ? s[b][j][r] : -INFINITY;
          }
        }
      }
      float mx = s[b][0][0];
#pragma unroll
      for (int e = 1; e < 8; e++) mx = fmaxf(mx, s[b][e / 4][e % 4]);
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      // m only has to keep 2^(s - m) in range: it moves when a row's maximum passes it by 8 (weights up
      // to 2^8), and the rows are rescaled only then. -inf while no key of the run is visible to the
      // row; m_use keeps -inf - -inf out, and 2^(-inf) = 0 needs no test per masked key.
      if (__any(mx > m_run[b] + 8.f)) {
        const float m_new = mx > m_run[b] + 8.f ? mx : m_run[b];
        const float corr = __builtin_amdgcn_exp2f(m_run[b] - (m_new == -INFINITY ? 0.f : m_new));
        l_run[b] *= corr;
        m_run[b] = m_new;
#pragma unroll
        for (int i = 0; i < 8; i++) o[b][i] *= corr;
      }
      const float m_use = m_run[b] == -INFINITY ? 0.f : m_run[b];
      float pv[8];
#pragma unroll
      for (int e = 0; e < 8; e++) pv[e] = __builtin_amdgcn_exp2f(s[b][e / 4][e % 4] - m_use);
      l_run[b] += ((pv[0] + pv[1]) + (pv[2] + pv[3])) + ((pv[4] + pv[5]) + (pv[6] + pv[7]));
      split8(pv, ph[b], pl[b]);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const uint16_t* at = vt + (16 * i + li) * VP + 8 * kg;
      const bf16x8 hi = *reinterpret_cast<const bf16x8*>(at);
      bf16x8 lo;
      if constexpr (!KV_BF16) lo = *reinterpret_cast<const bf16x8*>(at + D * VP);
#pragma unroll
      for (int b = 0; b < RB; b++) o[b][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, ph[b], o[b][i], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < RB; b++) o[b][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, pl[b], o[b][i], 0, 0, 0);
      if constexpr (!KV_BF16) {
#pragma unroll
        for (int b = 0; b < RB; b++) o[b][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, ph[b], o[b][i], 0, 0, 0);
      }
    }
    if (NB == 1) __syncthreads();  // every wave is done with this tile
    if ((NB == 1 || kh == 0) && more) stage();
    if (NB == 2) cur ^= 1;
  }
#pragma unroll
  for (int b = 0; b < RB; b++) {  // a lane's sum is over its own keys so far
    l_run[b] += __shfl_xor(l_run[b], 16);
    l_run[b] += __shfl_xor(l_run[b], 32);
  }
  // the two key halves of a row block meet in LDS; lane holds O^T[16 i + 4 kg + r][row], r < 4
  f32x4* ro = reinterpret_cast<f32x4*>(smem);
  float2* rml = reinterpret_cast<float2*>(ro + 4 * RB * 8 * 64);
  __syncthreads();
  if (kh == 1) {
#pragma unroll
    for (int b = 0; b < RB; b++) {
#pragma unroll
      for (int i = 0; i < 8; i++) ro[((rw * RB + b) * 8 + i) * 64 + lane] = o[b][i];
      if (kg == 0) rml[(rw * RB + b) * 16 + li] = make_float2(m_run[b], l_run[b]);
    }
  }
  __syncthreads();
  if (kh == 1) return;
#pragma unroll
  for (int b = 0; b < RB; b++) {
    if (tok[b] >= p.M) continue;
    const float2 ml = rml[(rw * RB + b) * 16 + li];
    const float m = fmaxf(m_run[b], ml.x), m_use = m == -INFINITY ? 0.f : m;
    const float e0 = __builtin_amdgcn_exp2f(m_run[b] - m_use), e1 = __builtin_amdgcn_exp2f(ml.x - m_use);
    const float l = l_run[b] * e0 + ml.y * e1;
#pragma unroll
    for (int i = 0; i < 8; i++) o[b][i] = o[b][i] * e0 + ro[((rw * RB + b) * 8 + i) * 64 + lane] * e1;
    const size_t vec = size_t(tok[b]) * p.n_heads + head[b];
    if (runs == 1) {
      const float inv = 1.0f / l;
      float* out = p.att + vec * D;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const f32x4 v = o[b][i] * inv;
        if (p.att_split) store_split4(out, 16 * i + 4 * kg, v[0], v[1], v[2], v[3]);
        else *reinterpret_cast<f32x4*>(out + 16 * i + 4 * kg) = v;
      }
    } else {
      float* out = p.part + (vec * runs + run) * kPartStride;
      if (kg == 0) {
        out[0] = m;
        out[1] = l;
      }
#pragma unroll
      for (int i = 0; i < 8; i++) *reinterpret_cast<f32x4*>(out + 4 + 16 * i + 4 * kg) = o[b][i];
    }
  }
}

// att[v] = sum_s e_s acc_s / sum_s e_s l_s over the runs of query vector v = (token, head),
// e_s = 2^(m_s - max m) (m in base-2 units); runs without a visible key (m = -inf) weigh 0. Eight
// query vectors per workgroup of 256 threads (four dims each); all U >= runs run loads are issued
// at once.
template <int U>
__global__ __launch_bounds__(256) void k_attn_merge_rows(const float* __restrict__ part, uint32_t runs,
                                                         uint32_t n_vec, float* __restrict__ att, int split) {
  const size_t v = min(blockIdx.x * 8 + (threadIdx.x >> 5), n_vec - 1);  // past the end: the last one again
  const uint32_t d = 4 * (threadIdx.x & 31);
  const float* base = part + v * runs * kPartStride;
  float2 ml[U];
  f32x4 av[U];
#pragma unroll
  for (int u = 0; u < U; u++) {
    const float* q = base + size_t(min(uint32_t(u), runs - 1)) * kPartStride;
    ml[u] = *reinterpret_cast<const float2*>(q);
    av[u] = *reinterpret_cast<const f32x4*>(q + 4 + d);
  }
  __builtin_amdgcn_sched_barrier(0);
  float M = -INFINITY;
#pragma unroll
  for (int u = 0; u < U; u++) M = uint32_t(u) < runs ? fmaxf(M, ml[u].x) : M;
  float L = 0.f;
  f32x4 A = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < U; u++) {  // m in base-2 units (k_attn_causal_bf)
    const float e = (uint32_t(u) < runs && ml[u].x != -INFINITY) ? exp2f(ml[u].x - M) : 0.f;
    L += e * ml[u].y;
#pragma unroll
    for (int r = 0; r < 4; r++) A[r] += e * av[u][r];
  }
#pragma unroll
  for (int r = 0; r < 4; r++) A[r] /= L;
  if (split) store_split4(att + v * kHeadDim, d, A[0], A[1], A[2], A[3]);
  else *reinterpret_cast<f32x4*>(att + v * kHeadDim + d) = A;
}

// tokens[r] = the greedy token of logits row r by the reference's scan (bench.rs:98-103,
// main.rs:37-42): the largest non-NaN value, lowest index on ties, and 0 when the row starts
// with NaN (or has nothing above -inf). Two launches: kArgParts workgroups per row each reduce
// one slice of the row to a (value, index) candidate, then one wave per row reduces the
// candidates. The comparison is a total order on (value, index) among non-NaN values, so the
// result does not depend on how the row is cut.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_row_argmax_part(const float* __restrict__ logits, uint32_t V, uint32_t S,
                                                         ArgCand* __restrict__ cand) {
  __shared__ float sv[4];
  __shared__ uint32_t si[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* x = logits + size_t(blockIdx.y) * V;
  const uint32_t beg = blockIdx.x * S, end = min(V, beg + S);
  float bv = -INFINITY;
  uint32_t bi = 0xFFFFFFFFu;
  constexpr int U = 4;
  for (uint32_t base = beg; base < end; base += 256u * U) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = x[min(base + uint32_t(tid) + 256u * u, V - 1)];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t i = base + uint32_t(tid) + 256u * u;
      if (i < end && cand_better(v[u], i, bv, bi)) { bv = v[u]; bi = i; }  // NaN never wins
    }
  }
  for (int o = 1; o < 64; o <<= 1) {
    const float ov = __shfl_xor(bv, o);
    const uint32_t oi = __shfl_xor(bi, o);
    if (cand_better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
  }
  if (lane == 0) { sv[wave] = bv; si[wave] = bi; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; w++)
      if (cand_better(sv[w], si[w], bv, bi)) { bv = sv[w]; bi = si[w]; }
    cand[size_t(blockIdx.y) * kArgParts + blockIdx.x] = ArgCand{bv, bi};
  }
}

// err_in / err_out (optional): workgroup 0 also copies the error word to err_out, so a host that
// waits for tokens (and err_out) in pinned memory learns of a failed pass without synchronizing
__global__ __launch_bounds__(64) void k_row_argmax_final(const ArgCand* __restrict__ cand,
                                                         const float* __restrict__ logits, uint32_t V,
                                                         uint32_t* __restrict__ tokens, const uint32_t* err_in,
                                                         uint32_t* err_out) {
  static_assert(kArgParts == 64, "one candidate per lane");
  const uint32_t row = blockIdx.x, lane = threadIdx.x;
  const ArgCand c = cand[size_t(row) * kArgParts + lane];
  const bool nan0 = isnan(logits[size_t(row) * V]);
  float bv = c.v;
  uint32_t bi = c.i;
  for (int o = 1; o < 64; o <<= 1) {
    const float ov = __shfl_xor(bv, o);
    const uint32_t oi = __shfl_xor(bi, o);
    if (cand_better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
  }
  if (lane == 0) tokens[row] = (nan0 || bi == 0xFFFFFFFFu) ? 0u : bi;
  if (err_out && row == 0 && lane == 0) __atomic_store_n(err_out, *err_in, __ATOMIC_RELAXED);
}

// x[m] = bf16 embedding row of ids[m] (cpu_inference.rs:109-111)
__global__ __launch_bounds__(256) void k_embed_rows(const uint16_t* __restrict__ table, const uint32_t* __restrict__ ids,
                                                    uint32_t M, uint32_t H, float* __restrict__ x) {
  const uint32_t m = blockIdx.y;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < H; i += gridDim.x * 256)
    x[size_t(m) * H + i] = bf16f(table[size_t(ids[m]) * H + i]);
}

// the same with the ids in the kernel argument
__global__ __launch_bounds__(256) void k_embed_rows_v(const uint16_t* __restrict__ table, TokenIds ids, uint32_t H,
                                                      float* __restrict__ x) {
  const uint32_t m = blockIdx.y;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < H; i += gridDim.x * 256)
    x[size_t(m) * H + i] = bf16f(table[size_t(ids.id[m]) * H + i]);
}

// ---------------------------------------------------------------------------------------------
// Matvec over the NV = M token rows of a short verify pass or chunk (M <= kMvRowsMaxM, with a residual
// kMvResAddMaxM): the decode step's matvec layout. A row group of TPR threads covers one weight row in 8-column
// chunks (CPT per thread) and RR rows per group; each weight chunk is loaded once (128-bit) and
// multiplied by the NV token rows in f32 FMA, so the weights stream once per pass as in a decode
// step. With NORM every row group computes the sum of squares of each token row over its own
// chunks (which cover the row) and scales the dot products, s * sum_c W[r,c] (x_c * g_c)
// (cpu_inference.rs:189-194, 225-257). All loads are issued before the first use. Each token row
// costs every wave its own products and lane reductions, so past a few rows the matrix cores
// (k_gemm_kslice) are faster.
// ---------------------------------------------------------------------------------------------
template <int TPR, int CPT, int RR, int NV, bool NORM, int EPI, int SM = 0>
__global__ __launch_bounds__(256) void k_mv_rows(MvRowsParams p) {
  constexpr int NG = 256 / TPR, WPG = TPR / 64, NS = NV * (RR + 1);
  __shared__ float red[4][NS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int grp = tid / TPR, t = tid % TPR;
  const uint32_t nch = p.cols >> 3;
  const uint32_t row0 = (blockIdx.x * NG + uint32_t(grp)) * RR;
  uint32_t cc[CPT];
#pragma unroll
  for (int k = 0; k < CPT; k++) cc[k] = min(uint32_t(t) + uint32_t(TPR) * k, nch - 1);

  // SM > 0: x is merged from the attention's partials (SM slots per chunk, the split kernel's
  // layout), loaded before the weights as the decode step's o_proj does
  float2 ml[SM > 0 ? NV : 1][CPT][SM > 0 ? SM : 1];
  float4 a0[SM > 0 ? NV : 1][CPT][SM > 0 ? SM : 1], a1[SM > 0 ? NV : 1][CPT][SM > 0 ? SM : 1];
  if constexpr (SM > 0) {
    const uint32_t S = p.attn_splits, th = p.tok_heads, GT = uint32_t(NV) * th;
#pragma unroll
    for (int v = 0; v < NV; v++) {
#pragma unroll
      for (int k = 0; k < CPT; k++) {
        const uint32_t h = cc[k] >> 4, d0 = (cc[k] & 15) * 8, g = h / th, j = uint32_t(v) * th + h % th;
#pragma unroll
        for (int s = 0; s < SM; s++) {
          const float* q = p.attn_part + ((size_t(g) * S + min(uint32_t(s), S - 1)) * GT + j) * kPartStride;
          ml[v][k][s] = *reinterpret_cast<const float2*>(q);
          a0[v][k][s] = *reinterpret_cast<const float4*>(q + 4 + d0);
          a1[v][k][s] = *reinterpret_cast<const float4*>(q + 8 + d0);
        }
      }
    }
  }
  const uint4* W = reinterpret_cast<const uint4*>(p.w);
  uint4 wv[RR][CPT];
#pragma unroll
  for (int r = 0; r < RR; r++) {
    const size_t row = min(row0 + uint32_t(r), p.rows - 1);
#pragma unroll
    for (int k = 0; k < CPT; k++) wv[r][k] = W[row * nch + cc[k]];
  }
  const float4* X = reinterpret_cast<const float4*>(p.x);
  float4 xa[NV][CPT], xb[NV][CPT];
  if constexpr (SM == 0) {
#pragma unroll
    for (int v = 0; v < NV; v++) {
#pragma unroll
      for (int k = 0; k < CPT; k++) {
        xa[v][k] = X[size_t(v) * (p.cols >> 2) + 2 * cc[k]];
        xb[v][k] = X[size_t(v) * (p.cols >> 2) + 2 * cc[k] + 1];
      }
    }
  }
  uint4 gains[CPT];
  if constexpr (NORM) {
#pragma unroll
    for (int k = 0; k < CPT; k++) gains[k] = reinterpret_cast<const uint4*>(p.gain)[cc[k]];
  }
  float res[NV][RR];
  if constexpr (EPI == kGemmResAdd) {
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int r = 0; r < RR; r++) res[v][r] = p.out[size_t(v) * p.ldo + min(row0 + uint32_t(r), p.rows - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (SM > 0) {
    // x = sum_s e_s acc_s / sum_s e_s l_s, e_s = exp(m_s - max m) (cpu_inference.rs:153-160 over
    // the runs); empty runs (m = -inf) and slots past the last run weigh 0
    const uint32_t S = p.attn_splits;
#pragma unroll
    for (int v = 0; v < NV; v++) {
#pragma unroll
      for (int k = 0; k < CPT; k++) {
        float M = -INFINITY;
#pragma unroll
        for (int s = 0; s < SM; s++) M = uint32_t(s) < S ? fmaxf(M, ml[v][k][s].x) : M;
        float L = 0.f;
        float4 A0 = make_float4(0.f, 0.f, 0.f, 0.f), A1 = A0;
#pragma unroll
        for (int s = 0; s < SM; s++) {
          const float e = (uint32_t(s) < S && ml[v][k][s].x != -INFINITY) ? expf(ml[v][k][s].x - M) : 0.f;
          L += e * ml[v][k][s].y;
          A0.x += e * a0[v][k][s].x; A0.y += e * a0[v][k][s].y; A0.z += e * a0[v][k][s].z; A0.w += e * a0[v][k][s].w;
          A1.x += e * a1[v][k][s].x; A1.y += e * a1[v][k][s].y; A1.z += e * a1[v][k][s].z; A1.w += e * a1[v][k][s].w;
        }
        const float inv = 1.0f / L;
        xa[v][k] = make_float4(A0.x * inv, A0.y * inv, A0.z * inv, A0.w * inv);
        xb[v][k] = make_float4(A1.x * inv, A1.y * inv, A1.z * inv, A1.w * inv);
      }
    }
  }

  if (uint32_t(TPR) * CPT > nch) {  // chunks past the row end contribute 0
#pragma unroll
    for (int k = 0; k < CPT; k++) {
      // component-wise: a ternary between float4 objects selects their addresses and sends the
      // arrays to scratch memory
      const bool in = uint32_t(t) + uint32_t(TPR) * k < nch;
#pragma unroll
      for (int v = 0; v < NV; v++) {
        const float4 a = xa[v][k], b = xb[v][k];
        xa[v][k] = make_float4(in ? a.x : 0.f, in ? a.y : 0.f, in ? a.z : 0.f, in ? a.w : 0.f);
        xb[v][k] = make_float4(in ? b.x : 0.f, in ? b.y : 0.f, in ? b.z : 0.f, in ? b.w : 0.f);
      }
    }
  }
  float ss[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    ss[v] = 0.f;
    if constexpr (NORM) {
#pragma unroll
      for (int k = 0; k < CPT; k++) {
        const float4 a = xa[v][k], b = xb[v][k];
        ss[v] += (a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w) + (b.x * b.x + b.y * b.y + b.z * b.z + b.w * b.w);
        const uint4 g = gains[k];
        xa[v][k] = make_float4(a.x * __uint_as_float(g.x << 16), a.y * __uint_as_float(g.x & 0xFFFF0000u),
                               a.z * __uint_as_float(g.y << 16), a.w * __uint_as_float(g.y & 0xFFFF0000u));
        xb[v][k] = make_float4(b.x * __uint_as_float(g.z << 16), b.y * __uint_as_float(g.z & 0xFFFF0000u),
                               b.z * __uint_as_float(g.w << 16), b.w * __uint_as_float(g.w & 0xFFFF0000u));
      }
      ss[v] = wave_sum(ss[v]);
    }
  }
  float acc[NV][RR];
#pragma unroll
  for (int v = 0; v < NV; v++)
#pragma unroll
    for (int r = 0; r < RR; r++) {
      float a = 0.f;
#pragma unroll
      for (int k = 0; k < CPT; k++) a = dot8(wv[r][k], xa[v][k], xb[v][k], a);
      acc[v][r] = wave_sum(a);
    }
  if constexpr (WPG > 1) {
    if (lane == 0) {
#pragma unroll
      for (int v = 0; v < NV; v++) {
#pragma unroll
        for (int r = 0; r < RR; r++) red[wave][v * (RR + 1) + r] = acc[v][r];
        red[wave][v * (RR + 1) + RR] = ss[v];
      }
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int r = 0; r <= RR; r++) {
        float a = 0.f;
#pragma unroll
        for (int w = 0; w < WPG; w++) a += red[grp * WPG + w][v * (RR + 1) + r];
        if (r < RR) acc[v][r] = a;
        else ss[v] = a;
      }
  }
  if (t != 0) return;
#pragma unroll
  for (int v = 0; v < NV; v++) {
    float sc = 1.f;
    if constexpr (NORM) sc = 1.0f / sqrtf(ss[v] / float(p.cols) + p.eps);
    float* o = p.out + size_t(v) * p.ldo;
    if constexpr (EPI == kGemmSiluPair) {
#pragma unroll
      for (int r = 0; r + 1 < RR; r += 2) {
        const uint32_t row = row0 + uint32_t(r);
        if (row + 1 < p.rows) {
          const float g = acc[v][r] * sc;
          o[row >> 1] = g / (1.0f + expf(-g)) * (acc[v][r + 1] * sc);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < RR; r++) {
        const uint32_t row = row0 + uint32_t(r);
        if (row < p.rows) o[row] = EPI == kGemmResAdd ? res[v][r] + acc[v][r] * sc : acc[v][r] * sc;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// final RMSNorm + lm_head over the NV token rows of a short verify pass: the decode step's lm_head
// matvec (k_matvec<R, CPL, kNorm, ..>: each wave R rows, lane l the 16-byte chunks l, l + 64, ..)
// with the NV normalized rows staged in LDS, so the 311 MB of weights stream once for all rows.
// Each row's norm and dot products are summed in the decode step's order, so a row's logits equal
// that step's bit for bit. out[v][row] = logits, ldo per token row.
// ---------------------------------------------------------------------------------------------
template <int R, int CPL, int NV>
__global__ __launch_bounds__(256) void k_lm_head_rows(MvRowsParams p) {
  extern __shared__ __align__(16) float xs[];  // [NV][cols]
  __shared__ float red[NV][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t nch = p.cols >> 3;
  const uint32_t row0 = (blockIdx.x * 4u + uint32_t(wave)) * R;
  const uint4* W = reinterpret_cast<const uint4*>(p.w);
  uint4 wv[R][CPL];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const uint32_t row = min(row0 + uint32_t(r), p.rows - 1);  // past the end: re-read the last row
    const uint4* wr = W + size_t(row) * nch;
#pragma unroll
    for (int k = 0; k < CPL; k++) wv[r][k] = ld_stream(&wr[min(uint32_t(lane) + 64u * k, nch - 1)]);  // (as k_matvec)
  }
  const float4* x4 = reinterpret_cast<const float4*>(p.x);
  float4* xs4 = reinterpret_cast<float4*>(xs);
  const uint32_t c4 = p.cols / 4;
  // no gain: the rows come normalized (the fused verify pass's final reduce applied the norm)
  const bool norm = p.gain != nullptr;
#pragma unroll
  for (int v = 0; v < NV; v++) {
    float ss = 0.f;
    for (uint32_t i = tid; i < c4; i += 256) {
      const float4 a = x4[size_t(v) * c4 + i];
      xs4[v * c4 + i] = a;
      ss += a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w;
    }
    if (norm) {
      ss = wave_sum(ss);
      if (lane == 0) red[v][wave] = ss;
    }
  }
  __syncthreads();
  if (norm) {
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const float tot = (red[v][0] + red[v][1]) + (red[v][2] + red[v][3]);
      const float sc = 1.0f / sqrtf(tot / float(p.cols) + p.eps);
      for (uint32_t i = tid; i < p.cols; i += 256) xs[v * p.cols + i] = xs[v * p.cols + i] * sc * bf16f(p.gain[i]);
    }
    __syncthreads();
  }
  float acc[NV][R];
#pragma unroll
  for (int v = 0; v < NV; v++)
#pragma unroll
    for (int r = 0; r < R; r++) acc[v][r] = 0.f;
#pragma unroll
  for (int k = 0; k < CPL; k++) {
    const uint32_t c = uint32_t(lane) + 64u * k;
    if (c < nch) {
#pragma unroll
      for (int v = 0; v < NV; v++) {
        const float4 a = xs4[v * c4 + 2 * c], b = xs4[v * c4 + 2 * c + 1];
#pragma unroll
        for (int r = 0; r < R; r++) acc[v][r] = dot8(wv[r][k], a, b, acc[v][r]);
      }
    }
  }
#pragma unroll
  for (int v = 0; v < NV; v++)
#pragma unroll
    for (int r = 0; r < R; r++) acc[v][r] = wave_sum(acc[v][r]);
  if (lane == 0) {
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int r = 0; r < R; r++) {
        const uint32_t row = row0 + uint32_t(r);
        if (row < p.rows) p.out[size_t(v) * p.ldo + row] = acc[v][r];
      }
  }
  if (p.cand) {  // each token row's best (value, row) of this workgroup, NaN never (k_matvec kLogits)
    __shared__ ArgCand cb[NV][4];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      float bv = -INFINITY;
      uint32_t bi = 0xFFFFFFFFu;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const uint32_t row = row0 + uint32_t(r);
        if (row < p.rows && !isnan(acc[v][r]) && cand_better(acc[v][r], row, bv, bi)) {
          bv = acc[v][r];
          bi = row;
        }
      }
      if (lane == 0) cb[v][wave] = ArgCand{bv, bi};
    }
    __syncthreads();
    if (tid < NV) {
      ArgCand b = cb[tid][0];
      for (int w = 1; w < 4; w++)
        if (cand_better(cb[tid][w].v, cb[tid][w].i, b.v, b.i)) b = cb[tid][w];
      p.cand[size_t(tid) * gridDim.x + blockIdx.x] = b;
    }
  }
}

// tokens[row] from the row's candidates: the first maximum, NaN never wins, a NaN first logit or
// no candidate above -inf gives 0 (main.rs:37-42; k_argmax's reduction, one workgroup per row)
__global__ __launch_bounds__(1024) void k_cand_argmax(const ArgCand* __restrict__ cand, uint32_t n_cand,
                                                      const float* __restrict__ logits, uint32_t V,
                                                      uint32_t* __restrict__ tokens, const uint32_t* err_in,
                                                      uint32_t* err_out) {
  __shared__ float sv[16];
  __shared__ uint32_t si[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t row = blockIdx.x;
  cand += size_t(row) * n_cand;
  float bv = -INFINITY;
  uint32_t bi = 0xFFFFFFFFu;
  constexpr int U = 16;
  for (uint32_t base = 0; base < n_cand; base += 1024u * U) {
    ArgCand c[U];
#pragma unroll
    for (int u = 0; u < U; u++) c[u] = cand[min(base + uint32_t(tid) + 1024u * u, n_cand - 1)];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (cand_better(c[u].v, c[u].i, bv, bi)) { bv = c[u].v; bi = c[u].i; }
  }
  for (int o = 1; o < 64; o <<= 1) {
    const float ov = __shfl_xor(bv, o);
    const uint32_t oi = __shfl_xor(bi, o);
    if (cand_better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
  }
  if (lane == 0) { sv[wave] = bv; si[wave] = bi; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 16; w++)
      if (cand_better(sv[w], si[w], bv, bi)) { bv = sv[w]; bi = si[w]; }
    tokens[row] = (isnan(logits[size_t(row) * V]) || bi == 0xFFFFFFFFu) ? 0u : bi;
    if (err_out && row == 0) __atomic_store_n(err_out, *err_in, __ATOMIC_RELAXED);
  }
}

template <int TPR, int CPT, int RR, int NV, bool NORM, int EPI>
hipError_t launch_mv_rows_t(const MvRowsParams& p, hipStream_t st) {
  constexpr int rows_per_block = (256 / TPR) * RR;
  hipLaunchKernelGGL((k_mv_rows<TPR, CPT, RR, NV, NORM, EPI>), dim3(ceil_div(p.rows, rows_per_block)), dim3(256), 0,
                     st, p);
  return hipGetLastError();
}

// the decode matvec's shapes: an exact fit of threads x chunks where one exists; silu rows pair up
template <int NV, bool NORM, int EPI>
hipError_t launch_mv_rows_cols(const MvRowsParams& p, hipStream_t st) {
  const uint32_t nch = p.cols / 8;
  constexpr bool SILU = EPI == kGemmSiluPair;
  if (nch <= 64) return launch_mv_rows_t<64, 1, 2, NV, NORM, EPI>(p, st);
  if (nch <= 128) {
    if (SILU) return launch_mv_rows_t<64, 2, 2, NV, NORM, EPI>(p, st);
    return launch_mv_rows_t<128, 1, 2, NV, NORM, EPI>(p, st);
  }
  if (nch <= 256) return launch_mv_rows_t<256, 1, SILU ? 2 : 1, NV, NORM, EPI>(p, st);
  if (nch == 384) return launch_mv_rows_t<128, 3, 2, NV, NORM, EPI>(p, st);
  if (nch <= 512) return launch_mv_rows_t<256, 2, SILU ? 2 : 1, NV, NORM, EPI>(p, st);
  return hipErrorInvalidValue;
}

template <int NV>
hipError_t launch_mv_rows_nv(const MvRowsParams& p, bool norm, int epi, hipStream_t st) {
  if (norm && epi == kGemmStore) return launch_mv_rows_cols<NV, true, kGemmStore>(p, st);
  if (norm && epi == kGemmSiluPair) return launch_mv_rows_cols<NV, true, kGemmSiluPair>(p, st);
  if (!norm && epi == kGemmResAdd) return launch_mv_rows_cols<NV, false, kGemmResAdd>(p, st);
  if (!norm && epi == kGemmStore) return launch_mv_rows_cols<NV, false, kGemmStore>(p, st);
  return hipErrorInvalidValue;
}

// o_proj with the attention merge: four rows per workgroup amortize the merge, which every
// workgroup repeats for all heads of its token rows
template <int NV, int SM>
hipError_t launch_mv_merge_t(const MvRowsParams& p, hipStream_t st) {
  const uint32_t nch = p.cols / 8;
  if (nch <= 128) {
    hipLaunchKernelGGL((k_mv_rows<128, 1, 4, NV, false, kGemmResAdd, SM>), dim3(ceil_div(p.rows, 8u)), dim3(256), 0,
                       st, p);
  } else {
    hipLaunchKernelGGL((k_mv_rows<256, 1, 4, NV, false, kGemmResAdd, SM>), dim3(ceil_div(p.rows, 4u)), dim3(256), 0,
                       st, p);
  }
  return hipGetLastError();
}

uint32_t mv_merge_slots(uint32_t splits) { return splits <= 4 ? 4 : splits <= 8 ? 8 : 16; }

template <int NV>
hipError_t launch_mv_merge_nv(const MvRowsParams& p, hipStream_t st) {
  const uint32_t sm = mv_merge_slots(p.attn_splits);
  if (sm == 4) return launch_mv_merge_t<NV, 4>(p, st);
  if constexpr (NV <= 2) {
    if (sm == 8) return launch_mv_merge_t<NV, 8>(p, st);
  }
  if constexpr (NV == 1) return launch_mv_merge_t<NV, 16>(p, st);
  return hipErrorNotSupported;
}

}  // namespace

bool mv_rows_merge_fits(uint32_t M, uint32_t splits) {
  return M >= 1 && M <= kMvRowsMaxM && splits >= 1 && splits <= uint32_t(kAttnMaxMergeSplits) &&
         M * mv_merge_slots(splits) <= 16;
}

hipError_t launch_mv_rows_merge(const MvRowsParams& p, hipStream_t st) {
  if (!p.w || !p.out || !p.attn_part || p.M == 0 || p.M > kMvRowsMaxM || p.rows == 0 || p.cols == 0 ||
      p.ldo < p.rows || p.attn_splits == 0 || p.tok_heads == 0)
    return hipErrorInvalidValue;
  if (p.cols % kHeadDim || p.cols / 8 > 256 || !mv_rows_merge_fits(p.M, p.attn_splits)) return hipErrorNotSupported;
  switch (p.M) {
    case 1: return launch_mv_merge_nv<1>(p, st);
    case 2: return launch_mv_merge_nv<2>(p, st);
    case 3: return launch_mv_merge_nv<3>(p, st);
    default: return launch_mv_merge_nv<4>(p, st);
  }
}

uint32_t lm_head_rows_workgroups(uint32_t rows) { return ceil_div(rows, 4u * 4u); }

hipError_t launch_cand_argmax(const ArgCand* cand, uint32_t n_cand, const float* logits, uint32_t rows, uint32_t V,
                              uint32_t* tokens, hipStream_t st, const uint32_t* err_in, uint32_t* err_out) {
  if (!cand || !logits || !tokens || n_cand == 0 || rows == 0 || V == 0 || rows > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_cand_argmax, dim3(rows), dim3(1024), 0, st, cand, n_cand, logits, V, tokens, err_in, err_out);
  return hipGetLastError();
}

hipError_t launch_lm_head_rows(const MvRowsParams& p, hipStream_t st) {
  if (!p.w || !p.x || !p.out || p.M == 0 || p.M > kMvRowsMaxM || p.rows == 0 || p.cols == 0 ||
      p.cols % 8 || p.ldo < p.rows)
    return hipErrorInvalidValue;
  if (p.cols / 8 > 128) return hipErrorNotSupported;  // the decode lm_head's shape: 2 chunks per lane
  constexpr int CPL = 2, R = 4;
  const dim3 grid(ceil_div(p.rows, 4u * R));
  const size_t lds = size_t(p.M) * p.cols * 4;
  switch (p.M) {
    case 1: hipLaunchKernelGGL((k_lm_head_rows<R, CPL, 1>), grid, dim3(256), lds, st, p); break;
    case 2: hipLaunchKernelGGL((k_lm_head_rows<R, CPL, 2>), grid, dim3(256), lds, st, p); break;
    case 3: hipLaunchKernelGGL((k_lm_head_rows<R, CPL, 3>), grid, dim3(256), lds, st, p); break;
    default: hipLaunchKernelGGL((k_lm_head_rows<R, CPL, 4>), grid, dim3(256), lds, st, p); break;
  }
  return hipGetLastError();
}

hipError_t launch_mv_rows(const MvRowsParams& p, bool norm, int epi, hipStream_t st) {
  const uint32_t max_m = !norm && epi == kGemmResAdd ? kMvResAddMaxM : kMvRowsMaxM;
  if (!p.w || !p.x || !p.out || (norm && !p.gain) || p.M == 0 || p.M > max_m || p.rows == 0 || p.cols == 0 ||
      p.cols % 8 || p.cols / 8 > 512 || (epi == kGemmSiluPair ? p.rows % 2 || p.ldo < p.rows / 2 : p.ldo < p.rows))
    return hipErrorInvalidValue;
  switch (p.M) {
    case 1: return launch_mv_rows_nv<1>(p, norm, epi, st);
    case 2: return launch_mv_rows_nv<2>(p, norm, epi, st);
    case 3: return launch_mv_rows_nv<3>(p, norm, epi, st);
    case 4: return launch_mv_rows_nv<4>(p, norm, epi, st);
    case 5: return launch_mv_rows_cols<5, false, kGemmResAdd>(p, st);
    default: return launch_mv_rows_cols<6, false, kGemmResAdd>(p, st);
  }
}

namespace {

hipError_t check_grid(uint64_t wgs, uint32_t threads) {
  return wgs * threads < (uint64_t(1) << 32) ? hipSuccess : hipErrorInvalidValue;
}

template <bool NORM, int EPI, int MT, int NT, int NW, int NS>
hipError_t launch_kslice_t(const GemmParams& p, hipStream_t st) {
  const uint64_t wgs = (uint64_t(p.M) + 16 * MT - 1) / (16 * MT) * ((uint64_t(p.N) + 16 * NT - 1) / (16 * NT));
  if (hipError_t e = check_grid(wgs, 64 * NW)) return e;
  if constexpr (MT == 1) {
    if (p.M <= 8) {
      hipLaunchKernelGGL((k_gemm_kslice<NORM, EPI, MT, NT, NW, NS, true>), dim3(uint32_t(wgs)), dim3(64 * NW), 0, st, p.A, p.W,
                         p.gain, p.C, p.lda, p.M, p.N, p.K, p.ldc, p.eps);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((k_gemm_kslice<NORM, EPI, MT, NT, NW, NS, false>), dim3(uint32_t(wgs)), dim3(64 * NW), 0, st, p.A, p.W,
                     p.gain, p.C, p.lda, p.M, p.N, p.K, p.ldc, p.eps);
  return hipGetLastError();
}

template <bool NORM, int EPI>
hipError_t launch_kslice(const GemmParams& p, hipStream_t st) {
  if (NORM && p.K > uint32_t(kGemmNormMaxK)) return hipErrorInvalidValue;
  switch (slice_tile(p.M, p.N, p.K)) {
    case 0: return launch_kslice_t<NORM, EPI, 1, 1, 8, 4>(p, st);
    case 1: return launch_kslice_t<NORM, EPI, 1, 2, 8, 2>(p, st);
    case 2: return launch_kslice_t<NORM, EPI, 2, 2, 8, 2>(p, st);
    case 3: return launch_kslice_t<NORM, EPI, 2, 3, 8, 2>(p, st);
    case 4: return launch_kslice_t<NORM, EPI, 2, 4, 8, 2>(p, st);
    case 5: return launch_kslice_t<NORM, EPI, 3, 4, 8, 1>(p, st);
    case 6: return launch_kslice_t<NORM, EPI, 4, 4, 8, 1>(p, st);
    case 7: return launch_kslice_t<NORM, EPI, 1, 8, 4, 2>(p, st);
    case 8: return launch_kslice_t<NORM, EPI, 2, 8, 4, 2>(p, st);
    case 9: return launch_kslice_t<NORM, EPI, 3, 8, 4, 2>(p, st);
    default: return launch_kslice_t<NORM, EPI, 4, 8, 4, 2>(p, st);
  }
}

template <int EPI, bool SPLIT, int BM, int BN, int NS>
hipError_t launch_wide_t(const GemmParams& p, uint32_t splits, const BatchAttnParams& qa, hipStream_t st) {
  const uint64_t wgs = (uint64_t(p.M) + BM - 1) / BM * ((uint64_t(p.N) + BN - 1) / BN) * splits;
  if (hipError_t e = check_grid(wgs, 512)) return e;
  auto* k = p.kz % 64 ? &k_gemm_wide<EPI, SPLIT, BM, BN, NS, true> : &k_gemm_wide<EPI, SPLIT, BM, BN, NS, false>;
  hipLaunchKernelGGL(k, dim3(uint32_t(wgs)), dim3(512), 0, st, p.A, p.W, p.gain, p.C, p.lda, p.M, p.N, p.K, p.ldc, p.kz,
                     qa);
  return hipGetLastError();
}

template <int EPI, bool SPLIT>
hipError_t launch_wide(GemmParams p, uint32_t splits, const BatchAttnParams& qa, hipStream_t st) {
  if (splits == 0 || p.K % splits || p.K / splits % (splits == 1 ? 32 : 64)) return hipErrorInvalidValue;
  p.kz = p.K / splits;
  if constexpr (EPI == kGemmStore) {
    const GemmTile two = wide_pair_tile(p.M, p.N, p.K);
    if (two.bn == 128) return launch_wide_t<EPI, SPLIT, 64, 128, 2>(p, splits, qa, st);
    if (two.bn == 192) return launch_wide_t<EPI, SPLIT, 64, 192, 2>(p, splits, qa, st);
  }
  const GemmTile t = wide_tile(p.M, p.N, p.kz, splits, EPI == kGemmQkRope);
  if (t.bm == 64 && t.bn == 128) return launch_wide_t<EPI, SPLIT, 64, 128, 4>(p, splits, qa, st);
  if (t.bm == 128 && t.bn == 128) return launch_wide_t<EPI, SPLIT, 128, 128, 3>(p, splits, qa, st);
  if (t.bm == 128 && t.bn == 256) return launch_wide_t<EPI, SPLIT, 128, 256, 2>(p, splits, qa, st);
  if constexpr (EPI != kGemmQkRope) {  // (whole heads)
    if (t.bm == 64 && t.bn == 192) return launch_wide_t<EPI, SPLIT, 64, 192, 3>(p, splits, qa, st);
    if (t.bm == 128 && t.bn == 192) return launch_wide_t<EPI, SPLIT, 128, 192, 2>(p, splits, qa, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_gemm(const GemmParams& p, bool norm, int epi, hipStream_t st) {
  if (p.M == 0 || p.N == 0 || p.N % 2 || p.K % 32 || p.K == 0 || p.lda % 4 || !p.A || !p.W || !p.C)
    return hipErrorInvalidValue;
  if (norm && !p.gain) return hipErrorInvalidValue;
  if (norm && epi == kGemmStore) return launch_kslice<true, kGemmStore>(p, st);
  if (norm && epi == kGemmSiluPair) return launch_kslice<true, kGemmSiluPair>(p, st);
  if (!norm && epi == kGemmResAdd) return launch_kslice<false, kGemmResAdd>(p, st);
  if (norm || epi != kGemmStore) return hipErrorInvalidValue;
  return gemm_on_wide(p.M, p.N, p.K) ? launch_wide<kGemmStore, false>(p, 1, BatchAttnParams{}, st)
                                     : launch_kslice<false, kGemmStore>(p, st);
}

hipError_t launch_gemm_split(const GemmParams& p, uint32_t splits, hipStream_t st) {
  if (p.M == 0 || p.N == 0 || p.N % 2 || p.lda % 4 || !p.A || !p.W || !p.C) return hipErrorInvalidValue;
  return launch_wide<kGemmPartial, true>(p, splits, BatchAttnParams{}, st);
}

hipError_t launch_gemm_silu_split(const GemmParams& p, hipStream_t st) {
  if (p.M == 0 || p.N == 0 || p.N % 16 || p.lda % 4 || p.ldc % 8 || !p.A || !p.W || !p.C) return hipErrorInvalidValue;
  return launch_wide<kGemmSiluSplit, true>(p, 1, BatchAttnParams{}, st);
}

L2Prefetch gemm_prefetch_target(const uint16_t* W, uint32_t M, uint32_t N, uint32_t K) {
  if (!W) return L2Prefetch{};
  const uint32_t z = gemm_splits(M, N, K), bn = wide_tile(M, N, K / z, z, false).bn, tiles = ceil_div(N, bn);
  // workgroup (j, y, z) runs on XCD (j + tiles (y + row tiles x z)) % 8: j % 8 when tiles is a
  // multiple of 8
  if (tiles % 8) return L2Prefetch{};
  return L2Prefetch{W, N * (K / 8), bn * (K / 8), tiles};
}

uint32_t tile_prefetch_slots(const L2Prefetch* pf, int n) {
  uint64_t tot = 0;  // XCD 0 has the most consumers
  for (int i = 0; i < n; i++)
    if (pf[i].w && pf[i].n_cwg) tot += uint64_t(ceil_div(pf[i].n_cwg, 8u)) * pf[i].cw_chunks;
  return uint32_t(std::min<uint64_t>(64, (tot + 4095) / 4096));
}

hipError_t launch_resadd_norm_split(float* x, const float* part, uint32_t splits, uint32_t M, uint32_t N, float eps,
                                    const uint16_t* gain, float* out, hipStream_t st) {
  if (!M || N % 8 || N > 4096 || !x || (splits && !part) || (gain && !out)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_resadd_norm_split, dim3(M), dim3(256), 0, st, x, part, splits, M, N, eps, gain, out);
  return hipGetLastError();
}

hipError_t launch_gemm_qk_rope(const GemmParams& g, const BatchAttnParams& a, hipStream_t st) {
  if (g.M == 0 || g.M != a.M || g.N != (a.n_heads + 2 * a.n_kv) * kHeadDim || !a.q || !a.q_norm || !a.k_norm ||
      !a.rope || !a.k_cache || !a.v_cache || g.lda % 4 || !g.A || !g.W)
    return hipErrorInvalidValue;
  if (uint64_t(a.start) + a.M > a.max_seq) return hipErrorInvalidValue;  // the K/V rows must fit the cache
  return launch_wide<kGemmQkRope, true>(g, 1, a, st);
}

hipError_t launch_qk_rope(const BatchAttnParams& p, hipStream_t st) {
  const uint32_t items = p.M * (p.n_heads + 2 * p.n_kv);
  hipLaunchKernelGGL(k_qk_rope, dim3(ceil_div(items, 4)), dim3(256), 0, st, p);
  return hipGetLastError();
}

// Row blocks per wave of k_attn_causal_bf: two (each LDS fragment feeds twice the MFMAs, each staged
// tile twice the rows) from 1024 rows, whatever the heads (prefill from position 0, two / one block: 700 rows
// 1.00 to 1.02, 1024 0.98 to 1.004, 2048 0.92 to 0.98, over 8 to 32 q heads on 1 to 16 KV heads; 16 over 8, us: 512
// rows 2426 / 2370, 1024 3850 / 3897, 2048 7270 / 7530). After 2048 cached positions two would pay from 512
// rows at 16 q heads (3024 / 3203), not at 8.
uint32_t attn_row_blocks(uint32_t M) { return M >= 1024 ? 2 : 1; }

template <int G, int RB>
hipError_t launch_attn_causal_t(const BatchAttnParams& p, bool rope, dim3 grid, hipStream_t st) {
  auto* k = p.kv_bf16 ? &k_attn_causal_bf<G, true, RB, false> : &k_attn_causal_bf<G, false, RB, false>;
  if constexpr (RB == 1) {
    if (rope) k = p.kv_bf16 ? &k_attn_causal_bf<G, true, RB, true> : &k_attn_causal_bf<G, false, RB, true>;
  }
  hipLaunchKernelGGL(k, grid, dim3(512), 0, st, rope ? p.qkv : p.q, p.k_cache, p.v_cache, p.start, p.M, p.max_seq,
                     p.key_run, p.runs, p.n_heads, p.n_kv, p);
  return hipGetLastError();
}

hipError_t launch_attn_causal(const BatchAttnParams& p, bool rope, uint32_t runs, hipStream_t st) {
  if (rope && (!p.qkv || !p.q_norm || !p.k_norm || !p.rope || uint64_t(p.start) + p.M > p.max_seq))
    return hipErrorInvalidValue;
  if (!p.n_kv || p.n_heads % p.n_kv || runs == 0 || runs > uint32_t(kBatchMaxRuns) || (runs > 1 && !p.part))
    return hipErrorInvalidValue;
  const uint32_t G = p.n_heads / p.n_kv;
  BatchAttnParams q = p;
  // runs of whole 64-position tiles covering positions 0 .. start + M - 1, none of them empty
  const uint32_t tiles = ceil_div(p.start + p.M, 64), per_run = ceil_div(tiles, runs);
  runs = ceil_div(tiles, per_run);
  q.key_run = 64 * per_run;
  q.runs = runs;
  if (q.pf.slots > 64) return hipErrorInvalidValue;
  const uint32_t RB = rope ? 1 : attn_row_blocks(p.M);
  const uint32_t gy = ceil_div(p.M, 64 * RB / G);
  // prefetch workgroups: whole planes after the runs' (8 x slots of them at consecutive ids)
  const uint32_t planes = q.pf.slots ? ceil_div(8 * q.pf.slots, p.n_kv * gy) : 0;
  const dim3 grid(p.n_kv, gy, runs + planes);
  hipError_t e = hipErrorInvalidValue;
  if (G == 1) e = RB == 2 ? launch_attn_causal_t<1, 2>(q, rope, grid, st) : launch_attn_causal_t<1, 1>(q, rope, grid, st);
  if (G == 2) e = RB == 2 ? launch_attn_causal_t<2, 2>(q, rope, grid, st) : launch_attn_causal_t<2, 1>(q, rope, grid, st);
  if (G == 4) e = RB == 2 ? launch_attn_causal_t<4, 2>(q, rope, grid, st) : launch_attn_causal_t<4, 1>(q, rope, grid, st);
  if (G == 8) e = RB == 2 ? launch_attn_causal_t<8, 2>(q, rope, grid, st) : launch_attn_causal_t<8, 1>(q, rope, grid, st);
  if (e != hipSuccess || runs == 1) return e;
  const uint32_t n_vec = p.M * p.n_heads;
  const dim3 mg(ceil_div(n_vec, 8));
  if (runs <= 4) hipLaunchKernelGGL((k_attn_merge_rows<4>), mg, dim3(256), 0, st, p.part, runs, n_vec, p.att, p.att_split);
  else if (runs <= 8) hipLaunchKernelGGL((k_attn_merge_rows<8>), mg, dim3(256), 0, st, p.part, runs, n_vec, p.att, p.att_split);
  else if (runs <= 16) hipLaunchKernelGGL((k_attn_merge_rows<16>), mg, dim3(256), 0, st, p.part, runs, n_vec, p.att, p.att_split);
  else hipLaunchKernelGGL((k_attn_merge_rows<32>), mg, dim3(256), 0, st, p.part, runs, n_vec, p.att, p.att_split);
  return hipGetLastError();
}

uint32_t attn_causal_runs(uint32_t M, uint32_t start, uint32_t n_heads, uint32_t n_kv) {
  if (!M || !n_kv || n_heads % n_kv || n_heads / n_kv > 16) return 1;
  // what fits one workgroup per CU (two f32 tiles are 140 KB of LDS): a second round or more partials
  // cost more than longer runs (2048 tokens in chunks of 512: 1, 2 and 4 runs 9.68, 9.29, 10.46 ms; in
  // one chunk of 2048: 1 and 2 runs 7.62, 8.09)
  const uint32_t wgs = n_kv * ceil_div(M, 64 * attn_row_blocks(M) / (n_heads / n_kv));
  const uint32_t runs = std::min(std::max(256 / wgs, 1u), uint32_t(kBatchMaxRuns));
  // a short pass is a few workgroups whose time is one tile's latency after the other: runs of one tile
  const uint32_t least = M <= kGemmSliceMaxM ? 64 : 128;
  return std::max(1u, std::min(runs, ceil_div(start + M, least)));
}

hipError_t launch_row_argmax(const float* logits, uint32_t rows, uint32_t V, uint32_t* tokens, ArgCand* cand,
                             hipStream_t st, const uint32_t* err_in, uint32_t* err_out) {
  if (!rows || !V || !cand || rows > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_row_argmax_part, dim3(kArgParts, rows), dim3(256), 0, st, logits, V, ceil_div(V, kArgParts),
                     cand);
  hipLaunchKernelGGL(k_row_argmax_final, dim3(rows), dim3(64), 0, st, cand, logits, V, tokens, err_in, err_out);
  return hipGetLastError();
}

hipError_t launch_embed_rows(const uint16_t* table, const uint32_t* ids, uint32_t M, uint32_t H, float* x,
                             hipStream_t st) {
  hipLaunchKernelGGL(k_embed_rows, dim3(ceil_div(H, 256), M), dim3(256), 0, st, table, ids, M, H, x);
  return hipGetLastError();
}

hipError_t launch_embed_rows(const uint16_t* table, const TokenIds& ids, uint32_t M, uint32_t H, float* x,
                             hipStream_t st) {
  if (M == 0 || M > kIdsByValue) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_embed_rows_v, dim3(ceil_div(H, 256), M), dim3(256), 0, st, table, ids, H, x);
  return hipGetLastError();
}

}  // namespace qe
