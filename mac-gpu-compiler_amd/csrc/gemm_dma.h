// Device code of the GEMMs C = A' W^T on bf16 matrix cores whose operands reach LDS by the wave's
// own direct-to-LDS loads (gfx950: 16 bytes per lane). A is f32 and is split into hi + lo bf16, so
// every product takes two MFMAs against the same W fragment and keeps ~16 mantissa bits of A.
//
// Why through LDS: an MFMA operand wants lane l to hold row l % 16. Loaded from global memory in
// that shape, neighbouring lanes read rows 2 K bytes apart and the address unit takes one lane a
// clock: 38 B/ns per CU on an L2-resident buffer, whatever the number of waves. The same bytes with
// neighbouring lanes on one row read at 70-108 B/ns into registers and 98-125 into LDS.
#pragma once

#include <hip/hip_runtime.h>

#include "batch.h"
#include "device_common.h"

namespace qe {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The GEMMs' arguments, as plain values that are in scalar registers when a wave starts (14 dwords with the
// one that follows): no first load waits for a load of the argument block (with the attention's the
// same way: verify of 5 rows 1325 -> 1270 us, 512-token prefill 2540 -> 2372).
#define QE_GEMM_ARGS                                                                                        \
  const float *A, const uint16_t *W, const uint16_t *gain, float *C, uint32_t lda, uint32_t M, uint32_t N, \
      uint32_t K, uint32_t ldc

// 8 floats -> (hi, lo) bf16x8 with hi = bf16(v), lo = bf16(v - hi), both rounded to nearest
// even by the hardware pair conversion (v_cvt_pk_bf16_f32); hi + lo keeps ~16 mantissa bits
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8& hi, bf16x8& lo) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  u32x4 h, l;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const uint32_t hb = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{v[2 * e], v[2 * e + 1]}), bf16x2));
    const float r0 = v[2 * e] - __uint_as_float(hb << 16), r1 = v[2 * e + 1] - __uint_as_float(hb & 0xFFFF0000u);
    h[e] = hb;
    l[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{r0, r1}), bf16x2));
  }
  hi = __builtin_bit_cast(bf16x8, h);
  lo = __builtin_bit_cast(bf16x8, l);
}

// Split rows: a row of n floats (n a multiple of 8) held as its two bf16 halves in the same n x 4
// bytes, per 8 values the 8 hi then the 8 lo. A producer that writes them saves every reader the
// split, and the halves of 8 consecutive k are the 16-byte pieces an MFMA operand wants.
// store_split2 / 4: elements i, i + 1 (i even) / i .. i + 3 (i a multiple of 4) of the row at `row`.
__device__ __forceinline__ uint32_t split_pair(float a, float b, uint32_t& lo) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
  const float ra = a - __uint_as_float(hi << 16), rb = b - __uint_as_float(hi & 0xFFFF0000u);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{ra, rb}), bf16x2));
  return hi;
}
__device__ __forceinline__ void store_split2(float* row, uint32_t i, float a, float b) {
  uint32_t* o = reinterpret_cast<uint32_t*>(row) + (i >> 3) * 8 + ((i & 7) >> 1);
  uint32_t lo;
  o[0] = split_pair(a, b, lo);
  o[4] = lo;
}
__device__ __forceinline__ void store_split4(float* row, uint32_t i, float a, float b, float c, float d) {
  uint2* o = reinterpret_cast<uint2*>(row) + (i >> 3) * 4 + ((i & 7) >> 2);
  uint2 hi, lo;
  hi.x = split_pair(a, b, lo.x);
  hi.y = split_pair(c, d, lo.y);
  o[0] = hi;
  o[2] = lo;
}

// One direct-to-LDS load of a wave: lane l's 16 bytes at `src` go to LDS byte address lds + 16 l.
// The compiler does not count it: a reader waits with wait_dma first. (No output registers.)
__device__ __forceinline__ void dma16(uint32_t lds, const void* src) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return uint32_t(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)p));
}
template <int N>
__device__ __forceinline__ void wait_dma() {  // all but the wave's last N vector memory operations are done
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds() {  // the wave's LDS reads have returned
  asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
}
// wait until at most `steps` (capped at NS - 1) later steps of X loads each are in flight
template <int X, int NS>
__device__ __forceinline__ void wait_steps(uint32_t steps) {
  if constexpr (NS == 1) {
    wait_dma<0>();
  } else {
    if (steps >= NS - 1) wait_dma<(NS - 1) * X>();
    else wait_steps<X, NS - 1>(steps);
  }
}

// Writes columns n .. n + 3 (n a multiple of 4, N even) of row m < M: one 16-byte store whatever the
// alignment of C and its rows (four dword stores at a stride of 16 bytes: 430 x 2526 x 320 8.9 us, so 7.1;
// 575 x 3230 x 1664 22.8 and 20.3). kGemmSiluPair: columns 2i / 2i + 1 are gate_i / up_i
// (cpu_inference.rs:170); kGemmSiluSplit: the same as a split row (N a multiple of 4).
template <int EPI>
__device__ __forceinline__ void emit4(const GemmParams& p, uint32_t m, uint32_t n, f32x4 v) {
  typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
  if constexpr (EPI == kGemmSiluPair) {
    float* c = p.C + size_t(m) * p.ldc + (n >> 1);
    if (n < p.N) c[0] = v[0] / (1.0f + expf(-v[0])) * v[1];
    if (n + 2 < p.N) c[1] = v[2] / (1.0f + expf(-v[2])) * v[3];
  } else if constexpr (EPI == kGemmSiluSplit) {
    if (n < p.N)
      store_split2(p.C + size_t(m) * p.ldc, n >> 1, v[0] / (1.0f + expf(-v[0])) * v[1],
                   v[2] / (1.0f + expf(-v[2])) * v[3]);
  } else {
    float* c = p.C + size_t(m) * p.ldc + n;
    if (n + 3 < p.N) {
      if constexpr (EPI == kGemmResAdd) v += f32x4(*reinterpret_cast<const f32x4a4*>(c));
      *reinterpret_cast<f32x4a4*>(c) = v;
    } else {
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (n + r < p.N) c[r] = EPI == kGemmResAdd ? c[r] + v[r] : v[r];
    }
  }
}

// ---------------------------------------------------------------------------------------------
// GEMM with K sliced over the waves of a workgroup: tile 16 MT (m) x 16 NT (n), NW waves; wave w
// takes the 64-deep k blocks w, w + NW, ... in 32-deep steps and multiplies the whole tile. Each
// wave fills its own ring of NS step slots in LDS and reads it back as MFMA operands, so every
// fragment is read from LDS once and the waves never wait for each other until their sums meet in
// LDS at the end (in wave order: the result does not depend on scheduling). K may be any multiple
// of 32 (the last block is then one step).
// Step slot: A rows of 128 bytes (32 f32, chunk c of 16 bytes at place c ^ (row & 7)), then W rows
// of 64 bytes (chunk c at place c ^ ((row >> 1) & 3)): the chunks of a fragment read then fall into
// distinct banks.
// The MFMA's first operand is W: lane l of a block holds columns n + 4 (l / 16) + r of row l % 16.
// NORM: A' = A x gain[k], C scaled by s[m] = 1 / sqrt(mean_k A^2 + eps), the squares summed over
// the same slices (s applied after the sum, a reassociation of the reference's f32 product,
// cpu_inference.rs:189-194).
// HALF (M <= 8): rows 8 .. 15 of the A tile are not loaded and have no place in the slot. Their lanes
// multiply what lies there (W), which reaches only the sums of those rows, and those are not written.
// Bound: at these sizes the bytes each CU pulls from L2 (about 50 B/ns with all CUs loading); the
// tile is the one with the fewest on the busiest CU (slice_tile).
// ---------------------------------------------------------------------------------------------
template <bool NORM, int EPI, int MT, int NT, int NW, int NS, bool HALF>
__global__ __launch_bounds__(64 * NW) void k_gemm_kslice(QE_GEMM_ARGS, float eps) {
  const GemmParams p{A, lda, gain, W, M, N, K, C, ldc, eps, 0};
  constexpr int BM = 16 * MT, BN = 16 * NT;
  constexpr int AI = HALF ? 1 : 2 * MT, WI = NT, X = AI + WI;  // loads per step
  static_assert(!HALF || MT == 1, "HALF: rows 8 .. 15 of the only row block are not there");
  constexpr uint32_t ABYTES = AI * 1024, SBYTES = ABYTES + BN * 64;
  constexpr uint32_t RING = NW * NS * SBYTES, SUMS = MT * NT * NW * 1024, TOP = RING > SUMS ? RING : SUMS;
  // the rings, later the sums
  __shared__ __align__(16) uint8_t smem[TOP];
  __shared__ __align__(16) uint16_t gains[NORM ? kGemmNormMaxK : 8];
  __shared__ float squares[NORM ? NW * BM : 1];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t ncol = ceil_div(p.N, uint32_t(BN));
  const uint32_t m0 = blockIdx.x / ncol * BM, n0 = blockIdx.x % ncol * BN;
  const uint32_t kb = ceil_div(p.K, 64u);
  uint32_t nst = uint32_t(wave) < kb ? 2 * ceil_div(kb - wave, uint32_t(NW)) : 0;  // this wave's steps
  if (p.K % 64 && (kb - 1) % NW == uint32_t(wave)) nst--;
  const uint32_t lds0 = lds_address(smem) + wave * NS * SBYTES;
  const uint8_t* const my = smem + wave * NS * SBYTES;
  // sources of this lane (rows past M or N: the last one), advanced with the steps
  const uint8_t *asrc[AI], *wsrc[WI];
#pragma unroll
  for (int i = 0; i < AI; i++) {
    const uint32_t r = 8 * i + (lane >> 3), c = (lane & 7) ^ (r & 7);
    asrc[i] = reinterpret_cast<const uint8_t*>(p.A + size_t(min(m0 + r, p.M - 1)) * p.lda + 64 * wave) + c * 16;
  }
#pragma unroll
  for (int i = 0; i < WI; i++) {
    const uint32_t r = 16 * i + (lane >> 2), c = (lane & 3) ^ ((r >> 1) & 3);
    wsrc[i] = reinterpret_cast<const uint8_t*>(p.W + size_t(min(n0 + r, p.N - 1)) * p.K + 64 * wave) + c * 16;
  }
  // the next step's loads into `slot`: steps come in pairs (the two halves of a 64-deep block)
  auto issue = [&](uint32_t t, uint32_t slot) __attribute__((always_inline)) {
    const uint32_t l = lds0 + slot * SBYTES, adv = t & 1 ? 64 * NW - 32 : 32;
#pragma unroll
    for (int i = 0; i < WI; i++) {
      dma16(l + ABYTES + i * 1024, wsrc[i]);
      wsrc[i] += adv * 2;
    }
#pragma unroll
    for (int i = 0; i < AI; i++) {
      dma16(l + i * 1024, asrc[i]);
      asrc[i] += adv * 4;
    }
  };
  if constexpr (NORM) {  // the gains first: all waves read all of them
    for (uint32_t i = wave; i < ceil_div(p.K, 512u); i += NW)
      dma16(lds_address(gains) + i * 1024, p.gain + min(512 * i + 8 * lane, p.K - 8));
  }
#pragma unroll
  for (int i = 0; i < NS; i++)
    if (uint32_t(i) < nst) issue(i, i);
  if constexpr (NORM) {
    wait_steps<X, NS + 1>(nst);
    __syncthreads();
  }

  f32x4 acc[MT][NT];
  float ss[MT];
#pragma unroll
  for (int i = 0; i < MT; i++) {
    ss[i] = 0.f;
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const uint32_t a0 = li * 128 + ((2 * kg) ^ (li & 7)) * 16, a1 = li * 128 + ((2 * kg + 1) ^ (li & 7)) * 16;
  const uint32_t w0 = ABYTES + li * 64 + ((kg ^ ((li >> 1) & 3)) * 16);
  uint32_t slot = 0;
  for (uint32_t t = 0; t < nst; t++) {
    wait_steps<X, NS>(nst - 1 - t);
    const uint8_t* sp = my + slot * SBYTES;
    f32x4 ra[MT][2];
    bf16x8 w[NT];
    u32x4 g;
#pragma unroll
    for (int i = 0; i < MT; i++) {
      ra[i][0] = *reinterpret_cast<const f32x4*>(sp + a0 + i * 2048);
      ra[i][1] = *reinterpret_cast<const f32x4*>(sp + a1 + i * 2048);
    }
#pragma unroll
    for (int j = 0; j < NT; j++) w[j] = *reinterpret_cast<const bf16x8*>(sp + w0 + j * 1024);
    if constexpr (NORM)
      g = *reinterpret_cast<const u32x4*>(gains + 64 * (wave + NW * (t >> 1)) + 32 * (t & 1) + 8 * kg);
    wait_lds();
    if (t + NS < nst) issue(t + NS, slot);
#pragma unroll
    for (int i = 0; i < MT; i++) {
      float v[8] = {ra[i][0][0], ra[i][0][1], ra[i][0][2], ra[i][0][3],
                    ra[i][1][0], ra[i][1][1], ra[i][1][2], ra[i][1][3]};
      if constexpr (NORM) {
#pragma unroll
        for (int e = 0; e < 8; e++) ss[i] += v[e] * v[e];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          v[2 * e] *= __uint_as_float(g[e] << 16);
          v[2 * e + 1] *= __uint_as_float(g[e] & 0xFFFF0000u);
        }
      }
      bf16x8 hi, lo;
      split8(v, hi, lo);
#pragma unroll
      for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], hi, acc[i][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], lo, acc[i][j], 0, 0, 0);
    }
    slot = slot == NS - 1 ? 0 : slot + 1;
  }

  // the sums meet over the rings (every load into them has landed and been read): block b = i NT + j
  // of wave w at [b][w][lane], finished by wave b % NW
  f32x4* red = reinterpret_cast<f32x4*>(smem);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MT; i++) {
#pragma unroll
    for (int j = 0; j < NT; j++) red[((i * NT + j) * NW + wave) * 64 + lane] = acc[i][j];
    if constexpr (NORM) {
      float q = ss[i];
      q += __shfl_xor(q, 16);
      q += __shfl_xor(q, 32);
      if (kg == 0) squares[wave * BM + 16 * i + li] = q;
    }
  }
  __syncthreads();
#pragma unroll
  for (int b0 = 0; b0 < MT * NT; b0 += NW) {
    const int b = b0 + wave;
    if (b >= MT * NT) break;
    f32x4 s = red[b * NW * 64 + lane];
#pragma unroll
    for (int v = 1; v < NW; v++) s += red[(b * NW + v) * 64 + lane];
    const int row = 16 * (b / NT) + li;
    if constexpr (NORM) {
      float q = 0.f;
#pragma unroll
      for (int v = 0; v < NW; v++) q += squares[v * BM + row];
      s *= 1.0f / sqrtf(q / float(p.K) + p.eps);
    }
    if (m0 + row < p.M) emit4<EPI>(p, m0 + row, n0 + uint32_t(16 * (b % NT) + 4 * kg), s);
  }
}

// ---------------------------------------------------------------------------------------------
// GEMM for many rows: tile BM (m) x BN (n), eight waves as 2 x 2 (a quarter of the tile each) x the two
// 32-deep halves of every 64-deep stage. TAIL: K is an odd number of halves and the last stage has one (its
// upper places are filled with the lower half again, which nothing reads; as a test in every stage of one
// kernel it cost the other shapes 2 to 5%). 2048 x 6144 x 1056: 61 us, 82 k-sliced; 2048 x 6144 x 96 18.7, 31.
// The stages of both operands are loaded straight into a ring of NS LDS slots, NS - 1 ahead, one barrier per
// stage, in whole 128-byte lines
// (with every CU loading, L2 gives a CU 115 B/ns in lines and 70 in halves of them): A rows of 256
// bytes (chunk c of 16 bytes at place (c & 8) | ((c ^ row) & 7)), then W rows of 128 bytes (chunk c at
// place c ^ (row & 7)).
// SPLIT: A rows are split rows, whose lanes read hi and lo where an f32 row's hold their eight
// floats; otherwise A is f32 and split here.
// C = (sum over the even 32-k blocks) + (sum over the odd ones), or the other way round: the two
// waves of a quarter hand each other half of their rows at the end.
// kGemmQkRope: a tile holds whole heads; the columns of a wave are dims d and d + 64 of its head(s).
// Bound: 25 us per 1024 of K at 2048 x 4096 are 1375 TFLOP/s of MFMAs, against 1590 of a large plain
// library product and 2055 of MFMAs alone on random operands (2430 on zeros: the clock gives way to
// power). Two other schedules of the same tiles (the two halves in antiphase; fragments read a stage
// ahead) ran at the same rate per stage and started 0.6 - 1.1 us later.
// ---------------------------------------------------------------------------------------------
template <int EPI, bool SPLIT, int BM, int BN, int NS, bool TAIL>
__global__ __launch_bounds__(512) void k_gemm_wide(QE_GEMM_ARGS, uint32_t kz, BatchAttnParams qa) {
  const GemmParams p{A, lda, gain, W, M, N, K, C, ldc, 0.f, kz};
  constexpr int MT = BM / 32, NT = BN / 32;
  constexpr int AI = BM / 32, WI = BN / 64;  // loads per wave and stage
  static_assert(AI * 32 == BM && WI * 64 == BN && MT % 2 == 0, "tile");
  constexpr uint32_t ABYTES = BM * 256, SBYTES = ABYTES + BN * 128;
  static_assert(uint32_t(BM) * BN * 4 <= NS * SBYTES, "the sums meet over the ring");
  constexpr bool HALF_HEADS = EPI == kGemmQkRope && BN == kHeadDim;  // two waves share a head
  static_assert(EPI != kGemmQkRope || BN == kHeadDim || BN == 2 * kHeadDim, "whole heads");
  __shared__ __align__(16) uint8_t smem[NS * SBYTES];
  __shared__ float squares[HALF_HEADS ? 2 * BM : 1];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, wm = wave & 1, wn = (wave >> 1) & 1;
  const uint32_t ncol = ceil_div(p.N, uint32_t(BN)), tiles = ncol * ceil_div(p.M, uint32_t(BM));
  const uint32_t z = blockIdx.x / tiles, t = blockIdx.x % tiles, m0 = t / ncol * BM, n0 = t % ncol * BN;
  const uint32_t nst = TAIL ? p.kz / 64 + 1 : p.kz / 64, lds0 = lds_address(smem);
  // tile column of fragment j's first column
  auto col = [&](int j) __attribute__((always_inline)) {
    return HALF_HEADS ? 64 * (j / (NT / 2)) + 32 * wn + 16 * (j % (NT / 2)) : 16 * (wn * NT + j);
  };

  const uint8_t *asrc[AI], *wsrc[WI];  // of the next stage to load (rows past M or N: the last one)
#pragma unroll
  for (int i = 0; i < AI; i++) {
    const uint32_t r = 4 * (wave + 8 * i) + (lane >> 4), c = lane & 15, lc = (c & 8) | ((c ^ r) & 7);
    asrc[i] = reinterpret_cast<const uint8_t*>(p.A + size_t(min(m0 + r, p.M - 1)) * p.lda + size_t(z) * p.kz) + lc * 16;
  }
#pragma unroll
  for (int i = 0; i < WI; i++) {
    const uint32_t r = 8 * (wave + 8 * i) + (lane >> 3), lc = (lane & 7) ^ (r & 7);
    wsrc[i] = reinterpret_cast<const uint8_t*>(p.W + size_t(min(n0 + r, p.N - 1)) * p.K + size_t(z) * p.kz) + lc * 16;
  }
  auto issue = [&](uint32_t s, uint32_t slot) __attribute__((always_inline)) {
    const uint32_t l = lds0 + slot * SBYTES;
    if (TAIL && s == nst - 1) {  // lanes of the upper half (lc & 8, lc & 4 above) stay within the row
#pragma unroll
      for (int i = 0; i < AI; i++) asrc[i] -= lane & 8 ? 128 : 0;
#pragma unroll
      for (int i = 0; i < WI; i++) wsrc[i] -= (lane ^ (lane >> 3)) & 4 ? 64 : 0;
    }
#pragma unroll
    for (int i = 0; i < AI; i++) {
      dma16(l + uint32_t(wave + 8 * i) * 1024, asrc[i]);
      asrc[i] += 256;
    }
#pragma unroll
    for (int i = 0; i < WI; i++) {
      dma16(l + ABYTES + uint32_t(wave + 8 * i) * 1024, wsrc[i]);
      wsrc[i] += 128;
    }
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t ar = (16 * wm * MT + li) * 256 + grp * 128;
  const uint32_t a0 = ar + ((2 * kg) ^ (li & 7)) * 16, a1 = ar + ((2 * kg + 1) ^ (li & 7)) * 16;
  const uint32_t w0 = ABYTES + li * 128 + ((4 * grp + kg) ^ (li & 7)) * 16;
#pragma unroll
  for (int i = 0; i < NS - 1; i++)
    if (uint32_t(i) < nst) issue(i, i);
  uint32_t slot = 0;
  for (uint32_t s = 0; s < nst; s++) {
    // this wave's loads of stage s have landed and its reads of the previous stage have returned;
    // after the barrier that holds for all waves
    wait_steps<AI + WI, NS - 1>(nst - 1 - s);
    wait_lds();
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
    if (TAIL && s == nst - 1 && grp) break;  // (the last stage: nothing is left to issue)
    const uint8_t* sp = smem + slot * SBYTES;
    f32x4 x[MT], y[MT];
    bf16x8 w[NT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
      x[i] = *reinterpret_cast<const f32x4*>(sp + a0 + i * 4096);
      y[i] = *reinterpret_cast<const f32x4*>(sp + a1 + i * 4096);
    }
#pragma unroll
    for (int j = 0; j < NT; j++) w[j] = *reinterpret_cast<const bf16x8*>(sp + w0 + col(j) * 128);
    if (s + NS - 1 < nst) issue(s + NS - 1, slot == 0 ? NS - 1 : slot - 1);
#pragma unroll
    for (int i = 0; i < MT; i++) {
      bf16x8 hi, lo;
      if constexpr (SPLIT) {
        hi = __builtin_bit_cast(bf16x8, x[i]);
        lo = __builtin_bit_cast(bf16x8, y[i]);
      } else {
        const float v[8] = {x[i][0], x[i][1], x[i][2], x[i][3], y[i][0], y[i][1], y[i][2], y[i][3]};
        split8(v, hi, lo);
      }
#pragma unroll
      for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], hi, acc[i][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], lo, acc[i][j], 0, 0, 0);
    }
    slot = slot == NS - 1 ? 0 : slot + 1;
  }

  f32x4* red = reinterpret_cast<f32x4*>(smem);
  const int pr = wave & 3;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MT / 2; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) {
      // component-wise: a ternary between vector objects would select their addresses (scratch)
      f32x4 give, keep;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float a = acc[i][j][r], b = acc[i + MT / 2][j][r];
        give[r] = grp ? a : b;
        keep[r] = grp ? b : a;
      }
      red[((grp * 4 + pr) * (MT / 2 * NT) + i * NT + j) * 64 + lane] = give;
      acc[i][j] = keep;
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MT / 2; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] += red[(((1 - grp) * 4 + pr) * (MT / 2 * NT) + i * NT + j) * 64 + lane];
  const uint32_t mrow = 16 * (wm * MT + grp * (MT / 2)) + li;  // tile row of acc[0]
  if constexpr (EPI == kGemmQkRope) {
    // per-head q/k RMSNorm, RoPE and the K/V append (cpu_inference.rs:134-141, 189-215)
    const uint32_t hh = (n0 + (HALF_HEADS ? 0 : wn * kHeadDim)) / kHeadDim;  // head of [q | k | v]
    const bool isq = hh < qa.n_heads, isk = !isq && hh < qa.n_heads + qa.n_kv, isv = !isq && !isk;
    constexpr int NH = NT / 2;
    auto dim = [&](int j) __attribute__((always_inline)) { return (HALF_HEADS ? col(j) : 16 * j) + 4 * kg; };
    float q[MT / 2];
#pragma unroll
    for (int i = 0; i < MT / 2; i++) {
      q[i] = 0.f;
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) q[i] += acc[i][j][r] * acc[i][j][r];
      q[i] += __shfl_xor(q[i], 16);
      q[i] += __shfl_xor(q[i], 32);
      if (HALF_HEADS && kg == 0) squares[wn * BM + mrow + 16 * i] = q[i];
    }
    if constexpr (HALF_HEADS) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < MT / 2; i++) q[i] = squares[mrow + 16 * i] + squares[BM + mrow + 16 * i];
    }
#pragma unroll
    for (int i = 0; i < MT / 2; i++) {
      const uint32_t m = m0 + mrow + 16 * i, pos = qa.start + min(m, p.M - 1);
      if (!isv) {
        const uint16_t* gain = isq ? qa.q_norm : qa.k_norm;
        const float sc = 1.0f / sqrtf(q[i] / float(kHeadDim) + qa.eps);
        const float* rope = qa.rope + size_t(pos) * kHeadDim;  // (cos, sin) of dims 0 .. 63
#pragma unroll
        for (int j = 0; j < NH; j++) {
          const f32x4 c01 = *reinterpret_cast<const f32x4*>(rope + 2 * dim(j));
          const f32x4 c23 = *reinterpret_cast<const f32x4*>(rope + 2 * dim(j) + 4);
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const float cs = r < 2 ? c01[2 * r] : c23[2 * r - 4], sn = r < 2 ? c01[2 * r + 1] : c23[2 * r - 3];
            const float a = acc[i][j][r] * sc * bf16f(gain[dim(j) + r]);
            const float b = acc[i][j + NH][r] * sc * bf16f(gain[dim(j + NH) + r]);
            acc[i][j][r] = a * cs - b * sn;
            acc[i][j + NH][r] = b * cs + a * sn;
          }
        }
      }
      if (m >= p.M || hh >= qa.n_heads + 2 * qa.n_kv) continue;  // (a tile's second head may lie past N)
      const uint32_t kvh = isk ? hh - qa.n_heads : hh - qa.n_heads - qa.n_kv;
      const size_t slot = isq ? (size_t(m) * qa.n_heads + hh) * kHeadDim : (size_t(kvh) * qa.max_seq + pos) * kHeadDim;
      void* out = isq ? qa.q : isk ? qa.k_cache : qa.v_cache;
#pragma unroll
      for (int j = 0; j < NT; j++) {
        if (!isq && qa.kv_bf16) {
          uint16_t* o = static_cast<uint16_t*>(out) + slot + dim(j);
          const uint32_t lo = f32_to_bf16(acc[i][j][0]) | uint32_t(f32_to_bf16(acc[i][j][1])) << 16;
          const uint32_t hi = f32_to_bf16(acc[i][j][2]) | uint32_t(f32_to_bf16(acc[i][j][3])) << 16;
          *reinterpret_cast<uint2*>(o) = make_uint2(lo, hi);
        } else {
          *reinterpret_cast<f32x4*>(static_cast<float*>(out) + slot + dim(j)) = acc[i][j];
        }
      }
    }
  } else {
    GemmParams q = p;
    if (EPI == kGemmPartial) q.C += size_t(z) * p.M * p.ldc;
#pragma unroll
    for (int i = 0; i < MT / 2; i++) {
      const uint32_t m = m0 + mrow + 16 * i;
#pragma unroll
      for (int j = 0; j < NT; j++)
        if (m < p.M) emit4<EPI>(q, m, n0 + uint32_t(col(j) + 4 * kg), acc[i][j]);
    }
  }
}

}  // namespace
}  // namespace qe
