// Fused passes of the spectral neural operator at its matrix-core size: 64
// channels, 128 retained modes (256 real DFT rows), 128 head units, P = n*n
// points with P % 16 == 0.  Other sizes run the general GEMM and elementwise
// kernels (nn.hip).
//
// What bounds it: the activations are (B, 64, P) and every product has a short
// side of 64-320, so one pass over them costs more than its arithmetic.  The
// general path made eleven passes over FP32 (B, 64, P) or (B, 128, P) arrays
// per layer and direction (GEMM result, beta add, bias and GELU, gradient of
// GELU, channel sums, casts); here each product carries its neighbours:
//   lift        rho -> first activations
//   dft         v (64 x P) against the 256 DFT rows, reduction split over
//               grid.x; in the backward also the 64 rows of the layer's input,
//               i.e. the pointwise weight gradient, from the same loads
//   mix         per mode: sum of the dft's partial results, BF16 rounding,
//               128 x 128 channel mixing
//   out         (64 x 256) spectrum against the inverse basis plus the 64 x 64
//               pointwise map (one reduction of 320), then bias, GELU and the
//               BF16 activations - or, backward, GELU' of the layer below,
//               the BF16 gradient and its channel sums
//   head_fwd    64 -> 128, GELU, sums over P: no (B, 128, P) array
//   head_bwd    recomputes the 128 pre-activations, GELU', both products that
//               need them (the second takes the first's accumulators as its
//               operand without leaving registers), channel sums
// BF16 operands, FP32 accumulation (v_mfma_f32_32x32x16_bf16); biases, GELU,
// pre-activations and sums FP32, as in the general path.  Partial sums are
// folded in a fixed order, so results do not depend on scheduling; the order
// does depend on a sample's place in its batch (dft's first step), so the same
// sample at two places differs by FP32 rounding and what BF16 makes of it.
// Batch 64 of 128^2 points, 4 layers, forward + every gradient: 10.77 -> 3.02
// ms; one sample's forward and input gradient 0.89 -> 0.45 ms.
// Per launch at that batch: dft 61 us, with the weight gradient 107, out 185 us,
// backward out 242 us, head forward 157 us, head backward 550 us (134 MB of BF16
// and 268 MB of FP32 activations are 26 and 52 us at the rate of a large copy).
// The vector work of GELU and of the operand conversions bounds them, and the
// head backward with gradients its registers too: 256 VGPRs and 47 spilled (192 B
// of scratch per lane) beside 32 persistent accumulators.
//
// MFMA fragments (32x32x16): lane l holds A row / B column l & 31, reduction
// elements 8 (l >> 5) .. + 7; result column l & 31, rows 8 (r >> 2) +
// 4 (l >> 5) + (r & 3).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.h"
#include "meep_surrogate.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace mt {
namespace {

constexpr int NC = 64;        // channels
constexpr int NK = 256;       // real DFT rows
constexpr int NH = 128;       // head units
constexpr int PT = 128;       // points per tile (32 per wave)
constexpr int LDX = NC + 8;   // LDS row pitch of a [point][channel] tile
constexpr int LDU = NK + 8;   // ... of the [channel][row] spectrum

union Frag {
  uint4 u;
  uint2 h[2];
  uint16_t s[8];
  bf16x8 v;
};

__device__ __forceinline__ uint16_t bf(float f) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f)); }
__device__ __forceinline__ float f32(uint16_t h) { return __uint_as_float((unsigned)h << 16); }
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float x) {
  return 0.5f * (1.f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}
__device__ __forceinline__ f32x16 zero16() {
  f32x16 a;
#pragma unroll
  for (int r = 0; r < 16; ++r) a[r] = 0.f;
  return a;
}
__device__ __forceinline__ uint4 ld16(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ int crow(int r, int hi) { return 8 * (r >> 2) + 4 * hi + (r & 3); }

// Sum of v over the 32 lanes of a half wave, in lane 31 of the half: shifted
// adds within rows of 16 lanes, then lane 15's total into the next row (VALU
// only; as cross-lane LDS permutes the channel sums took a sixth of the pass).
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float half_sum(float v) {
  v = dpp_add<0x111>(v);   // row_shr:1
  v = dpp_add<0x112>(v);
  v = dpp_add<0x114>(v);
  v = dpp_add<0x118>(v);
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xa, 0xf, false));  // row_bcast:15
}

// *p += v in LDS without waiting for the old value.  Each word is only ever
// added to by one lane, so the order of the sum is the program's.
__device__ __forceinline__ void lds_add(float* p, float v) { unsafeAtomicAdd(p, v); }

// X[c][p0 .. p0 + PT) of 64 channel rows (pitch P) -> LDS [point][channel]:
// two rows at a time, so that a pair of channels is one 32-bit LDS write;
// points from P on are zero.
__device__ __forceinline__ void load_points(const uint16_t* X, int P, int p0, uint16_t* sX) {
  uint32_t* s32 = reinterpret_cast<uint32_t*>(sX);
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int idx = threadIdx.x + it * 256, cp = idx & 31, po = idx >> 5;
    Frag a, b;
    a.u = b.u = make_uint4(0, 0, 0, 0);
    if (p0 + po * 8 < P) {
      const uint16_t* x = X + (long long)(2 * cp) * P + p0 + po * 8;
      a.u = ld16(x);
      b.u = ld16(x + P);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) s32[(po * 8 + q) * (LDX / 2) + cp] = a.s[q] | ((uint32_t)b.s[q] << 16);
  }
}

// ---------------------------------------------------------------- lift
// x = [rho, (i+0.5)/n, (j+0.5)/n] in BF16; v = W x + b in BF16.
__global__ __launch_bounds__(256) void lift_kernel(const float* rho, const uint16_t* w, const float* bias,
                                                   uint16_t* x16, uint16_t* v, int n, int P) {
  const int p = blockIdx.x * 256 + threadIdx.x, b = blockIdx.y;
  if (p >= P) return;
  const int i = p / n, j = p - i * n;
  const uint16_t h0 = bf(rho[(long long)b * P + p]), h1 = bf(((float)i + 0.5f) / (float)n),
                 h2 = bf(((float)j + 0.5f) / (float)n);
  uint16_t* x = x16 + (long long)b * 3 * P + p;
  x[0] = h0, x[P] = h1, x[2 * P] = h2;
  const float x0 = f32(h0), x1 = f32(h1), x2 = f32(h2);
  v += (long long)b * NC * P + p;
  for (int c = 0; c < NC; ++c)
    v[(long long)c * P] = bf(f32(w[3 * c]) * x0 + f32(w[3 * c + 1]) * x1 + f32(w[3 * c + 2]) * x2 + bias[c]);
}

// d/d(rho) = sum_c W[c][0] dv[c]
__global__ __launch_bounds__(256) void lift_back_kernel(const uint16_t* dv, const uint16_t* w, float* drho, int P) {
  const int p = blockIdx.x * 256 + threadIdx.x, b = blockIdx.y;
  if (p >= P) return;
  dv += (long long)b * NC * P + p;
  float s = 0.f;
  for (int c = 0; c < NC; ++c) s += f32(w[3 * c]) * f32(dv[(long long)c * P]);
  drho[(long long)b * P + p] = s;
}

// ----------------------------------------------------------------- dft
// part[split][b][row][c] = sum over the split's points of basis[row][p] X[b][c][p]
// (waves 0-3, 64 rows each), and with W the fifth wave's
// wpart[split][b][c'][c] = sum_p X[b][c'][p] Y[b][c][p].
// Every operand is contiguous along the reduction.  64 points (one cache line
// per row) of all rows are staged through LDS per step: eight lanes read one
// line, while a fragment read straight from memory touches 32 lines per
// instruction and was bound by the L1 (64 x 128^2 points: 143 us).  The next
// step's lines are in flight while this one multiplies.  The rows lie 2 P
// bytes apart (32 KiB at n = 128) and the splits a multiple of 4 KiB, so
// walked from the start every workgroup would be on the same L2 channel at a
// time: each starts at its own step and wraps around (143 -> 60 us in all).
template <bool W>
__global__ __launch_bounds__(W ? 320 : 256) void dft_kernel(const uint16_t* X, const uint16_t* basis,
                                                            const uint16_t* Y, float* part, float* wpart, int P,
                                                            int chunk) {
  constexpr int ROWS = NK + NC + (W ? NC : 0), NT = W ? 320 : 256, LD = 64 + 8;
  constexpr int NL = (ROWS * 8 + NT - 1) / NT;   // 16-byte pieces per thread and step
  __shared__ __align__(16) uint16_t sm[ROWS * LD];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
  const int split = blockIdx.x, b = blockIdx.y, B = gridDim.y;
  const int k0 = split * chunk, k1 = min(P, k0 + chunk);
  const int steps = k1 > k0 ? (k1 - k0 + 63) / 64 : 0, first = steps ? (split * 5 + b * 3) % steps : 0;
  const uint16_t* xb = X + (long long)b * NC * P;
  const uint16_t* yb = W ? Y + (long long)b * NC * P : nullptr;
  Frag f[NL];
  auto fetch = [&](int i) {
    const int st = first + i, k = k0 + 64 * (st < steps ? st : st - steps);
#pragma unroll
    for (int q = 0; q < NL; ++q) {
      const int idx = threadIdx.x + q * NT, row = idx >> 3, kk = k + (idx & 7) * 8;
      f[q].u = make_uint4(0, 0, 0, 0);
      if (row < ROWS && kk < k1) {
        const uint16_t* r = row < NK ? basis + (long long)row * P
                                     : (!W || row < NK + NC ? xb + (long long)(row - NK) * P
                                                            : yb + (long long)(row - NK - NC) * P);
        f[q].u = ld16(r + kk);
      }
    }
  };
  // rows of this wave's operands
  const int ra = (!W || wave < 4 ? wave * 64 : NK) + l31, rb = (!W || wave < 4 ? NK : NK + NC) + l31;
  f32x16 acc[2][2] = {{zero16(), zero16()}, {zero16(), zero16()}};
  if (steps) fetch(0);
  for (int i = 0; i < steps; ++i) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NL; ++q) {
      const int idx = threadIdx.x + q * NT;
      if (idx < ROWS * 8) *reinterpret_cast<uint4*>(&sm[(idx >> 3) * LD + (idx & 7) * 8]) = f[q].u;
    }
    __syncthreads();
    if (i + 1 < steps) fetch(i + 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      Frag A0, A1, B0, B1;
      A0.u = ld16(&sm[ra * LD + 16 * q + hi * 8]);
      A1.u = ld16(&sm[(ra + 32) * LD + 16 * q + hi * 8]);
      B0.u = ld16(&sm[rb * LD + 16 * q + hi * 8]);
      B1.u = ld16(&sm[(rb + 32) * LD + 16 * q + hi * 8]);
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A0.v, B0.v, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A0.v, B1.v, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A1.v, B0.v, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A1.v, B1.v, acc[1][1], 0, 0, 0);
    }
  }
  float* o = (!W || wave < 4) ? part + (((long long)split * B + b) * NK + wave * 64) * NC
                              : wpart + ((long long)split * B + b) * NC * NC;
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[(32 * m + crow(r, hi)) * NC + 32 * n + l31] = acc[m][n][r];
}

// ----------------------------------------------------------------- mix
// Mode m, 32 batch rows: in[b][k] = BF16(sum_split part[split][b][2m..2m+1][c])
// (k = 128 values, also stored), out[b][n] = sum_k in[b][k] W[m][n][k] in BF16.
__global__ __launch_bounds__(256) void mix_kernel(const float* part, int splits, const uint16_t* W, uint16_t* in16,
                                                  uint16_t* out16, int B) {
  __shared__ __align__(16) uint16_t sA[32][128 + 8];
  const int m = blockIdx.x, b0 = blockIdx.y * 32;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
  const uint16_t* w = W + ((long long)m * 128 + wave * 32 + l31) * 128 + hi * 8;
  Frag bw[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) bw[q].u = ld16(w + 16 * q);
  const int k = threadIdx.x & 127;
  for (int i = threadIdx.x >> 7; i < 32; i += 2) {
    float s = 0.f;
    if (b0 + i < B) {
      const float* p = part + ((long long)(b0 + i) * NK + 2 * m) * NC + k;
      const long long st = (long long)B * NK * NC;
      int q = 0;
      for (; q + 4 <= splits; q += 4) {   // four loads in flight, added in order
        const float v0 = p[q * st], v1 = p[(q + 1) * st], v2 = p[(q + 2) * st], v3 = p[(q + 3) * st];
        s = (((s + v0) + v1) + v2) + v3;
      }
      for (; q < splits; ++q) s += p[q * st];
      in16[((long long)(b0 + i) * NK + 2 * m) * NC + k] = bf(s);
    }
    sA[i][k] = bf(s);
  }
  __syncthreads();
  f32x16 acc = zero16();
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    Frag a;
    a.u = ld16(&sA[l31][16 * q + hi * 8]);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, bw[q].v, acc, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int b = b0 + crow(r, hi);
    if (b < B) out16[((long long)b * NK + 2 * m) * NC + wave * 32 + l31] = bf(acc[r]);
  }
}

// ----------------------------------------------------------------- out
// Tile of 128 points of batch b: acc[c][p] = sum_k U[b][k][c] basisT[p][k] +
// sum_c' W[c][c'] X[b][c'][p].
//   forward (BACK = false): u = acc + bias -> pre (if given), gelu(u) or u -> y16
//   backward: d = acc * gelu'(pre) or acc -> y16, and part[tile][b][c] = sum_p d
// basisT is stored in fragment order (32-point tile, 16-row step, lane): a
// fragment load is 1 KiB in a row, where rows of (P, 256) touched 32 lines.
template <bool BACK>
__global__ __launch_bounds__(256, 3) void out_kernel(const uint16_t* U, const uint16_t* basisT, const uint16_t* W,
                                                  const uint16_t* X, const float* bias, float* pre, uint16_t* y16,
                                                  float* part, int P, int act, int ntile) {
  __shared__ __align__(16) uint16_t sU[NC * LDU];
  __shared__ __align__(16) uint16_t sX[PT * LDX];
  __shared__ float sS[4][NC];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
  const int tile = blockIdx.x, b = blockIdx.y, p0 = tile * PT, p = p0 + wave * 32 + l31;
  const uint16_t* g = basisT + ((long long)(tile * 4 + wave) * (NK / 16) * 64 + lane) * 8;
  const bool ok = p < P;
  load_points(X + (long long)b * NC * P, P, p0, sX);
  {  // U [k][c] -> LDS [c][k], two rows at a time
    const uint16_t* u = U + (long long)b * NK * NC;
    uint32_t* s32 = reinterpret_cast<uint32_t*>(sU);
    const int kp = threadIdx.x & 127;
#pragma unroll
    for (int cq = threadIdx.x >> 7; cq < 8; cq += 2) {
      Frag a, c;
      a.u = ld16(u + (2 * kp) * NC + cq * 8);
      c.u = ld16(u + (2 * kp + 1) * NC + cq * 8);
#pragma unroll
      for (int q = 0; q < 8; ++q) s32[(cq * 8 + q) * (LDU / 2) + kp] = a.s[q] | ((uint32_t)c.s[q] << 16);
    }
  }
  // the epilogue's operands, loaded before the products
  const long long base = (long long)b * NC * P + min(p, P - 1);
  float ep[2][16];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int c = 32 * t + crow(r, hi);
      ep[t][r] = BACK ? (act ? pre[base + (long long)c * P] : 0.f) : bias[c];
    }
  __syncthreads();
  f32x16 acc[2] = {zero16(), zero16()};
#pragma unroll 8
  for (int q = 0; q < NK / 16; ++q) {
    Frag bb, a0, a1;
    bb.u = ld16(g + q * 512);
    a0.u = ld16(&sU[l31 * LDU + 16 * q + hi * 8]);
    a1.u = ld16(&sU[(32 + l31) * LDU + 16 * q + hi * 8]);
    acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0.v, bb.v, acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1.v, bb.v, acc[1], 0, 0, 0);
  }
#pragma unroll
  for (int kk = 0; kk < NC; kk += 16) {
    Frag bb, a0, a1;
    bb.u = ld16(&sX[(wave * 32 + l31) * LDX + kk + hi * 8]);
    a0.u = ld16(W + l31 * NC + kk + hi * 8);
    a1.u = ld16(W + (32 + l31) * NC + kk + hi * 8);
    acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0.v, bb.v, acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1.v, bb.v, acc[1], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    if constexpr (BACK) {
      float d[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) d[r] = ok ? acc[t][r] : 0.f;
      if (act) {
#pragma unroll
        for (int r = 0; r < 16; ++r) d[r] *= gelu_d(ep[t][r]);
      }
      if (ok) {
#pragma unroll
        for (int r = 0; r < 16; ++r) y16[base + (long long)(32 * t + crow(r, hi)) * P] = bf(d[r]);
      }
      if (part) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float s = half_sum(d[r]);
          if (l31 == 31) sS[wave][32 * t + crow(r, hi)] = s;
        }
      }
    } else if (ok) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const long long o = base + (long long)(32 * t + crow(r, hi)) * P;
        const float u = acc[t][r] + ep[t][r];
        if (pre) pre[o] = u;
        y16[o] = bf(act ? gelu(u) : u);
      }
    }
  }
  if (BACK && part) {
    __syncthreads();
    if (threadIdx.x < NC)
      part[((long long)b * ntile + tile) * NC + threadIdx.x] =
          ((sS[0][threadIdx.x] + sS[1][threadIdx.x]) + sS[2][threadIdx.x]) + sS[3][threadIdx.x];
  }
}

// ---------------------------------------------------------------- head
// part[b][chunk][h] = sum over the chunk's points of gelu(Wq v + bq)
__global__ __launch_bounds__(256) void head_fwd_kernel(const uint16_t* V, const uint16_t* Wq, const float* bq,
                                                       float* part, int P, int ntile, int tiles) {
  __shared__ __align__(16) uint16_t sX[PT * LDX];
  __shared__ float sB[NH], sS[4][NH];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
  const int b = blockIdx.y, t0 = blockIdx.x * tiles, t1 = min(ntile, t0 + tiles);
  if (threadIdx.x < NH) sB[threadIdx.x] = bq[threadIdx.x];
  float s[4][16];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[t][r] = 0.f;
  for (int tile = t0; tile < t1; ++tile) {
    __syncthreads();
    load_points(V + (long long)b * NC * P, P, tile * PT, sX);
    __syncthreads();
    const bool ok = tile * PT + wave * 32 + l31 < P;
    Frag bb[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) bb[q].u = ld16(&sX[(wave * 32 + l31) * LDX + 16 * q + hi * 8]);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x16 acc = zero16();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        Frag a;
        a.u = ld16(Wq + (32 * t + l31) * NC + 16 * q + hi * 8);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, bb[q].v, acc, 0, 0, 0);
      }
      if (ok) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[t][r] += gelu(acc[r] + sB[32 * t + crow(r, hi)]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float v = half_sum(s[t][r]);
      if (l31 == 31) sS[wave][32 * t + crow(r, hi)] = v;
    }
  __syncthreads();
  if (threadIdx.x < NH)
    part[((long long)b * gridDim.x + blockIdx.x) * NH + threadIdx.x] =
        ((sS[0][threadIdx.x] + sS[1][threadIdx.x]) + sS[2][threadIdx.x]) + sS[3][threadIdx.x];
}

// hm = mean over P in BF16, out = Wo hm + bo
__global__ __launch_bounds__(NH) void head_out_kernel(const float* part, int chunks, const uint16_t* Wo,
                                                      const float* bo, uint16_t* hm16, float* out, int n_out,
                                                      float scale) {
  __shared__ float sh[NH];
  const int b = blockIdx.x, h = threadIdx.x;
  float s = 0.f;
#pragma unroll 16
  for (int q = 0; q < chunks; ++q) s += part[((long long)b * chunks + q) * NH + h];
  const uint16_t m = bf(s * scale);
  hm16[b * NH + h] = m;
  sh[h] = f32(m);
  __syncthreads();
  for (int n = threadIdx.x; n < n_out; n += NH) {
    float v = 0.f;
    for (int q = 0; q < NH; ++q) v += sh[q] * f32(Wo[n * NH + q]);
    out[(long long)b * n_out + n] = v + bo[n];
  }
}

// Blocks 0 .. n_out-1 (with grads): row n of dWo = dout16^T hm16 and dbo;
// the rest: dhm[b] = dout16[b] Wo.
__global__ __launch_bounds__(NH) void head_grad_kernel(const float* dout, const uint16_t* Wo, const uint16_t* hm16,
                                                       float* dWo, float* dbo, float* dhm, int B, int n_out) {
  const int h = threadIdx.x;
  int blk = blockIdx.x;
  if (dWo) {
    if (blk < n_out) {
      float s = 0.f, sb = 0.f;
      for (int b = 0; b < B; ++b) {
        const float d = dout[(long long)b * n_out + blk];
        s += f32(bf(d)) * f32(hm16[b * NH + h]);
        sb += d;
      }
      dWo[blk * NH + h] = s;
      if (h == 0) dbo[blk] = sb;
      return;
    }
    blk -= n_out;
  }
  float s = 0.f;
  for (int n = 0; n < n_out; ++n) s += f32(bf(dout[(long long)blk * n_out + n])) * f32(Wo[n * NH + h]);
  dhm[blk * NH + h] = s;
}

// Backward of the head over the tiles of one chunk of batch b: recompute
// h = Wq v + bq, dq = dhm / P * gelu'(h); dv = Wq^T dq in BF16; with G the
// chunk's sums of dq (bq), dv (bias of the last layer) and dq v^T (Wq).
// dq leaves the first product with point = lane and eight consecutive units
// per lane pair of register groups, which is a B operand of the second product
// for the unit order 8 (g + (i >> 2)) + 4 hi + (i & 3): Wq^T is loaded in that
// order, and dq needs no transpose.
template <bool G>
__global__ __launch_bounds__(256, 2) void head_bwd_kernel(const uint16_t* V, const uint16_t* Wq, const uint16_t* WqT,
                                                       const float* bq, const float* dhm, uint16_t* dv16,
                                                       float* qbpart, float* vbpart, float* qwpart, int P, int ntile,
                                                       int tiles, float scale) {
  constexpr int LDD = PT + 8;
  __shared__ __align__(16) uint16_t sX[PT * LDX];
  __shared__ __align__(16) uint16_t sD[G ? NH * LDD : 8];
  __shared__ float sB[NH], sG[NH], sS[4][NH + NC];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
  const int b = blockIdx.y, t0 = blockIdx.x * tiles, t1 = min(ntile, t0 + tiles);
  const uint16_t* v = V + (long long)b * NC * P;
  if (threadIdx.x < NH) {
    sB[threadIdx.x] = bq[threadIdx.x];
    sG[threadIdx.x] = dhm[b * NH + threadIdx.x] * scale;
  }
  f32x16 gw[2] = {zero16(), zero16()};
  if constexpr (G)   // per-wave sums of dq and dv over the chunk, one tile's total at a time
    for (int x = threadIdx.x; x < 4 * (NH + NC); x += 256) sS[x / (NH + NC)][x % (NH + NC)] = 0.f;
  for (int tile = t0; tile < t1; ++tile) {
    const int p0 = tile * PT, p = p0 + wave * 32 + l31;
    const bool ok = p < P;
    __syncthreads();
    load_points(v, P, p0, sX);
    __syncthreads();
    Frag bb[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) bb[q].u = ld16(&sX[(wave * 32 + l31) * LDX + 16 * q + hi * 8]);
    f32x16 dv[2] = {zero16(), zero16()};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x16 acc = zero16();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        Frag a;
        a.u = ld16(Wq + (32 * t + l31) * NC + 16 * q + hi * 8);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, bb[q].v, acc, 0, 0, 0);
      }
      Frag d[2];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int h = 32 * t + crow(r, hi);
        const float x = ok ? sG[h] * gelu_d(acc[r] + sB[h]) : 0.f;
        if constexpr (G) {
          const float tot = half_sum(x);
          if (l31 == 31) lds_add(&sS[wave][h], tot);
        }
        d[r >> 3].s[r & 7] = bf(x);
        if constexpr (G) sD[h * LDD + wave * 32 + l31] = d[r >> 3].s[r & 7];
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {   // units 32 t + 16 j ..
        const uint16_t* w0 = WqT + l31 * NH + 32 * t + 16 * j + 4 * hi;
        Frag a0, a1;
        a0.h[0] = *reinterpret_cast<const uint2*>(w0);
        a0.h[1] = *reinterpret_cast<const uint2*>(w0 + 8);
        a1.h[0] = *reinterpret_cast<const uint2*>(w0 + 32 * NH);
        a1.h[1] = *reinterpret_cast<const uint2*>(w0 + 32 * NH + 8);
        dv[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0.v, d[j].v, dv[0], 0, 0, 0);
        dv[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1.v, d[j].v, dv[1], 0, 0, 0);
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int c = 32 * t + crow(r, hi);
        if (ok) dv16[(long long)b * NC * P + (long long)c * P + p] = bf(dv[t][r]);
        if constexpr (G) {   // zero past P
          const float tot = half_sum(dv[t][r]);
          if (l31 == 31) lds_add(&sS[wave][NH + c], tot);
        }
      }
    if constexpr (G) {
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 8; ++q) {   // units 32 wave .. x channels, over the tile's points
        Frag a, b0, b1;
        a.u = ld16(&sD[(32 * wave + l31) * LDD + 16 * q + hi * 8]);
        b0.u = b1.u = make_uint4(0, 0, 0, 0);
        const int pp = p0 + 16 * q + hi * 8;
        if (pp < P) {
          b0.u = ld16(v + (long long)l31 * P + pp);
          b1.u = ld16(v + (long long)(32 + l31) * P + pp);
        }
        gw[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b0.v, gw[0], 0, 0, 0);
        gw[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b1.v, gw[1], 0, 0, 0);
      }
    }
  }
  if constexpr (G) {
    const long long blk = (long long)b * gridDim.x + blockIdx.x;
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        qwpart[blk * NH * NC + (32 * wave + crow(r, hi)) * NC + 32 * n + l31] = gw[n][r];
    __syncthreads();
    const int x = threadIdx.x;
    if (x < NH + NC) {
      const float v4 = ((sS[0][x] + sS[1][x]) + sS[2][x]) + sS[3][x];
      if (x < NH) qbpart[blk * NH + x] = v4;
      else vbpart[blk * NC + x - NH] = v4;
    }
  }
}

// ---------------------------------------------------------------- folds
// Column sums of part (rows `stride` rows apart): a block sums 64 columns of
// a slab of `rows` rows, dealt to four groups of threads whose sums are added
// in group order.  With several slabs each writes its sum to its own first
// row, and a second launch adds those.
constexpr int kSlab = 128;
__global__ __launch_bounds__(256) void fold_kernel(float* part, int Q, int n, int stride, int rows,
                                                   float* out) {
  __shared__ float s[4][64];
  const int i = blockIdx.x * 64 + (threadIdx.x & 63), g = threadIdx.x >> 6;
  const int q0 = blockIdx.y * rows, q1 = min(Q, q0 + rows);
  float v = 0.f;
  if (i < n) {
    const float* p = part + i;
    const long long st = (long long)stride * n;
    int q = q0 + g;
    for (; q + 28 < q1; q += 32) {   // eight loads in flight, added in order
      float t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) t[u] = p[(q + 4 * u) * st];
#pragma unroll
      for (int u = 0; u < 8; ++u) v += t[u];
    }
    for (; q < q1; q += 4) v += p[q * st];
  }
  s[g][threadIdx.x & 63] = v;
  __syncthreads();
  if (g == 0 && i < n) {
    const int x = threadIdx.x;
    const float t = ((s[0][x] + s[1][x]) + s[2][x]) + s[3][x];
    if (out) out[i] = t;
    else part[(long long)q0 * n + i] = t;
  }
}

// BF16 copies of the packed spectral weights (mt_pack_spectral), plain and
// transposed per mode: the mixing kernel reads weight rows along its
// reduction, forward from the transpose, backward from the plain form.  The
// weights lie along the modes, the copies along the channels: a block takes 32
// modes of one input channel (blockIdx.z 0: two rows of every plain block) or
// one output channel (1: two rows of the transposes) through LDS, so that both
// sides are read and written in lines.  64 channels, 128 modes, per layer:
// 17.8 us element by element, 9.5 this way (the plain copy alone 9.8); two
// channels per store are no faster.
__global__ __launch_bounds__(256) void pack_both_kernel(const float* wre, const float* wim, uint16_t* wp,
                                                        uint16_t* wt, int C, int Mo) {
  constexpr int TM = 32, TA = 64;
  __shared__ float re[TA][TM + 1], im[TA][TM + 1];
  const int ch = blockIdx.x, m0 = blockIdx.y * TM;
  const bool t = blockIdx.z;
  uint16_t* out = t ? wt : wp;
  for (int a0 = 0; a0 < C; a0 += TA) {
    const int na = min(TA, C - a0), nm = min(TM, Mo - m0);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < TA * TM / 256; ++it) {
      const int x = threadIdx.x + it * 256, a = x / TM, m = x % TM;
      if (a < na && m < nm) {
        const long long w = ((long long)(t ? a0 + a : ch) * C + (t ? ch : a0 + a)) * Mo + m0 + m;
        re[a][m] = wre[w];
        im[a][m] = wim[w];
      }
    }
    __syncthreads();
    // rows r * C + ch, columns h * C + a: real where r == h, else +-imaginary
    const int a = threadIdx.x % TA, h = threadIdx.x / TA & 1, r = threadIdx.x / (2 * TA);
    const bool neg = t ? h > r : r > h;
    if (a < na)
      for (int m = 0; m < nm; ++m) {
        const float v = r == h ? re[a][m] : neg ? -im[a][m] : im[a][m];
        out[((long long)(m0 + m) * 2 * C + r * C + ch) * 2 * C + h * C + a0 + a] = bf(v);
      }
  }
}

// y = BF16 of x (R, C) where given, and yt its transpose
__global__ void cast_transpose_kernel(const float* x, uint16_t* y, uint16_t* yt, int R, int C) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= R * C) return;
  const uint16_t v = bf(x[e]);
  if (y) y[e] = v;
  yt[(e % C) * R + e / C] = v;
}

bool al16(const void* p) { return p && (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int shape_ok(int B, int P) {
  if (B < 1 || P < 16 || P % 16) return fail(MT_EINVAL, "fno: needs B >= 1 and P a multiple of 16");
  if (B > 65535) return fail(MT_EINVAL, "fno: batch too large");
  return MT_OK;
}

}  // namespace
}  // namespace mt

using namespace mt;

#define U16(p) static_cast<const uint16_t*>(p)
#define M16(p) static_cast<uint16_t*>(p)

extern "C" int mt_fno_lift(const float* rho, const void* w, const float* bias, void* x16, void* v16, int B, int n,
                           void* stream) {
  const int P = n * n;
  int rc = shape_ok(B, P);
  if (rc) return rc;
  if (!rho || !w || !bias || !x16 || !v16) return fail(MT_EINVAL, "fno_lift: null pointer");
  hipLaunchKernelGGL(lift_kernel, dim3((P + 255) / 256, B), dim3(256), 0, static_cast<hipStream_t>(stream), rho,
                     U16(w), bias, M16(x16), M16(v16), n, P);
  return check_launch("fno_lift");
}

extern "C" int mt_fno_lift_back(const void* dv16, const void* w, float* drho, int B, int P, void* stream) {
  int rc = shape_ok(B, P);
  if (rc) return rc;
  if (!dv16 || !w || !drho) return fail(MT_EINVAL, "fno_lift_back: null pointer");
  hipLaunchKernelGGL(lift_back_kernel, dim3((P + 255) / 256, B), dim3(256), 0, static_cast<hipStream_t>(stream),
                     U16(dv16), U16(w), drho, P);
  return check_launch("fno_lift_back");
}

extern "C" int mt_fno_dft(const void* x16, const void* basis, const void* y16, float* part, float* wpart, int B,
                          int P, int splits, void* stream) {
  int rc = shape_ok(B, P);
  if (rc) return rc;
  if (!al16(x16) || !al16(basis) || (y16 && (!al16(y16) || !wpart)) || !part || splits < 1)
    return fail(MT_EINVAL, "fno_dft: bad arguments");
  const int chunk = ((P / 16 + splits - 1) / splits) * 16;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (y16)
    hipLaunchKernelGGL(dft_kernel<true>, dim3(splits, B), dim3(320), 0, s, U16(x16), U16(basis), U16(y16), part,
                       wpart, P, chunk);
  else
    hipLaunchKernelGGL(dft_kernel<false>, dim3(splits, B), dim3(256), 0, s, U16(x16), U16(basis), U16(y16), part,
                       wpart, P, chunk);
  return check_launch("fno_dft");
}

extern "C" int mt_fno_mix(const float* part, int splits, const void* w, void* in16, void* out16, int B, int Mo,
                          void* stream) {
  if (!part || splits < 1 || !al16(w) || !in16 || !out16 || B < 1 || Mo != NK / 2)
    return fail(MT_EINVAL, "fno_mix: bad arguments");
  hipLaunchKernelGGL(mix_kernel, dim3(Mo, (B + 31) / 32), dim3(256), 0, static_cast<hipStream_t>(stream), part,
                     splits, U16(w), M16(in16), M16(out16), B);
  return check_launch("fno_mix");
}

extern "C" int mt_fno_out(const void* u16, const void* basis_t, const void* w, const void* x16, const float* bias,
                          float* pre, void* y16, int B, int P, int act, void* stream) {
  int rc = shape_ok(B, P);
  if (rc) return rc;
  if (!al16(u16) || !al16(basis_t) || !al16(w) || !al16(x16) || !bias || !y16)
    return fail(MT_EINVAL, "fno_out: bad arguments");
  const int nt = (P + PT - 1) / PT;
  hipLaunchKernelGGL(out_kernel<false>, dim3(nt, B), dim3(256), 0, static_cast<hipStream_t>(stream), U16(u16),
                     U16(basis_t), U16(w), U16(x16), bias, pre, M16(y16), (float*)nullptr, P, act, nt);
  return check_launch("fno_out");
}

extern "C" int mt_fno_out_back(const void* u16, const void* basis_t, const void* w, const void* x16,
                               const float* pre, void* y16, float* part, int B, int P, int act, void* stream) {
  int rc = shape_ok(B, P);
  if (rc) return rc;
  if (!al16(u16) || !al16(basis_t) || !al16(w) || !al16(x16) || !y16 || (act && !pre))
    return fail(MT_EINVAL, "fno_out_back: bad arguments");
  const int nt = (P + PT - 1) / PT;
  hipLaunchKernelGGL(out_kernel<true>, dim3(nt, B), dim3(256), 0, static_cast<hipStream_t>(stream), U16(u16),
                     U16(basis_t), U16(w), U16(x16), (const float*)nullptr, const_cast<float*>(pre), M16(y16), part,
                     P, act, nt);
  return check_launch("fno_out_back");
}

extern "C" int mt_fno_head(const void* v16, const void* wq, const float* bq, const void* wo, const float* bo,
                           float* part, int chunks, void* hm16, float* out, int B, int P, int n_out, void* stream) {
  int rc = shape_ok(B, P);
  if (rc) return rc;
  if (!al16(v16) || !al16(wq) || !bq || !wo || !bo || !part || chunks < 1 || !hm16 || !out || n_out < 1)
    return fail(MT_EINVAL, "fno_head: bad arguments");
  const int nt = (P + PT - 1) / PT, tiles = (nt + chunks - 1) / chunks;
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(head_fwd_kernel, dim3(chunks, B), dim3(256), 0, s, U16(v16), U16(wq), bq, part, P, nt, tiles);
  hipLaunchKernelGGL(head_out_kernel, dim3(B), dim3(NH), 0, s, part, chunks, U16(wo), bo, M16(hm16), out, n_out,
                     1.0f / (float)P);
  return check_launch("fno_head");
}

extern "C" int mt_fno_head_back(const float* dout, const void* v16, const void* wq, const void* wq_t,
                                const float* bq, const void* wo, const void* hm16, float* dwo, float* dbo,
                                float* dhm, void* dv16, float* qbpart, float* vbpart, float* qwpart, int chunks,
                                int B, int P, int n_out, void* stream) {
  int rc = shape_ok(B, P);
  if (rc) return rc;
  const bool grads = dwo != nullptr;
  if (!dout || !al16(v16) || !al16(wq) || !al16(wq_t) || !bq || !wo || !hm16 || !dhm || !dv16 || chunks < 1 ||
      n_out < 1 || (grads && (!dbo || !qbpart || !vbpart || !qwpart)))
    return fail(MT_EINVAL, "fno_head_back: bad arguments");
  const int nt = (P + PT - 1) / PT, tiles = (nt + chunks - 1) / chunks;
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(head_grad_kernel, dim3((grads ? n_out : 0) + B), dim3(NH), 0, s, dout, U16(wo), U16(hm16), dwo,
                     dbo, dhm, B, n_out);
  if (grads)
    hipLaunchKernelGGL(head_bwd_kernel<true>, dim3(chunks, B), dim3(256), 0, s, U16(v16), U16(wq), U16(wq_t), bq, dhm,
                       M16(dv16), qbpart, vbpart, qwpart, P, nt, tiles, 1.0f / (float)P);
  else
    hipLaunchKernelGGL(head_bwd_kernel<false>, dim3(chunks, B), dim3(256), 0, s, U16(v16), U16(wq), U16(wq_t), bq,
                       dhm, M16(dv16), qbpart, vbpart, qwpart, P, nt, tiles, 1.0f / (float)P);
  return check_launch("fno_head_back");
}

extern "C" int mt_fno_fold(float* part, int Q, int n, float* out, void* stream) {
  if (!part || !out || Q < 1 || n < 1) return fail(MT_EINVAL, "fno_fold: bad arguments");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned cols = (unsigned)((n + 63) / 64);
  int stride = 1;
  if (Q > kSlab) {
    const int slabs = (Q + kSlab - 1) / kSlab;
    if (slabs > 65535) return fail(MT_EINVAL, "fno_fold: too many rows");
    hipLaunchKernelGGL(fold_kernel, dim3(cols, slabs), dim3(256), 0, s, part, Q, n, 1, kSlab, (float*)nullptr);
    Q = slabs;
    stride = kSlab;
  }
  hipLaunchKernelGGL(fold_kernel, dim3(cols), dim3(256), 0, s, part, Q, n, stride, Q, out);
  return check_launch("fno_fold");
}

extern "C" int mt_fno_pack(const float* wre, const float* wim, void* wp, void* wp_t, int C, int Mo, void* stream) {
  if (!wre || !wim || !wp || !wp_t || C < 1 || Mo < 1) return fail(MT_EINVAL, "fno_pack: bad arguments");
  if ((Mo + 31) / 32 > 65535) return fail(MT_EINVAL, "fno_pack: too many modes");
  hipLaunchKernelGGL(pack_both_kernel, dim3(C, (Mo + 31) / 32, 2), dim3(256), 0, static_cast<hipStream_t>(stream), wre,
                     wim, M16(wp), M16(wp_t), C, Mo);
  return check_launch("fno_pack");
}

extern "C" int mt_cast_transpose_bf16(const float* x, void* y, void* y_t, int R, int C, void* stream) {
  if (!x || !y_t || R < 1 || C < 1) return fail(MT_EINVAL, "cast_transpose_bf16: bad arguments");
  hipLaunchKernelGGL(cast_transpose_kernel, dim3((R * C + 255) / 256), dim3(256), 0,
                     static_cast<hipStream_t>(stream), x, M16(y), M16(y_t), R, C);
  return check_launch("cast_transpose_bf16");
}

extern "C" int mt_transpose_bf16(const float* x, void* y, int R, int C, void* stream) {
  if (!y) return fail(MT_EINVAL, "transpose_bf16: bad arguments");
  return mt_cast_transpose_bf16(x, nullptr, y, R, C, stream);
}
