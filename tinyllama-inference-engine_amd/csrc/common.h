// Shared device helpers for the gfx950 kernels: storage types, wave64 and block reductions.
//
// Storage is float or bfloat16; arithmetic that the engine promises in 32-bit (softmax, norms,
// rotation angles, the residual sum) is done on floats obtained with to_float().
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

namespace tlie {

constexpr int kWave = 64;

// dtype codes of the C interface
constexpr int kF32 = 0;
constexpr int kBF16 = 1;

typedef __hip_bfloat16 bf16;

__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(bf16 v) { return __bfloat162float(v); }

template <typename T> __device__ __forceinline__ T from_float(float v);
template <> __device__ __forceinline__ float from_float<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 from_float<bf16>(float v) { return __float2bfloat16(v); }

// bfloat16 bits <-> float without going through the class type (for packed 16-byte loads)
__device__ __forceinline__ float bf16_bits_to_float(uint16_t bits) {
  return __uint_as_float(static_cast<uint32_t>(bits) << 16);
}
__device__ __forceinline__ float bf16_lo(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t pair) { return __uint_as_float(pair & 0xffff0000u); }

// two floats to two bfloat16 (round to nearest even) in one instruction, v_cvt_pk_bf16_f32
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float floatx2;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const bf16x2 r = __builtin_convertvector((floatx2{lo, hi}), bf16x2);
  return *reinterpret_cast<const uint32_t*>(&r);
}

// Eight consecutive elements (the address a multiple of 16 bytes for bfloat16, of 32 for float) as floats.
__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
  const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void load8(const bf16* p, float (&v)[8]) {
  const uint4 u = *reinterpret_cast<const uint4*>(p);
  v[0] = bf16_lo(u.x); v[1] = bf16_hi(u.x); v[2] = bf16_lo(u.y); v[3] = bf16_hi(u.y);
  v[4] = bf16_lo(u.z); v[5] = bf16_hi(u.z); v[6] = bf16_lo(u.w); v[7] = bf16_hi(u.w);
}
// Four consecutive elements as floats (the address a multiple of 16 bytes for float, of 8 for bfloat16).
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 load4(const bf16* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return make_float4(bf16_lo(u.x), bf16_hi(u.x), bf16_lo(u.y), bf16_hi(u.y));
}
__device__ __forceinline__ void store8(float* p, const float (&v)[8]) {
  reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
  reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void store8(bf16* p, const float (&v)[8]) {
  *reinterpret_cast<uint4*>(p) = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
}
__device__ __forceinline__ void store4(float* p, float a, float b, float c, float d) {
  *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
}
__device__ __forceinline__ void store4(bf16* p, float a, float b, float c, float d) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16(a, b), pack_bf16(c, d));
}

// A barrier for what a workgroup hands on through LDS alone: it waits for this wave's LDS accesses, and not, as
// __syncthreads() does, for its loads from memory on their way (data asked for ahead then stays on its way).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// What matrix instructions have left in v, ready to be read.  A result must not be read for up to 12 states after its
// instruction; the compiler (ROCm 7.2.0, AMD clang 22.0.0git) puts in that wait, but counts it along one path only where two
// branches meet again: with code for the wait on the longer of the two and none on the shorter, the reader behind them comes too
// early on the shorter (10 states wanted, 2 left; the last element of the result was wrong).  So whatever reads results behind a
// branch that came after their instruction asks for them here: the first empty statements stand behind the instructions, the
// last ones in front of the readers, and the wait between the two.  16 states, some 7 ns.
template <typename V, int N>
__device__ __forceinline__ void settle(V (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
  asm volatile("s_nop 15");
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
}
template <typename V, int N, int M>
__device__ __forceinline__ void settle(V (&v)[N][M]) {
#pragma unroll
  for (int i = 0; i < N * M; ++i) asm volatile("" : "+v"(v[i / M][i % M]));
  asm volatile("s_nop 15");
#pragma unroll
  for (int i = 0; i < N * M; ++i) asm volatile("" : "+v"(v[i / M][i % M]));
}

// a's lanes 32 .. 63 with b's 0 .. 31; a's odd sixteens of lanes with b's even ones.
__device__ __forceinline__ void swap32(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
}
// A lane of the quarter g (lanes 16 g ..) holds the values 4 g .. 4 g + 3 of sixteen; afterwards it holds g, 4 + g, 8 + g,
// 12 + g: what it gives to four matrix instructions of four k each, so that these take the k in their order.
__device__ __forceinline__ void to_quarters(float& a, float& b, float& c, float& d) {
  swap32(a, c);
  swap32(b, d);
  swap16(a, b);
  swap16(c, d);
}
__device__ __forceinline__ void to_quarters(float (&v)[4]) { to_quarters(v[0], v[1], v[2], v[3]); }
__device__ __forceinline__ void to_quarters(float4& v) { to_quarters(v.x, v.y, v.z, v.w); }

// Reductions over a whole wave (every lane active), a value with that of lane ^ 32, then ^ 16, 8, 4, 2 and 1, between registers: a
// shuffle goes through the LDS unit and waits for it six times in a row, 0.25 us that a kernel of 4 us feels.  Once a step has made the
// lanes of a sixteen repeat, a rotation within the sixteen is the exchange that the next step wants.
template <typename Join>
__device__ __forceinline__ float wave_join(float v, Join join) {
  float a = v, b = v;
  swap32(a, b);
  v = a = join(a, b), b = v;
  swap16(a, b);
  v = join(a, b);
#define TLIE_STEP(control) v = join(v, __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), control, 0xf, 0xf, true)));
  TLIE_STEP(0x128)                                       // row_ror:8
  TLIE_STEP(0x124)                                       // row_ror:4
  TLIE_STEP(0x4e)                                        // quad_perm 2 3 0 1
  TLIE_STEP(0xb1)                                        // quad_perm 1 0 3 2
#undef TLIE_STEP
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
  return wave_join(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_join(v, [](float a, float b) { return fmaxf(a, b); });
}

// Block-wide reductions over up to 16 waves; `scratch` holds at least 16 floats of LDS.
// Every thread of the block must call them; every thread gets the result.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int waves = (blockDim.x + kWave - 1) / kWave;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < waves; ++w) total += scratch[w];
  return total;
}
__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int waves = (blockDim.x + kWave - 1) / kWave;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = -INFINITY;
  for (int w = 0; w < waves; ++w) total = fmaxf(total, scratch[w]);
  return total;
}

// The sum over `nsplit` partial results that lie `stride` elements apart, four loads in flight at a
// time.  The order of the additions is fixed (four interleaved chains, then their sum), so the
// result does not vary from run to run.
template <typename D>
__device__ __forceinline__ float sum_splits(const D* __restrict__ first, int nsplit, size_t stride) {
  if (nsplit == 1) return to_float(first[0]);
  float a = 0.f, b = 0.f, c = 0.f, d = 0.f;
  int s = 0;
  for (; s + 3 < nsplit; s += 4) {
    a += to_float(first[(s + 0) * stride]);
    b += to_float(first[(s + 1) * stride]);
    c += to_float(first[(s + 2) * stride]);
    d += to_float(first[(s + 3) * stride]);
  }
  for (; s < nsplit; ++s) a += to_float(first[s * stride]);
  return (a + b) + (c + d);
}

// Eight neighbouring elements summed over the parts of a split product, in the order of their index.  The parts are asked for eight at a
// time: one after the other, each waits for the one before, and a kernel of few rows is little else than that chain (the norm after a
// product of 64 rows in 8 parts, 2048 columns, 5.2 us one by one, 4.7 so).  They take 64 registers, with which half as many waves fit a
// compute unit: PARTS false for a product that comes whole, as those of many rows do (2048 x 2048 floats normed 14.3 us with them, 12.6 without).
template <bool PARTS, typename D>
__device__ __forceinline__ void load8_splits(const D* __restrict__ part, int nsplit, size_t stride, float (&d)[8]) {
  load8(part, d);
  if (!PARTS) return;
  constexpr int kTogether = sizeof(D) < sizeof(float) ? 1 : 8;       // (the products of this library leave their parts as floats)
  for (int s = 1; s < nsplit; s += kTogether) {
    float more[kTogether][8];
#pragma unroll
    for (int u = 0; u < kTogether; ++u)
      if (s + u < nsplit) load8(part + (s + u) * stride, more[u]);       // (the same for the whole grid)
#pragma unroll
    for (int u = 0; u < kTogether; ++u) {
      if (s + u >= nsplit) break;
#pragma unroll
      for (int j = 0; j < 8; ++j) d[j] += more[u][j];
    }
  }
}

// Of a kernel's two forms, the one for this product.
#define TLIE_PARTS_FORM(nsplit, KERNEL, ...) ((nsplit) == 1 ? &KERNEL<__VA_ARGS__, false> : &KERNEL<__VA_ARGS__, true>)

// The sum of squares of four, or eight, neighbouring columns of the 32-bit path's norms: one order for every kernel that forms it.
__device__ __forceinline__ float squares_of4(float a, float b, float c, float d) { return fmaf(a, a, b * b) + fmaf(c, c, d * d); }
__device__ __forceinline__ float squares_of8(const float (&v)[8]) {
  return squares_of4(v[0], v[1], v[2], v[3]) + squares_of4(v[4], v[5], v[6], v[7]);
}

// The gate of a gated feed-forward, from a gate g and an up u (both float).
// kind 0: silu(g) * u (reference: (g / (1 + exp(-g))) * u in float, src/cuda/kernels.cu:198-206).
// kind 1: g and u clamped first, g from above only (g = min(g, limit), u in [-limit, limit]), then
//         g * sigmoid(alpha * g) * (u + 1).
__device__ __forceinline__ float gated_value(float g, float u, int kind, float alpha, float limit) {
  if (kind == 0) return (g / (1.f + expf(-g))) * u;
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return (g / (1.f + expf(-alpha * g))) * (u + 1.f);
}

constexpr int kGateSilu = 0, kGateClampedSwish = 1;

// Error codes returned by the C entry points (0 = launched).
constexpr int kOk = 0;
constexpr int kBadArgument = -1;   // a size or dtype the kernel does not take
constexpr int kLaunchFailed = -2;  // hipGetLastError() reported an error after the launch
constexpr int kScratchTooSmall = -4;  // the sizes need more scratch memory than the library's own array holds

inline int launch_status() { return hipGetLastError() == hipSuccess ? kOk : kLaunchFailed; }

}  // namespace tlie
