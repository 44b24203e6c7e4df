// y[M, N] = x[M, K] . W[N, K]^T (+ bias[N]) with every product and sum in true 32-bit, on the matrix
// cores' 32-bit instruction (v_mfma_f32_16x16x4_f32): values widened to float, no reduced-precision mode.  Optionally the gated feed-forward's activation in the same kernel.
//
// reference: the only product of the reference's device path is a library call with 16-bit
// inputs and 32-bit accumulation (GemmFp16RowMajor, src/cuda/kernels.cu:342-368); its 32-bit
// model multiplies row by vector in a plain loop (src/model.cpp:65-72).
//
// What a 32-bit matrix instruction computes was measured on an MI355X, on 250 thousand results each of
// ordinary values, of exponents spread over 40 powers of two and of denormals: bit for bit the chain of fused
// multiply-adds fma(a[k], b[k], .) in the order of k, starting from C.  So the kernels here give the bits that a
// plain loop of v_fma_f32 over k gives, at twice its rate (packed 32-bit instructions are not used in this
// library): 143 TFLOP/s over the chip in chains of such instructions.
//
// The order of the sum of one output is fixed by K alone: K is cut into blocks of 512 from index 0;
// within a block the products are added one by one in index order (a chain of fused multiply-adds
// that starts at zero), and the blocks' sums are added to a total, which starts at zero, in index
// order.  Whatever M and N are, and whichever of the kernels below runs, an output gets the same
// bits: a token's result does not depend on what else is in the batch.  (Blocks, and not one chain
// over all of K, so that a product of few rows can give the blocks to different waves.)
#include "common.h"

#include <cmath>

namespace tlie {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kBlockK = 512;          // the blocks of K whose sums are formed apart (a multiple of every tile's width)
constexpr int kNoGate = -1;           // else a gate of common.h: W's rows alternate gate and up, y is [M, N / 2]

// Four consecutive values of a row as floats; the row is `K` long and the four may reach past its end: what lies
// there is read from inside the row and must be dropped by the caller.  WIDE: K and k are multiples of 4 and the
// rows are aligned for four values, so the four lie all inside or all past the end.
template <bool WIDE, typename T>
__device__ __forceinline__ float4 fetch4(const T* __restrict__ row, int k, int K) {
  if (WIDE) return load4(row + min(k, K - 4));
  return make_float4(to_float(row[min(k, K - 1)]), to_float(row[min(k + 1, K - 1)]), to_float(row[min(k + 2, K - 1)]),
                     to_float(row[min(k + 3, K - 1)]));
}

__device__ __forceinline__ float4 inside(float4 v, int k, int K) {
  return make_float4(k < K ? v.x : 0.f, k + 1 < K ? v.y : 0.f, k + 2 < K ? v.z : 0.f, k + 3 < K ? v.w : 0.f);
}

// ---- what a product of few rows may do beside (a layer's neighbouring arithmetic) ---------------------------
// Each saves a launch of 5 us whose own work is some kilobytes, and gives the bits of the kernel that it stands in for:
//   before   x is residual * norm weight and `ssq` [M][K / 8] the sums of squares of the residual's rows by eights; the rows of x are
//            multiplied by rsqrt(mean of squares + eps), the sum formed as in the norm kernel (`block_of_squares` in elementwise.hip)
//   after    kFoldResidual: residual [M][N] += result; with next_weight also xg = residual * next_weight and `ssq_out` for the
//            product that the next norm stands before.  kFoldRotation: W is a fused q/k/v weight with rows in paired order; rotation
//            and cache write of rope_cache.hip
constexpr int kFoldStore = 0, kFoldResidual = 1, kFoldRotation = 2;

struct RowsFold {
  const float* ssq;
  float eps;
  int kind;
  int squares_at;                     // where the blocks' sums of squares lie in LDS
  int rows;                           // rows of W a workgroup: even, at most the kernel's R; for ssq_out a multiple of 8
  float* residual;
  const float* next_weight;
  float* xg;
  float* ssq_out;
  const int* positions;
  const int* slot_map;
  const float* inv_freq;
  float* q_out;
  float* cache;
  int rot_dim, nq, nkv, d, page_size;
};

// What a thread's four neighbouring columns n .. n + 3 of row m need beside their sums, asked for before W (behind it the wait for
// these would be a way to memory of its own, twice for the rotation).
struct FoldAhead {
  float4 bias, residual, weight;
  float sine[2], cosine[2];
  int slot;
};

__device__ __forceinline__ FoldAhead fold_ahead(const RowsFold& fold, const float* __restrict__ bias, int m, int n, int N) {
  FoldAhead a;
  a.bias = make_float4(0.f, 0.f, 0.f, 0.f);
  if (bias) a.bias = make_float4(bias[n], bias[min(n + 1, N - 1)], bias[min(n + 2, N - 1)], bias[min(n + 3, N - 1)]);
  if (fold.kind == kFoldResidual) {
    a.residual = *reinterpret_cast<const float4*>(fold.residual + static_cast<size_t>(m) * N + n);
    if (fold.next_weight != nullptr) a.weight = *reinterpret_cast<const float4*>(fold.next_weight + n);
  } else if (fold.kind == kFoldRotation) {
    a.slot = fold.slot_map[m];
    a.cosine[0] = static_cast<float>(fold.positions[m]);   // (turned into sines by `fold_angles`)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int c = (n + 2 * e) % fold.d;
      a.sine[e] = fold.inv_freq != nullptr && c < fold.rot_dim ? fold.inv_freq[c / 2] : 0.f;
    }
  }
  return a;
}

__device__ __forceinline__ void fold_angles(const RowsFold& fold, FoldAhead& a) {
  if (fold.kind != kFoldRotation || fold.inv_freq == nullptr) return;
  const float position = a.cosine[0];
#pragma unroll
  for (int e = 0; e < 2; ++e) sincosf(position * a.sine[e], &a.sine[e], &a.cosine[e]);
}

// N a multiple of 4; with next_weight of 8, and the neighbouring thread holds the other half of the eight.
__device__ __forceinline__ void fold_residual(const RowsFold& fold, const FoldAhead& a, const float (&sum)[4], int m, int n, int N) {
  const float v[4] = {a.residual.x + sum[0], a.residual.y + sum[1], a.residual.z + sum[2], a.residual.w + sum[3]};
  store4(fold.residual + static_cast<size_t>(m) * N + n, v[0], v[1], v[2], v[3]);
  if (fold.next_weight == nullptr) return;                 // (the same for the whole grid)
  store4(fold.xg + static_cast<size_t>(m) * N + n, v[0] * a.weight.x, v[1] * a.weight.y, v[2] * a.weight.z, v[3] * a.weight.w);
  const float half = squares_of4(v[0], v[1], v[2], v[3]), other = __shfl_xor(half, 1, 64);
  if ((n & 4) == 0) fold.ssq_out[static_cast<size_t>(m) * (N / 8) + n / 8] = half + other;
}

// Two pairs of columns n, n + 1 and n + 2, n + 3 of token m (n and d even).
__device__ __forceinline__ void fold_rotation(const RowsFold& fold, const FoldAhead& a, const float (&sum)[4], int m, int n, int n_end) {
  const int slot = a.slot, half = fold.rot_dim / 2;
  const size_t head_stride = static_cast<size_t>(fold.page_size) * fold.d;
  float* page = fold.cache + static_cast<size_t>(slot < 0 ? 0 : slot / fold.page_size) * 2 * fold.nkv * head_stride;
  const int row = slot < 0 ? 0 : slot % fold.page_size;
#pragma unroll
  for (int e = 0; e < 4; e += 2) {
    if (n + e >= n_end) break;
    const int head = (n + e) / fold.d, c = (n + e) % fold.d;
    if (head >= fold.nq && slot < 0) continue;
    if (head >= fold.nq + fold.nkv) {                      // a value head lies transposed, after the key heads
      float* out = page + (head - fold.nq) * head_stride + static_cast<size_t>(c) * fold.page_size + row;
      out[0] = sum[e], out[fold.page_size] = sum[e + 1];
      continue;
    }
    float* out = head < fold.nq ? fold.q_out + (static_cast<size_t>(m) * fold.nq + head) * fold.d
                                : page + (head - fold.nq) * head_stride + static_cast<size_t>(row) * fold.d;
    if (fold.inv_freq != nullptr && c < fold.rot_dim) {
      const float sn = a.sine[e / 2], cs = a.cosine[e / 2];
      out[c / 2] = sum[e] * cs - sum[e + 1] * sn;
      out[c / 2 + half] = sum[e + 1] * cs + sum[e] * sn;
    } else {
      out[c] = sum[e], out[c + 1] = sum[e + 1];
    }
  }
}

// ---- few rows of x (decoding, short portions) ------------------------------------------------------------
// Bound by reading W.  A workgroup owns R rows of W (columns of y) and all M <= 16 MT rows of x; its waves take the blocks
// of K in turn, each block one chain of matrix instructions whose operands go straight from memory into registers: a
// lane asks for 16 bytes of a row (a wave for 16 rows by 64 bytes) and four swaps between lanes put 16 k in the order of
// the chain.  RING such loads of W are on their way per wave, and x (which comes from the caches) some ahead; no barrier
// until the blocks' sums meet in LDS, where the first waves add them in index order and apply bias and gate.
// PAIR (at most 8 rows of x, R = 8): of the instruction's 16 x 16 results two quarters of 8 x 8 are used, one for each of
// two blocks of K: lanes 0 .. 7 of a sixteen bring both operands' rows from the one block, lanes 8 .. 15 from the other.
// Twice the workgroups of R = 16, and no lane brings what another one has.
// FOLD: a layer's neighbouring arithmetic in the same kernel, described by `RowsFold` (at most 16 rows of x, all in 32 bits; the bits
// are those of the kernels it stands in for).
template <typename X, typename W, typename O, int MT, int R, bool PAIR, int RING, int WAVES, bool WIDE, bool FOLD = false>
__global__ void __launch_bounds__(64 * WAVES)
gemm_generic_few_kernel(const X* __restrict__ x, const W* __restrict__ w, const W* __restrict__ bias,
                        O* __restrict__ y, int M, int N, int K, int gate, float alpha, float limit, int jobs_at_once, RowsFold fold) {
  static_assert(!PAIR || (MT == 1 && R == 8), "two blocks at once: 8 rows of W, 8 of x");
  static_assert(!FOLD || (MT == 1 && WIDE), "folds: at most 16 rows of x, 16-byte loads");
  // Folded: x goes through a ring of its own, both rings 8 deep and asked for four pieces at a time.  Loads come back in the order they
  // were asked for, so that with W 16 groups ahead and x 8 the wait for x leaves only 8 of W's on their way; and a shorter ring is
  // half the code, most of which runs once or twice and comes from memory itself.  8 rows: 11264 x 2048 gated 26.9 us (rings of 16 with
  // x 8 ahead 31.7, one piece at a time 29.3), 2048 x 5632 17.6 (22.1, 19.1; two blocks at once with rings of 16 19.7), 2560 x 2048 11.2.
  constexpr bool kTogether = FOLD;
  constexpr int SC = kTogether ? RING : (8 / MT < RING / 2 ? 8 / MT : RING / 2);     // loads of x asked for together
  constexpr int kJobK = PAIR ? 2 * kBlockK : kBlockK, kPartK = 16 * RING;
  extern __shared__ __attribute__((aligned(16))) float sums[];   // [block][rows of x][R rows of W]
  constexpr int kNormRows = PAIR ? 8 : 16;
  float* squares = sums + fold.squares_at;                       // [block][rows of x]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int here = FOLD ? fold.rows : R;                   // rows of W of this workgroup (even, at most R)
  const int n0 = blockIdx.x * here, n_end = min(N, n0 + here);
  const W* w_row = w + static_cast<size_t>(min(n0 + (FOLD ? min(r % R, here - 1) : r % R), N - 1)) * K;
  const X* x_row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) x_row[i] = x + static_cast<size_t>(min(16 * i + (PAIR ? r & 7 : r), M - 1)) * K;
  const int jobs = (K + kJobK - 1) / kJobK;                // of one block of K, or of two
  const int first = (PAIR ? (r >> 3) * kBlockK : 0) + 4 * g;     // this lane's k within a job's first 16
  float4 ring[RING], xs[kTogether ? 1 : 2][SC][MT];
  int k0 = wave * kJobK;
  constexpr int kQuads = R / 4, kRows = PAIR ? 8 : 16 * MT;
  FoldAhead ahead;
  // the norm before this product: a lane sums the squares of its row of x over its quarter of a block of K, asked for ahead of W (its
  // first job's; those of further ones behind); code that runs once is kept short, its way from memory is what it costs
  const int chunks = K / 8;
  const bool normed = FOLD && fold.ssq != nullptr;         // (the same for the whole grid)
  auto part_of_block = [&](int k, float4 (&v)[4]) {
    const float* row = fold.ssq + static_cast<size_t>(min(PAIR ? r & 7 : r, M - 1)) * chunks;
    const int c0 = (k + first - 4 * g) / 8 + 4 * g;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = load4(row + min(c0 + 16 * j, chunks - 4));
  };
  float4 square[4];
  if constexpr (FOLD) {
    const int m = threadIdx.x / kQuads, n = n0 + threadIdx.x % kQuads * 4;
    if (m < M && n < n_end && threadIdx.x < kQuads * kRows) ahead = fold_ahead(fold, bias, m, n, N);
    if (normed && k0 < K) part_of_block(k0, square);
  }
  if (k0 < K) {
    if (!kTogether) {
#pragma unroll
      for (int c = 0; c < SC; ++c)
#pragma unroll
        for (int i = 0; i < MT; ++i) xs[0][c][i] = fetch4<WIDE>(x_row[i], k0 + first + 16 * c, K);
    }
#pragma unroll
    for (int c = 0; c < RING; ++c) {
      ring[c] = fetch4<WIDE>(w_row, k0 + first + 16 * c, K);
      if (kTogether) xs[0][c][0] = fetch4<WIDE>(x_row[0], k0 + first + 16 * c, K);
    }
  }
  float x_scale = 1.f;                                     // of this lane's row of x
  if constexpr (FOLD) {
    if (normed) {
      for (int job = wave; job < (K + kJobK - 1) / kJobK; job += waves) {
        if (job != wave) part_of_block(job * kJobK, square);
        const int c0 = (job * kJobK + first - 4 * g) / 8 + 4 * g;
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          sum += c0 + 16 * j < chunks ? (square[j].x + square[j].z) + (square[j].y + square[j].w) : 0.f;
        float a = sum, b = sum;
        swap16(a, b);
        a = b = a + b;
        swap32(a, b);
        if (lane < 16) squares[(PAIR ? 2 * job + (r >> 3) : job) * kNormRows + (PAIR ? r & 7 : r)] = a + b;
      }
      lds_barrier();
      float total = 0.f;
#pragma unroll 4
      for (int b = 0; b < (K + kBlockK - 1) / kBlockK; ++b) total += squares[b * kNormRows + (PAIR ? r & 7 : r)];
      x_scale = rsqrtf(total / static_cast<float>(K) + fold.eps);
    }
    if (wave == 0) fold_angles(fold, ahead);
  }
  // (the blocks' sums of one pass fit LDS; only a K of more than 64 blocks, with MT = 1, takes several: 512 x 40000 at 1 row 63 us,
  // at 16 rows 155, in tiles 540; 128 x 33000 46, 358)
  const int blocks = (K + kBlockK - 1) / kBlockK, pass = min(jobs, jobs_at_once);
  float4 before = make_float4(0.f, 0.f, 0.f, 0.f);         // this thread's sums of earlier passes (then it has one place at most)
  int job = wave;
  for (int first_job = 0; first_job < jobs; first_job += pass) {
    for (; job < min(jobs, first_job + pass); job += waves) {
      const int end = min(job * kJobK + kBlockK, K), slot = job - first_job;
      floatx4 acc[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
      while (k0 < end) {                                     // (all of these the same for the whole wave)
        const int next = k0 + kPartK < end ? k0 + kPartK : (job + waves) * kJobK;
        const bool more = next < K, edge = k0 + kPartK + (PAIR ? kBlockK : 0) > K;
#pragma unroll
        for (int c = 0; c < RING; ++c) {
          if (!kTogether && c % SC == 0) {                   // the next few pieces of x
            const int to = (c / SC + 1) & 1;
            const int from = (c + SC < RING ? k0 + 16 * (c + SC) : next) + first;
            if (c + SC < RING || more) {
#pragma unroll
              for (int e = 0; e < SC; ++e)
#pragma unroll
                for (int i = 0; i < MT; ++i) xs[to][e][i] = fetch4<WIDE>(x_row[i], from + 16 * e, K);
            }
          }
          float4 a = ring[c], b[MT];
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            b[i] = xs[kTogether ? 0 : (c / SC) & 1][c % SC][i];
            if (FOLD) b[i].x *= x_scale, b[i].y *= x_scale, b[i].z *= x_scale, b[i].w *= x_scale;
          }
          if (edge) {                                        // past the end of K: zeros
            a = inside(a, k0 + first + 16 * c, K);
#pragma unroll
            for (int i = 0; i < MT; ++i) b[i] = inside(b[i], k0 + first + 16 * c, K);
          }
          if (more && !kTogether) ring[c] = fetch4<WIDE>(w_row, next + first + 16 * c, K);
          to_quarters(a);
#pragma unroll
          for (int i = 0; i < MT; ++i) to_quarters(b[i]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32((&a.x)[e], (&b[i].x)[e], acc[i], 0, 0, 0);
          if (kTogether && more && c % 4 == 3) {
#pragma unroll
            for (int e = c - 3; e <= c; ++e) ring[e] = fetch4<WIDE>(w_row, next + first + 16 * e, K);
#pragma unroll
            for (int e = c - 3; e <= c; ++e) xs[0][e][0] = fetch4<WIDE>(x_row[0], next + first + 16 * e, K);
          }
        }
        k0 = next;
      }
      settle(acc);
      // lane (r, g) holds what the instruction's rows 4 g .. 4 g + 3 (of W) have for its column r (of x)
      if (PAIR) {
        if ((r >> 3) == (g >> 1))
          *reinterpret_cast<float4*>(sums + (2 * slot + (r >> 3)) * 64 + (r & 7) * 8 + 4 * (g & 1)) = make_float4(acc[0][0], acc[0][1], acc[0][2], acc[0][3]);
      } else {
#pragma unroll
        for (int i = 0; i < MT; ++i)
          *reinterpret_cast<float4*>(sums + (slot * MT + i) * 256 + r * 16 + 4 * g) = make_float4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
      }
    }
    __syncthreads();
    const bool last = first_job + pass >= jobs;
    const int blocks_here = last ? blocks - first_job * (kJobK / kBlockK) : pass * (kJobK / kBlockK);
    for (int t = threadIdx.x; t < kQuads * kRows; t += blockDim.x) {
      const int m = t / kQuads, j = t % kQuads * 4, n = n0 + j;       // four neighbouring columns of y
      if (m >= M || n >= n_end) continue;
      float4 v = before;
      for (int b = 0; b < blocks_here; ++b) {                // in index order
        const float4 s = *reinterpret_cast<const float4*>(sums + (b * kRows + m) * R + j);
        v.x += s.x, v.y += s.y, v.z += s.z, v.w += s.w;
      }
      if (!last) {
        before = v;
        continue;
      }
      const float out[4] = {v.x, v.y, v.z, v.w};
      if constexpr (FOLD) {
        if (fold.kind != kFoldStore) {
          float sum[4] = {out[0], out[1], out[2], out[3]};
          if (bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += (&ahead.bias.x)[e];
          }
          if (fold.kind == kFoldResidual) fold_residual(fold, ahead, sum, m, n, N);
          else fold_rotation(fold, ahead, sum, m, n, n_end);
          continue;
        }
      }
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        float p = out[e], u = out[e + 1];
        if (n + e >= n_end) break;
        if (bias) {
          p += to_float(bias[n + e]);
          if (n + e + 1 < n_end) u += to_float(bias[n + e + 1]);
        }
        if (gate != kNoGate) {
          y[static_cast<size_t>(m) * (N / 2) + (n + e) / 2] = from_float<O>(gated_value(p, u, gate, alpha, limit));
        } else {
          y[static_cast<size_t>(m) * N + n + e] = from_float<O>(p);
          if (n + e + 1 < n_end) y[static_cast<size_t>(m) * N + n + e + 1] = from_float<O>(u);
        }
      }
    }
    if (!last) __syncthreads();                              // (the sums have been read)
  }
}

// ---- many rows of x (prompts) ------------------------------------------------------------------------------
// Bound by the matrix cores.  A workgroup of four waves makes TN columns by TM rows of y, a wave a quarter of that in
// tiles of 16 by 16 (of 32 by 32, whose instruction is 5% faster alone, a wave would have one chain where it has four:
// 11264 x 2048 at 1000 rows 475 us against 424); 32 k of both operands lie in LDS, twice, one barrier a turn; D turns'
// loads are on their way in registers (a turn of a 64 x 64 tile is 0.4 us of products, a load from memory takes one to
// two).  Within 16 k a row lies as 0 4 8 12 1 5 ..: one 16-byte read then gives a lane what four matrix instructions take
// from it, in the order of k.  Rows are 36 floats apart, so that eight rows' reads cover the banks once.
// Measured beside the plain multiply-adds before (64 x 64 tiles, loads a turn of 16 k ahead): 1000 rows by 11264 x 2048
// 424 us against 805 (109 TFLOP/s), by 2048 x 5632 222 against 880, 2048 rows by 11264 x 2048 835 against 1489.
constexpr int kStepK = 32, kStride = kStepK + 4;

template <typename X, typename W, typename O, int TN, int TM, int D, bool WIDE>
__global__ void __launch_bounds__(256)
gemm_generic_kernel(const X* __restrict__ x, const W* __restrict__ w, const W* __restrict__ bias,
                    O* __restrict__ y, int M, int N, int K, int gate, float alpha, float limit) {
  constexpr int A = TN / 32, B = TM / 32;            // a wave's tiles
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* ws = lds;                                         // [2][TN][kStride]
  float* xs = lds + 2 * TN * kStride;                      // [2][TM][kStride]
  // workgroups go to the chip's eight dies in turn: each die gets a stretch of neighbouring tiles, rows of y first, so
  // that its cache holds their rows of W
  const int m_tiles = (M + TM - 1) / TM, tiles = m_tiles * ((N + TN - 1) / TN);
  const int each = tiles / 8, over = tiles % 8, die = blockIdx.x % 8;
  const int tile = die * each + min(die, over) + blockIdx.x / 8;
  const int n0 = tile / m_tiles * TN, m0 = tile % m_tiles * TM;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = threadIdx.x >> 3, piece = threadIdx.x & 7;           // 32 rows a pass, eight 16-byte pieces a row
  const W* w_row[TN / 32];
  const X* x_row[TM / 32];
#pragma unroll
  for (int p = 0; p < TN / 32; ++p) w_row[p] = w + static_cast<size_t>(min(n0 + row + 32 * p, N - 1)) * K;
#pragma unroll
  for (int p = 0; p < TM / 32; ++p) x_row[p] = x + static_cast<size_t>(min(m0 + row + 32 * p, M - 1)) * K;
  float4 w_next[D][TN / 32], x_next[D][TM / 32];
  auto ask = [&](int slot, int step) {
    const int k = step * kStepK + 4 * piece;
#pragma unroll
    for (int p = 0; p < TN / 32; ++p) w_next[slot][p] = fetch4<WIDE>(w_row[p], k, K);
#pragma unroll
    for (int p = 0; p < TM / 32; ++p) x_next[slot][p] = fetch4<WIDE>(x_row[p], k, K);
  };
  auto put_row = [&](float* at, const float4& v) {
    at += (piece >> 2) * 16 + (piece & 3);
    at[0] = v.x, at[4] = v.y, at[8] = v.z, at[12] = v.w;
  };
  auto put = [&](int slot, int step) {
    const int k = step * kStepK + 4 * piece, buffer = step & 1;
    if (step * kStepK + kStepK > K) {                      // (the last: what lies past K is zero)
#pragma unroll
      for (int p = 0; p < TN / 32; ++p) w_next[slot][p] = inside(w_next[slot][p], k, K);
#pragma unroll
      for (int p = 0; p < TM / 32; ++p) x_next[slot][p] = inside(x_next[slot][p], k, K);
    }
#pragma unroll
    for (int p = 0; p < TN / 32; ++p) put_row(ws + (buffer * TN + row + 32 * p) * kStride, w_next[slot][p]);
#pragma unroll
    for (int p = 0; p < TM / 32; ++p) put_row(xs + (buffer * TM + row + 32 * p) * kStride, x_next[slot][p]);
  };
  floatx4 acc[A][B] = {}, total[A][B] = {};
  const int steps = (K + kStepK - 1) / kStepK;
  const float* my_w = ws + ((wave & 1) * (TN / 2) + (lane & 15)) * kStride + (lane >> 4) * 4;
  const float* my_x = xs + ((wave >> 1) * (TM / 2) + (lane & 15)) * kStride + (lane >> 4) * 4;
#pragma unroll
  for (int j = 0; j < D; ++j)
    if (j < steps) ask(j, j);
  put(0, 0);
  if (D < steps) ask(0, D);
  for (int base = 0; base < steps; base += D) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int s = base + j;
      if (s >= steps) break;                               // (the same for the whole workgroup)
      lds_barrier();                                       // this turn's tiles are whole, the last turn's have been read
      if (s > 0 && s % (kBlockK / kStepK) == 0) {          // a block of K has ended: its sums join the totals
        settle(acc);
#pragma unroll
        for (int i = 0; i < A; ++i)
#pragma unroll
          for (int u = 0; u < B; ++u) total[i][u] += acc[i][u], acc[i][u] = floatx4{};
      }
      if (s + 1 < steps) put((j + 1) % D, s + 1);
      if (s + 1 + D < steps) ask((j + 1) % D, s + 1 + D);
      const float* wt = my_w + (s & 1) * TN * kStride;
      const float* xt = my_x + (s & 1) * TM * kStride;
#pragma unroll
      for (int e = 0; e < kStepK; e += 16) {
        float4 a[A], b[B];
#pragma unroll
        for (int i = 0; i < A; ++i) a[i] = *reinterpret_cast<const float4*>(wt + 16 * i * kStride + e);
#pragma unroll
        for (int i = 0; i < B; ++i) b[i] = *reinterpret_cast<const float4*>(xt + 16 * i * kStride + e);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int i = 0; i < A; ++i)
#pragma unroll
            for (int u = 0; u < B; ++u) acc[i][u] = __builtin_amdgcn_mfma_f32_16x16x4f32((&a[i].x)[c], (&b[u].x)[c], acc[i][u], 0, 0, 0);
      }
    }
  }
  settle(acc);
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int u = 0; u < B; ++u) total[i][u] += acc[i][u];
  // a lane holds four neighbouring columns of one row of each tile
  const bool whole = (N & 3) == 0;
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int m = m0 + (wave >> 1) * (TM / 2) + 16 * u + (lane & 15);
      const int n = n0 + (wave & 1) * (TN / 2) + 16 * i + 4 * (lane >> 4);
      if (m >= M || n >= N) continue;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = total[i][u][e];
        if (bias && n + e < N) v[e] += to_float(bias[n + e]);
      }
      if (gate != kNoGate) {
        O* at = y + static_cast<size_t>(m) * (N / 2) + n / 2;
        at[0] = from_float<O>(gated_value(v[0], v[1], gate, alpha, limit));
        if (n + 2 < N) at[1] = from_float<O>(gated_value(v[2], v[3], gate, alpha, limit));
      } else if (whole) {
        store4(y + static_cast<size_t>(m) * N + n, v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) y[static_cast<size_t>(m) * N + n + e] = from_float<O>(v[e]);
      }
    }
}

template <typename X, typename W, typename O, int MT, int R, bool PAIR, int RING, int WAVES, bool WIDE>
int launch_few(const X* x, const W* w, const W* bias, O* y, int M, int N, int K, int gate, float alpha, float limit, hipStream_t s) {
  const int job_k = PAIR ? 2 * kBlockK : kBlockK, jobs = (K + job_k - 1) / job_k, turns = (jobs + WAVES - 1) / WAVES;
  const int waves = (jobs + turns - 1) / turns;            // as many for each turn
  const int job_bytes = (PAIR ? 2 * 64 : 16 * MT * R) * static_cast<int>(sizeof(float));
  const int at_once = jobs <= 64 * 1024 / job_bytes ? jobs : 64 * 1024 / job_bytes;
  const int bytes = at_once * job_bytes;
  hipLaunchKernelGGL((gemm_generic_few_kernel<X, W, O, MT, R, PAIR, RING, WAVES, WIDE>), dim3((N + R - 1) / R), dim3(64 * waves), bytes, s,
                     x, w, bias, y, M, N, K, gate, alpha, limit, at_once, RowsFold{});
  return launch_status();
}

template <int R, bool PAIR, int WAVES>
int launch_folded(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int gate, float alpha, float limit,
                  const RowsFold& fold, hipStream_t s) {
  const int job_k = PAIR ? 2 * kBlockK : kBlockK, jobs = (K + job_k - 1) / job_k, turns = (jobs + WAVES - 1) / WAVES;
  const int waves = (jobs + turns - 1) / turns;
  const int job_bytes = (PAIR ? 2 * 64 : 16 * R) * static_cast<int>(sizeof(float));
  const int squares = fold.ssq != nullptr ? jobs * 16 * static_cast<int>(sizeof(float)) : 0, room = 64 * 1024 - squares;
  if (room < job_bytes) return kBadArgument;               // (K of half a million)
  const int at_once = jobs <= room / job_bytes ? jobs : room / job_bytes;
  RowsFold placed = fold;
  placed.squares_at = at_once * job_bytes / static_cast<int>(sizeof(float));
  hipLaunchKernelGGL((gemm_generic_few_kernel<float, float, float, 1, R, PAIR, 8, WAVES, true, true>), dim3((N + fold.rows - 1) / fold.rows),
                     dim3(64 * waves), at_once * job_bytes + squares, s, x, w, bias, y, M, N, K, gate, alpha, limit, at_once, placed);
  return launch_status();
}

// ---- embedding of few rows with the first norm's inputs ------------------------------------------------------
__global__ void embed_rows_float_kernel(const int* __restrict__ tokens, const float* __restrict__ table, const float* __restrict__ weight,
                                        float* __restrict__ residual, float* __restrict__ xg, float* __restrict__ ssq, int hidden) {
  const int t = blockIdx.y, chunk = blockIdx.x * blockDim.x + threadIdx.x;
  if (chunk * 8 >= hidden) return;
  const size_t at = static_cast<size_t>(t) * hidden + chunk * 8;
  float v[8], w[8];
  load8(table + static_cast<size_t>(tokens[t]) * hidden + chunk * 8, v);
  load8(weight + chunk * 8, w);
  store8(residual + at, v);
  ssq[static_cast<size_t>(t) * (hidden / 8) + chunk] = squares_of8(v);
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] *= w[j];
  store8(xg + at, v);
}

template <typename X, typename W, typename O, int TN, int TM, int D, bool WIDE>
int launch_tiles(const X* x, const W* w, const W* bias, O* y, int M, int N, int K, int gate, float alpha, float limit, hipStream_t s) {
  const long long tiles = static_cast<long long>((M + TM - 1) / TM) * ((N + TN - 1) / TN);
  if (tiles > 0x7fffffff) return kBadArgument;
  constexpr int kBytes = 2 * (TN + TM) * kStride * static_cast<int>(sizeof(float));
  static_assert(kBytes <= 64 * 1024, "within what a launch may ask for without an attribute");
  hipLaunchKernelGGL((gemm_generic_kernel<X, W, O, TN, TM, D, WIDE>), dim3(static_cast<unsigned>(tiles)), dim3(256), kBytes, s, x, w, bias,
                     y, M, N, K, gate, alpha, limit);
  return launch_status();
}

template <typename X, typename W, typename O, bool WIDE>
int launch_product(const X* x, const W* w, const W* bias, O* y, int M, int N, int K, int gate, float alpha, float limit,
                   int compute_units, hipStream_t s) {
  const long long blocks = (K + kBlockK - 1) / kBlockK;
  // Few rows of x: the kernel that reads W straight into registers; more than 16, while the sums of the blocks fit LDS.  A matrix of at
  // most 8 rows a compute unit takes two blocks at once (2048 x 2048, 8 rows of x: 10.1 us against 12.0; 2560 x 2048, where
  // some units would get two workgroups: 14.8 against 12.3).  More than 16 rows of x go there only while W has at most 16 rows
  // a unit: every workgroup reads all of x (64 rows, 2048 x 2048: 24.7 us against 34.4 in tiles; 11264 x 2048: 70.1 against 46.1).
  // One block of K or less gives a workgroup one wave: such products go in tiles (96 x 96, 16 rows: 3.3 us against 4.0).
  const int mt = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
  if (M <= 64 && blocks > 1 && (mt == 1 || (blocks * mt * 1024 <= 64 * 1024 && (N + 15) / 16 <= compute_units))) {
    constexpr int kRing = WIDE ? 16 : 8;
    if (mt == 4) return launch_few<X, W, O, 4, 16, false, 8, 8, WIDE>(x, w, bias, y, M, N, K, gate, alpha, limit, s);
    if (mt == 2) return launch_few<X, W, O, 2, 16, false, 8, WIDE ? 12 : 8, WIDE>(x, w, bias, y, M, N, K, gate, alpha, limit, s);
    if (M <= 8 && (N + 7) / 8 <= compute_units) return launch_few<X, W, O, 1, 8, true, kRing, 12, WIDE>(x, w, bias, y, M, N, K, gate, alpha, limit, s);
    return launch_few<X, W, O, 1, 16, false, kRing, 12, WIDE>(x, w, bias, y, M, N, K, gate, alpha, limit, s);
  }
  // Tiles of 64 x 64, 64 x 32 or 32 x 32: alone on its compute unit a tile takes 50, 40 or 35 us for K = 2048 (the way of its
  // loads), of which its products are 28.6, 14.3 and 7.2; several tiles to a unit reach 0.75, 0.69 and 0.62 of the matrix
  // cores' rate (measured at 11264 x 2048 and 1000 rows: 424, 459 and 510 us).  The least of the three estimates:
  const double rows[3] = {64, 64, 32}, cols[3] = {64, 32, 32}, alone[3] = {50, 40, 35}, busy[3] = {28.6 / 0.75, 14.3 / 0.69, 7.2 / 0.62};
  int best = 0;
  double least = 0;
  for (int i = 0; i < 3; ++i) {
    const double tiles = ceil(N / rows[i]) * ceil(M / cols[i]), time = fmax(alone[i], busy[i] * ceil(tiles / compute_units));
    if (i == 0 || time < least) best = i, least = time;
  }
  if (best == 0) return launch_tiles<X, W, O, 64, 64, 2, WIDE>(x, w, bias, y, M, N, K, gate, alpha, limit, s);
  if (best == 1) return launch_tiles<X, W, O, 64, 32, 4, WIDE>(x, w, bias, y, M, N, K, gate, alpha, limit, s);
  return launch_tiles<X, W, O, 32, 32, 4, WIDE>(x, w, bias, y, M, N, K, gate, alpha, limit, s);
}

}  // namespace tlie

using namespace tlie;

extern "C" int tlie_gemm_generic(const void* x, int x_dtype, const void* w, int w_dtype, const void* bias,
                                 void* y, int y_dtype, int M, int N, int K, int gate, float alpha, float limit, int compute_units,
                                 void* stream) {
  if (M <= 0 || N <= 0 || K <= 0 || compute_units <= 0) return kBadArgument;
  if (gate < kNoGate || gate > kGateClampedSwish || (gate != kNoGate && N % 2 != 0)) return kBadArgument;
  hipStream_t s = (hipStream_t)stream;
#define TLIE_CASE(XC, X, WC, W, OC, O)                                                                       \
  if (x_dtype == XC && w_dtype == WC && y_dtype == OC) {                                                     \
    /* four values of a row in one load where every row of both operands is aligned for it */               \
    const bool wide = (K & 3) == 0 && reinterpret_cast<uintptr_t>(x) % (4 * sizeof(X)) == 0 &&               \
                      reinterpret_cast<uintptr_t>(w) % (4 * sizeof(W)) == 0;                                 \
    return wide ? launch_product<X, W, O, true>((const X*)x, (const W*)w, (const W*)bias, (O*)y, M, N, K, gate, alpha, limit, compute_units, s)   \
                : launch_product<X, W, O, false>((const X*)x, (const W*)w, (const W*)bias, (O*)y, M, N, K, gate, alpha, limit, compute_units, s); \
  }
  TLIE_CASE(kF32, float, kF32, float, kF32, float)
  TLIE_CASE(kBF16, bf16, kBF16, bf16, kBF16, bf16)
  TLIE_CASE(kBF16, bf16, kBF16, bf16, kF32, float)
  TLIE_CASE(kBF16, bf16, kF32, float, kBF16, bf16)
  TLIE_CASE(kBF16, bf16, kF32, float, kF32, float)
#undef TLIE_CASE
  return kBadArgument;
}

// The product of at most 16 rows with a layer's neighbouring arithmetic, all in 32 bits (see `RowsFold`).  K % 4 == 0 (ssq: % 32) and
// 16-byte aligned rows; N % 4 == 0 for the residual, % 8 with next_weight; d even for the rotation.
extern "C" int tlie_gemm_generic_rows(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int gate, float alpha,
                                      float limit, const float* ssq, float eps, int kind, float* residual, const float* next_weight, float* xg,
                                      float* ssq_out, const int* positions, const int* slot_map, const float* inv_freq, int rot_dim, float* q_out,
                                      float* cache, int nq, int nkv, int d, int page_size, int compute_units, void* stream) {
  if (M <= 0 || M > 16 || N <= 0 || K <= 0 || K % 4 != 0 || compute_units <= 0) return kBadArgument;
  if (gate < kNoGate || gate > kGateClampedSwish || (gate != kNoGate && (N % 2 != 0 || kind != kFoldStore))) return kBadArgument;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 != 0 || (ssq != nullptr && (K % 32 != 0 || reinterpret_cast<uintptr_t>(ssq) % 16 != 0))) return kBadArgument;
  if (kind == kFoldStore) {
    if (y == nullptr) return kBadArgument;
  } else if (kind == kFoldResidual) {
    if (residual == nullptr || N % 4 != 0 || (next_weight != nullptr && (N % 8 != 0 || xg == nullptr || ssq_out == nullptr))) return kBadArgument;
    if ((reinterpret_cast<uintptr_t>(residual) | reinterpret_cast<uintptr_t>(next_weight) | reinterpret_cast<uintptr_t>(xg)) % 16 != 0) return kBadArgument;
  } else if (kind == kFoldRotation) {
    if (positions == nullptr || slot_map == nullptr || q_out == nullptr || cache == nullptr || nq <= 0 || nkv <= 0 || d <= 0 || d % 2 != 0 ||
        page_size <= 0 || rot_dim < 0 || rot_dim > d || rot_dim % 2 != 0 || N != (nq + 2 * nkv) * d)
      return kBadArgument;
  } else {
    return kBadArgument;
  }
  hipStream_t s = (hipStream_t)stream;
  RowsFold fold{ssq, eps, kind, 0, 16, residual, next_weight, xg, ssq_out, positions, slot_map, inv_freq, q_out, cache, rot_dim, nq, nkv, d, page_size};
  if (M <= 8 && K > kBlockK && (N + 7) / 8 <= compute_units) {       // (the lines of `launch_product`)
    fold.rows = 8;
    return launch_folded<8, true, 12>(x, w, bias, y, M, N, K, gate, alpha, limit, fold, s);
  }
  // where strips of 16 rows leave units without a workgroup, even shares of the rows instead
  const int strips = (N + 15) / 16, share = ((N + compute_units - 1) / compute_units + 1) / 2 * 2;
  if (kind != kFoldResidual && strips < compute_units && 2 * strips > compute_units && share < 16) fold.rows = share < 8 ? 8 : share;
  return launch_folded<16, false, 12>(x, w, bias, y, M, N, K, gate, alpha, limit, fold, s);
}

// The embedding of few rows with the first norm's inputs: residual [rows][hidden] = table's rows, xg = residual * weight, ssq the sums
// of squares by eights; hidden % 8 == 0, 32-byte aligned arrays.
extern "C" int tlie_embed_rows_float(const int* tokens, const float* table, const float* weight, float* residual, float* xg, float* ssq,
                                     int rows, int hidden, void* stream) {
  if (rows <= 0 || rows > 65535 || hidden <= 0 || hidden % 8 != 0) return kBadArgument;
  if ((reinterpret_cast<uintptr_t>(table) | reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(residual) | reinterpret_cast<uintptr_t>(xg)) & 31)
    return kBadArgument;
  hipLaunchKernelGGL(embed_rows_float_kernel, dim3((hidden / 8 + 63) / 64, rows), dim3(64), 0, (hipStream_t)stream, tokens, table, weight, residual,
                     xg, ssq, hidden);
  return launch_status();
}
