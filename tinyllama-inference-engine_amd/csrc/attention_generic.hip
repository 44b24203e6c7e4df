// Paged causal grouped-query attention, the plain kernel: any storage type, any head size up to
// the block size, any number of tokens per sequence.  It is the whole 32-bit path's attention and
// the fallback of the bfloat16 path for sizes the tiled kernels refuse.
//
// reference: AttentionDecodeKernel (src/cuda/kernels.cu:147-196): one block per query head,
// scores = (q . k) * rsqrt(d) over positions 0..pos, max, exp, sum, normalise, then one thread
// per output dimension sums p * v serially.  That kernel keeps all scores of the context in
// shared memory and serves one token; this one walks the context in chunks of 64, 128 or 256 keys
// (the least that holds the head size) with running maxima and sums (so the context length is
// unbounded), serves every token of a step in one launch, finds keys through the block table, and
// optionally limits the keys to a window.  Chunks start at multiples of their size counted from
// position 0, so the order of the sums for a given (sequence, position) never depends on how the
// step was cut.
#include "common.h"

#include <type_traits>

namespace tlie {

// q: [tokens][nq][d]; a page of the cache holds nkv planes of keys, [row][d], and after them nkv planes
// of values, transposed, [dv][row] (with dv = d that is [pages][2][nkv][page_size * d]);
// out: [tokens][nq][dv].
// token_seq[t]: row of the block table; positions[t]: absolute position of the token.
// window <= 0: all keys 0..pos; otherwise keys pos-window+1..pos.
// chunk > 0: only keys of the query's own chunk of positions, pos - pos % chunk .. pos (chunks are
// counted from position 0 of the sequence).
// sink (or null): one number per query head that joins the softmax's denominator as exp(sink): it has
// no key and no value and is not scaled.
// softcap > 0: a scaled score s becomes softcap * tanh(s / softcap) before the softmax.
// A workgroup of 256 threads serves one (token, head).  Its threads form 256 / CHUNK groups of
// CHUNK threads (CHUNK >= d); chunk c of the context (keys c * CHUNK ..) belongs to group
// c % groups, and every group keeps a running maximum, sum and output of its own over its chunks,
// in the order of their index; at the end the groups' results are put together in the order of
// the groups.  Which keys meet in which sum, and in which order, depends on the positions alone.
// seq_start (or null) with min_tokens: the step's cumulative token counts per sequence; tokens of
// sequences that bring min_tokens tokens or more are then left to the kernel of many tokens below, which
// is launched beside this one for the same step and leaves the others to this one.
// The attended values go out in the activation type, or, when the caller works on with them in 32-bit (two
// maps of attention whose difference is normed), as floats: `out` then points to floats whatever T is.
template <typename T>
__device__ __forceinline__ void store_result(T* out, size_t index, float value, int out_f32) {
  if (out_f32) reinterpret_cast<float*>(out)[index] = value;
  else out[index] = from_float<T>(value);
}

template <typename T, int CHUNK>
__global__ void __launch_bounds__(256)
attention_generic_kernel(const T* __restrict__ q, const T* __restrict__ cache, const int* __restrict__ block_table,
                         int max_blocks, const int* __restrict__ token_seq, const int* __restrict__ positions,
                         T* __restrict__ out, int nq, int nkv, int d, int dv, int page_size, int window, int chunk,
                         const float* __restrict__ sink, float scale, float softcap,
                         const int* __restrict__ seq_start, int min_tokens, int vshare, int out_f32) {
  constexpr int kGroups = 256 / CHUNK, kWavesPerGroup = CHUNK / 64;
  if (seq_start != nullptr) {                      // (the same for the whole workgroup)
    const int seq = token_seq[blockIdx.x];
    if (seq_start[seq + 1] - seq_start[seq] >= min_tokens) return;
  }
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* q_row = lds;                              // d
  float* prob = q_row + d;                         // 256: a group's probabilities of its current chunk
  float* wave_part = prob + 256;                   // 4: one value per wave, for the reductions within a group
  float* group_stat = wave_part + 4;               // kGroups x 2: maximum, sum
  float* group_out = group_stat + 2 * kGroups;     // kGroups x dv
  const int t = blockIdx.x, h = blockIdx.y;
  const int group = threadIdx.x / CHUNK, place = threadIdx.x % CHUNK;       // place: key of the chunk, then dim of the output
  const int wave = threadIdx.x / 64, first_wave = group * kWavesPerGroup;
  const int kv_head = h / (nq / nkv);
  const int pos = positions[t];
  const int* pages = block_table + static_cast<size_t>(token_seq[t]) * max_blocks;
  int lo = window > 0 ? max(0, pos - window + 1) : 0;
  if (chunk > 0) lo = max(lo, pos - pos % chunk);
  // (vshare key heads in a row read one value head: a page then holds nkv planes of keys and nkv / vshare of values)
  const size_t page_stride = static_cast<size_t>(page_size) * (static_cast<size_t>(nkv) * d + static_cast<size_t>(nkv / vshare) * dv);
  const size_t head_offset = static_cast<size_t>(kv_head) * page_size * d;
  const size_t v_offset = static_cast<size_t>(nkv) * page_size * d + static_cast<size_t>(kv_head / vshare) * page_size * dv;

  for (int i = threadIdx.x; i < d; i += 256) q_row[i] = to_float(q[(static_cast<size_t>(t) * nq + h) * d + i]);
  __syncthreads();
  // whole 16-byte loads of keys and values where everything is a multiple of four floats
  const bool wide = (d & 3) == 0 && (page_size & 3) == 0 && (reinterpret_cast<uintptr_t>(cache) & 15) == 0;

  // the reductions over a group: over each of its waves by shuffles, then over its waves through LDS
  // (every thread of the workgroup takes part in every call: the barriers are the workgroup's)
  auto over_group = [&](float value, bool maximum) {
    value = maximum ? wave_max(value) : wave_sum(value);
    if (kWavesPerGroup == 1) return value;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) wave_part[wave] = value;
    __syncthreads();
    float total = wave_part[first_wave];
    for (int w = 1; w < kWavesPerGroup; ++w) total = maximum ? fmaxf(total, wave_part[first_wave + w]) : total + wave_part[first_wave + w];
    return total;
  };

  float running_max = -INFINITY, running_sum = 0.f, acc = 0.f;
  constexpr int kRound = CHUNK * kGroups;          // keys all groups take in one turn of the loop
  for (int base = (lo / kRound) * kRound; base <= pos; base += kRound) {
    const int start = base + group * CHUNK;        // (a group whose chunk lies outside lo..pos goes along with nothing to add)
    const int j = start + place;
    const bool valid = j >= lo && j <= pos;
    float score = -INFINITY;
    if (valid) {
      const T* key = cache + static_cast<size_t>(pages[j / page_size]) * page_stride + head_offset +
                     static_cast<size_t>(j % page_size) * d;
      float dot = 0.f;
      int i = 0;
      if (std::is_same<T, float>::value && wide) {
        // (four dims a load; the additions stay in the order of the dims)
#pragma unroll 4
        for (; i + 4 <= d; i += 4) {
          const float4 kv = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(key) + i);
          const float4 qv = *reinterpret_cast<const float4*>(q_row + i);
          dot += qv.x * kv.x;
          dot += qv.y * kv.y;
          dot += qv.z * kv.z;
          dot += qv.w * kv.w;
        }
      }
      for (; i < d; ++i) dot += q_row[i] * to_float(key[i]);
      score = dot * scale;
      if (softcap > 0.f) score = softcap * tanhf(score / softcap);
    }
    const float new_max = fmaxf(running_max, over_group(score, true));
    const float p = valid ? expf(score - new_max) : 0.f;
    prob[threadIdx.x] = p;
    const float chunk_sum = over_group(p, false);
    __syncthreads();                               // prob[] is written
    // nothing seen yet (new_max = -inf): nothing to rescale, nothing to add
    const float alpha = new_max == -INFINITY ? 1.f : expf(running_max - new_max);   // 0 when this chunk is the group's first with keys
    running_sum = running_sum * alpha + chunk_sum;
    running_max = new_max;
    if (place < dv) {
      acc *= alpha;
      const int first = max(0, lo - start), last = min(CHUNK, pos - start + 1);
      int jj = first;
      if (std::is_same<T, float>::value && wide) {
        // (four keys a load where they lie on one page, four to a boundary: chunks start at multiples of
        // 64 and pages hold a multiple of four rows; the additions stay in the order of the keys)
        for (; jj < last && (jj & 3) != 0; ++jj) {
          const int key_pos = start + jj;
          const T* value = cache + static_cast<size_t>(pages[key_pos / page_size]) * page_stride + v_offset +
                           static_cast<size_t>(place) * page_size + key_pos % page_size;
          acc += prob[group * CHUNK + jj] * to_float(*value);
        }
#pragma unroll 4
        for (; jj + 4 <= last; jj += 4) {
          const int key_pos = start + jj;
          const float* value = reinterpret_cast<const float*>(cache) + static_cast<size_t>(pages[key_pos / page_size]) * page_stride +
                               v_offset + static_cast<size_t>(place) * page_size + key_pos % page_size;
          const float4 vv = *reinterpret_cast<const float4*>(value);
          const float4 pv = *reinterpret_cast<const float4*>(prob + group * CHUNK + jj);
          acc += pv.x * vv.x;
          acc += pv.y * vv.y;
          acc += pv.z * vv.z;
          acc += pv.w * vv.w;
        }
      }
      for (; jj < last; ++jj) {
        const int key_pos = start + jj;
        const T* value = cache + static_cast<size_t>(pages[key_pos / page_size]) * page_stride + v_offset +
                         static_cast<size_t>(place) * page_size + key_pos % page_size;
        acc += prob[group * CHUNK + jj] * to_float(*value);
      }
    }
    __syncthreads();                               // prob[] is read
  }
  // the groups' results into one, in the order of the groups
  if (place == 0) group_stat[2 * group] = running_max, group_stat[2 * group + 1] = running_sum;
  if (place < dv) group_out[group * dv + place] = acc;
  __syncthreads();
  if (threadIdx.x < dv) {
    float top = -INFINITY;
    for (int g = 0; g < kGroups; ++g) top = fmaxf(top, group_stat[2 * g]);
    float total = 0.f, result = 0.f;
    if (sink != nullptr) {                         // the sink counts once: exp(sink) in the denominator, nothing in the sum of values
      top = fmaxf(top, sink[h]);
      total = expf(sink[h] - top);
    }
    for (int g = 0; g < kGroups; ++g) {
      const float m = group_stat[2 * g];
      if (m == -INFINITY) continue;                // a group that saw no key
      const float w = expf(m - top);
      total += w * group_stat[2 * g + 1];
      result += w * group_out[g * dv + threadIdx.x];
    }
    store_result(out, (static_cast<size_t>(t) * nq + h) * dv + threadIdx.x, result / total, out_f32);
  }
}

// ---- head sizes up to 64, on the matrix cores' 32-bit instruction ------------------------------------------
// v_mfma_f32_16x16x4_f32 gives, bit for bit, the chain of fused multiply-adds over k in their order, starting from C
// (measured; see the 32-bit products).  Scores are therefore instructions over a head's dims, and values instructions over
// a chunk's keys that continue a state's sums: the sums of the kernel above, operation for operation.  A column, a (token,
// query head) pair, is one of an instruction's sixteen; chunk c of 64 keys belongs to the column's running state c % 4; the
// maximum and the sum of a chunk's probabilities are taken over the key's bits in the order wave_sum takes them; the four
// states meet in the same order at the end.  Both kernels below and the one above give a column the same bits, and a step may
// take whichever is faster.
typedef float floatx4 __attribute__((ext_vector_type(4)));

// The sum and the maximum with the lane 32 (then 16) away: for keys, with the key whose bit 3 (then bit 2) differs.
__device__ __forceinline__ float sum_quarters(float v) {
  float a = v, b = v;
  swap32(a, b);
  v = a + b, a = v, b = v;
  swap16(a, b);
  return a + b;
}
__device__ __forceinline__ float max_quarters(float v) {
  float a = v, b = v;
  swap32(a, b);
  v = fmaxf(a, b), a = v, b = v;
  swap16(a, b);
  return fmaxf(a, b);
}

// Four values of a row from i on, of which `count` exist (the others are zero and not read).  `wide`: four that exist lie
// aligned for one load.
template <typename T>
__device__ __forceinline__ void row4(float (&v)[4], const T* __restrict__ row, int i, int count, bool wide) {
  if (wide && i + 4 <= count) {
    const float4 f = load4(row + i);
    v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = i + e < count ? to_float(row[i + e]) : 0.f;
}

// One running state of a column: lane (column l & 15, quarter g) keeps the dims 16 t + 4 g .. + 3 of its sum of values.
template <int KD>
struct ColumnState {
  float top = -INFINITY, sum = 0.f;
  floatx4 acc[KD] = {};
};

// A chunk's scores (dot[t]: keys 16 t + 4 g .. + 3, from `start`) become probabilities, in place, and the state takes in their
// maximum and sum; its values are scaled and wait for the chunk's.
template <bool CAP, int KD>
__device__ __forceinline__ void take_scores(floatx4 (&dot)[4], ColumnState<KD>& state, int start, int lo, int pos, int g, float scale, float softcap) {
  settle(dot);
  settle(state.acc);
  float top = -INFINITY;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = start + 16 * t + 4 * g + i;
      const float score = CAP && softcap > 0.f ? softcap * tanhf(dot[t][i] * scale / softcap) : dot[t][i] * scale;
      dot[t][i] = j >= lo && j <= pos ? score : -INFINITY;
      top = fmaxf(top, dot[t][i]);
    }
  const float new_max = fmaxf(state.top, max_quarters(top));
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = start + 16 * t + 4 * g + i;
      const float weight = expf(dot[t][i] - new_max);
      dot[t][i] = j >= lo && j <= pos ? weight : 0.f;
    }
  // over the key's bits 5, 4, 3, 2, 1, 0, as wave_sum over one key a lane
  float part[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) part[i] = sum_quarters((dot[0][i] + dot[2][i]) + (dot[1][i] + dot[3][i]));
  const float chunk_sum = (part[0] + part[2]) + (part[1] + part[3]);
  const float alpha = new_max == -INFINITY ? 1.f : expf(state.top - new_max);
  state.sum = state.sum * alpha + chunk_sum;
  state.top = new_max;
#pragma unroll
  for (int u = 0; u < KD; ++u) state.acc[u] *= alpha;
}

// ---- many tokens a sequence ----
// A workgroup of four waves serves up to 64 columns, of up to 64 / heads consecutive tokens of the step and the heads of
// one kv head (or 64 of them), a wave 16 of them, and brings every chunk of 64 keys and values through LDS once for all (the
// kernel above reads each key and value again for every column: a prompt of 2048 tokens would be 34 GB of cache traffic a
// layer).  Bound by the matrix cores: a chunk is 128 instructions of 32 clocks a wave.  The chunk after the next is asked for, and the
// next stored behind a barrier, before a chunk's products.  Rows lie in LDS 16 dims (keys) at a time as 0 4 8 12 1 5 ..: one
// 16-byte read gives a lane what four instructions take from it; 68 floats apart, sixteen rows' reads cover the banks once.
// Later tokens see more keys: workgroups are taken from the step's end, in rounds of one for each compute unit, every second
// round backwards, so that the two that share a unit add up to the same length.
// 32 heads of 64 on 4, beside the form of plain multiply-adds before: a prompt of 1000 tokens 75 us against 493, of 2048 237 (73
// TFLOP/s) against 1756; without groups 84 against 942.
// Tokens of a workgroup that belong to different sequences are served one run of equal sequences after the other.
// C > 0: both head sizes are 16 C, a page holds a power of two of rows, 16 at least, cache and queries are aligned for loads of
// four, and scores have no cap: a chunk's sixteen rows a piece then lie on one page.  C = 0: everything else.
// KD: sixteens of dims that either head size has at most.
constexpr int kTiledCols = 64, kTiledWaves = 4, kRowStride = 68;
template <typename T, int C, int KD>
__global__ void __launch_bounds__(64 * kTiledWaves)
attention_generic_tiled_kernel(const T* __restrict__ q, const T* __restrict__ cache, const int* __restrict__ block_table,
                               int max_blocks, const int* __restrict__ token_seq, const int* __restrict__ positions,
                               T* __restrict__ out, int tokens, int nq, int nkv, int d, int dv, int page_size, int window,
                               int chunk, const float* __restrict__ sink, float scale, float softcap, int tokens_per_block, int heads_per_block, const int* __restrict__ seq_start, int min_tokens,
                               int vshare, int out_f32, int units) {
  __shared__ __attribute__((aligned(16))) float k_tile[2][64 * kRowStride];      // [key][dims]
  __shared__ __attribute__((aligned(16))) float v_tile[2][64 * kRowStride];      // [dim][keys]
  __shared__ int infinite[2];                      // the last chunk in this half of v_tile that held a value that is not finite
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int G = nq / nkv;
  const int round = blockIdx.x / units, in_round = blockIdx.x - round * units;
  const int place = round % 2 == 0 ? blockIdx.x : round * units + min(units, static_cast<int>(gridDim.x) - round * units) - 1 - in_round;
  const int kv_head = place % nkv, tok0 = ((static_cast<int>(gridDim.x) - 1 - place) / nkv) * tokens_per_block, head0 = blockIdx.z * heads_per_block;
  const int ntok = min(tokens_per_block, tokens - tok0), nheads = min(heads_per_block, G - head0);
  const int ncols = ntok * nheads;                 // column c = (token c / nheads, head c % nheads)
  // (vshare key heads in a row read one value head: a page then holds nkv planes of keys and nkv / vshare of values)
  const size_t page_stride = static_cast<size_t>(page_size) * (static_cast<size_t>(nkv) * d + static_cast<size_t>(nkv / vshare) * dv);
  const T* keys = cache + static_cast<size_t>(kv_head) * page_size * d;
  const T* values = cache + static_cast<size_t>(nkv) * page_size * d + static_cast<size_t>(kv_head / vshare) * page_size * dv;
  static_assert(C == 0 || C == KD, "known sizes");
    const int page_bits = 31 - __builtin_clz(page_size), in_page = page_size - 1;        // (where pages hold a power of two)
  const bool whole_bits = (page_size & in_page) == 0;
  // where key j lies: its page's place in the table, its row there
  auto page_at = [&](int j) { return whole_bits ? j >> page_bits : j / page_size; };
  auto row_in = [&](int j) { return whole_bits ? j & in_page : j % page_size; };
  // whole loads of four where rows allow them
  const bool aligned = C > 0 || ((reinterpret_cast<uintptr_t>(cache) % (4 * sizeof(T))) == 0 && (page_size & 3) == 0);
  const bool wide_k = aligned && (d & 3) == 0, wide_q = C > 0 || ((d & 3) == 0 && (reinterpret_cast<uintptr_t>(q) % (4 * sizeof(T))) == 0);
  if (threadIdx.x < 2) infinite[threadIdx.x] = -1;

  // this wave's columns
  const int column = wave * 16 + r;
  const int col_tok = column < ncols ? column / nheads : -1, col_head = kv_head * G + head0 + max(column, 0) % nheads;
  const int col_pos = col_tok >= 0 ? positions[tok0 + col_tok] : -1;
  int col_lo = window > 0 ? max(0, col_pos - window + 1) : 0;
  if (chunk > 0 && col_pos >= 0) col_lo = max(col_lo, col_pos - col_pos % chunk);
  float query[KD][4];                           // dims 16 c + 4 j + g
#pragma unroll
  for (int c = 0; c < KD; ++c) {
    row4(query[c], q + (static_cast<size_t>(tok0 + max(col_tok, 0)) * nq + col_head) * d, 16 * c + 4 * g, C > 0 ? 16 * C : (col_tok >= 0 ? d : 0), wide_q);
    to_quarters(query[c]);
  }
  ColumnState<KD> kept0, kept1, kept2, kept3;          // (not an array: the compiler would keep it in memory)

  int stamp = 0;                                   // chunks so far
  int run_first = 0;
  while (run_first < ntok) {                       // (the same for every thread: the barriers below are the workgroup's)
    const int seq = token_seq[tok0 + run_first];
    int run_end = run_first + 1;
    while (run_end < ntok && token_seq[tok0 + run_end] == seq) ++run_end;
    if (seq_start != nullptr && seq_start[seq + 1] - seq_start[seq] < min_tokens) {   // left to the kernel of few tokens (the same for every thread)
      run_first = run_end;
      continue;
    }
    // the keys the run's columns see: from the least lower bound to the last position; those that all of them see: from the
    // greatest lower bound to the first position
    int hi = -1, lo = 1 << 30, all_hi = 1 << 30, all_lo = 0;
    for (int t = run_first; t < run_end; ++t) {
      const int pos = positions[tok0 + t];
      int bound = window > 0 ? max(0, pos - window + 1) : 0;
      if (chunk > 0) bound = max(bound, pos - pos % chunk);
      hi = max(hi, pos), lo = min(lo, bound), all_hi = min(all_hi, pos), all_lo = max(all_lo, bound);
    }
    if (run_end - run_first < ntok) all_hi = -1;   // (columns of another run are in the same instructions)
    const bool mine = col_tok >= run_first && col_tok < run_end;
    const int my_pos = mine ? col_pos : -1;
    const int* pages = block_table + static_cast<size_t>(seq) * max_blocks;
    const int first = lo / 256 * 256, chunks = (hi - first) / 64 + 1;      // (chunk n of the walk belongs to state n % 4)

    float k_next[4][4], v_next[4][4];
    int page_of[4];                                // (C > 0) the pages of the sixteens of the chunk that is asked for next
    auto look_up = [&](int n) {
      if (C > 0) {
#pragma unroll
        for (int p = 0; p < 4; ++p) page_of[p] = pages[min(max(first + 64 * n + 16 * p, lo), hi) >> page_bits];
      }
    };
    auto ask = [&](int n) {                        // a thread brings four pieces of four of either
      const int start = first + 64 * n, piece = threadIdx.x & 15;
      if (C > 0) {
        // keys: rows tid / 16 of the four sixteens; values: the four keys of this thread's piece, of dims tid / 16 + 16 p.
        // What lies outside lo .. hi is read from within the same pages, and masked (keys) or set to zero (values).
        const int row = threadIdx.x >> 4;
        const int mine = piece >> 2, v_page = mine == 0 ? page_of[0] : (mine == 1 ? page_of[1] : (mine == 2 ? page_of[2] : page_of[3]));
        const int jv = start + 4 * piece;
        const T* v_at = values + static_cast<size_t>(v_page) * page_stride + (jv & in_page);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const int j = start + 16 * p + row;
          if (4 * piece < 16 * C) {
            const float4 f = load4(keys + static_cast<size_t>(page_of[p]) * page_stride + static_cast<size_t>(j & in_page) * (16 * C) + 4 * piece);
            k_next[p][0] = f.x, k_next[p][1] = f.y, k_next[p][2] = f.z, k_next[p][3] = f.w;
          }
          if (p < C) {
            const float4 f = load4(v_at + static_cast<size_t>(row + 16 * p) * page_size);
            v_next[p][0] = f.x, v_next[p][1] = f.y, v_next[p][2] = f.z, v_next[p][3] = f.w;
          }
        }
        return;
      }
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int row = (threadIdx.x >> 4) + 16 * p;
        const int j = min(max(start + row, lo), hi);                       // (a key outside is masked: any that was written will do)
        row4(k_next[p], keys + static_cast<size_t>(pages[page_at(j)]) * page_stride + static_cast<size_t>(row_in(j)) * d, 4 * piece, d, wide_k);
        if (p >= KD) continue;                     // (no dims there)
        const int jv = start + 4 * piece;          // keys jv .. jv + 3 of dim `row`
        if (aligned && jv >= lo && jv + 3 <= hi) {
          row4(v_next[p], values + static_cast<size_t>(pages[page_at(jv)]) * page_stride + static_cast<size_t>(row) * page_size + row_in(jv), 0, row < dv ? 4 : 0, true);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int je = jv + e;
            v_next[p][e] = row < dv && je >= lo && je <= hi
                ? to_float(values[static_cast<size_t>(pages[page_at(je)]) * page_stride + static_cast<size_t>(row) * page_size + row_in(je)]) : 0.f;
          }
        }
      }
    };
    auto put = [&](int n, int half) {
      const int start = first + 64 * n, piece = threadIdx.x & 15;
      const bool outside = start < lo || start + 63 > hi, partial = start < all_lo || start + 63 > all_hi;     // (uniform)
      bool odd = false;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int at = ((threadIdx.x >> 4) + 16 * p) * kRowStride + (piece >> 2) * 16 + (piece & 3);
        if (4 * piece < 16 * KD) {
#pragma unroll
          for (int e = 0; e < 4; ++e) k_tile[half][at + 4 * e] = k_next[p][e];
        }
        if (p < KD) {
          if (C > 0 && outside) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v_next[p][e] = start + 4 * piece + e >= lo && start + 4 * piece + e <= hi ? v_next[p][e] : 0.f;
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) v_tile[half][at + 4 * e] = v_next[p][e];
          if (partial) {
#pragma unroll
            for (int e = 0; e < 4; ++e) odd |= !(fabsf(v_next[p][e]) < INFINITY);
          }
        }
      }
      if (odd) infinite[half] = stamp + n;
    };
    __syncthreads();                               // (the run before is done with LDS; `infinite` is set)
    // state by state, the chunks of each in their order: n, n + 4, .., then the next state's (one copy of the code, and one
    // state in the works; the others wait in `kept`)
    auto after = [&](int n) { return n + 4 < chunks ? n + 4 : (n & 3) + 1 + ((n & 3) == 3 ? chunks : 0); };
    int n = 0, n1 = after(0), half = 0;            // this chunk, the next (chunks or more: none)
    look_up(0);
    ask(0);
    look_up(n1);
    put(0, 0);
    if (n1 < chunks) ask(n1);
    ColumnState<KD> own = kept0;
    while (n < chunks) {                           // (uniform)
      const int n2 = n1 < chunks ? after(n1) : n1;
      lds_barrier();                               // chunk n is whole, the one before has been read
      if (n1 < chunks) put(n1, half ^ 1);
      look_up(n2);
      if (n2 < chunks) ask(n2);
      const int start = first + 64 * n;
      if (!__all(my_pos < start || col_lo > start + 63)) {                 // (else no column of the wave sees it)
        floatx4 dot[4] = {};
        const float* key = k_tile[half] + r * kRowStride + 4 * g;
#pragma unroll
        for (int c = 0; c < KD; ++c) {
          if (16 * c >= d) break;                  // (dims past d are zeros)
          float4 a[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) a[t] = *reinterpret_cast<const float4*>(key + 16 * t * kRowStride + 16 * c);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int t = 0; t < 4; ++t) dot[t] = __builtin_amdgcn_mfma_f32_16x16x4f32((&a[t].x)[e], query[c][e], dot[t], 0, 0, 0);
        }
        take_scores<C == 0>(dot, own, start, col_lo, my_pos, g, scale, softcap);
        if (infinite[half] != stamp + n) {
          const float* value = v_tile[half] + r * kRowStride + 4 * g;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            float weight[4] = {dot[t][0], dot[t][1], dot[t][2], dot[t][3]};
            to_quarters(weight);
            float4 a[KD];
#pragma unroll
            for (int u = 0; u < KD; ++u) a[u] = *reinterpret_cast<const float4*>(value + 16 * u * kRowStride + 16 * t);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int u = 0; u < KD; ++u) own.acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32((&a[u].x)[e], weight[e], own.acc[u], 0, 0, 0);
          }
        } else {
          // a value that is not finite, among keys that some column must not see: zero times it would be no zero there, so every
          // column adds its own keys and no others, in the same order
#pragma unroll
          for (int t = 0; t < 4; ++t)
            for (int from = 0; from < 4; ++from)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int at = 16 * t + 4 * from + i, j = start + at;
                const float weight = __shfl(dot[t][i], 16 * from + r, 64);
                if (j < col_lo || j > my_pos) continue;
#pragma unroll
                for (int u = 0; u < KD; ++u)
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                    own.acc[u][e] = fmaf(weight, v_tile[half][(16 * u + 4 * g + e) * kRowStride + 16 * t + 4 * i + from], own.acc[u][e]);
              }
        }
      }
      if (n1 >= chunks || (n1 & 3) != (n & 3)) {   // the state's last chunk
        settle(own.acc);
        if ((n & 3) == 0) kept0 = own, own = kept1;
        else if ((n & 3) == 1) kept1 = own, own = kept2;
        else if ((n & 3) == 2) kept2 = own, own = kept3;
        else kept3 = own;
      }
      n = n1, n1 = n2, half ^= 1;
    }
    stamp += chunks;
    run_first = run_end;
  }
  if (col_tok < 0) return;
  if (seq_start != nullptr) {                      // a token of a sequence that brings few tokens is the other kernel's
    const int seq = token_seq[tok0 + col_tok];
    if (seq_start[seq + 1] - seq_start[seq] < min_tokens) return;
  }
  // the four states of a column into one, in their order
  float top = fmaxf(fmaxf(kept0.top, kept1.top), fmaxf(kept2.top, kept3.top)), total = 0.f;
  floatx4 result[KD] = {};
  if (sink != nullptr) {
    top = fmaxf(top, sink[col_head]);
    total = expf(sink[col_head] - top);
  }
  auto join = [&](const ColumnState<KD>& one) {
    if (one.top == -INFINITY) return;
    const float w = expf(one.top - top);
    total += w * one.sum;
#pragma unroll
    for (int u = 0; u < KD; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) result[u][e] += w * one.acc[u][e];
  };
  join(kept0);
  join(kept1);
  join(kept2);
  join(kept3);
  const size_t row = (static_cast<size_t>(tok0 + col_tok) * nq + col_head) * dv;
#pragma unroll
  for (int u = 0; u < KD; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int dim = 16 * u + 4 * g + e;
      if (dim < dv) store_result(out, row + dim, result[u][e] / total, out_f32);
    }
}

// ---- few tokens a sequence (decoding) ----
// A workgroup of four waves serves one token and up to 16 heads of one kv head; wave w takes the chunks of state w, with keys
// and values straight from the cache into registers (a lane asks for 16 bytes of a key or of a dim's row of values), the next
// chunk's asked for while this one's products run.  The kernel of one head a workgroup reads a key once for each of the heads that
// share it; what a chunk takes here (some 4 us) does not fall with the number of heads, so that kernel stays for steps of little
// work (the line is drawn where it is launched).  C as above, but never 0: with sizes that are not known beforehand it is the slower
// one throughout (64 tokens of 200 keys, 16 heads of 48 on 8: 36 us against 15).
template <typename T, int C>
__global__ void __launch_bounds__(256)
attention_generic_few_kernel(const T* __restrict__ q, const T* __restrict__ cache, const int* __restrict__ block_table,
                             int max_blocks, const int* __restrict__ token_seq, const int* __restrict__ positions,
                             T* __restrict__ out, int nq, int nkv, int d, int dv, int page_size, int window, int chunk,
                             const float* __restrict__ sink, float scale, float softcap,
                             const int* __restrict__ seq_start, int min_tokens, int vshare, int out_f32) {
  __shared__ __attribute__((aligned(16))) float states[4][16][68];        // [state][column][64 dims, maximum, sum]
  const int t0 = blockIdx.x, seq = token_seq[t0];
  if (seq_start != nullptr && seq_start[seq + 1] - seq_start[seq] >= min_tokens) return;      // (the same for the whole workgroup)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int G = nq / nkv, kv_head = blockIdx.y, head0 = blockIdx.z * 16, nheads = min(16, G - head0);
  const int pos = positions[t0];
  int lo = window > 0 ? max(0, pos - window + 1) : 0;
  if (chunk > 0) lo = max(lo, pos - pos % chunk);
  const int* pages = block_table + static_cast<size_t>(seq) * max_blocks;
  const size_t page_stride = static_cast<size_t>(page_size) * (static_cast<size_t>(nkv) * d + static_cast<size_t>(nkv / vshare) * dv);
  const T* keys = cache + static_cast<size_t>(kv_head) * page_size * d;
  const T* values = cache + static_cast<size_t>(nkv) * page_size * d + static_cast<size_t>(kv_head / vshare) * page_size * dv;
  const int page_bits = 31 - __builtin_clz(page_size), in_page = page_size - 1;
  float query[C][4];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    row4(query[c], q + (static_cast<size_t>(t0) * nq + kv_head * G + head0 + min(r, nheads - 1)) * d, 16 * c + 4 * g, 16 * C, true);
    to_quarters(query[c]);
  }
  const int first = lo / 256 * 256 + 64 * wave;
  float k_next[4][C][4], v_next[4][C][4];
  int page_of[4];                                  // the pages of the four sixteens of the chunk that is asked for next
  auto look_up = [&](int start) {
#pragma unroll
    for (int t = 0; t < 4; ++t) page_of[t] = pages[min(max(start + 16 * t, lo), pos) >> page_bits];
  };
  auto ask_keys = [&](int start) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const T* row = keys + static_cast<size_t>(page_of[t]) * page_stride + static_cast<size_t>((start + 16 * t + r) & in_page) * (16 * C);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const float4 f = load4(row + 16 * c + 4 * g);
        k_next[t][c][0] = f.x, k_next[t][c][1] = f.y, k_next[t][c][2] = f.z, k_next[t][c][3] = f.w;
      }
    }
  };
  // (a value outside lo .. pos counts as zero: `hide` sets it to zero before it is used)
  auto ask_values = [&](int start) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int jv = start + 16 * t + 4 * g;
      const T* at = values + static_cast<size_t>(page_of[t]) * page_stride + static_cast<size_t>(r) * page_size + (jv & in_page);
#pragma unroll
      for (int u = 0; u < C; ++u) {
        const float4 f = load4(at + static_cast<size_t>(16 * u) * page_size);
        v_next[t][u][0] = f.x, v_next[t][u][1] = f.y, v_next[t][u][2] = f.z, v_next[t][u][3] = f.w;
      }
    }
  };
  auto hide = [&](int start) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int u = 0; u < C; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = start + 16 * t + 4 * g + e;
          v_next[t][u][e] = j >= lo && j <= pos ? v_next[t][u][e] : 0.f;
        }
  };
  ColumnState<C> state;
  if (first <= pos) {
    look_up(first);
    ask_keys(first);
    ask_values(first);
    look_up(first + 256);
  }
  for (int start = first; start <= pos; start += 256) {
    const bool more = start + 256 <= pos, partial = start < lo || start + 63 > pos;      // (uniform)
    floatx4 dot[4] = {};
#pragma unroll
    for (int c = 0; c < C; ++c) {
#pragma unroll
      for (int t = 0; t < 4; ++t) to_quarters(k_next[t][c]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < 4; ++t) dot[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k_next[t][c][e], query[c][e], dot[t], 0, 0, 0);
    }
    if (more) ask_keys(start + 256);
    take_scores<false>(dot, state, start, lo, pos, g, scale, softcap);
    if (partial) hide(start);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float weight[4] = {dot[t][0], dot[t][1], dot[t][2], dot[t][3]};
      to_quarters(weight);
#pragma unroll
      for (int u = 0; u < C; ++u) to_quarters(v_next[t][u]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int u = 0; u < C; ++u) state.acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(v_next[t][u][e], weight[e], state.acc[u], 0, 0, 0);
    }
    if (more) {
      ask_values(start + 256);
      look_up(start + 512);
    }
  }
  settle(state.acc);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < C; ++u)
    *reinterpret_cast<float4*>(&states[wave][r][16 * u + 4 * g]) = make_float4(state.acc[u][0], state.acc[u][1], state.acc[u][2], state.acc[u][3]);
  if (g == 0) states[wave][r][64] = state.top, states[wave][r][65] = state.sum;
  __syncthreads();
  // the four states into one, in their order: a wave a column, a lane a dim
  for (int column = wave; column < nheads; column += 4) {
    const int head = kv_head * G + head0 + column;
    float top = -INFINITY;
#pragma unroll
    for (int s = 0; s < 4; ++s) top = fmaxf(top, states[s][column][64]);
    float total = 0.f, result = 0.f;
    if (sink != nullptr) {                         // the sink counts once: exp(sink) in the denominator, nothing in the sum of values
      top = fmaxf(top, sink[head]);
      total = expf(sink[head] - top);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float m = states[s][column][64];
      if (m == -INFINITY) continue;                // a state that saw no key
      const float w = expf(m - top);
      total += w * states[s][column][65];
      result += w * states[s][column][lane];
    }
    if (lane < dv) store_result(out, (static_cast<size_t>(t0) * nq + head) * dv + lane, result / total, out_f32);
  }
}

}  // namespace tlie

using namespace tlie;

extern "C" int tlie_attention_generic(const void* q, const void* cache, int dtype, const int* block_table,
                                      int max_blocks, const int* token_seq, const int* positions, void* out,
                                      int tokens, int nq, int nkv, int d, int dv, int page_size, int window, int chunk,
                                      const float* sink, float scale, int tiled, int tile_tokens, const int* seq_start, int min_tokens,
                                      int vshare, int out_f32, float softcap, int compute_units, void* stream) {
  // tiled 0: the kernel of one (token, head) a workgroup; 1: the kernel that shares keys among a
  // sequence's tokens (head sizes up to 64); 2: both, each token served by one of them: the second
  // takes the sequences that bring min_tokens tokens or more (seq_start: int32 [sequences + 1], the
  // step's cumulative token counts), the first the others.  A token gets the same bits from either.
  // tile_tokens: at most so many tokens a workgroup of the second (0: as many as its 64 columns hold).  It serves the sequences
  // that its tokens belong to one after the other, so where they bring few tokens each, a workgroup of one sequence ends the
  // sooner: 16 sequences of 32 tokens behind 200, 16 heads of 20, 33 us with 32 tokens a workgroup against 59 with 64.
  // (d only bounds the length of a dot product; dv is served by one thread a dim of a group of at most 256)
  if (tokens <= 0 || nq <= 0 || nkv <= 0 || nq % nkv != 0 || d <= 0 || d > 4096 || dv <= 0 || dv > 256 || page_size <= 0 ||
      max_blocks <= 0 || chunk < 0 || compute_units <= 0 || vshare <= 0 || nkv % vshare != 0 || softcap < 0.f)
    return kBadArgument;
  if (tiled < 0 || tiled > 2 || (tiled == 2 && (seq_start == nullptr || min_tokens < 1))) return kBadArgument;
  if (dtype != kF32 && dtype != kBF16) return kBadArgument;
  if (d > 64 || dv > 64) tiled = 0;
  const int* select = tiled == 2 ? seq_start : nullptr;
  // sixteens of dims where the kernels for head sizes up to 64 know the sizes beforehand (see there), else 0
  const bool known = d == dv && d % 16 == 0 && d <= 64 && page_size >= 16 && (page_size & (page_size - 1)) == 0 &&
                     (reinterpret_cast<uintptr_t>(cache) | reinterpret_cast<uintptr_t>(q)) % (dtype == kF32 ? 16 : 8) == 0 && softcap == 0.f;
  const int sixteens = known && d != 48 ? d / 16 : 0;
#define TLIE_BY_TYPE(LAUNCH, C, KD) \
  { if (dtype == kF32) LAUNCH(float, C, KD); else LAUNCH(bf16, C, KD); }
  if (tiled) {
    // (the same bits as the kernel below, for steps whose sequences bring several tokens each)
    const int G = nq / nkv;
    const int heads_per_block = G < kTiledCols ? G : kTiledCols;
    int tokens_per_block = kTiledCols / heads_per_block;
    const int least = (16 + heads_per_block - 1) / heads_per_block;                // (a wave's columns)
    if (tile_tokens > 0) tokens_per_block = tile_tokens >= tokens_per_block ? tokens_per_block : (tile_tokens > least ? tile_tokens : least);
    const long long blocks = static_cast<long long>((tokens + tokens_per_block - 1) / tokens_per_block) * nkv;
    if (blocks > 0x7fffffff) return kBadArgument;
    const dim3 grid(static_cast<unsigned>(blocks), 1, (G + heads_per_block - 1) / heads_per_block);
    const int widest = d > dv ? d : dv;
#define TLIE_TILED(T, C, KD)                                                                                                   \
  hipLaunchKernelGGL((attention_generic_tiled_kernel<T, C, KD>), grid, dim3(64 * kTiledWaves), 0, (hipStream_t)stream, (const T*)q,      \
                     (const T*)cache, block_table, max_blocks, token_seq, positions, (T*)out, tokens, nq, nkv, d, dv, page_size,      \
                     window, chunk, sink, scale, softcap, tokens_per_block, heads_per_block, select, min_tokens, vshare, out_f32, compute_units)
    if (sixteens == 1) TLIE_BY_TYPE(TLIE_TILED, 1, 1)
    else if (sixteens == 2) TLIE_BY_TYPE(TLIE_TILED, 2, 2)
    else if (sixteens == 4) TLIE_BY_TYPE(TLIE_TILED, 4, 4)
    else if (widest <= 16) TLIE_BY_TYPE(TLIE_TILED, 0, 1)
    else if (widest <= 32) TLIE_BY_TYPE(TLIE_TILED, 0, 2)
    else if (widest <= 48) TLIE_BY_TYPE(TLIE_TILED, 0, 3)
    else TLIE_BY_TYPE(TLIE_TILED, 0, 4)
#undef TLIE_TILED
    const int status = launch_status();
    if (status != kOk || tiled == 1) return status;
  }
  // Known sizes: the kernel that serves a kv head's query heads together, where they are several and the step has work for four
  // workgroups a compute unit in the kernel of one head each (64 tokens of 500 keys, 32 heads on 4: 17.4 us against
  // 54; 8 tokens of 100 keys 9.0 against 6.7; 64 tokens of 500 keys, 32 heads on 32: 144 against 116).  A single chunk of keys
  // takes it longer (48 tokens of 3 keys, 32 heads on 4: 9.6 us against 8.7), so that where no sequence has more, it wants
  // sixteen a unit.
  const long long enough = static_cast<long long>(max_blocks) * page_size <= 64 ? 16LL * compute_units : 4LL * compute_units;
  if (sixteens > 0 && nq / nkv >= 2 && static_cast<long long>(tokens) * nq >= enough) {
    const dim3 grid(tokens, nkv, (nq / nkv + 15) / 16);
    if (grid.y > 65535 || grid.z > 65535) return kBadArgument;
#define TLIE_FEW(T, C, KD)                                                                                                         \
  hipLaunchKernelGGL((attention_generic_few_kernel<T, C>), grid, dim3(256), 0, (hipStream_t)stream, (const T*)q, (const T*)cache,    \
                     block_table, max_blocks, token_seq, positions, (T*)out, nq, nkv, d, dv, page_size, window, chunk, sink, scale,  \
                     softcap, select, min_tokens, vshare, out_f32)
    if (sixteens == 1) TLIE_BY_TYPE(TLIE_FEW, 1, 1)
    else if (sixteens == 2) TLIE_BY_TYPE(TLIE_FEW, 2, 2)
    else TLIE_BY_TYPE(TLIE_FEW, 4, 4)
#undef TLIE_FEW
    return launch_status();
  }
  // keys a group of threads takes in one turn: the least of 64, 128, 256 that holds both head sizes (beyond 256 dims of
  // a key: 256)
  const int widest = d > dv ? d : dv;
  const int keys = widest <= 64 ? 64 : (widest <= 128 ? 128 : 256);
  const int groups = 256 / keys;
  const size_t lds = (static_cast<size_t>(d) + 256 + 4 + 2 * groups + static_cast<size_t>(groups) * dv) * sizeof(float);
  if (lds > 64 * 1024) return kBadArgument;
  hipStream_t s = (hipStream_t)stream;
#define TLIE_LAUNCH(T, CHUNK)                                                                                         \
  hipLaunchKernelGGL((attention_generic_kernel<T, CHUNK>), dim3(tokens, nq), dim3(256), lds, s, (const T*)q,           \
                     (const T*)cache, block_table, max_blocks, token_seq, positions, (T*)out, nq, nkv, d, dv, page_size, \
                     window, chunk, sink, scale, softcap, select, min_tokens, vshare, out_f32)
  if (dtype == kF32) {
    if (keys == 64) TLIE_LAUNCH(float, 64); else if (keys == 128) TLIE_LAUNCH(float, 128); else TLIE_LAUNCH(float, 256);
  } else if (dtype == kBF16) {
    if (keys == 64) TLIE_LAUNCH(bf16, 64); else if (keys == 128) TLIE_LAUNCH(bf16, 128); else TLIE_LAUNCH(bf16, 256);
  }
  else
    return kBadArgument;
#undef TLIE_LAUNCH
#undef TLIE_BY_TYPE
  return launch_status();
}
