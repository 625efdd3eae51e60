// Column sums over an example's rows of output gradients: the per-example
// bias gradient sum_t G_i[t, m].  The norm pass (gram.hip) and the clipped sum
// (gemm.hip) both take them from this routine, so the value whose norm is
// measured is the value that is summed, bit for bit.
//
// A workgroup sums 128 columns: the rows are dealt to row groups (group r
// takes rows r, r + R, ...; R = 32 for bf16 and 16 for fp32 with 16-byte
// loads, 8 where rows are not 16-byte aligned), each group adds its rows in
// order in fp32, and the groups' sums are added in order through LDS.  The
// sums are memory-bound; one thread per column walking all T rows, as before,
// kept one 2-byte load in flight per lane: [24, 197, 3072] bf16 took 574 us
// in the norm pass and 48 us in the clipped sum (now 7.3 and 7.0, 4.1 TB/s).
#pragma once

#include "common.h"

constexpr int kBiasThreads = 512;
constexpr int kBiasCols = 128;
constexpr int kBiasSlots = 32;  // partial squared norms kept per example
constexpr int kBiasRedFloats = 32 * kBiasCols;

template <typename In>
DPC_DEVICE void bias_chunk_f32(u32x4_t c, float* v) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t w = c[k];
    if constexpr (sizeof(In) == 2) {
      v[2 * k] = __builtin_bit_cast(float, w << 16);
      v[2 * k + 1] = __builtin_bit_cast(float, w & 0xffff0000u);
    } else {
      v[k] = __builtin_bit_cast(float, w);
    }
  }
}

// Sum over t < T of g[t * dout + c0 + tid] in threads tid < kBiasCols (0 past
// the last column); called by all kBiasThreads threads.  red: kBiasRedFloats
// floats of LDS.
template <typename In>
DPC_DEVICE float bias_column_sum(const In* g, int T, int dout, int c0, float* red) {
  constexpr int V = 16 / (int)sizeof(In);
  constexpr int kLanes = kBiasCols / V;
  constexpr int kGroups = kBiasThreads / kLanes;
  const int tid = threadIdx.x;
  int groups;
  if (dout % V == 0 && (reinterpret_cast<uintptr_t>(g) & 15) == 0) {
    groups = kGroups;
    const int rg = tid / kLanes, cl = V * (tid % kLanes);
    float s[V];
#pragma unroll
    for (int k = 0; k < V; ++k) s[k] = 0.0f;
    if (c0 + cl < dout) {
      const In* p = g + c0 + cl;
      constexpr int kAhead = 4;
      int t = rg;
      for (; t + (kAhead - 1) * kGroups < T; t += kAhead * kGroups) {
        u32x4_t c[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
          c[j] = *global_ptr<const u32x4_t>(p + (size_t)(t + j * kGroups) * dout);
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
          float v[V];
          bias_chunk_f32<In>(c[j], v);
#pragma unroll
          for (int k = 0; k < V; ++k) s[k] += v[k];
        }
      }
      for (; t < T; t += kGroups) {
        float v[V];
        bias_chunk_f32<In>(*global_ptr<const u32x4_t>(p + (size_t)t * dout), v);
#pragma unroll
        for (int k = 0; k < V; ++k) s[k] += v[k];
      }
    }
#pragma unroll
    for (int k = 0; k < V; ++k) red[rg * kBiasCols + cl + k] = s[k];
  } else {
    groups = kBiasThreads / 64;
    const int rg = tid >> 6, cl = tid & 63;
    float s[2] = {0.0f, 0.0f};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = c0 + cl + 64 * h;
      if (c < dout) {
#pragma unroll 8
        for (int t = rg; t < T; t += kBiasThreads / 64) {
          const In x = global_ptr<const In>(g + c)[(size_t)t * dout];
          if constexpr (sizeof(In) == 2)
            s[h] += bf16_bits_to_f32(x);
          else
            s[h] += x;
        }
      }
      red[rg * kBiasCols + cl + 64 * h] = s[h];
    }
  }
  __syncthreads();
  float col = 0.0f;
  if (tid < kBiasCols)
    for (int r = 0; r < groups; ++r) col += red[r * kBiasCols + tid];
  __syncthreads();
  return col;
}
