// Routing of one token by one wave, and the workgroup scan the dispatch orders use.
#pragma once

#include "common.hpp"

namespace anna {

// LDS scratch route_token needs per wave, in floats
__host__ __device__ constexpr int route_scratch(int64_t E) { return (int)((E + 3) / 4 * 4) + 128; }

// Softmax over the E logits of token t and its top_k (ties to the lower expert index), by one
// wave; lane l holds experts l, l + 64, ...  Lane j < top_k returns route j's weight (normalized
// over the top_k when asked) and expert.  The top_k is found by rank, not by k rounds of a
// cross-lane argmax: the probabilities go to the wave's LDS scratch sp (route_scratch(E)
// floats), every lane counts for each of its experts how many experts beat it (a larger
// probability, or an equal one at a lower index), and an expert of rank j < top_k is route j.
// Every logit row gives top_k different experts: a row with a NaN or +inf logit, whose
// probabilities are all NaN, ranks each of them as -1 (below every probability, ties by index) and
// returns NaN weights, so that it spoils its own token only.
// MAXV: experts per lane, E <= 64 MAXV (instantiated for E <= 64, 128, 256 and 1024).
template <int LDT, int MAXV>
__device__ __forceinline__ void route_token(const typename Elem<LDT>::T* __restrict__ logits, int64_t t, int64_t E,
                                            int64_t ls, int64_t top_k, int normalize, int lane, float* sp,
                                            float& w_out, int64_t& e_out) {
  float v[MAXV];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int64_t e = lane + 64 * i;
    v[i] = e < E ? Elem<LDT>::load(logits, t * ls + e) : -INFINITY;
    mx = fmaxf(mx, v[i]);
  }
  mx = wave_max(mx);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int64_t e = lane + 64 * i;
    v[i] = e < E ? expf(v[i] - mx) : 0.f;
    s += v[i];
  }
  const float inv = 1.0f / wave_sum(s);
  const int E4 = (int)((E + 3) / 4 * 4);
  float* stp = sp + E4;                 // route j's probability
  int* ste = (int*)(sp + E4 + 64);      // route j's expert
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int e = lane + 64 * i;
    const float p = v[i] * inv;
    if (e < E) sp[e] = p == p ? p : -1.0f;
    else if (e < E4) sp[e] = -2.0f;     // padding: beats nothing, ties nothing
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (int e = lane; e < E; e += 64) {
    const float p = sp[e];
    int rank = 0;
    for (int j = 0; j < E4; j += 4) {
      const float4 q = *(const float4*)(sp + j);
      rank += (q.x > p || (q.x == p && j < e)) + (q.y > p || (q.y == p && j + 1 < e)) +
              (q.z > p || (q.z == p && j + 2 < e)) + (q.w > p || (q.w == p && j + 3 < e));
    }
    if (rank < top_k) {
      stp[rank] = p < 0.f ? __builtin_nanf("") : p;
      ste[rank] = e;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float top_sum = 0.f;  // in route order (descending), as the k rounds of argmax summed them
  for (int64_t j = 0; j < top_k; ++j) top_sum += stp[j];
  const float scale = normalize && top_sum > 0.f ? 1.0f / top_sum : 1.0f;
  w_out = lane < top_k ? stp[lane] * scale : 0.f;
  e_out = lane < top_k ? ste[lane] : 0;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();  // sp is reused by the wave's next token
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Experts per lane for E experts (the route_token instantiations).
inline int route_maxv(int64_t E) { return E <= 64 ? 1 : E <= 128 ? 2 : E <= 256 ? 4 : 16; }
#define ANNA_DISPATCH_MAXV(E, NAME, ...)                                  \
  switch (route_maxv(E)) {                                                \
    case 1: { constexpr int NAME = 1; __VA_ARGS__; break; }               \
    case 2: { constexpr int NAME = 2; __VA_ARGS__; break; }               \
    case 4: { constexpr int NAME = 4; __VA_ARGS__; break; }               \
    default: { constexpr int NAME = 16; __VA_ARGS__; break; }             \
  }

// Exclusive prefix sum of v over the 1024 threads of a workgroup (s: 16 ints of LDS); *total
// receives the sum.
__device__ __forceinline__ int block_exclusive_scan(int v, int* s, int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(inc, off, 64);
    if (lane >= off) inc += o;
  }
  if (lane == 63) s[wave] = inc;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    before += w < wave ? s[w] : 0;
    all += s[w];
  }
  __syncthreads();  // s may be reused by the caller
  *total = all;
  return before + inc - v;
}

}  // namespace anna
