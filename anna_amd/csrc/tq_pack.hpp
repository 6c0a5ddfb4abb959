// Packing of TurboQuant codes into cache rows, shared by the quantizers and the cache writers.
#pragma once

#include <math.h>

#include "common.hpp"

namespace anna {

__host__ __device__ inline int storage_bits(int bits) { return bits == 2 ? 2 : 4; }

// The E codes of every lane of a wave (lane l: elements l*E ..), sb bits each, packed in element
// order into dst (D * sb / 8 bytes).  The whole wave takes part (sub-byte lanes combine by shuffles).
template <int E>
__device__ __forceinline__ void store_codes_wave(const uint32_t (&code)[E], int sb, uint8_t* dst, int lane) {
  const int nbits = E * sb;
  uint64_t pk = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) pk |= (uint64_t)code[e] << (sb * e);
  if (nbits == 8) {
    dst[lane] = (uint8_t)pk;
  } else if (nbits == 16) {
    ((uint16_t*)dst)[lane] = (uint16_t)pk;
  } else if (nbits > 8) {
    for (int k = 0; k < nbits / 8; ++k) dst[lane * (nbits / 8) + k] = (uint8_t)(pk >> (8 * k));
  } else {
    const int per = 8 / nbits;  // lanes per byte
    uint32_t b = (uint32_t)pk << (nbits * (lane % per));
    for (int m = 1; m < per; m <<= 1) b |= (uint32_t)__shfl_xor((int)b, m, 64);
    if (lane % per == 0) dst[lane / per] = (uint8_t)b;
  }
}

// Groups g0 .. g0 + gpt - 1 of one vector (`src`, D elements): min/max, scale and zero point
// (rounded to the value dtype), codes packed into `data` (the vector's packed row).  The run
// ends on a packed-byte boundary, so runs of one vector can be done by different threads.
template <int DT>
__device__ void quantize_value_run(const typename Elem<DT>::T* __restrict__ src, int64_t D, int bits, int64_t gsz,
                                   int64_t g0, int64_t gpt, uint8_t* __restrict__ data,
                                   typename Elem<DT>::T* __restrict__ scales, typename Elem<DT>::T* __restrict__ zeros) {
  const float levels = (float)((1 << bits) - 1);
  const int sb = storage_bits(bits), per = 8 / sb;
  uint32_t byte = 0;
  for (int64_t g = g0; g < g0 + gpt; ++g) {
    float vmin = INFINITY, vmax = -INFINITY;
    for (int64_t j = 0; j < gsz; ++j) {
      const float f = Elem<DT>::to_f32(src[g * gsz + j]);
      vmin = fminf(vmin, f);
      vmax = fmaxf(vmax, f);
    }
    float sc = __fdiv_rn(__fsub_rn(vmax, vmin), levels);
    sc = sc < 1e-8f ? 1e-8f : sc;
    const typename Elem<DT>::T sc_s = Elem<DT>::cvt(sc), z_s = Elem<DT>::cvt(vmin);
    scales[g] = sc_s;
    zeros[g] = z_s;
    const float scf = Elem<DT>::to_f32(sc_s), zf = Elem<DT>::to_f32(z_s);
    for (int64_t j = 0; j < gsz; ++j) {
      const int64_t d = g * gsz + j;
      float q = rintf(__fdiv_rn(__fsub_rn(Elem<DT>::to_f32(src[d]), zf), scf));
      q = fminf(fmaxf(q, 0.f), levels);
      byte |= (uint32_t)q << (sb * (d % per));
      if (d % per == per - 1) {
        data[d / per] = (uint8_t)byte;
        byte = 0;
      }
    }
  }
}

// Groups per run: 1 when a group fills whole packed bytes, else the whole vector.
__host__ __device__ inline int64_t value_groups_per_run(int bits, int64_t D, int64_t gsz) {
  return gsz % (8 / storage_bits(bits)) == 0 ? 1 : D / gsz;
}

}  // namespace anna
