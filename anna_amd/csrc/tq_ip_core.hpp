// Building blocks of the TurboQuant inner-product quantizer (definition and arithmetic order in
// tq_ip.hip), shared by the quantizers on flat vectors and by the cache writer.
//
// The two D x D products of a tile of TV vectors (rho . G^T for the signs, signs . G for the
// reconstruction) run on the fp32 matrix instruction: v_mfma_f32_16x16x4_f32 adds its four k as
// one fma chain in ascending k from the accumulator, subnormals and overflow included (compared
// bit by bit with the scalar chain on this chip), so the order the oracle fixes is kept while the
// matrix is read once per 16 to 64 vectors instead of once per 4, and at twice the rate that
// scalar fp32 fma issues at (154 TFLOP/s against 77).
#pragma once

#include "common.hpp"
#include "tq_hadamard.hpp"

namespace anna {

constexpr int IP_WAVES = 8;  // waves of a workgroup of the tile kernels

// Vectors of a tile: few calls' worth of vectors take tiles of 16, which spread over the chip and hold
// the matrices in registers; larger calls take tiles that read the matrices less often and leave two
// workgroups to a compute unit (D = 256: 32 against 64 vectors is 126 against 125 us at 32,256
// vectors and 65 against 71 at 15,104).
constexpr int ip_tile(int E, bool small) { return small || E >= 16 ? 16 : E >= 4 ? 32 : 64; }
// Tiles of 16 while one compute unit gets at most two of them.
inline bool ip_small_tiles(int64_t vectors) { return vectors <= 256 * 32; }
// LDS row of a tile: 4 floats of padding put the 16 rows x 4 chunks of an operand read on distinct banks
template <int E> constexpr int IP_ROW = 64 * E + 4;
template <int E> constexpr size_t ip_lds_bytes(int TV) { return (size_t)TV * IP_ROW<E> * 4; }

// Position of k in a row of the product's left operand: the four k of one instruction go to the
// four 16-lane groups, so groups of 16 k are transposed and one 16-byte read feeds four of them.
__device__ __forceinline__ int ip_pos(int k) { return (k & ~15) | ((k & 3) << 2) | ((k >> 2) & 3); }

// y = fl(1/sqrt(D)) * FWHT(s .* x), as the TQ-MSE quantizer forms it
template <int NV, int E>
__device__ __forceinline__ void rotate_wave_n(const float (&x)[NV][E], const float* __restrict__ signs, float inv,
                                              float (&y)[NV][E]) {
  const int lane = threadIdx.x & 63;
  float sg[E];
#pragma unroll
  for (int e = 0; e < E; ++e) sg[e] = signs[lane * E + e];
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int e = 0; e < E; ++e) y[n][e] = x[n][e] * sg[e];
  fwht_wave_n<NV, E>(y);
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int e = 0; e < E; ++e) y[n][e] = y[n][e] * inv;
}

// The centroid of a code: lane l < 16 of `table` holds centroid l (a gather from memory per element
// waited for the caches twice per vector).
__device__ __forceinline__ float ip_centroid_table(const float* __restrict__ cent, int bits) {
  return cent[threadIdx.x & ((1 << (bits - 1)) - 1)];
}
__device__ __forceinline__ float ip_centroid(float table, uint32_t code) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute((int)(code << 2), __float_as_int(table)));
}

// MSE stage of NV vectors of the wave (lane's E elements each): codes, norms, the rotated residual
// and residual_norm = |rho| / norm.
template <int NV, int E>
__device__ __forceinline__ void ip_mse_stage(const float (&x)[NV][E], const float* __restrict__ signs,
                                             const float* __restrict__ thr, float ctab, int nthr,
                                             uint32_t (&code)[NV][E], float (&nrm)[NV], float (&rho)[NV][E],
                                             float (&rn)[NV]) {
  float ss[NV];
  sumsq_wave_n<NV, E>(x, ss);
#pragma unroll
  for (int n = 0; n < NV; ++n) nrm[n] = __builtin_sqrtf(ss[n]);
  float y[NV][E];
  rotate_wave_n<NV, E>(x, signs, tq_inv_sqrt(64 * E), y);
  count_thresholds_n<NV, E>(y, thr, nthr, nrm, code);
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int e = 0; e < E; ++e) rho[n][e] = __builtin_fmaf(-ip_centroid(ctab, code[n][e]), nrm[n], y[n][e]);
  float gg[NV];
  sumsq_wave_n<NV, E>(rho, gg);
#pragma unroll
  for (int n = 0; n < NV; ++n) rn[n] = nrm[n] > 0.f ? __fdiv_rn(__builtin_sqrtf(gg[n]), nrm[n]) : 0.f;
}

// The E bytes of a lane (elements lane * E ..) at dst + lane * E, dst 64 * E-byte rows
template <int E>
__device__ __forceinline__ void store_bytes_wave(const uint32_t (&v)[E], uint8_t* dst, int lane) {
  if constexpr (E == 1) {
    dst[lane] = (uint8_t)v[0];
  } else if constexpr (E == 2) {
    ((uint16_t*)dst)[lane] = (uint16_t)(v[0] | (v[1] << 8));
  } else {
#pragma unroll
    for (int e = 0; e < E; e += 4)
      ((uint32_t*)dst)[lane * (E / 4) + e / 4] = v[e] | (v[e + 1] << 8) | (v[e + 2] << 16) | (v[e + 3] << 24);
  }
}

// A wave's CT column tiles of the product cover columns 16 CT wave .. + 16 CT, column r of tile c
// being 16 CT wave + CT r + c: a lane's elements of a matrix row are then CT consecutive floats, and
// 16 lanes read a whole 128-byte line from CT = 2 on.  (With D = 64 only the first four waves have
// a tile.)
template <int E> constexpr int IP_CT = E >= 2 ? E / 2 : 1;
template <int E>
__device__ __forceinline__ bool ip_has_tile(int wave) { return E >= 2 || wave < 4; }
template <int E>
__device__ __forceinline__ int ip_col(int wave, int c, int r) { return (wave * 16 + r) * IP_CT<E> + c; }
// W consecutive floats of a matrix row
template <int W>
__device__ __forceinline__ void ip_load_row(const float* p, float (&b)[W]) {
  typedef float FV __attribute__((ext_vector_type(W)));
  if constexpr (W == 1) {
    b[0] = *p;
  } else {
    const FV v = *(const FV*)p;
#pragma unroll
    for (int i = 0; i < W; ++i) b[i] = v[i];
  }
}

// The matrix elements one wave's lanes need for its column tiles, all k.  A tile of 16 vectors does
// too little with each element to hide its latency behind the products (a decode step's matrices
// often come from beyond the L2: 45 us a call at D = 256 with 32 k in flight), so it loads
// the first matrix whole at the start of the kernel and the second one during the first product.
// 512 threads then hold 128 registers of it at D = 256; larger D keep the loop below.
template <int E> constexpr bool IP_WHOLE = E <= 4;
template <int E>
struct IpMatrix {
  float b[16 * E][IP_CT<E>];
  __device__ __forceinline__ void load(const float* __restrict__ M, int wave) {
    constexpr int D = 64 * E;
    const int lane = threadIdx.x & 63;
    if (!ip_has_tile<E>(wave)) wave = 0;  // (loaded and not used)
    const float* p = M + (lane >> 4) * D + ip_col<E>(wave, 0, lane & 15);
#pragma unroll
    for (int s = 0; s < 16 * E; ++s) ip_load_row(p + 4 * s * D, b[s]);
  }
};
template <int E>
__device__ __forceinline__ void ip_product_whole(const IpMatrix<E>& m, const float* lds, f32x4 (&acc)[IP_CT<E>][1]) {
  const int lane = threadIdx.x & 63;
  const float* arow = lds + (lane & 15) * IP_ROW<E> + 4 * (lane >> 4);
#pragma unroll
  for (int c = 0; c < IP_CT<E>; ++c) acc[c][0] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < 4 * E; ++kk) {
    const f32x4 a = *(const f32x4*)(arow + 16 * kk);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int c = 0; c < IP_CT<E>; ++c)
        acc[c][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], m.b[4 * kk + s][c], acc[c][0], 0, 0, 0);
  }
}

// acc[c][n]: rows 16 n .. of `lds` (ip_pos order) times M (row-major D x D, k = row), column tile c
// of this wave, each element one fma chain over k ascending from 0.  C layout: column
// ip_col of lane & 15, rows 4 (lane >> 4) + e.
template <int E, int NT>
__device__ __forceinline__ void ip_product(const float* __restrict__ M, const float* lds, int wave,
                                           f32x4 (&acc)[IP_CT<E>][NT]) {
  constexpr int D = 64 * E, CT = IP_CT<E>;
  constexpr int CG = CT < 2 ? 1 : 2;  // column tiles together: one read of the left operand feeds both
  constexpr int KU = 32;  // k per step: the next step's matrix elements are in flight during this one
  const int lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4;
  const float* arow = lds + r * IP_ROW<E> + 4 * kq;
#pragma unroll
  for (int c0 = 0; c0 < CT; c0 += CG) {
    const float* bcol = M + kq * D + ip_col<E>(wave, c0, r);
    float b[KU / 4][CG], bn[KU / 4][CG];
#pragma unroll
    for (int c = 0; c < CG; ++c)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[c0 + c][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KU / 4; ++s) ip_load_row(bcol + 4 * s * D, b[s]);
#pragma unroll 1
    for (int k0 = 0; k0 < D; k0 += KU) {
      const int kn = k0 + KU < D ? k0 + KU : k0;  // (the last step reloads itself)
#pragma unroll
      for (int s = 0; s < KU / 4; ++s) ip_load_row(bcol + (kn + 4 * s) * D, bn[s]);
#pragma unroll
      for (int kk = 0; kk < KU; kk += 16) {
        f32x4 a[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) a[n] = *(const f32x4*)(arow + n * 16 * IP_ROW<E> + k0 + kk);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int c = 0; c < CG; ++c)
#pragma unroll
            for (int n = 0; n < NT; ++n)
              acc[c0 + c][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[n][s], b[kk / 4 + s][c], acc[c0 + c][n], 0, 0, 0);
      }
#pragma unroll
      for (int s = 0; s < KU / 4; ++s)
#pragma unroll
        for (int c = 0; c < CG; ++c) b[s][c] = bn[s][c];
    }
  }
}

// Whether a tile of TV vectors holds its matrices whole
template <int E, int TV> constexpr bool ip_whole() { return TV == 16 && IP_WHOLE<E>; }

// acc of a tile, from the matrix in registers (ip_whole) or from memory
template <int E, int TV>
__device__ __forceinline__ void ip_tile_product(const float* __restrict__ M, const IpMatrix<E>& m, const float* lds,
                                                int wave, f32x4 (&acc)[IP_CT<E>][TV / 16]) {
  if constexpr (ip_whole<E, TV>()) ip_product_whole<E>(m, lds, acc);
  else ip_product<E, TV / 16>(M, lds, wave, acc);
}

// Signs stage of a tile: `lds` holds rho of TV vectors (ip_pos order, every wave's rows written, no
// barrier yet); leaves +-1 (z >= 0) there in the same order, after a barrier.  m: gt, loaded by the
// caller (ip_whole only); `next`, if given, replaces it once it is used.
template <int E, int TV>
__device__ __forceinline__ void ip_signs(const float* __restrict__ gt, IpMatrix<E>& m, const float* __restrict__ next,
                                         float* lds, int wave) {
  constexpr int NT = TV / 16, CT = IP_CT<E>;
  const int lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4;
  uint32_t pos[CT][NT];  // bit e: element e of the C fragment is >= 0
  __syncthreads();
  if (ip_has_tile<E>(wave)) {
    f32x4 acc[CT][NT];
    ip_tile_product<E, TV>(gt, m, lds, wave, acc);
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        pos[c][n] = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) pos[c][n] |= acc[c][n][e] >= 0.f ? 1u << e : 0u;
      }
  }
  if constexpr (ip_whole<E, TV>()) {
    if (next) {
      m.load(next, wave);
      __builtin_amdgcn_sched_barrier(0);  // in flight while the signs are exchanged
    }
  }
  __syncthreads();  // every read of rho is done
  if (ip_has_tile<E>(wave)) {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int col = ip_pos(ip_col<E>(wave, c, r));
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          lds[(16 * n + 4 * kq + e) * IP_ROW<E> + col] = (pos[c][n] >> e) & 1u ? 1.f : -1.f;
    }
  }
  __syncthreads();
}

// Projection stage: `lds` holds the +-1 signs of TV vectors (ip_pos order, after a barrier); leaves
// w = signs . G there in plain order, after a barrier.  m: g, loaded by the caller (ip_whole only).
template <int E, int TV>
__device__ __forceinline__ void ip_project(const float* __restrict__ g, const IpMatrix<E>& m, float* lds, int wave) {
  constexpr int NT = TV / 16, CT = IP_CT<E>;
  const int lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4;
  f32x4 acc[CT][NT];
  if (ip_has_tile<E>(wave)) ip_tile_product<E, TV>(g, m, lds, wave, acc);
  __syncthreads();  // every read of the signs is done
  if (ip_has_tile<E>(wave)) {
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) lds[(16 * n + 4 * kq + e) * IP_ROW<E> + ip_col<E>(wave, c, r)] = acc[c][n][e];
  }
  __syncthreads();
}

// Reconstruction of one vector from its w row: lane's E elements of norm * R^T(c + k0 rn w).
template <int E>
__device__ __forceinline__ void ip_reconstruct(const float* wrow, const float (&c)[E], float coef, float nrm,
                                               const float (&sg)[E], int lane, float (&out)[E]) {
  float u[1][E];
#pragma unroll
  for (int e = 0; e < E; ++e) u[0][e] = __builtin_fmaf(coef, wrow[lane * E + e], c[e]);
  fwht_wave_n<1, E>(u);
  const float inv = tq_inv_sqrt(64 * E);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    float t = u[0][e] * inv;
    t = t * sg[e];
    out[e] = nrm * t;
  }
}

inline float ip_k0(int64_t D) { return (float)(1.2533141373155002512 / (double)D); }  // fl(sqrt(pi/2) / D)

}  // namespace anna
