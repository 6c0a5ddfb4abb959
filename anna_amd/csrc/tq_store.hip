// Tokens joining the TurboQuant cache of a layer, on gfx950: one launch for every sequence.
//
// A layer's slab holds, per (sequence, KV head), `capacity` quantized slots and a ring of the R
// newest tokens (token j at ring slot j % R).  When T tokens join a sequence of L, the tokens
// max(0, L - R) <= j < max(0, L + T - R) leave the window: each is read from the ring (j < L) or
// from the new tokens, quantized into slot j, and -- if it came from the ring -- replaced there by
// the one new token that ends up in its ring slot.  While L < R, ring slots L .. are filled too.
// (reference: Qwen3DynamicCache._update_turboquant_layer looping TurboQuantKVRow.append,
// src/anna/model/ops.py:618-661, turboquant.py:1027-1140.)
//
// The launch has three kinds of 512-thread workgroups: tiles of keys, values, and ring fills.  A
// ring slot is read and written by one wave only (its reading lanes are its writing lanes), so the
// kinds need no order among them.  Lengths are read from one array and the new ones written to
// another, so no workgroup can see a length another has already raised; a third one, which stays the
// same from launch to launch, is for the decode.
//
// What bounds it.  Inner-product keys: the two D x D fp32 products of a vector (4 D^2 flops) on the
// matrix cores.  2 x 8064 leaving tokens of 2 KV heads, D = 256: 125 us, of which the products are
// 55 us at the fp32 matrix rate and 70 us as measured (the call without them: 56 us; keys only: 121
// us); the transforms before and after run in the same workgroups and overlap with them only across
// the two workgroups of a compute unit.  Few vectors (a decode step): one tile of 16, bound by one
// compute unit's fetch of the two matrices and its matrix rate (2 x 2 vectors, D = 256: 27 us with
// the caches flushed between calls, 45 us before the matrices were loaded whole; 8 x 2 vectors,
// D = 128: 15 us; with the matrices in the L2 20 and 10).  TQ-MSE keys and values: transform and min/max arithmetic (8,192 vectors of 128
// at 4 bits, keys and values: 8.1 us under the tracer, 6.6 back to back).  A step of 8 sequences (D = 128, 2 KV heads, 4 bits) was ~30
// launches and 370 us before this kernel.
#include <math.h>

#include <type_traits>

#include "common.hpp"
#include "tq_hadamard.hpp"
#include "tq_ip_core.hpp"
#include "tq_pack.hpp"

namespace anna {
namespace {

constexpr int ST_THREADS = 64 * IP_WAVES;
constexpr int ST_MSE_NV = 4;  // TQ-MSE key vectors per wave

struct StoreGrid {
  uint32_t key_wgs, value_wgs;  // then the ring fills
  uint32_t vectors;             // rows * kv_heads * max_leaving (the bound the caller gives)
};

template <int XDT, int E>
__device__ __forceinline__ void load_elems(const typename Elem<XDT>::T* p, float (&x)[E]) {
  using T = typename Elem<XDT>::T;
  constexpr int W = E < 8 ? E : 8;  // (rows are 16-byte aligned: checked by the launcher)
  typedef T TV __attribute__((ext_vector_type(W)));
#pragma unroll
  for (int e = 0; e < E; e += W) {
    if constexpr (W == 1) {
      x[e] = Elem<XDT>::to_f32(p[e]);
    } else {
      const TV v = *(const TV*)(p + e);
#pragma unroll
      for (int i = 0; i < W; ++i) x[e + i] = Elem<XDT>::to_f32(v[i]);
    }
  }
}
template <int XDT, int E>
__device__ __forceinline__ void copy_elems(const typename Elem<XDT>::T* src, typename Elem<XDT>::T* dst) {
  using T = typename Elem<XDT>::T;
  constexpr int W = E < 8 ? E : 8;
  typedef T TV __attribute__((ext_vector_type(W)));
#pragma unroll
  for (int e = 0; e < E; e += W) {
    if constexpr (W == 1) dst[e] = src[e];
    else *(TV*)(dst + e) = *(const TV*)(src + e);
  }
}

// Where leaving vector v (of rows x kv_heads x max_leaving) comes from and goes to.
template <typename T>
struct Leaving {
  const T* src;        // a valid row also when !ok
  T* ring;             // the ring row to refill after reading it, or null
  const T* refill;     // its new content
  int64_t slot;        // destination row of the quantized arrays: (b * H + h) * capacity + j
  bool ok;
};

template <typename T, bool VALUE>
__device__ __forceinline__ Leaving<T> leaving(const anna_mi_tq_store_args& a, uint32_t v, bool in_range) {
  const uint32_t nq = (uint32_t)a.max_leaving, H = (uint32_t)a.kv_heads;
  const uint32_t bh = v / nq, i = v - bh * nq, br = bh / H, h = bh - br * H;
  const int R = (int)a.residual_capacity, T_ = (int)a.tokens;
  const int64_t b = a.row0 + br;
  const int L = a.seq_in ? a.seq_in[b] : 0;
  const int j0 = L > R ? L - R : 0, j1 = L + T_ > R ? L + T_ - R : 0;
  const int j = j0 + (int)i;
  const T* fresh = VALUE ? (const T*)a.new_value + br * a.value_stride_row + h * a.value_stride_head
                         : (const T*)a.new_key + br * a.key_stride_row + h * a.key_stride_head;
  const int64_t st = VALUE ? a.value_stride_token : a.key_stride_token;
  const int64_t row = b * H + h;
  T* const ring0 = (T*)(VALUE ? a.residual_value : a.residual_key) + row * R * a.head_dim;
  Leaving<T> o;
  o.ok = in_range && j < j1 && j < (int)a.capacity;
  o.slot = row * a.capacity + j;
  o.ring = nullptr;
  o.src = o.refill = fresh;
  if (o.ok) {
    if (j < L) {
      o.ring = ring0 + (int64_t)((uint32_t)j % (uint32_t)R) * a.head_dim;
      o.src = o.ring;
      // the last token of the sequence whose ring slot is j's
      const int last = L + T_ - 1;
      o.refill = fresh + (int64_t)(last - (int)((uint32_t)(last - j) % (uint32_t)R) - L) * st;
    } else {
      o.src = fresh + (int64_t)(j - L) * st;
    }
  }
  return o;
}

// ---- keys, inner-product format: a tile of TV vectors, TV / 8 of them per wave
template <int XDT, int E, int TV>
__device__ __forceinline__ void store_ip_keys(const anna_mi_tq_store_args& a, const StoreGrid& g, float* lds) {
  using T = typename Elem<XDT>::T;
  constexpr int D = 64 * E, VW = TV / IP_WAVES, NB = VW < 4 ? VW : 4;
  constexpr int CW = E <= 8 ? 1 : 2;  // words of 4-bit codes per vector and lane
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int nthr = (1 << (a.key_bits - 1)) - 1;
  IpMatrix<E> m;
  if constexpr (ip_whole<E, TV>()) {
    m.load(a.gaussian_t, wave);
    __builtin_amdgcn_sched_barrier(0);  // before anything waits
  }
  const float ctab = ip_centroid_table(a.centroids, a.key_bits);
  uint32_t codes[VW][CW];
  float nrm[VW], rnv[VW];
#pragma unroll
  for (int n0 = 0; n0 < VW; n0 += NB) {
    float x[NB][E], rho[NB][E], nb[NB], rb[NB];
    uint32_t cb[NB][E];
    Leaving<T> lv[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const uint32_t v = blockIdx.x * TV + wave * VW + n0 + n;
      lv[n] = leaving<T, false>(a, v < g.vectors ? v : g.vectors - 1, v < g.vectors);
      load_elems<XDT, E>(lv[n].src + lane * E, x[n]);
    }
    ip_mse_stage<NB, E>(x, a.signs, a.thresholds, ctab, nthr, cb, nb, rho, rb);
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      float* my = lds + (wave * VW + n0 + n) * IP_ROW<E>;
#pragma unroll
      for (int w = 0; w < CW; ++w) codes[n0 + n][w] = 0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        my[ip_pos(lane * E + e)] = rho[n][e];
        codes[n0 + n][e / 8] |= cb[n][e] << (4 * (e & 7));
      }
      nrm[n0 + n] = nb[n];
      rnv[n0 + n] = rb[n];
      if (!lv[n].ok) continue;
      if (lv[n].ring) copy_elems<XDT, E>(lv[n].refill + lane * E, lv[n].ring + lane * E);
      store_bytes_wave<E>(cb[n], a.key_codes + lv[n].slot * D, lane);
      if (lane == 0) {
        ((float*)a.key_norms)[lv[n].slot] = nb[n];
        a.key_residual_norms[lv[n].slot] = rb[n];
      }
    }
  }
  ip_signs<E, TV>(a.gaussian_t, m, a.gaussian, lds, wave);
#pragma unroll
  for (int n = 0; n < VW; ++n) {
    const uint32_t v = blockIdx.x * TV + wave * VW + n;
    if (v >= g.vectors) break;
    const Leaving<T> lv = leaving<T, false>(a, v, true);
    if (!lv.ok) continue;
    uint32_t q[E];
#pragma unroll
    for (int e = 0; e < E; ++e) q[e] = lds[(wave * VW + n) * IP_ROW<E> + ip_pos(lane * E + e)] > 0.f ? 1u : 0u;
    store_bytes_wave<E>(q, a.key_signs + lv.slot * D, lane);
  }
  ip_project<E, TV>(a.gaussian, m, lds, wave);
  float sg[E];
#pragma unroll
  for (int e = 0; e < E; ++e) sg[e] = a.signs[lane * E + e];
  const float k0 = a.k0;
#pragma unroll
  for (int n = 0; n < VW; ++n) {
    const uint32_t v = blockIdx.x * TV + wave * VW + n;
    if (v >= g.vectors) break;
    const Leaving<T> lv = leaving<T, false>(a, v, true);
    if (!lv.ok) continue;
    float c[E], out[E];
#pragma unroll
    for (int e = 0; e < E; ++e) c[e] = ip_centroid(ctab, (codes[n][e / 8] >> (4 * (e & 7))) & 15u);
    ip_reconstruct<E>(lds + (wave * VW + n) * IP_ROW<E>, c, k0 * rnv[n], nrm[n], sg, lane, out);
    constexpr int W = E < 8 ? E : 8;
    typedef T TVec __attribute__((ext_vector_type(W)));
    T* dst = (T*)a.key_dense + lv.slot * D + lane * E;
#pragma unroll
    for (int e = 0; e < E; e += W) {
      if constexpr (W == 1) {
        dst[e] = Elem<XDT>::cvt(out[e]);
      } else {
        TVec t;
#pragma unroll
        for (int i = 0; i < W; ++i) t[i] = Elem<XDT>::cvt(out[e + i]);
        *(TVec*)(dst + e) = t;
      }
    }
  }
}

// ---- keys, TQ-MSE format: ST_MSE_NV vectors per wave, no LDS
template <int XDT, int E>
__device__ __forceinline__ void store_mse_keys(const anna_mi_tq_store_args& a, const StoreGrid& g) {
  using T = typename Elem<XDT>::T;
  constexpr int D = 64 * E, NV = ST_MSE_NV;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t v0 = (blockIdx.x * IP_WAVES + wave) * NV;
  if (v0 >= g.vectors) return;
  float x[NV][E], nrm[NV];
  uint32_t code[NV][E];
  Leaving<T> lv[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const uint32_t v = v0 + n;
    lv[n] = leaving<T, false>(a, v < g.vectors ? v : g.vectors - 1, v < g.vectors);
    load_elems<XDT, E>(lv[n].src + lane * E, x[n]);
  }
  hadamard_codes_wave_n<NV, E>(x, a.signs, a.thresholds, (1 << a.key_bits) - 1, tq_inv_sqrt(D), code, nrm);
  const int sb = storage_bits(a.key_bits);
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    if (!lv[n].ok) continue;
    if (lv[n].ring) copy_elems<XDT, E>(lv[n].refill + lane * E, lv[n].ring + lane * E);
    store_codes_wave<E>(code[n], sb, a.key_codes + lv[n].slot * (D * sb / 8), lane);
    if (lane == 0) ((uint16_t*)a.key_norms)[lv[n].slot] = f32_to_f16_bits(nrm[n]);
  }
}

// ---- values.  Groups of 8 .. 512 elements (a power of two): a lane takes 8 consecutive elements,
// the lanes of a group meet in xor steps (min and max are exact in any order) and every lane packs
// its own 8 codes.  Other group sizes: one wave per vector, runs of groups by lane.
constexpr int ST_VALUE_WAVE_ELEMS = 512;

template <int XDT, int E>
__device__ __forceinline__ void store_values(const anna_mi_tq_store_args& a, const StoreGrid& g, uint32_t wg) {
  using T = typename Elem<XDT>::T;
  constexpr int D = 64 * E;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int gs = (int)a.value_group_size, ng = D / gs, sb = storage_bits(a.value_bits);
  const int64_t pb = D * sb / 8;
  if (a.value_lane_groups) {
    const int64_t el = ((int64_t)(wg * IP_WAVES + wave)) * ST_VALUE_WAVE_ELEMS + lane * 8;
    const uint32_t v = (uint32_t)(el / D), d0 = (uint32_t)(el % D);
    const Leaving<T> lv = leaving<T, true>(a, v < g.vectors ? v : g.vectors - 1, v < g.vectors);
    float x[8];
    load_elems<XDT, 8>(lv.src + d0, x);
    float lo = INFINITY, hi = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      lo = fminf(lo, x[i]);
      hi = fmaxf(hi, x[i]);
    }
    for (int m = 1; m < gs / 8; m <<= 1) {  // gs is uniform
      lo = fminf(lo, __shfl_xor(lo, m, 64));
      hi = fmaxf(hi, __shfl_xor(hi, m, 64));
    }
    const float levels = (float)((1 << a.value_bits) - 1);
    float sc = __fdiv_rn(__fsub_rn(hi, lo), levels);
    sc = sc < 1e-8f ? 1e-8f : sc;
    const T sc_s = Elem<XDT>::cvt(sc), z_s = Elem<XDT>::cvt(lo);
    const float scf = Elem<XDT>::to_f32(sc_s), zf = Elem<XDT>::to_f32(z_s);
    uint32_t w = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float q = rintf(__fdiv_rn(__fsub_rn(x[i], zf), scf));
      q = fminf(fmaxf(q, 0.f), levels);
      w |= (uint32_t)q << (sb * i);
    }
    if (!lv.ok) return;
    if (lv.ring) copy_elems<XDT, 8>(lv.refill + d0, lv.ring + d0);
    uint8_t* data = a.value_data + lv.slot * pb;
    if (sb == 2) ((uint16_t*)data)[d0 / 8] = (uint16_t)w;
    else ((uint32_t*)data)[d0 / 8] = w;
    if (d0 % (uint32_t)gs == 0) {
      ((T*)a.value_scales)[lv.slot * ng + d0 / gs] = sc_s;
      ((T*)a.value_zeros)[lv.slot * ng + d0 / gs] = z_s;
    }
    return;
  }
  const uint32_t v = wg * IP_WAVES + wave;
  if (v >= g.vectors) return;
  const Leaving<T> lv = leaving<T, true>(a, v, true);
  if (!lv.ok) return;
  const int64_t gpt = value_groups_per_run(a.value_bits, D, gs);
  for (int64_t r = lane; r < ng / gpt; r += 64)
    quantize_value_run<XDT>(lv.src, D, a.value_bits, gs, r * gpt, gpt, a.value_data + lv.slot * pb,
                            (T*)a.value_scales + lv.slot * ng, (T*)a.value_zeros + lv.slot * ng);
  if (lv.ring) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // the lanes' reads of the row come first
    __builtin_amdgcn_wave_barrier();
    copy_elems<XDT, E>(lv.refill + lane * E, lv.ring + lane * E);
  }
}

// ---- ring slots a sequence shorter than the window fills for the first time: one wave per
// (row, KV head, slot), keys and values
template <int XDT, int E>
__device__ __forceinline__ void fill_ring(const anna_mi_tq_store_args& a, uint32_t wg) {
  using T = typename Elem<XDT>::T;
  constexpr int D = 64 * E;
  const int lane = threadIdx.x & 63;
  const uint32_t w = wg * IP_WAVES + (threadIdx.x >> 6), nf = (uint32_t)a.max_fill, H = (uint32_t)a.kv_heads;
  const uint32_t bh = w / nf, i = w - bh * nf, br = bh / H, h = bh - br * H;
  if (br >= (uint32_t)a.rows) return;
  const int R = (int)a.residual_capacity, T_ = (int)a.tokens;
  const int64_t b = a.row0 + br;
  const int L = a.seq_in ? a.seq_in[b] : 0;
  const int s = L + (int)i;  // ring slot
  if (s >= R || s >= L + T_) return;
  const int last = L + T_ - 1;
  const int64_t t = last - (int)((uint32_t)(last - s) % (uint32_t)R) - L;  // the new token that stays there
  const int64_t dst = ((b * H + h) * R + s) * D + lane * E;
  copy_elems<XDT, E>((const T*)a.new_key + br * a.key_stride_row + h * a.key_stride_head + t * a.key_stride_token + lane * E,
                     (T*)a.residual_key + dst);
  copy_elems<XDT, E>((const T*)a.new_value + br * a.value_stride_row + h * a.value_stride_head +
                         t * a.value_stride_token + lane * E,
                     (T*)a.residual_value + dst);
}

// TV: vectors of an inner-product key tile, 0 for TQ-MSE keys
template <int XDT, int E, int TV>
__global__ __launch_bounds__(ST_THREADS, TV > 16 ? 4 : 1) void tq_store_kernel(const anna_mi_tq_store_args a, const StoreGrid g) {
  extern __shared__ __attribute__((aligned(16))) float st_lds[];
  if (blockIdx.x == 0) {
    for (int b = threadIdx.x; b < (int)a.batch; b += ST_THREADS) {
      const bool mine = b >= a.row0 && b < a.row0 + a.rows;
      const int L = a.seq_in ? a.seq_in[b] : 0;
      if (a.past_out) a.past_out[b] = L;
      if (mine || a.seq_in) {
        const int n = L + (mine ? (int)a.tokens : 0);
        a.seq_out[b] = n;
        if (a.seq_lengths) a.seq_lengths[b] = n;
      }
    }
  }
  if (blockIdx.x < g.key_wgs) {
    if constexpr (TV > 0) store_ip_keys<XDT, E, TV>(a, g, st_lds);
    else store_mse_keys<XDT, E>(a, g);
  } else if (blockIdx.x < g.key_wgs + g.value_wgs) {
    store_values<XDT, E>(a, g, blockIdx.x - g.key_wgs);
  } else {
    if (a.max_fill > 0) fill_ring<XDT, E>(a, blockIdx.x - g.key_wgs - g.value_wgs);
  }
}

template <int XDT, int E, int TV>
int launch_store(const anna_mi_tq_store_args& a, hipStream_t st) {
  StoreGrid g;
  const int64_t vectors = a.rows * a.kv_heads * a.max_leaving;
  g.vectors = (uint32_t)vectors;
  const int64_t per_key_wg = TV > 0 ? TV : IP_WAVES * ST_MSE_NV;
  g.key_wgs = (uint32_t)((vectors + per_key_wg - 1) / per_key_wg);
  const int64_t vw = a.value_lane_groups ? (vectors * 64 * E + ST_VALUE_WAVE_ELEMS - 1) / ST_VALUE_WAVE_ELEMS : vectors;
  g.value_wgs = (uint32_t)((vw + IP_WAVES - 1) / IP_WAVES);
  const int64_t fw = a.rows * a.kv_heads * a.max_fill;
  int64_t wgs = (int64_t)g.key_wgs + g.value_wgs + (fw + IP_WAVES - 1) / IP_WAVES;
  if (wgs == 0) wgs = 1;  // only the lengths change
  constexpr size_t lds = TV > 0 ? ip_lds_bytes<E>(TV) : 0;
  auto kern = tq_store_kernel<XDT, E, TV>;
  if constexpr (lds > 0) {
    ANNA_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) ==
                   hipSuccess,
               "anna_mi_tq_store: cannot raise the LDS limit");
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(ST_THREADS), lds, st, a, g);
  return ANNA_MI_OK;
}

}  // namespace
}  // namespace anna

using namespace anna;

extern "C" int64_t anna_mi_sizeof_tq_store_args(void) { return (int64_t)sizeof(anna_mi_tq_store_args); }

extern "C" int anna_mi_tq_store(const anna_mi_tq_store_args* ap, void* stream) {
  ANNA_CHECK(ap != nullptr, "anna_mi_tq_store: null args");
  anna_mi_tq_store_args a = *ap;
  const bool ip = a.key_format == 1;
  ANNA_CHECK(valid_dtype(a.dtype), "anna_mi_tq_store: bad dtype code");
  ANNA_CHECK(a.key_format == 0 || a.key_format == 1, "anna_mi_tq_store: key_format must be 0 (TQ-MSE) or 1 (inner product)");
  const int64_t D = a.head_dim;
  ANNA_CHECK(D == 64 || D == 128 || D == 256 || D == 512 || D == 1024,
             "anna_mi_tq_store: head_dim must be a power of two in [64, 1024]");
  ANNA_CHECK(a.key_bits >= (ip ? 2 : 1) && a.key_bits <= 4, "anna_mi_tq_store: bad key bits");
  ANNA_CHECK(a.value_bits >= 2 && a.value_bits <= 4, "anna_mi_tq_store: value bits must be 2..4");
  // (no values are grouped while nothing leaves the window)
  ANNA_CHECK(a.max_leaving == 0 || (a.value_group_size > 0 && D % a.value_group_size == 0),
             "anna_mi_tq_store: value_group_size must divide head_dim");
  ANNA_CHECK(a.batch > 0 && a.kv_heads > 0 && a.rows > 0 && a.row0 >= 0 && a.row0 + a.rows <= a.batch,
             "anna_mi_tq_store: bad row range");
  ANNA_CHECK(a.tokens > 0 && a.residual_capacity > 0 && a.capacity >= 0 && a.max_leaving >= 0 && a.max_fill >= 0,
             "anna_mi_tq_store: bad lengths");
  // every index the kernel forms in 32 bits: lengths, vectors of the call, 8-element pieces of them
  ANNA_CHECK(a.tokens < (1ll << 29) && a.residual_capacity < (1ll << 29) && a.capacity < (1ll << 30) &&
                 a.kv_heads < (1ll << 20) && a.rows < (1ll << 20) && a.max_leaving < (1ll << 30) &&
                 a.max_fill <= a.residual_capacity && a.rows * a.kv_heads * a.max_leaving < (1ll << 31) / (D / 64) &&
                 a.rows * a.kv_heads * a.max_fill < (1ll << 31),
             "anna_mi_tq_store: too many tokens for one call");
  ANNA_CHECK(a.max_leaving == 0 || a.capacity > 0, "anna_mi_tq_store: tokens leave the window but there are no slots");
  ANNA_CHECK(a.new_key && a.new_value && a.residual_key && a.residual_value && a.seq_out && a.signs && a.thresholds,
             "anna_mi_tq_store: null pointer");
  ANNA_CHECK(a.max_leaving == 0 || (a.key_codes && a.key_norms && a.value_data && a.value_scales && a.value_zeros),
             "anna_mi_tq_store: null quantized storage");
  ANNA_CHECK(!ip || (a.centroids && a.gaussian && a.gaussian_t), "anna_mi_tq_store: null quantizer tables");
  ANNA_CHECK(!ip || a.max_leaving == 0 || (a.key_signs && a.key_residual_norms && a.key_dense),
             "anna_mi_tq_store: null key state");
  ANNA_CHECK(a.seq_out != a.seq_in && (!a.seq_lengths || a.seq_lengths != a.seq_in),
             "anna_mi_tq_store: the new lengths need an array of their own");
  const int64_t es = a.dtype == ANNA_MI_F32 ? 4 : 2, per = 16 / es;
  auto aligned = [&](const void* p, int64_t s0, int64_t s1, int64_t s2) {
    return (uintptr_t)p % 16 == 0 && s0 % per == 0 && s1 % per == 0 && s2 % per == 0;
  };
  ANNA_CHECK(aligned(a.new_key, a.key_stride_row, a.key_stride_head, a.key_stride_token) &&
                 aligned(a.new_value, a.value_stride_row, a.value_stride_head, a.value_stride_token) &&
                 aligned(a.residual_key, 0, 0, 0) && aligned(a.residual_value, 0, 0, 0) && aligned(a.key_dense, 0, 0, 0),
             "anna_mi_tq_store: rows must be 16-byte aligned");
  ANNA_CHECK((uintptr_t)a.key_codes % 4 == 0 && (uintptr_t)a.key_signs % 4 == 0 && (uintptr_t)a.value_data % 4 == 0,
             "anna_mi_tq_store: code rows must be 4-byte aligned");
  const int64_t gs = a.value_group_size;
  a.value_lane_groups = gs >= 8 && gs <= ST_VALUE_WAVE_ELEMS && (gs & (gs - 1)) == 0;
  a.k0 = ip_k0(D);
  const bool small = ip_small_tiles(a.rows * a.kv_heads * a.max_leaving);
  int rc = ANNA_MI_OK;
  ANNA_DISPATCH_DTYPE(a.dtype, XDT, {
    auto go = [&](auto e_tag) {
      constexpr int E = decltype(e_tag)::value;
      if (!ip) return launch_store<XDT, E, 0>(a, as_stream(stream));
      return small ? launch_store<XDT, E, ip_tile(E, true)>(a, as_stream(stream))
                   : launch_store<XDT, E, ip_tile(E, false)>(a, as_stream(stream));
    };
    switch (D) {
      case 64: rc = go(std::integral_constant<int, 1>{}); break;
      case 128: rc = go(std::integral_constant<int, 2>{}); break;
      case 256: rc = go(std::integral_constant<int, 4>{}); break;
      case 512: rc = go(std::integral_constant<int, 8>{}); break;
      default: rc = go(std::integral_constant<int, 16>{}); break;
    }
  });
  if (rc != ANNA_MI_OK) return rc;
  ANNA_LAUNCH_CHECK("tq_store_kernel");
  return ANNA_MI_OK;
}
