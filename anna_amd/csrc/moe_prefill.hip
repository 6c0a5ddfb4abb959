// The sparse MoE block for many routes per expert (prefill) on gfx950: routing, dispatch, grouped int4
// SwiGLU MLP and combine in five launches, for 16-bit hidden states and group 128.
//
//   moe_pf_route    one wave per token (softmax, top-k, renorm as moe_router_kernel); each workgroup
//                   keeps its tokens' expert counts in LDS and writes them out -- global atomics on
//                   128 counters serialized 16,384 routes (35 us at 2048 tokens).
//   moe_pf_gather   the same token ranges: a workgroup adds up the counts of the ranges before its own,
//                   ranks its routes in (expert, token, k) order and copies each token's row, read
//                   once, to its routes' places, in the order of the weight fragments, with the sums
//                   of its 128-k groups (which the products need once per route, not per tile).
//   moe_pf_gemm     the two products, below.
//   moe_pf_combine  out[t] = sum of its routes' rows.
//
// moe_pf_gemm.  A 4-wave workgroup takes (expert, item, sweep): an item is one or more consecutive tiles of
// 256 rows of W -- 128 of the gate and the same of the up matrix, or 256 of the down matrix -- and a sweep
// up to 48 of the expert's routes (its 16-route chunks split evenly over its sweeps).  Each wave holds 64
// rows of W as four MFMA operands, so that one read of an x operand from LDS feeds four instructions and a
// nibble conversion up to three; two workgroups share a compute unit and fill each other's barriers and
// waits.  The steps of an item's tiles (one group of K each) form one pipeline: W two steps ahead into a
// ring of the wave's own in LDS, x two steps ahead through registers into a double-buffered,
// chunk-swizzled LDS tile, scales and zero points a step ahead in registers, the sums of all groups in
// LDS from the start.  The scale and zero point are applied per group in fp32 as
// s (sum x (off + q) - (off + z) sum x); the activation between the products is bf16, as in the other
// forms (moe.hip).  What bounds it: issue, ~6.5 VALU instructions (conversion, scaling, addresses) to an
// MFMA.  2048 tokens, 128 experts, top 8, 2048 x 512, traced: gate/up 152 us, down 98, gather 33, route 15,
// combine 13; the block with fp32 scales 289 to 307 us, with the forms of moe.hip 429 to 439; 32 experts of 768
// 318 and 1077.  Measured and not kept: 8 waves of two operands against
// up to 128 routes in one workgroup per compute unit (181 + 140 us; W is converted once, but nothing fills
// the barriers).
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "int4_frag.hpp"
#include "moe_route.hpp"

namespace anna {
namespace {

constexpr int PF_WAVES = 4, PF_ROWS = 256, PF_NC = 3;   // gemm: waves, W rows, 16-route chunks per sweep
constexpr int PF_GMAX = 32;                              // gemm: groups of K
// gemm LDS: x (two passes), W (three 4 KB stages per wave), the waves' activation sums, x's group sums
constexpr int PF_X_BYTES = 2 * 16 * PF_NC * 128 * 2, PF_W_BYTES = PF_WAVES * 3 * 4096, PF_S_BYTES = PF_WAVES * 16 * PF_NC * 4;
constexpr int pf_gemm_lds(int G) { return PF_X_BYTES + PF_W_BYTES + PF_S_BYTES + G * 16 * PF_NC * 4; }
static_assert(2 * pf_gemm_lds(PF_GMAX) <= 160 * 1024, "two workgroups per compute unit");
typedef __attribute__((address_space(3))) void* pf_lds_ptr;
constexpr int PF_RT_WAVES = 16;                          // route / gather: waves, one token at a time each
constexpr int PF_RT_ROUTES = 1024;                       // routes of one route / gather workgroup at most

// position of element e of an 8-element chunk in interleave_x's order
__device__ __forceinline__ int pf_pos(int e) { return e < 4 ? 2 * e : 2 * (e - 4) + 1; }

struct PfPlan {
  int64_t tokens, experts, top_k, hidden, inter, routes;
  int64_t wg_tokens, wgs;  // tokens per route / gather workgroup, their number
};

template <int LDT, int MAXV>
__global__ __launch_bounds__(64 * PF_RT_WAVES) void moe_pf_route(const PfPlan p, const typename Elem<LDT>::T* __restrict__ logits,
                                                                 int64_t ls, int normalize, float* __restrict__ weights,
                                                                 int32_t* __restrict__ selected, int32_t* __restrict__ counts) {
  __shared__ int s_cnt[512];
  extern __shared__ float r_scratch[];  // PF_RT_WAVES x route_scratch(E)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int e = threadIdx.x; e < 512; e += 64 * PF_RT_WAVES) s_cnt[e] = 0;
  __syncthreads();
  const int64_t t0 = blockIdx.x * p.wg_tokens, t1 = t0 + p.wg_tokens < p.tokens ? t0 + p.wg_tokens : p.tokens;
  for (int64_t t = t0 + wave; t < t1; t += PF_RT_WAVES) {
    float w;
    int64_t e;
    route_token<LDT, MAXV>(logits, t, p.experts, ls, p.top_k, normalize, lane, r_scratch + wave * route_scratch(p.experts), w, e);
    if (lane < p.top_k) {
      weights[t * p.top_k + lane] = w;
      selected[t * p.top_k + lane] = (int32_t)e;
      atomicAdd(&s_cnt[e], 1);
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < (int)p.experts; e += 64 * PF_RT_WAVES) counts[blockIdx.x * p.experts + e] = s_cnt[e];
}

template <int HDT>
__global__ __launch_bounds__(64 * PF_RT_WAVES) void moe_pf_gather(
    const PfPlan p, const uint16_t* __restrict__ hidden, int64_t hs, const float* __restrict__ weights,
    const int32_t* __restrict__ selected, const int32_t* __restrict__ counts, const int64_t* __restrict__ slots,
    uint16_t* __restrict__ xg, float* __restrict__ sums, uint16_t* __restrict__ cw, int32_t* __restrict__ route_pos,
    int32_t* __restrict__ items) {
  __shared__ int s_scan[16], s_first[512], s_before[512], s_sel[PF_RT_ROUTES], s_pos[PF_RT_ROUTES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int E = (int)p.experts, e = threadIdx.x, k = (int)p.top_k;
  const int64_t t0 = blockIdx.x * p.wg_tokens, t1 = t0 + p.wg_tokens < p.tokens ? t0 + p.wg_tokens : p.tokens;
  const int n = (int)(t1 - t0) * k;
  if (e < n) s_sel[e] = selected[t0 * k + e];
  // expert counts of all ranges and of those before this one: 1024 / EP threads share an expert
  const int EP = E <= 64 ? 64 : E <= 128 ? 128 : E <= 256 ? 256 : 512;
  if (e < 512) s_first[e] = s_before[e] = 0;
  __syncthreads();
  if ((e & (EP - 1)) < E) {
    int total = 0, before = 0;
#pragma unroll 16
    for (int w = e / EP; w < (int)p.wgs; w += 1024 / EP) {
      const int c = counts[(int64_t)w * E + (e & (EP - 1))];
      total += c;
      before += w < (int)blockIdx.x ? c : 0;
    }
    atomicAdd(&s_first[e & (EP - 1)], total);
    atomicAdd(&s_before[e & (EP - 1)], before);
  }
  __syncthreads();
  const int total = e < E ? s_first[e] : 0, before = e < E ? s_before[e] : 0;
  int all, nact;
  const int start = block_exclusive_scan(total, s_scan, &all);
  const int j = block_exclusive_scan(total > 0 ? 1 : 0, s_scan, &nact);
  if (e < E) {
    s_first[e] = start + before;
    if (blockIdx.x == 0 && total > 0) *(int4*)(items + 4 + 4 * j) = make_int4((int)slots[e], start, start + total, 0);
  }
  if (blockIdx.x == 0 && e == 0) items[0] = nact;
  __syncthreads();
  if (e < n) {
    const int er = s_sel[e];
    int rank = 0;
    for (int q = 0; q < e; ++q) rank += s_sel[q] == er;
    const int pos = s_first[er] + rank;
    s_pos[e] = pos;
    route_pos[t0 * k + e] = pos;
    cw[pos] = Elem<HDT>::cvt(weights[t0 * k + e]);
  }
  __syncthreads();
  const int H = (int)p.hidden;
  for (int64_t t = t0 + wave; t < t1; t += PF_RT_WAVES) {
    const uint16_t* src = hidden + t * hs;
    const int* pos = s_pos + (t - t0) * k;
    for (int c = lane * 8; c < H; c += 512) {  // (H % 128 == 0: whole 16-lane groups take part)
      const u32x4 v = *(const u32x4*)(src + c);
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s += Elem<HDT>::to_f32((uint16_t)(v[i] & 0xFFFFu));
        s += Elem<HDT>::to_f32((uint16_t)(v[i] >> 16));
      }
      s += dpp_move<0xB1>(s);
      s += dpp_move<0x4E>(s);
      s += dpp_move<0x141>(s);
      s += dpp_move<0x140>(s);
      const u32x4 x = interleave_x(v);
      for (int q = 0; q < k; ++q) {
        const int64_t at = pos[q];
        *(u32x4*)(xg + at * H + c) = x;
        if ((lane & 15) == 0) sums[(int64_t)(c >> 7) * p.routes + at] = s;
      }
    }
  }
}

__device__ __forceinline__ float pf_silu(float g) { return g / (1.0f + expf(-g)); }

struct PfGemm {
  const uint16_t* x;     // [routes][K], interleaved
  const float* sums;     // [K / 128][routes]
  const uint16_t* cw;    // down: routing weights in the hidden dtype
  const int32_t* items;  // {nact}, then {slot, start, end, -} each
  const int32_t* qw[2];  // gate, up; or down
  const void* qs[2];
  const int8_t* qz[2];
  int64_t N, K, pc, routes;  // rows and columns of a matrix, packed words per row
  uint32_t slot_bytes_w;     // bytes of a slot's matrix
  int sweeps;                // workgroups per (expert, item)
  int tiles;                 // consecutive tiles of an item: one pipeline over their steps
  uint16_t* out;             // act [routes][N] bf16 interleaved, or [routes][N] in the hidden dtype
  float* act_sums;           // gate/up: [N / 128][routes]
};

template <int SDT>
struct PfScales {
  typename Elem<SDT>::T s[4];
  int8_t z[4];
};

template <int HDT, int SDT, bool GU, int NC>
__device__ __forceinline__ void pf_sweep(const PfGemm& a, uint16_t* xs, unsigned char* ws, float* s_x, float (*s_sum)[16 * PF_NC],
                                         uint32_t slot, int tile0, int ntile, int64_t c0, int R) {
  constexpr int MDT = GU ? HDT : ANNA_MI_BF16;
  constexpr float OFF = MDT == ANNA_MI_BF16 ? 128.0f : 1024.0f;
  using ST = typename Elem<SDT>::T;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r = lane & 15, kq = lane >> 4;
  const int N = (int)a.N, K = (int)a.K, G = K / 128;
  // the wave's four 16-row operands: gate rows n, n + 16 and the same up rows, or 64 down rows
  int nf[4];
#pragma unroll
  for (int f = 0; f < 4; ++f)
    nf[f] = GU ? tile0 * 128 + wave * 32 + 16 * (f & 1) + r : tile0 * 256 + wave * 64 + 16 * f + r;
  __amdgpu_buffer_rsrc_t rw[2], rs[2], rz[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int q = GU ? m : 0;
    rw[m] = __builtin_amdgcn_make_buffer_rsrc((char*)const_cast<int32_t*>(a.qw[q]) + (uint64_t)slot * a.slot_bytes_w, 0,
                                              (int)a.slot_bytes_w, 0x00020000);
    rs[m] = __builtin_amdgcn_make_buffer_rsrc((char*)const_cast<void*>(a.qs[q]) + (uint64_t)slot * G * N * sizeof(ST), 0,
                                              (int)(G * N * sizeof(ST)), 0x00020000);
    rz[m] = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.qz[q]) + (uint64_t)slot * G * N, 0, G * N, 0x00020000);
  }
  // rows past N read other rows' scales and no weights (past the buffer: zero), and are not stored
  constexpr int ROWS = GU ? PF_ROWS / 2 : PF_ROWS;
  const int tile_w = ROWS * (int)a.pc * 4;
  uint32_t wo[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) wo[f] = (uint32_t)((nf[f] * (int)a.pc + kq * 4) * 4);
  // x: chunk i of this thread is row (t + 256 i) / 16, 16-byte chunk (t + 256 i) % 16 of the pass; rows
  // past the sweep's repeat the last one (their results are not stored)
  // (32-bit offsets from the sweep's first row)
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.x + c0 * K), 0, R * K * 2, 0x00020000);
  uint32_t xo[NC];
  int xl[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int e = (int)threadIdx.x + 256 * i, row = e >> 4, ch = e & 15;
    xo[i] = (uint32_t)(((row < R ? row : R - 1) * K + ch * 8) * 2);
    xl[i] = row * 128 + ((ch ^ (row & 15)) * 8);
  }
  // W of group g into stage st of the wave's ring (every lane reads back its own 16 bytes)
  unsigned char* const wl = ws + wave * (3 * 4096);
  // a step: group g of tile t (past the last one: the last one again)
  struct Step {
    int t, g;
  };
  auto advance = [&](Step& p) {
    if (p.g + 1 < G) ++p.g;
    else if (p.t + 1 < ntile) ++p.t, p.g = 0;
  };
  auto load = [&](const Step& p, int st, u32x4 (&xr)[NC]) {
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const int m = GU ? f >> 1 : 0;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw[m], (pf_lds_ptr)(wl + st * 4096 + f * 1024), 16, wo[f],
                                               p.t * tile_w + p.g * 64, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);  // W of a step is requested before its x (see pass)
#pragma unroll
    for (int i = 0; i < NC; ++i)
      xr[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, xo[i], p.g * 256, 0));
  };
  auto load_scales = [&](const Step& p, PfScales<SDT>& P) {
    const int row = p.g * N + p.t * ROWS;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const int m = GU ? f >> 1 : 0;
      if constexpr (sizeof(ST) == 4) P.s[f] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs[m], nf[f] * 4, row * 4, 0));
      else P.s[f] = (ST)__builtin_amdgcn_raw_buffer_load_b16(rs[m], nf[f] * 2, row * 2, 0);
      P.z[f] = (int8_t)__builtin_amdgcn_raw_buffer_load_b8(rz[m], nf[f], row, 0);
    }
  };
  auto store_x = [&](const u32x4 (&xr)[NC], int buf) {
#pragma unroll
    for (int i = 0; i < NC; ++i) *(u32x4*)(xs + buf * (16 * PF_NC * 128) + xl[i]) = xr[i];
  };
  f32x4 out[NC][4];
  auto clear = [&]() {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int f = 0; f < 4; ++f) out[c][f] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  auto compute = [&](const PfScales<SDT>& P, int g, int st, int buf) {
    u32x4 wq[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) wq[f] = *(const u32x4*)(wl + st * 4096 + f * 1024 + lane * 16);
    const uint16_t* xb = xs + buf * (16 * PF_NC * 128) + r * 128;
    f32x4 acc[NC][4];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int f = 0; f < 4; ++f) acc[c][f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      u32x4 wf[4], xa[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) xa[c] = *(const u32x4*)(xb + c * 16 * 128 + (((kq * 4 + s) ^ r) * 8));
#pragma unroll
      for (int f = 0; f < 4; ++f) wf[f] = nibbles_to_frag<MDT>(wq[f][s]);
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[c][f] = mfma16<MDT>(xa[c], wf[f], acc[c][f]);
    }
    f32x4 sx[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) sx[c] = *(const f32x4*)(s_x + g * (16 * PF_NC) + 16 * c + 4 * kq);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const float sf = Elem<SDT>::to_f32(P.s[f]), zf = -(OFF + (float)P.z[f]);
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) out[c][f][i] = fmaf(sf, fmaf(zf, sx[c][i], acc[c][f][i]), out[c][f][i]);
    }
  };
  // LDS writes done, then the barrier (the loads ahead stay in flight)
  auto meet = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  // C layout: lane (r, kq) element i is route c0 + 16 c + 4 kq + i of W row nf (of tile t)
  auto finish = [&](int t) {
    int base = (int)c0, left = R, nn = N;
    asm volatile("" : "+s"(base), "+s"(left), "+s"(nn));
    if constexpr (GU) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = 16 * c + 4 * kq + i;
          float both = 0.f;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int n = nf[h] + t * ROWS;
            const uint16_t v = f32_to_bf16_bits(pf_silu(out[c][h][i]) * out[c][h + 2][i]);
            both += n < nn ? bf16_bits_to_f32(v) : 0.f;
            if (m < left && n < nn) a.out[(int64_t)(base + m) * nn + (n & ~7) + pf_pos(n & 7)] = v;
          }
          both += dpp_move<0xB1>(both);
          both += dpp_move<0x4E>(both);
          both += dpp_move<0x141>(both);
          both += dpp_move<0x140>(both);
          if (r == 0) s_sum[wave][m] = both;
        }
      __syncthreads();
      if ((int)threadIdx.x < left)
        a.act_sums[(int64_t)(tile0 + t) * a.routes + c0 + threadIdx.x] =
            (s_sum[0][threadIdx.x] + s_sum[1][threadIdx.x]) + (s_sum[2][threadIdx.x] + s_sum[3][threadIdx.x]);
    } else {
      using HT = typename Elem<HDT>::T;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = 16 * c + 4 * kq + i;
          if (m >= left) continue;
          const float wr = s_sum[0][m];  // the routing weight
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            const int n = nf[f] + t * ROWS;
            if (n < nn) ((HT*)a.out)[(int64_t)(base + m) * nn + n] = Elem<HDT>::cvt(out[c][f][i] * wr);
          }
        }
    }
  };
  PfScales<SDT> A, B;
  u32x4 XA[NC], XB[NC];
  Step ahead1{0, 0}, ahead2{0, 0};  // the steps whose scales, and whose W and x, are requested next
  load_scales(ahead1, A);
  advance(ahead1);
  load(ahead2, 0, XA);
  advance(ahead2);
  __builtin_amdgcn_sched_barrier(0);
  load(ahead2, 1, XB);
  advance(ahead2);
  __builtin_amdgcn_sched_barrier(0);
  for (int i = threadIdx.x; i < G * 16 * NC; i += 64 * PF_WAVES) {
    const int g = i / (16 * NC), m = i - g * (16 * NC);
    s_x[g * (16 * PF_NC) + m] = m < R ? a.sums[(int64_t)g * a.routes + c0 + m] : 0.f;
  }
  if constexpr (!GU) {
    if ((int)threadIdx.x < R) s_sum[0][threadIdx.x] = Elem<HDT>::to_f32(a.cw[c0 + threadIdx.x]);
  }
  store_x(XA, 0);
  meet();
  // Step q (group g of tile t): request the scales of q + 1, then W and x of q + 2 (W into the stage step
  // q - 1 read), compute q, publish x of q + 1 (its buffer was last read in step q - 1).  Loads complete in
  // order and a step's W is requested before its x, so a wave that has x of a step in registers, as it must
  // to publish it a step ahead, has the step's W in its ring.
  const int steps = ntile * G;
  int t = 0, g = 0, st = 0;
  auto pass = [&](int buf, const PfScales<SDT>& cur, PfScales<SDT>& next, const u32x4 (&xnext)[NC], u32x4 (&xahead)[NC]) {
    load_scales(ahead1, next);
    advance(ahead1);
    load(ahead2, st == 0 ? 2 : st - 1, xahead);
    advance(ahead2);
    __builtin_amdgcn_sched_barrier(0);
    compute(cur, g, st, buf);
    st = st == 2 ? 0 : st + 1;
    if (++g == G) {
      finish(t);
      clear();
      g = 0, ++t;
    }
    store_x(xnext, buf ^ 1);
    meet();
  };
  for (int q = 0; q < steps; q += 2) {
    pass(0, A, B, XB, XA);
    if (q + 1 < steps) pass(1, B, A, XA, XB);
  }
  // the last steps' repeated copies land in stages nobody reads: before the next sweep's first ones; and
  // s_sum is free
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

template <int HDT, int SDT, bool GU>
__global__ __launch_bounds__(64 * PF_WAVES, 2) void moe_pf_gemm(const PfGemm a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char pf_lds[];
  uint16_t* const xs = (uint16_t*)pf_lds;
  unsigned char* const ws = pf_lds + PF_X_BYTES;
  float(*const s_sum)[16 * PF_NC] = (float(*)[16 * PF_NC])(ws + PF_W_BYTES);
  float* const s_x = (float*)(ws + PF_W_BYTES + PF_S_BYTES);
  const int nact = a.items[0];
  const int rows = GU ? PF_ROWS / 2 : PF_ROWS, all = ((int)a.N + rows - 1) / rows;
  const int tiles = (all + a.tiles - 1) / a.tiles;  // items of a.tiles consecutive tiles
  // expert-major within a (tile, sweep): an expert's workgroups are nact apart, on one XCD where nact
  // is a multiple of 8, and share its L2 copy of the expert's x and W
  const int total = nact * tiles * a.sweeps;
  for (int it = blockIdx.x; it < total; it += gridDim.x) {
    const int rest = it / nact, tile = rest % tiles;
    const int4 e = *(const int4*)(a.items + 4 + 4 * (it - rest * nact));
    const uint32_t slot = __builtin_amdgcn_readfirstlane(e.x);
    const int start = __builtin_amdgcn_readfirstlane(e.y), end = __builtin_amdgcn_readfirstlane(e.z);
    const int chunks = (end - start + 15) / 16, nsw = (chunks + PF_NC - 1) / PF_NC;
    for (int sw = rest / tiles; sw < nsw; sw += a.sweeps) {
      // an even split whose terms stay below chunks (sw * chunks / nsw passes 2^31 from 1.3 M routes on)
      const int each = chunks / nsw, more = chunks - each * nsw;
      const int lo = sw * each + (sw < more ? sw : more), hi = lo + each + (sw < more ? 1 : 0);
      const int64_t c0 = start + 16 * lo;
      const int t0 = tile * a.tiles, nt = all - t0 < a.tiles ? all - t0 : a.tiles;
      const int R = (start + 16 * hi < end ? start + 16 * hi : end) - (int)c0;
      if (hi - lo == 1) pf_sweep<HDT, SDT, GU, 1>(a, xs, ws, s_x, s_sum, slot, t0, nt, c0, R);
      else if (hi - lo == 2) pf_sweep<HDT, SDT, GU, 2>(a, xs, ws, s_x, s_sum, slot, t0, nt, c0, R);
      else pf_sweep<HDT, SDT, GU, 3>(a, xs, ws, s_x, s_sum, slot, t0, nt, c0, R);
    }
  }
}

// One wave per (token, 512 columns): the token's rows in route order, fp32 sums (as moe_combine_kernel)
template <int HDT>
__global__ __launch_bounds__(256) void moe_pf_combine(const PfPlan p, const uint16_t* __restrict__ rows,
                                                      const int32_t* __restrict__ route_pos, uint16_t* __restrict__ out) {
  const int lane = threadIdx.x & 63, H = (int)p.hidden, cols = (H + 511) / 512;
  const int64_t w = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t t = w / cols;
  const int c = (int)(w - t * cols) * 512 + lane * 8;
  if (t >= p.tokens || c >= H) return;
  float s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) s[i] = 0.f;
#pragma unroll 4
  for (int q = 0; q < (int)p.top_k; ++q) {
    const u32x4 v = *(const u32x4*)(rows + (int64_t)route_pos[t * p.top_k + q] * H + c);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[2 * i] += Elem<HDT>::to_f32((uint16_t)(v[i] & 0xFFFFu));
      s[2 * i + 1] += Elem<HDT>::to_f32((uint16_t)(v[i] >> 16));
    }
  }
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = (uint32_t)Elem<HDT>::cvt(s[2 * i]) | ((uint32_t)Elem<HDT>::cvt(s[2 * i + 1]) << 16);
  *(u32x4*)(out + t * H + c) = o;
}

struct PfWorkspace {
  int64_t total = 0;
  int64_t take(int64_t bytes) {
    const int64_t at = total;
    total += (bytes + 255) & ~(int64_t)255;
    return at;
  }
};
struct PfLayout {
  int64_t weights, selected, counts, pos, items, cw, sums, act_sums, x, act, rows, total;
};

PfPlan pf_plan(const anna_mi_moe_prefill_args& a) {
  PfPlan p;
  p.tokens = a.tokens, p.experts = a.num_experts, p.top_k = a.top_k, p.hidden = a.hidden_dim, p.inter = a.intermediate_dim;
  p.routes = a.tokens * a.top_k;
  // one token per wave while that gives at most 256 workgroups
  const int64_t per = PF_RT_WAVES * ((a.tokens + PF_RT_WAVES * 256 - 1) / (PF_RT_WAVES * 256));
  p.wg_tokens = std::max<int64_t>(1, std::min(per, PF_RT_ROUTES / a.top_k));
  p.wgs = (a.tokens + p.wg_tokens - 1) / p.wg_tokens;
  return p;
}
PfLayout pf_layout(const PfPlan& p) {
  PfWorkspace w;
  PfLayout l;
  l.weights = w.take(p.routes * 4);
  l.selected = w.take(p.routes * 4);
  l.counts = w.take(p.wgs * p.experts * 4);
  l.pos = w.take(p.routes * 4);
  l.items = w.take((4 + 4 * p.experts) * 4);
  l.cw = w.take(p.routes * 2);
  l.sums = w.take(p.hidden / 128 * p.routes * 4);
  l.act_sums = w.take((p.inter + 127) / 128 * p.routes * 4);
  l.x = w.take(p.routes * p.hidden * 2);
  l.act = w.take(p.routes * p.inter * 2);
  l.rows = w.take(p.routes * p.hidden * 2);
  l.total = w.total;
  return l;
}

bool pf_shape_ok(const anna_mi_moe_prefill_args& a) {
  // 32-bit offsets into one slot's matrices; whole groups; the kernels' LDS
  const int64_t lim = 1ll << 30;
  return (a.dtype == ANNA_MI_BF16 || a.dtype == ANNA_MI_F16) && a.group_size == 128 && a.hidden_dim % 128 == 0 &&
         a.intermediate_dim % 128 == 0 && a.hidden_dim <= 128 * PF_GMAX && a.intermediate_dim <= 128 * PF_GMAX && a.tokens > 0 && a.num_experts > 0 && a.num_experts <= 512 && a.top_k > 0 &&
         a.top_k <= a.num_experts && a.top_k <= 64 && a.tokens * a.top_k < lim &&
         a.hidden_packed_cols % 4 == 0 && a.intermediate_packed_cols % 4 == 0 &&
         a.hidden_packed_cols * 8 >= a.hidden_dim && a.intermediate_packed_cols * 8 >= a.intermediate_dim &&
         a.hidden_groups * 128 == a.hidden_dim && a.intermediate_groups * 128 == a.intermediate_dim &&
         a.intermediate_dim * a.hidden_packed_cols * 4 < lim && a.hidden_dim * a.intermediate_packed_cols * 4 < lim &&
         a.intermediate_dim * a.hidden_groups * 4 < lim && a.hidden_dim * a.intermediate_groups * 4 < lim;
}
// rows and words are read 16 bytes at a time
bool pf_aligned(const anna_mi_moe_prefill_args& a) {
  return a.hidden_row_stride % 8 == 0 && (uintptr_t)a.hidden % 16 == 0 && (uintptr_t)a.gate_qweight % 16 == 0 &&
         (uintptr_t)a.up_qweight % 16 == 0 && (uintptr_t)a.down_qweight % 16 == 0;
}

}  // namespace
}  // namespace anna

using namespace anna;

extern "C" int64_t anna_mi_sizeof_moe_prefill_args(void) { return (int64_t)sizeof(anna_mi_moe_prefill_args); }

// Where this form is faster than those of moe.hip (us, this form and those; 738 shapes of 4 to 128 experts, hidden
// 512 to 4096, intermediate 256 to 4096, 18 to 128 routes per expert: 0.3% from the better one on average, and at
// most 12% slower than those where it is taken).  Never below 18 routes per expert (64 tokens of 32 experts, top 8 (16) 50 and 46); above:
//  - where moe.hip has its wide and resident forms (intermediate 256 or 512, hidden a multiple of 256): from
//    1024 x 512 on (128 experts of 2048 x 512, top 8, 18 routes 95 and 108, 64 302 and 440); narrower ones keep this
//    form's five launches too short of work until there are 36 routes or many tokens (16 experts of 512 x 256, 24
//    routes 45 and 39, 48 46 and 52; 32 of 2048 x 256, top 8, 96 tokens 70 and 64; 64 of 1024 x 256, top 2, 1024
//    tokens 60 and 68);
//  - else, where the 16-route kernels are the other form, by the work and the sweeps those need: 8 experts of
//    512 x 768, 24 routes 55 and 39, 64 55 and 56; 64 of 1024 x 768, 18 routes 59 and 81; 16 of 1024 x 768, 24
//    routes 48 and 43, 16 of 2048 x 1408 59 and 79.
static bool pf_faster(int64_t tokens, int64_t experts, int64_t top_k, int64_t hidden, int64_t inter) {
  const int64_t routes = tokens * top_k;
  if (routes < 18 * experts) return false;
  if (inter % 256 == 0 && inter <= 512 && hidden % 256 == 0)
    return (hidden >= 1024 && inter >= 512) || routes >= 36 * experts || tokens * hidden * inter >= 1ll << 27;
  return routes >= 64 * experts || (double)routes * routes / experts * hidden * inter >= 8589934592.0;
}

extern "C" int64_t anna_mi_moe_prefill_workspace(const anna_mi_moe_prefill_args* ap) {
  if (!ap || !pf_shape_ok(*ap) || !pf_aligned(*ap)) return 0;
  // ANNA_MI_MOE_FORM = P forces this form, anything else the ones of moe.hip (read on every call; the tests run
  // both on shapes small enough for the CPU oracle)
  const char* f = getenv("ANNA_MI_MOE_FORM");
  const bool take = f && *f ? f[0] == 'P'
                            : pf_faster(ap->tokens, ap->num_experts, ap->top_k, ap->hidden_dim, ap->intermediate_dim);
  if (!take) return 0;
  return pf_layout(pf_plan(*ap)).total;
}

extern "C" int anna_mi_moe_prefill(const anna_mi_moe_prefill_args* ap, void* stream) {
  ANNA_CHECK(ap != nullptr, "anna_mi_moe_prefill: null args");
  const anna_mi_moe_prefill_args& a = *ap;
  ANNA_CHECK(valid_dtype(a.logits_dtype) && valid_dtype(a.scale_dtype), "anna_mi_moe_prefill: bad dtype code");
  ANNA_CHECK(pf_shape_ok(a), "anna_mi_moe_prefill: shape not supported (see anna_mi_moe_prefill_workspace)");
  ANNA_CHECK(a.hidden && a.logits && a.out && a.workspace && a.slots && a.gate_qweight && a.gate_qscale && a.gate_qzeros &&
                 a.up_qweight && a.up_qscale && a.up_qzeros && a.down_qweight && a.down_qscale && a.down_qzeros,
             "anna_mi_moe_prefill: null pointer");
  ANNA_CHECK(pf_aligned(a) && a.hidden_row_stride >= a.hidden_dim && (uintptr_t)a.out % 16 == 0 &&
                 (uintptr_t)a.workspace % 256 == 0,
             "anna_mi_moe_prefill: rows and weights must be 16-byte aligned, the workspace 256-byte aligned");
  ANNA_CHECK(a.logits_row_stride >= a.num_experts, "anna_mi_moe_prefill: bad logits stride");
  const PfPlan p = pf_plan(a);
  const PfLayout l = pf_layout(p);
  hipStream_t st = as_stream(stream);
  char* const w = (char*)a.workspace;
  float* const weights = (float*)(w + l.weights);
  int32_t *const selected = (int32_t*)(w + l.selected), *const counts = (int32_t*)(w + l.counts),
                 *const pos = (int32_t*)(w + l.pos), *const items = (int32_t*)(w + l.items);
  ANNA_DISPATCH_DTYPE(a.logits_dtype, LDT, {
    ANNA_DISPATCH_MAXV(a.num_experts, MAXV, {
      hipLaunchKernelGGL((moe_pf_route<LDT, MAXV>), dim3((unsigned)p.wgs), dim3(64 * PF_RT_WAVES),
                         PF_RT_WAVES * route_scratch(a.num_experts) * sizeof(float), st, p,
                         (const typename Elem<LDT>::T*)a.logits, a.logits_row_stride, a.normalize, weights, selected, counts);
    });
  });
  ANNA_LAUNCH_CHECK("moe_pf_route");
  auto go = [&](auto h_tag, auto s_tag) {
    constexpr int HDT = decltype(h_tag)::value, SDT = decltype(s_tag)::value;
    hipLaunchKernelGGL((moe_pf_gather<HDT>), dim3((unsigned)p.wgs), dim3(64 * PF_RT_WAVES), 0, st, p, (const uint16_t*)a.hidden,
                       a.hidden_row_stride, weights, selected, counts, a.slots, (uint16_t*)(w + l.x), (float*)(w + l.sums),
                       (uint16_t*)(w + l.cw), pos, items);
    PfGemm g{};
    g.items = items;
    g.routes = p.routes;
    g.cw = (const uint16_t*)(w + l.cw);
    // workgroups per (expert, tile): the sweeps of an expert with half again the mean load
    g.sweeps = (int)std::max<int64_t>(1, (p.routes * 3 / 2 / a.num_experts + 16 * PF_NC - 1) / (16 * PF_NC));
    auto launch = [&](auto gu_tag) {
      constexpr bool GU = decltype(gu_tag)::value;
      // an item's steps fill the pipeline once: eight of them or more (the down product at K = 512, with bf16
      // scales: 132 us with 4 steps, 113 with 8, 107 with 16, which loses where items are few: 32 experts of 768
      // 372 against 345 us a block)
      g.tiles = (int)std::max<int64_t>(1, (8 * 128 + g.K - 1) / g.K);
      const int64_t all = (g.N + (GU ? 127 : 255)) / (GU ? 128 : 256), tiles = (all + g.tiles - 1) / g.tiles;
      const int64_t wgs = std::min<int64_t>(a.num_experts * tiles * g.sweeps, 1 << 16);
      auto kern = moe_pf_gemm<HDT, SDT, GU>;
      ANNA_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     pf_gemm_lds(PF_GMAX)) == hipSuccess,
                 "anna_mi_moe_prefill: cannot raise the LDS limit");
      hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(64 * PF_WAVES), pf_gemm_lds((int)(g.K / 128)), st, g);
      return ANNA_MI_OK;
    };
    g.x = (const uint16_t*)(w + l.x), g.sums = (const float*)(w + l.sums);
    g.qw[0] = a.gate_qweight, g.qw[1] = a.up_qweight;
    g.qs[0] = a.gate_qscale, g.qs[1] = a.up_qscale;
    g.qz[0] = a.gate_qzeros, g.qz[1] = a.up_qzeros;
    g.N = a.intermediate_dim, g.K = a.hidden_dim, g.pc = a.hidden_packed_cols;
    g.slot_bytes_w = (uint32_t)(g.N * g.pc * 4);
    g.out = (uint16_t*)(w + l.act), g.act_sums = (float*)(w + l.act_sums);
    if (const int rc = launch(std::integral_constant<bool, true>{}); rc != ANNA_MI_OK) return rc;
    g.x = (const uint16_t*)(w + l.act), g.sums = (const float*)(w + l.act_sums);
    g.qw[0] = g.qw[1] = a.down_qweight;
    g.qs[0] = g.qs[1] = a.down_qscale;
    g.qz[0] = g.qz[1] = a.down_qzeros;
    g.N = a.hidden_dim, g.K = a.intermediate_dim, g.pc = a.intermediate_packed_cols;
    g.slot_bytes_w = (uint32_t)(g.N * g.pc * 4);
    g.out = (uint16_t*)(w + l.rows), g.act_sums = nullptr;
    if (const int rc = launch(std::integral_constant<bool, false>{}); rc != ANNA_MI_OK) return rc;
    const int64_t waves = a.tokens * ((a.hidden_dim + 511) / 512);
    hipLaunchKernelGGL((moe_pf_combine<HDT>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, p,
                       (const uint16_t*)(w + l.rows), pos, (uint16_t*)a.out);
    return ANNA_MI_OK;
  };
  ANNA_DISPATCH_DTYPE(a.scale_dtype, SDT, {
    using ST = std::integral_constant<int, SDT>;
    const int rc = a.dtype == ANNA_MI_BF16 ? go(std::integral_constant<int, ANNA_MI_BF16>{}, ST{})
                                           : go(std::integral_constant<int, ANNA_MI_F16>{}, ST{});
    if (rc != ANNA_MI_OK) return rc;
  });
  ANNA_LAUNCH_CHECK("anna_mi_moe_prefill");
  return ANNA_MI_OK;
}
