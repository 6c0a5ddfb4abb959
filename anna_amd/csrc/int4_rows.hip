// W4A16 linear for groups of 32 or 64 and for activations that are not 16-byte aligned (odd K or row
// strides) on gfx950: y[M, N] = x[M, K] . ((q - z) s)[N, K]^T, 16-bit x, any M.
//
// The forms of int4_linear.hip multiply by "off + q" and take the zero point out once per 128-k block,
// which needs one scale per block.  Here W enters v_mfma_f32_16x16x32 as q - z itself (an integer of
// [-128, 143], exact in bf16 and f16), so that a product is exact, sums are fp32, and an infinity of x
// stays one as in the scalar kernel; every instruction's 32 k lie in one group, whose scale multiplies
// its sum in fp32.
//   - A workgroup of 8 waves owns NT 16-row tiles of W against MG 16-row groups of x; its waves take
//     the 128-k blocks in turn and meet once, in LDS.
//   - W: one 128-bit load per lane brings 32 nibbles of a row.  An instruction wants 8 nibbles of each
//     of four lane groups next to each other in k, so a block's four words are transposed between the
//     lane groups (four v_permlane swaps).  The next block's words, scales and zero points are loaded
//     while the current block computes.
//   - Padding rows, k past K, rows past N: buffer loads past the resource, which read zero.
// What bounds it: HBM for few rows (the memory of W once), the conversion (25 VALU instructions per 8
// nibbles and lane) above that, shared by the MG row groups.  Groups of 32, K = 4096,
// N = 6144, with the scalar kernel before: M = 1 46.7 -> 9.2 us, 8 140 -> 10.9, 16 276 -> 13.0, 48 820 -> 20.7,
// 100 1709 -> 40.3, 333 5561 -> 98; groups of 64, M = 8 137 -> 10.9, K = 1024, N = 4096 22.0 -> 3.5.
#include <type_traits>

#include "common.hpp"
#include "int4_frag.hpp"
#include "int4_gemm.hpp"

namespace anna {
namespace {

constexpr int RW_WAVES = 8;
constexpr uint32_t RW_OOB = 0x80000000u;  // buffer offset past any num_records: the load returns 0

typedef float f32x2r __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2r __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2r __attribute__((ext_vector_type(2)));

template <int XDT>
__device__ __forceinline__ uint32_t rw_pack2(float lo, float hi) {
  if constexpr (XDT == ANNA_MI_BF16)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2r){lo, hi}, bf16x2r));
  else
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2r){lo, hi}, f16x2r));
}

// q - z of the 8 nibbles of w, in k order.  off is 128, or 0 for z < -112, so that q + off - z is a
// byte; bias holds off - z in each of its bytes.
template <int XDT>
__device__ __forceinline__ u32x4 rw_frag(uint32_t w, uint32_t bias, float off) {
  const uint32_t lo = (w & 0x0F0F0F0Fu) + bias, hi = ((w >> 4) & 0x0F0F0F0Fu) + bias;
  u32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o[j] = rw_pack2<XDT>((float)((lo >> (8 * j)) & 0xFFu) - off, (float)((hi >> (8 * j)) & 0xFFu) - off);
  return o;
}

// ALIGNED: x is 16-byte aligned and K and its row stride are multiples of 8 (one load per fragment,
// else eight of two bytes).
template <int XDT, int SDT, int NT, int MG, bool ALIGNED>
__global__ __launch_bounds__(64 * RW_WAVES) void int4_rows_mfma(
    const uint16_t* __restrict__ x, int64_t M, int64_t K, int64_t xs, const uint32_t* __restrict__ qw, int64_t N,
    int64_t pc, const typename Elem<SDT>::T* __restrict__ qs, const int8_t* __restrict__ qz, int gshift, int G,
    uint16_t* __restrict__ y) {
  using ST = typename Elem<SDT>::T;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r = lane & 15, kq = lane >> 4;
  const int64_t n0 = xcd_tile(blockIdx.x, gridDim.x) * (16 * NT);
  const int64_t m0 = (int64_t)blockIdx.y * (16 * MG);
  const int64_t rows_x = M - m0 < 16 * MG ? M - m0 : 16 * MG, rows_w = N - n0 < 16 * NT ? N - n0 : 16 * NT;
  const int nblk = (int)((K + 127) >> 7), pc32 = (int)pc;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(x + m0 * xs), 0, (int)(((rows_x - 1) * xs + K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(qw + n0 * pc), 0, (int)(rows_w * pc * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<ST*>(qs), 0, (int)((int64_t)G * N * (int64_t)sizeof(ST)), 0x00020000);
  const __amdgpu_buffer_rsrc_t rz =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(qz), 0, (int)((int64_t)G * N), 0x00020000);

  struct Stage {
    u32x4 w[NT];                  // words 16 b + 4 kq .. + 3 of row n0 + 16 t + r
    uint32_t sc[NT][4], z[NT][4];  // raw, of the block's four 32-k steps
  };
  auto load_w = [&](int b, Stage& S) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int word = 16 * b + 4 * kq, row = 16 * t + r;
      const bool ok = word < pc32 && row < rows_w;
      S.w[t] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, ok ? (uint32_t)((row * pc32 + word) * 4) : RW_OOB, 0, 0));
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int g = (128 * b + 32 * s) >> gshift;
        const bool gok = g < G && row < rows_w;
        const uint32_t gi = (uint32_t)(g * (int)N + (int)n0 + row);
        if constexpr (sizeof(ST) == 4)
          S.sc[t][s] = __builtin_amdgcn_raw_buffer_load_b32(rs, gok ? gi * 4 : RW_OOB, 0, 0);
        else
          S.sc[t][s] = __builtin_amdgcn_raw_buffer_load_b16(rs, gok ? gi * 2 : RW_OOB, 0, 0);
        S.z[t][s] = __builtin_amdgcn_raw_buffer_load_b8(rz, gok ? gi : RW_OOB, 0, 0);
      }
    }
  };
  auto load_x = [&](int b, int s, int g) -> u32x4 {
    const int row = 16 * g + r, k = 128 * b + 32 * s + 8 * kq;
    if constexpr (ALIGNED) {
      const bool ok = row < rows_x && k < K;
      return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                           rx, ok ? (uint32_t)((row * xs + k) * 2) : RW_OOB, 0, 0));
    } else {
      u32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t o = (uint32_t)((row * xs + k + 2 * j) * 2);
        const uint32_t lo = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rx, row < rows_x && k + 2 * j < K ? o : RW_OOB, 0, 0);
        const uint32_t hi = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rx, row < rows_x && k + 2 * j + 1 < K ? o + 2 : RW_OOB, 0, 0);
        v[j] = lo | (hi << 16);
      }
      return v;
    }
  };

  f32x4 out[MG][NT];
#pragma unroll
  for (int g = 0; g < MG; ++g)
#pragma unroll
    for (int t = 0; t < NT; ++t) out[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto block = [&](int b, Stage& S, Stage& Snext) {
    u32x4 xa[MG][4];
#pragma unroll
    for (int g = 0; g < MG; ++g)
#pragma unroll
      for (int s = 0; s < 4; ++s) xa[g][s] = load_x(b, s, g);
    load_w(b + RW_WAVES, Snext);  // past the end: zeros, from no memory
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      // word 4 kq + s in register s -> word 4 s + kq in register s
      uint32_t w0 = S.w[t].x, w1 = S.w[t].y, w2 = S.w[t].z, w3 = S.w[t].w;
      auto p = __builtin_amdgcn_permlane32_swap(w0, w2, false, false);
      w0 = p[0], w2 = p[1];
      p = __builtin_amdgcn_permlane32_swap(w1, w3, false, false);
      w1 = p[0], w3 = p[1];
      p = __builtin_amdgcn_permlane16_swap(w0, w1, false, false);
      w0 = p[0], w1 = p[1];
      p = __builtin_amdgcn_permlane16_swap(w2, w3, false, false);
      w2 = p[0], w3 = p[1];
      const uint32_t wt[4] = {w0, w1, w2, w3};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int z = (int)(int8_t)S.z[t][s], off = z < -112 ? 0 : 128;
        const u32x4 bf = rw_frag<XDT>(wt[s], (uint32_t)(off - z) * 0x01010101u, (float)off);
        float sc;
        if constexpr (sizeof(ST) == 4) sc = __uint_as_float(S.sc[t][s]);
        else sc = Elem<SDT>::to_f32((ST)S.sc[t][s]);
#pragma unroll
        for (int g = 0; g < MG; ++g) {
          const f32x4 acc = mfma16<XDT>(xa[g][s], bf, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
          for (int i = 0; i < 4; ++i) out[g][t][i] = fmaf(sc, acc[i], out[g][t][i]);
        }
      }
    }
  };
  Stage S0, S1;
  load_w(wave, S0);
  for (int b = wave; b < nblk; b += 2 * RW_WAVES) {
    block(b, S0, S1);
    if (b + RW_WAVES >= nblk) break;
    block(b + RW_WAVES, S1, S0);
  }

  // C layout: lane holds rows 4 kq + i of column r of each 16 x 16 block.  Each wave sums a share of
  // the fragments over the eight waves.
  __shared__ float red[RW_WAVES][4 * NT][64];
#pragma unroll
  for (int g = 0; g < MG; ++g) {
    if (16 * g >= rows_x) break;
    if (g > 0) __syncthreads();  // the previous group's sums are read
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][4 * t + i][lane] = out[g][t][i];
    __syncthreads();
    for (int f = wave; f < 4 * NT; f += RW_WAVES) {
      float v = red[0][f][lane];
#pragma unroll
      for (int w = 1; w < RW_WAVES; ++w) v += red[w][f][lane];
      const int row = 16 * g + 4 * kq + (f & 3), col = 16 * (f >> 2) + r;
      if (row < rows_x && col < rows_w) y[(m0 + row) * N + n0 + col] = Elem<XDT>::cvt(v);
    }
  }
}

}  // namespace

bool int4_rows_supported(int x_dtype, int64_t M, int64_t N, int64_t K, int64_t xs, const void* qweight, int64_t pc,
                         int64_t G, int64_t gsz) {
  // 32-bit buffer offsets: 64 rows of x, 48 of W, the scale and zero-point arrays; grid limit of y
  const bool fits = 64 * xs * 2 + K * 2 < (1ll << 31) && 48 * pc * 4 < (1ll << 31) && G * N * 4 < (1ll << 31) &&
                    K < (1ll << 30) && (M + 15) / 16 < 65536;
  return (x_dtype == ANNA_MI_BF16 || x_dtype == ANNA_MI_F16) && gsz >= 32 && (gsz & (gsz - 1)) == 0 && pc % 4 == 0 &&
         (uintptr_t)qweight % 16 == 0 && fits;
}

int int4_rows_launch(const void* x, int x_dtype, int64_t M, int64_t K, int64_t xs, const int32_t* qweight, int64_t N,
                     int64_t pc, const void* qscale, int scale_dtype, const int8_t* qzeros, int64_t G, int64_t gsz,
                     void* y, hipStream_t st) {
  const bool aligned = (uintptr_t)x % 16 == 0 && xs % 8 == 0 && K % 8 == 0;
  const int gshift = __builtin_ctzll((unsigned long long)gsz);
  G = (K + gsz - 1) / gsz;  // a group past K is not read
  ANNA_DISPATCH_DTYPE(scale_dtype, SDT, {
    auto go = [&](auto xdt_tag, auto nt_tag, auto mg_tag, auto al_tag) {
      constexpr int XDT = decltype(xdt_tag)::value, NT = decltype(nt_tag)::value, MG = decltype(mg_tag)::value;
      constexpr bool AL = decltype(al_tag)::value;
      const dim3 grid((unsigned)((N + 16 * NT - 1) / (16 * NT)), (unsigned)((M + 16 * MG - 1) / (16 * MG)));
      hipLaunchKernelGGL((int4_rows_mfma<XDT, SDT, NT, MG, AL>), grid, dim3(64 * RW_WAVES), 0, st, (const uint16_t*)x,
                         M, K, xs, (const uint32_t*)qweight, N, pc, (const typename Elem<SDT>::T*)qscale, qzeros,
                         gshift, (int)G, (uint16_t*)y);
    };
    using T1 = std::integral_constant<int, 1>;
    using T2 = std::integral_constant<int, 2>;
    using T4 = std::integral_constant<int, 4>;
    auto go_mg = [&](auto xdt_tag, auto al_tag) {
      // one row group and one tile of W a workgroup while that is no more than two workgroups a compute
      // unit (K = 4095, N = 64, M = 64: 25 us; 84 in two workgroups of four groups, 67 with the scalar
      // kernel; N = 1024 21.6, 75 and 132); two tiles beyond, and two or four row groups for more rows (the
      // conversion is shared by them: M = 48, K = 4096, N = 6144 20.7 us against three times 13)
      if (((N + 15) / 16) * ((M + 15) / 16) <= 512) go(xdt_tag, T1{}, T1{}, al_tag);
      else if (M <= 16) go(xdt_tag, T2{}, T1{}, al_tag);
      else if (M <= 32) go(xdt_tag, T2{}, T2{}, al_tag);
      else go(xdt_tag, T2{}, T4{}, al_tag);
    };
    auto go_al = [&](auto xdt_tag) {
      if (aligned) go_mg(xdt_tag, std::true_type{});
      else go_mg(xdt_tag, std::false_type{});
    };
    if (x_dtype == ANNA_MI_BF16) go_al(std::integral_constant<int, ANNA_MI_BF16>{});
    else go_al(std::integral_constant<int, ANNA_MI_F16>{});
  });
  ANNA_LAUNCH_CHECK("int4_rows_mfma");
  return ANNA_MI_OK;
}

}  // namespace anna
