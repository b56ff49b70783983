// Pieces shared by the fp32 products: fragments, waits, the epilogue.
#pragma once
#include "pf_gemm_common.h"

namespace {

#define PF_LDS(T) __attribute__((address_space(3))) T*
typedef float float2_t __attribute__((ext_vector_type(2)));

// Fragments are read by inline assembly (the compiler would make an LDS read wait for every outstanding
// direct-to-LDS load); it takes their registers for complete where the read is issued.  arrived(), after the wait,
// keeps what uses them below it, and the registers theirs until then.
template <bool TRANS> struct FragF;
template <> struct FragF<false> {
  float4_t v;
  __device__ __forceinline__ float get(int e) const { return v[e]; }
  __device__ __forceinline__ void arrived() { asm volatile("" : "+v"(v)); }
  // zero the reduction indices from `left` on (k: the lane's first one)
  __device__ __forceinline__ void mask(int k, int left) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k + e < left ? v[e] : 0.f;
  }
};
template <> struct FragF<true> {
  float2_t lo, hi;
  __device__ __forceinline__ float get(int e) const { return e < 2 ? lo[e] : hi[e - 2]; }
  __device__ __forceinline__ void arrived() { asm volatile("" : "+v"(lo), "+v"(hi)); }
  __device__ __forceinline__ void mask(int, int) {}   // (k-rows past K arrive as zeros)
};
template <int N> __device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory"); }
template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// The epilogue of a lane's sums v, a vector of rows r per 16x16 block: row m0 + first + 16 i + r, column col0 + 16 j.  16 lanes cover 64 consecutive bytes of a
// row.  With fp32 operands throughout (vec_epi), everything one step reads is requested before any of it is used; the
// buffers' range checks drop rows past M (m0: the first of the tile's BM rows), columns past N are sent out of range.
typedef float float1_t __attribute__((ext_vector_type(1)));
template <int BM, int TM, int TN, typename V>
__device__ __forceinline__ void epilogue_f32(const pf_gemm_desc& p, const GemmGrid& g, V (&v)[TM][TN], const int64_t m0, const int first,
                                             const int64_t col0, const int64_t c_base) {
  constexpr int NR = sizeof(V) / 4;
  const Epi epi = make_epi(p);
  const int64_t M = p.M, N = p.N, row0 = m0 + first;
  if (!g.vec_epi) {
#pragma nounroll
    for (int h = 0; h < TM * TN; ++h) {
      V x;
      static_for<TM * TN>([&](auto hc) {
        constexpr int c = decltype(hc)::value;
        if (h == c) x = v[c / TN][c % TN];
      });
      const int64_t col = col0 + 16 * (h % TN);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const int64_t row = row0 + 16 * (h / TN) + r;
        if (row < M && col < N) epilogue_scalar(epi, c_base, row, col, x[r]);
      }
    }
    return;
  }
  const int rows_left = (int)(M - m0 < BM ? M - m0 : BM);
  auto buffer = [&](const void* x, int64_t ld) {   // rows m0 .. of an operand of C's shape
    return make_rsrc((const float*)x + m0 * ld, (uint32_t)(((rows_left - 1) * ld + N) * 4));
  };
  auto offset = [&](int i, int j, int r, int64_t ld) {
    const int64_t col = col0 + 16 * j;
    return col < N ? (int)(((first + 16 * i + r) * ld + col) * 4) : (int)0x80000000;
  };
  auto each = [&](auto&& f) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < NR; ++r) f(i, j, r);
  };
  V x[TM][TN];
  auto load = [&](const void* src, int64_t ld) {
    const __amdgpu_buffer_rsrc_t rs = buffer(src, ld);
    each([&](int i, int j, int r) { x[i][j][r] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, offset(i, j, r, ld), 0, 0)); });
  };
  each([&](int i, int j, int r) { v[i][j][r] *= epi.alpha; });
  if (epi.bias) {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(epi.bias, (uint32_t)(N * 4));
    float b[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) b[j] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)((col0 + 16 * j) * 4), 0, 0));
    each([&](int i, int j, int r) { v[i][j][r] += b[j]; });
  }
  if (epi.aux_out) {
    const __amdgpu_buffer_rsrc_t rs = buffer(epi.aux_out, epi.ld_aux_out);
    each([&](int i, int j, int r) { __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v[i][j][r]), rs, offset(i, j, r, epi.ld_aux_out), 0, 0); });
  }
  if (epi.act == PF_ACT_GELU) {
    each([&](int i, int j, int r) { v[i][j][r] = pf_gelu_erf(v[i][j][r]); });
  } else if (epi.act != PF_ACT_NONE) {
    each([&](int i, int j, int r) { v[i][j][r] = pf_act(epi.act, v[i][j][r]); });
  }
  if (epi.dact != PF_ACT_NONE) {
    load(epi.aux_in, epi.ld_aux_in);
    if (epi.dact == PF_ACT_GELU) each([&](int i, int j, int r) { v[i][j][r] *= pf_gelu_erf_grad(x[i][j][r]); });
    else each([&](int i, int j, int r) { v[i][j][r] *= pf_act_grad(epi.dact, x[i][j][r]); });
  }
  if (epi.residual) {
    load(epi.residual, epi.ld_res);
    each([&](int i, int j, int r) { v[i][j][r] += x[i][j][r]; });
  }
  const float* C = (const float*)epi.C + c_base;
  if (epi.beta) {
    load(C, epi.ldc);
    each([&](int i, int j, int r) { v[i][j][r] += x[i][j][r]; });
  }
  const __amdgpu_buffer_rsrc_t rs = buffer(C, epi.ldc);
  each([&](int i, int j, int r) { __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v[i][j][r]), rs, offset(i, j, r, epi.ldc), 0, 0); });
}

// what the vector epilogue needs of a product over tiles of bm rows: fp32 operands, byte offsets inside a tile in 31 bits
inline int epi_f32_vec_ok(const pf_gemm_desc& d, int bm) {
  const int64_t lim = (1ll << 31) / (4 * bm) - 1;
  return d.c_dtype == PF_F32 && (!d.bias || d.bias_dtype == PF_F32) && (!d.residual || d.res_dtype == PF_F32) && d.ldc < lim &&
         (!d.residual || d.ld_res < lim) && (!d.aux_in || d.ld_aux_in < lim) && (!d.aux_out || d.ld_aux_out < lim);
}

}  // namespace

// pf_gemm_f32_depth.hip: the tile it takes for a product, as the profiler prints it, and the launch
const char* pf_gemm_f32_depth_shape(const pf_gemm_desc& d);
int pf_gemm_f32_depth(const pf_gemm_desc& d, hipStream_t st);
