// Measurement aid: the matrix-instruction stream of a GEMM tile with nothing else around it.  Fragments stay in
// registers: no loads, no LDS, no barriers.  Timed on all CUs it gives the rate the MFMA pipes sustain under the
// board's power limit with this operand data, the ceiling any GEMM K loop on this device can approach (the published
// peak assumes the full boost clock).  mfma16_rate_kernel is the direct-to-LDS kernel's stream: v_mfma_f32_16x16x32, an
// 8 x 4 grid of 16x16 blocks per wavefront and two wavefronts per SIMD, as its eight-wavefront 256x256 tile has them.
// mfma_rate_kernel issues v_mfma_f32_32x32x16 on a 4 x 4 grid of 32x32 blocks, one wavefront per SIMD: the shape the
// register-staged and attention kernels use, for comparison.
#include "pf_gemm_common.h"

template <int DT>
__global__ __launch_bounds__(256, 1) void mfma_rate_kernel(const uint16_t* __restrict__ operands, int64_t iters,
                                                            float* __restrict__ sink) {
  typedef short short8_t __attribute__((ext_vector_type(8)));
  const int lane = threadIdx.x & 63;
  short8_t fa[4], fb[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    fa[i] = *(const short8_t*)(operands + ((i * 64 + lane) * 8));
    fb[i] = *(const short8_t*)(operands + ((256 + i * 64 + lane) * 8));
  }
  float16_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  for (int64_t it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = Mfma<DT>::run(__builtin_bit_cast(uint4, fa[i]), __builtin_bit_cast(uint4, fb[j]), acc[i][j]);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) s += acc[i][j][r];
  // every lane's share of the checksum keeps the loop alive; a wavefront's 64 values add up to
  // iters * sum_{i,j} sum(A_i . B_j)
  sink[(int64_t)blockIdx.x * 256 + threadIdx.x] = s;
}

template <int DT>
__global__ __launch_bounds__(512, 2) void mfma16_rate_kernel(const uint16_t* __restrict__ operands, int64_t iters,
                                                              float* __restrict__ sink) {
  typedef short short8_t __attribute__((ext_vector_type(8)));
  const int lane = threadIdx.x & 63;
  short8_t fa[8], fb[4];
#pragma unroll
  for (int i = 0; i < 8; ++i) fa[i] = *(const short8_t*)(operands + ((i * 64 + lane) * 8));
#pragma unroll
  for (int i = 0; i < 4; ++i) fb[i] = *(const short8_t*)(operands + ((512 + i * 64 + lane) * 8));
  float4_t acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
  for (int64_t it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = Mfma<DT>::run16(fa[i], fb[j], acc[i][j]);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) s += acc[i][j][r];
  sink[(int64_t)blockIdx.x * 512 + threadIdx.x] = s;   // (the checksum of mfma_rate_kernel)
}

extern "C" int pf_mfma_rate(int dtype, const void* operands, int64_t iters, int workgroups, float* sink, void* stream) {
  PF_REQUIRE(dtype == PF_F16 || dtype == PF_BF16, "pf_mfma_rate: dtype %d is not a 16-bit type", dtype);
  PF_REQUIRE(operands != nullptr && sink != nullptr && pf_aligned(operands, 16), "pf_mfma_rate: operands / sink missing or unaligned");
  PF_REQUIRE(iters > 0 && workgroups > 0 && workgroups <= 65536, "pf_mfma_rate: iters %lld, workgroups %d", (long long)iters, workgroups);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == PF_F16) mfma_rate_kernel<PF_F16><<<workgroups, 256, 0, st>>>((const uint16_t*)operands, iters, sink);
  else mfma_rate_kernel<PF_BF16><<<workgroups, 256, 0, st>>>((const uint16_t*)operands, iters, sink);
  PF_CHECK_LAUNCH("pf_mfma_rate");
  return PF_OK;
}

extern "C" int pf_mfma16_rate(int dtype, const void* operands, int64_t iters, int workgroups, float* sink, void* stream) {
  PF_REQUIRE(dtype == PF_F16 || dtype == PF_BF16, "pf_mfma16_rate: dtype %d is not a 16-bit type", dtype);
  PF_REQUIRE(operands != nullptr && sink != nullptr && pf_aligned(operands, 16), "pf_mfma16_rate: operands / sink missing or unaligned");
  PF_REQUIRE(iters > 0 && workgroups > 0 && workgroups <= 65536, "pf_mfma16_rate: iters %lld, workgroups %d", (long long)iters, workgroups);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == PF_F16) mfma16_rate_kernel<PF_F16><<<workgroups, 512, 0, st>>>((const uint16_t*)operands, iters, sink);
  else mfma16_rate_kernel<PF_BF16><<<workgroups, 512, 0, st>>>((const uint16_t*)operands, iters, sink);
  PF_CHECK_LAUNCH("pf_mfma16_rate");
  return PF_OK;
}
