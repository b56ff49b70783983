// Fused attention (forward, dQ, dK/dV) on gfx950 MFMA: softmax(Q K^T * scale [+ causal]) V
// without materialising the [B,H,Tq,Tk] score / probability matrices.
//
// All three kernels work in the "transposed world": score tiles are computed so that a
// lane owns ONE column of the tile (lane % 32) and 16 rows of it in registers.  The
// softmax statistics of that column are then a per-lane loop plus one exchange with
// lane ^ 32, and the probabilities can be fed straight back into the next MFMA as the
// B operand (the MFMA reduction index may be permuted freely as long as A and B agree),
// so P never goes through LDS.
//
//   forward / dQ kernel : tile = S^T[kv][q], column = query row   (workgroup = 128 queries)
//   dK/dV kernel        : tile = S[q][kv],   column = key row     (workgroup = 128 keys)
//
// Operands whose MFMA reduction index is NOT their contiguous dimension (V in forward,
// K in dQ, Q and dO in dK/dV) stay in their natural [token][hd] layout in LDS and are read
// with the transposing LDS read (ds_read_b64_tr_b16); no transposed copy exists anywhere.
//
// Q, K, V, O and their gradients are [B, H, T, hd] tensors addressed with element
// strides (batch, head, token) and unit stride along hd, so heads can live inside a
// packed qkv projection and the output can be token-major.

#include "pf_common.h"

namespace {

constexpr int KT = 64;        // keys (forward/dQ) or queries (dK/dV) per LDS tile
constexpr float LOG2E = 1.4426950408889634f;
constexpr float O_LO = 2048.f;   // scale of what rounding O lost: at most as large as O itself, in fp16 too

struct AttnArgs {
  const uint16_t* q; const uint16_t* k; const uint16_t* v; const uint16_t* o; const uint16_t* d_o;
  uint16_t* out; uint16_t* o_lo; uint16_t* dq; uint16_t* dk; uint16_t* dv;
  float* lse; float* delta;
  int64_t q_sb, q_sh, q_st, k_sb, k_sh, k_st, v_sb, v_sh, v_st, o_sb, o_sh, o_st;
  int64_t do_sb, do_sh, do_st, dq_sb, dq_sh, dq_st, dk_sb, dk_sh, dk_st, dv_sb, dv_sh, dv_st;
  int B, H, Tq, Tk, hd, causal;
  float scale;
};

template <int DT> struct M32;
template <> struct M32<PF_F16> {
  static __device__ __forceinline__ float16_t run(uint4 a, uint4 b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0,
                                                  0, 0);
  }
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) { return pf_pack2_f16(lo, hi); }
  static __device__ __forceinline__ float lo(uint32_t w) { return pf_f16_bits_to_f32((uint16_t)(w & 0xffffu)); }
  static __device__ __forceinline__ float hi(uint32_t w) { return pf_f16_bits_to_f32((uint16_t)(w >> 16)); }
};
template <> struct M32<PF_BF16> {
  static __device__ __forceinline__ float16_t run(uint4 a, uint4 b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) { return pf_pack2_bf16(lo, hi); }
  static __device__ __forceinline__ float lo(uint32_t w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
};

// registers r..r+7 of an accumulator tile -> one 16-byte MFMA operand (8 x 16-bit)
template <int DT>
__device__ __forceinline__ uint4 pack8(const float16_t& a, int r) {
  return make_uint4(M32<DT>::pack(a[r], a[r + 1]), M32<DT>::pack(a[r + 2], a[r + 3]),
                    M32<DT>::pack(a[r + 4], a[r + 5]), M32<DT>::pack(a[r + 6], a[r + 7]));
}

// row index inside a 32-row accumulator tile of register r for this lane
__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// 16-byte global load of 8 consecutive hd elements of one token row; zero when the
// token or the hd chunk is out of range
__device__ __forceinline__ uint4 load_row8(const uint16_t* base, int64_t st, int t, int T, int h0, int hd) {
  if (t < T && h0 < hd) return *(const uint4*)(base + (int64_t)t * st + h0);
  return make_uint4(0, 0, 0, 0);
}

template <int DT>
__device__ __forceinline__ void unpack8(const uint4& r, float (&v)[8]) {
  const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (DT == PF_F16) {
      v[2 * k] = pf_f16_bits_to_f32((uint16_t)(w[k] & 0xffffu));
      v[2 * k + 1] = pf_f16_bits_to_f32((uint16_t)(w[k] >> 16));
    } else {
      v[2 * k] = __uint_as_float(w[k] << 16);
      v[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
    }
  }
}

// One [ROWS tokens][HD] tile in flight: NV 16-byte vectors per thread, loaded from global into
// registers while the previous tile is being multiplied, stored to LDS ([KT][HD + 8]) afterwards.
// The loads go through a buffer descriptor at the tile's first row: an offset out of its range reads zeros, where a test in front of
// each load was a branch and a 64-bit product (2048 causal tokens x 128 heads of 64: forward 112 -> 106 us, backward 350 -> 332;
// 577 x 32 heads of 88: forward 23.0 -> 19.2).  FAR: tokens so far apart that a tile spans 2 GiB keep that form.
template <int HD, int ROWS = KT, bool FAR = false> struct Tile {
  static constexpr int LD = HD + 8, VPR = HD / 8, NV = (ROWS * VPR + 255) / 256;
  uint4 v[NV];
  __device__ __forceinline__ void load(const uint16_t* base, int64_t st, int t0, int T, int hd, int tid) {
    if constexpr (FAR) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = tid + i * 256;
        v[i] = (e < ROWS * VPR) ? load_row8(base, st, t0 + e / VPR, T, (e % VPR) * 8, hd) : make_uint4(0, 0, 0, 0);
      }
    } else {
      typedef int v4 __attribute__((ext_vector_type(4)));
      const __amdgpu_buffer_rsrc_t rs =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base + (int64_t)t0 * st), 0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = tid + i * 256, t = e / VPR, c = (e % VPR) * 8;
        const bool ok = e < ROWS * VPR && t0 + t < T && c < hd;
        const v4 x = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(ok ? (uint32_t)(t * (int)st + c) * 2u : 0x80000000u), 0, 0);
        v[i] = make_uint4((uint32_t)x.x, (uint32_t)x.y, (uint32_t)x.z, (uint32_t)x.w);
      }
    }
  }
  __device__ __forceinline__ void store(uint16_t* s, int tid) const {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = tid + i * 256;
      if (e < ROWS * VPR) *(uint4*)(s + (e / VPR) * LD + (e % VPR) * 8) = v[i];
    }
  }
};

#define PF_LDS16(T) __attribute__((address_space(3))) T*
typedef short short4v_t __attribute__((ext_vector_type(4)));

// Transposing LDS read.  The 16 lanes of a group each name an 8-byte chunk (4 elements);
// group lane j must point at row k0 + j/4, columns n0 + 4*(j%4); lane i of the group then
// receives the four elements (k0 .. k0+3, column n0 + i).
__device__ __forceinline__ uint2 lds_read_tr(const uint16_t* p) {
  const short4v_t r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PF_LDS16(short4v_t))(uintptr_t)p);
  return __builtin_bit_cast(uint2, r);
}

// A operand X^T[row = hd index][k = token] for the 16-token chunk starting at `t0` of a
// natural [token][LD] tile, hd rows o32 .. o32+31, with the token permutation of pack8():
// element i of the lane <-> token t0 + 8*(i/4) + 4*(lane/32) + (i%4)
template <int LD>
__device__ __forceinline__ uint4 frag_tr(const uint16_t* s, int t0, int o32, int lane) {
  const int g = lane >> 4, j = lane & 15;
  const uint16_t* p = s + (t0 + 4 * (g >> 1) + (j >> 2)) * LD + o32 + 16 * (g & 1) + 4 * (j & 3);
  const uint2 lo = lds_read_tr(p), hi = lds_read_tr(p + 8 * LD);
  return make_uint4(lo.x, lo.y, hi.x, hi.y);
}

// Workgroup -> (row block, batch*head).  The hardware starts workgroups in the order of their
// linear id (x fastest).  Under a causal mask the blocks of one head differ in work by up to the
// number of blocks (a query block sweeps the keys up to its diagonal, a key block the queries from
// its diagonal on): the heaviest blocks of EVERY head are started first, the lightest ones fill the
// tail.  Without a mask all blocks are alike and neighbours keep sharing a head's operands in L2.
__device__ __forceinline__ void attn_block(const AttnArgs& a, bool heavy_is_last, int& blk, int& bh) {
  blk = (int)blockIdx.x;
  bh = (int)blockIdx.y;
  if (a.causal) {
    const int id = (int)(blockIdx.y * gridDim.x + blockIdx.x), nbh = (int)gridDim.y;
    const int k = id / nbh;
    bh = id % nbh;
    blk = heavy_is_last ? (int)gridDim.x - 1 - k : k;
  }
}

// ---------------------------------------------------------------------------------
// forward: one workgroup = 128 queries of one (batch, head); wavefront w owns 32 of them
//
// Occupancy (second __launch_bounds__ argument) of the tiled kernels: a tile step is a chain of
// dependent MFMA -> softmax -> MFMA phases with LDS reads in between, so a SIMD that holds a single
// wavefront idles through every latency.  The register budget is set so that three (forward, head
// dim <= 64: 152 VGPRs) or two (dQ: 240, dK/dV: 247) wavefronts share a SIMD without spilling;
// measured on 2048 causal tokens x 64 heads: forward 76 -> 56 us, backward 280 -> 194 us.
// Head dims above 64 hold two (forward: 204 / 248 VGPRs at 96 / 128; dQ up to 96: 251), where the compiler left to
// itself takes registers for one: forward 577 tokens x 56 heads of 88 47 -> 28 us, 2048 causal tokens x 64 heads of
// 128 166 -> 104 us.  dQ of 128 and dK/dV above 96 would spill (dK/dV of 128 by 307 registers: 498 -> 793 us).
// ---------------------------------------------------------------------------------
template <int DT, int HD, bool FAR = false>
__global__ __launch_bounds__(256, HD <= 64 ? 3 : 2) void attn_fwd_kernel(const AttnArgs a) {
  constexpr int NC = HD / 16, NO = HD / 32, KLD = HD + 8;
  __shared__ __align__(16) uint16_t sK[KT * KLD];
  __shared__ __align__(16) uint16_t sV[KT * KLD];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int qb, bh;
  attn_block(a, true, qb, bh);
  const int b = bh / a.H, h = bh % a.H;
  const int q0 = qb * 128 + wave * 32;
  const int qi = q0 + (lane & 31);          // this lane's query row
  const uint16_t* Q = a.q + b * a.q_sb + h * a.q_sh;
  const uint16_t* K = a.k + b * a.k_sb + h * a.k_sh;
  const uint16_t* V = a.v + b * a.v_sb + h * a.v_sh;
  const float sc = a.scale * LOG2E;
  const int shift = a.Tk - a.Tq;            // causal: key j visible to query i iff j <= i + shift

  uint4 qf[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) qf[c] = load_row8(Q, a.q_st, qi, a.Tq, c * 16 + (lane >> 5) * 8, a.hd);

  float16_t oacc[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[o][r] = 0.f;
  float m = -INFINITY, l = 0.f;

  int k_end = a.Tk;
  if (a.causal) {
    const int last_q = min(qb * 128 + 127, a.Tq - 1);
    k_end = min(a.Tk, last_q + shift + 1);
  }
  Tile<HD, KT, FAR> tk, tv;
  tk.load(K, a.k_st, 0, a.Tk, a.hd, tid);
  tv.load(V, a.v_st, 0, a.Tk, a.hd, tid);
  for (int k0 = 0; k0 < k_end; k0 += KT) {
    __syncthreads();                     // previous tile's LDS reads are done
    tk.store(sK, tid);
    tv.store(sV, tid);
    if (k0 + KT < k_end) {               // next tile's global loads fly during this tile's math
      tk.load(K, a.k_st, k0 + KT, a.Tk, a.hd, tid);
      tv.load(V, a.v_st, k0 + KT, a.Tk, a.hd, tid);
    }
    __syncthreads();
    float16_t s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[t][r] = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const uint4 kf = *(const uint4*)(sK + (t * 32 + (lane & 31)) * KLD + c * 16 + (lane >> 5) * 8);
        s[t] = M32<DT>::run(kf, qf[c], s[t]);
      }
    }
    // only the tile on the causal diagonal and the ragged last tile need per-element masks
    const bool masked = (k0 + KT > a.Tk) || (a.causal && k0 + KT - 1 > q0 + shift);
    float mx = m;   // running maximum of the RAW scores (scale > 0, so the ordering is the same)
    if (masked) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kj = k0 + t * 32 + acc_row(r, lane);
          const bool ok = kj < a.Tk && (!a.causal || kj <= qi + shift);
          s[t][r] = ok ? s[t][r] : -INFINITY;
          mx = fmaxf(mx, s[t][r]);
        }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[t][r]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const bool dead = (mx == -INFINITY);
    const float moff = dead ? 0.f : -mx * sc;
    const float alpha = dead ? 1.f : __builtin_amdgcn_exp2f((m - mx) * sc);
    float psum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[t][r], sc, moff));   // masked entries: exp2(-inf) = 0
        s[t][r] = p;
        psum += p;
      }
    l = l * alpha + psum;
    m = mx;
    if (__any(alpha != 1.f)) {   // wavefront-uniform: once the maxima have settled nothing is rescaled
#pragma unroll
      for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[o][r] *= alpha;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint4 pf = pack8<DT>(s[j >> 1], 8 * (j & 1));
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        oacc[o] = M32<DT>::run(frag_tr<KLD>(sV, 16 * j, o * 32, lane), pf, oacc[o]);
      }
    }
  }
  l += __shfl_xor(l, 32, 64);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (qi < a.Tq) {
    uint16_t* O = a.out + b * a.o_sb + h * a.o_sh + (int64_t)qi * a.o_st;
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int h0 = o * 32 + 8 * g + 4 * (lane >> 5);
        if (h0 < a.hd) {
          const uint2 w = make_uint2(M32<DT>::pack(oacc[o][4 * g] * inv, oacc[o][4 * g + 1] * inv),
                                     M32<DT>::pack(oacc[o][4 * g + 2] * inv, oacc[o][4 * g + 3] * inv));
          *(uint2*)(O + h0) = w;
          if constexpr (HD > 96) {
            if (a.o_lo != nullptr) {
              auto rest = [&](float v, float kept) { return (v * inv - kept) * O_LO; };
              *(uint2*)(a.o_lo + (O - a.out) + h0) =
                  make_uint2(M32<DT>::pack(rest(oacc[o][4 * g], M32<DT>::lo(w.x)), rest(oacc[o][4 * g + 1], M32<DT>::hi(w.x))),
                             M32<DT>::pack(rest(oacc[o][4 * g + 2], M32<DT>::lo(w.y)), rest(oacc[o][4 * g + 3], M32<DT>::hi(w.y))));
            }
          }
        }
      }
    if ((lane >> 5) == 0) a.lse[((int64_t)bh) * a.Tq + qi] = (l > 0.f) ? (m * sc + log2f(l)) / LOG2E : -INFINITY;
  }
}

// ---------------------------------------------------------------------------------
// dQ: same tiling as forward (column = query); dQ^T[hd][q] += K^T[hd][kv] dS^T[kv][q]
//
// It holds its queries' rows of dO and so also forms delta[b,h,q] = sum_hd dO * O, for itself and for the dK/dV kernel that is launched
// after it; a kernel of its own read dO once more (7.2 us of 43 + 7 at 4096 x 20 heads of 64, 41 us beside another stage's work at
// 8192 x 32 heads; a step of 30 transformer blocks 50.1 -> 49.3 ms, a 1B decoder's 189.2 -> 188.5).  With o_lo, from O to
// twice its digits: where one key has most of a query's weight, dP - delta is a small difference, and the rounding of O is the
// largest error in it.
// ---------------------------------------------------------------------------------
template <int DT, int HD, bool FAR = false>
__global__ __launch_bounds__(256, HD <= 96 ? 2 : 1) void attn_dq_kernel(const AttnArgs a) {
  constexpr int NC = HD / 16, NO = HD / 32, KLD = HD + 8;
  __shared__ __align__(16) uint16_t sK[KT * KLD];
  __shared__ __align__(16) uint16_t sV[KT * KLD];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int qb, bh;
  attn_block(a, true, qb, bh);
  const int b = bh / a.H, h = bh % a.H;
  const int q0 = qb * 128 + wave * 32;
  const int qi = q0 + (lane & 31);
  const uint16_t* Q = a.q + b * a.q_sb + h * a.q_sh;
  const uint16_t* K = a.k + b * a.k_sb + h * a.k_sh;
  const uint16_t* V = a.v + b * a.v_sb + h * a.v_sh;
  const uint16_t* DO = a.d_o + b * a.do_sb + h * a.do_sh;
  const float sc = a.scale * LOG2E;
  const int shift = a.Tk - a.Tq;

  uint4 qf[NC], dof[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    qf[c] = load_row8(Q, a.q_st, qi, a.Tq, c * 16 + (lane >> 5) * 8, a.hd);
    dof[c] = load_row8(DO, a.do_st, qi, a.Tq, c * 16 + (lane >> 5) * 8, a.hd);
  }
  const bool qok = qi < a.Tq;
  // a query row past the end keeps lse = +inf so that its probabilities are exactly zero
  const float lse2 = qok ? a.lse[(int64_t)bh * a.Tq + qi] * LOG2E : INFINITY;
  float dlt = 0.f;
  {
    const uint16_t* O = a.o + b * a.o_sb + h * a.o_sh;
    uint4 of[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) of[c] = load_row8(O, a.o_st, qi, a.Tq, c * 16 + (lane >> 5) * 8, a.hd);
    // eight products to a chain of sums, then neighbours in pairs (one chain of the half row that a lane holds is 1.5 times as far from 64 bits at
    // head dim 64 in fp16, 9.7e-8 against 6.5e-8, and 1.9 times at 128, 1.4e-7 against 7.6e-8)
    float part[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float x[8], y[8];
      unpack8<DT>(of[c], x);
      unpack8<DT>(dof[c], y);
      if (a.o_lo != nullptr) {
        float z[8];
        unpack8<DT>(load_row8(a.o_lo + (O - a.o), a.o_st, qi, a.Tq, c * 16 + (lane >> 5) * 8, a.hd), z);
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] += z[k] * (1.f / O_LO);
      }
      part[c] = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) part[c] += x[k] * y[k];
      part[c] += __shfl_xor(part[c], 32, 64);   // (the chunk beside it)
    }
#pragma unroll
    for (int w = 1; w < NC; w *= 2)
#pragma unroll
      for (int c = 0; c + w < NC; c += 2 * w) part[c] += part[c + w];
    dlt = part[0];
    if (qok && (lane >> 5) == 0) a.delta[(int64_t)bh * a.Tq + qi] = dlt;
  }

  float16_t acc[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[o][r] = 0.f;

  int k_end = a.Tk;
  if (a.causal) {
    const int last_q = min(qb * 128 + 127, a.Tq - 1);
    k_end = min(a.Tk, last_q + shift + 1);
  }
  Tile<HD, KT, FAR> tk, tv;
  tk.load(K, a.k_st, 0, a.Tk, a.hd, tid);
  tv.load(V, a.v_st, 0, a.Tk, a.hd, tid);
  for (int k0 = 0; k0 < k_end; k0 += KT) {
    __syncthreads();
    tk.store(sK, tid);
    tv.store(sV, tid);
    if (k0 + KT < k_end) {
      tk.load(K, a.k_st, k0 + KT, a.Tk, a.hd, tid);
      tv.load(V, a.v_st, k0 + KT, a.Tk, a.hd, tid);
    }
    __syncthreads();
    const bool masked = (k0 + KT > a.Tk) || (a.causal && k0 + KT - 1 > q0 + shift);
    float16_t s[2], dp[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[t][r] = dp[t][r] = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int off = (t * 32 + (lane & 31)) * KLD + c * 16 + (lane >> 5) * 8;
        s[t] = M32<DT>::run(*(const uint4*)(sK + off), qf[c], s[t]);
        dp[t] = M32<DT>::run(*(const uint4*)(sV + off), dof[c], dp[t]);
      }
      if (masked) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kj = k0 + t * 32 + acc_row(r, lane);
          const bool ok = kj < a.Tk && (!a.causal || kj <= qi + shift);
          const float p = ok ? __builtin_amdgcn_exp2f(s[t][r] * sc - lse2) : 0.f;
          s[t][r] = p * (dp[t][r] - dlt);   // dS^T / scale (the scale is applied to dQ at the end)
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[t][r] = __builtin_amdgcn_exp2f(s[t][r] * sc - lse2) * (dp[t][r] - dlt);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint4 dsf = pack8<DT>(s[j >> 1], 8 * (j & 1));
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        acc[o] = M32<DT>::run(frag_tr<KLD>(sK, 16 * j, o * 32, lane), dsf, acc[o]);
      }
    }
  }
  if (qok) {
    uint16_t* DQ = a.dq + b * a.dq_sb + h * a.dq_sh + (int64_t)qi * a.dq_st;
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int h0 = o * 32 + 8 * g + 4 * (lane >> 5);
        if (h0 < a.hd)
          *(uint2*)(DQ + h0) = make_uint2(M32<DT>::pack(acc[o][4 * g] * a.scale, acc[o][4 * g + 1] * a.scale),
                                          M32<DT>::pack(acc[o][4 * g + 2] * a.scale, acc[o][4 * g + 3] * a.scale));
      }
  }
}

// ---------------------------------------------------------------------------------
// dK/dV: column = key row; S[q][kv] = Q K^T, dV^T[hd][kv] += dO^T[hd][q] P[q][kv],
//        dK^T[hd][kv] += Q^T[hd][q] dS[q][kv]
// ---------------------------------------------------------------------------------
// SPLITQ (few keys, many queries: cross attention to a short context): a workgroup owns ONE 32-key
// tile, its four wavefronts each take a quarter of every staged block of 128 queries, and their
// accumulators are added at the end through LDS in wavefront order, so that a head's dK/dV come
// from 4 x ceil(Tk / 32) wavefronts instead of ceil(Tk / 32).
template <int DT, int HD, bool SPLITQ = false, bool FAR = false>
__global__ __launch_bounds__(256, SPLITQ || HD > 96 ? 1 : 2) void attn_dkv_kernel(const AttnArgs a) {
  constexpr int NC = HD / 16, NO = HD / 32, QLD = HD + 8;
  constexpr int QT = SPLITQ ? 128 : KT;        // queries staged per iteration
  constexpr int NH = SPLITQ ? 1 : 2;           // 32-query halves per wavefront and iteration
  __shared__ __align__(16) uint16_t sQD[2 * QT * QLD];
  uint16_t* sQ = sQD;
  uint16_t* sDO = sQD + QT * QLD;
  __shared__ float sLse[QT], sDelta[QT];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int kb, bh;
  attn_block(a, false, kb, bh);
  const int b = bh / a.H, h = bh % a.H;
  const int kw0 = SPLITQ ? kb * 32 : kb * 128 + wave * 32;     // this wavefront's first key row
  const int qoff = SPLITQ ? wave * 32 : 0;                     // its first query row inside a staged block
  const int kj = kw0 + (lane & 31);                            // this lane's key row
  const uint16_t* Q = a.q + b * a.q_sb + h * a.q_sh;
  const uint16_t* K = a.k + b * a.k_sb + h * a.k_sh;
  const uint16_t* V = a.v + b * a.v_sb + h * a.v_sh;
  const uint16_t* DO = a.d_o + b * a.do_sb + h * a.do_sh;
  const float sc = a.scale * LOG2E;
  const int shift = a.Tk - a.Tq;
  const bool kok = kj < a.Tk;

  uint4 kf[NC], vf[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    kf[c] = load_row8(K, a.k_st, kj, a.Tk, c * 16 + (lane >> 5) * 8, a.hd);
    vf[c] = load_row8(V, a.v_st, kj, a.Tk, c * 16 + (lane >> 5) * 8, a.hd);
  }
  float16_t dk[NO], dv[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int r = 0; r < 16; ++r) dk[o][r] = dv[o][r] = 0.f;

  int q_begin = 0;
  if (a.causal) {  // queries i with i + shift >= first key of the block see it
    q_begin = max(0, (SPLITQ ? kb * 32 : kb * 128) - shift);
    q_begin = q_begin / QT * QT;
  }
  Tile<HD, QT, FAR> tq, tdo;
  float r_lse = 0.f, r_dlt = 0.f;
  auto prefetch = [&](int q0) {
    tq.load(Q, a.q_st, q0, a.Tq, a.hd, tid);
    tdo.load(DO, a.do_st, q0, a.Tq, a.hd, tid);
    if (tid < QT) {
      const int qi = q0 + tid;
      // rows past the end: Q and dO rows are zero, lse = +inf makes their P exactly zero
      r_lse = qi < a.Tq ? a.lse[(int64_t)bh * a.Tq + qi] * LOG2E : INFINITY;
      r_dlt = qi < a.Tq ? a.delta[(int64_t)bh * a.Tq + qi] : 0.f;
    }
  };
  if (q_begin < a.Tq) prefetch(q_begin);
  for (int q0 = q_begin; q0 < a.Tq; q0 += QT) {
    __syncthreads();
    tq.store(sQ, tid);
    tdo.store(sDO, tid);
    if (tid < QT) {
      sLse[tid] = r_lse;
      sDelta[tid] = r_dlt;
    }
    if (q0 + QT < a.Tq) prefetch(q0 + QT);
    __syncthreads();
    // causal: rows before `first` (of this lane's) do not see its key: a constant against a threshold that the compiler
    // cannot take apart (it would test `causal` again in every compare).  Each half's P and dS are multiplied before the next half's
    // scores exist: with both alive four registers spilled as soon as anything else changed, and their reloads wait
    // for the next tile's loads.  2048 causal tokens x 128 heads backward 350 -> 332 us with the loads through descriptors (see
    // Tile; without these two 349), 1024 x 80 heads 149 -> 137.
    int first = a.causal ? kj - (q0 + qoff + 4 * (lane >> 5) + shift) : 0;
    if constexpr (HD == 64) asm("" : "+v"(first));   // (96 has no register left for it)
#pragma unroll
    for (int t = 0; t < NH; ++t) {
      float16_t s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int off = (qoff + t * 32 + (lane & 31)) * QLD + c * 16 + (lane >> 5) * 8;
        s = M32<DT>::run(*(const uint4*)(sQ + off), kf[c], s);
        dp = M32<DT>::run(*(const uint4*)(sDO + off), vf[c], dp);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int ql = qoff + t * 32 + acc_row(r, lane);
        float p = __builtin_amdgcn_exp2f(s[r] * sc - sLse[ql]);
        if (t * 32 + 8 * (r >> 2) + (r & 3) < first) p = 0.f;
        s[r] = p;                                         // P
        dp[r] = p * (dp[r] - sDelta[ql]);              // dS / scale (applied to dK at the end)
      }
#pragma unroll
      for (int j = 2 * t; j < 2 * t + 2; ++j) {
        const uint4 pf = pack8<DT>(s, 8 * (j & 1));
        const uint4 dsf = pack8<DT>(dp, 8 * (j & 1));
#pragma unroll
        for (int o = 0; o < NO; ++o) {
          dv[o] = M32<DT>::run(frag_tr<QLD>(sDO, qoff + 16 * j, o * 32, lane), pf, dv[o]);
          dk[o] = M32<DT>::run(frag_tr<QLD>(sQ, qoff + 16 * j, o * 32, lane), dsf, dk[o]);
        }
      }
    }
  }
  if constexpr (SPLITQ) {
    // wavefront 0 adds the other three's accumulators in wavefront order: dV, then dK
    float* red = (float*)sQD;
    static_assert(3 * NO * 16 * 64 * 4 <= 2 * QT * QLD * 2, "reduction patch exceeds the operand tiles");
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
      __syncthreads();   // the tiles (or the previous pass's patch) are no longer read
      if (wave > 0) {
#pragma unroll
        for (int o = 0; o < NO; ++o)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            red[(((wave - 1) * NO + o) * 16 + r) * 64 + lane] = pass == 0 ? dv[o][r] : dk[o][r];
      }
      __syncthreads();
      if (wave == 0) {
#pragma unroll
        for (int w = 0; w < 3; ++w)
#pragma unroll
          for (int o = 0; o < NO; ++o)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const float x = red[((w * NO + o) * 16 + r) * 64 + lane];
              if (pass == 0) dv[o][r] += x; else dk[o][r] += x;
            }
      }
    }
    if (wave != 0) return;
  }
  if (kok) {
    uint16_t* DK = a.dk + b * a.dk_sb + h * a.dk_sh + (int64_t)kj * a.dk_st;
    uint16_t* DV = a.dv + b * a.dv_sb + h * a.dv_sh + (int64_t)kj * a.dv_st;
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int h0 = o * 32 + 8 * g + 4 * (lane >> 5);
        if (h0 < a.hd) {
          *(uint2*)(DK + h0) = make_uint2(M32<DT>::pack(dk[o][4 * g] * a.scale, dk[o][4 * g + 1] * a.scale),
                                          M32<DT>::pack(dk[o][4 * g + 2] * a.scale, dk[o][4 * g + 3] * a.scale));
          *(uint2*)(DV + h0) = make_uint2(M32<DT>::pack(dv[o][4 * g], dv[o][4 * g + 1]),
                                          M32<DT>::pack(dv[o][4 * g + 2], dv[o][4 * g + 3]));
        }
      }
  }
}


// =================================================================================
// Short sequences (Tq, Tk <= SHORT_T, e.g. ViT's 197 or 257 tokens): the two operands a workgroup
// sweeps over (K and V, or Q and dO) are loaded into LDS ONCE, whole, in their natural
// [token][hd] layout; after a single barrier every wavefront runs its tile loop without
// any further synchronisation.  Operands the MFMA needs transposed (V^T, K^T, Q^T, dO^T)
// are read from the natural layout with the transposing LDS read (ds_read_b64_tr_b16),
// so no transposed copy is made.
// =================================================================================
constexpr int SHORT_T = 288;   // 2 operands x 288 rows x (96 + 8) x 2 bytes = 117 KB of the 160 KB

// One head's [T][hd] operand for 16-byte loads without a branch: rows past T and chunks past hd get an offset out of the
// buffer's range, which reads zeros.  (T * st * 2 bytes are below 2 GiB, see short_ok.)
struct HeadRows {
  __amdgpu_buffer_rsrc_t rs;
  uint32_t st2;
  int T, hd;
  __device__ __forceinline__ HeadRows(const uint16_t* x, int64_t st, int T_, int hd_) : st2((uint32_t)(st * 2)), T(T_), hd(hd_) {
    rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, (int)((uint32_t)(T - 1) * st2 + (uint32_t)hd_ * 2u), 0x00020000);
  }
  __device__ __forceinline__ uint4 load(int t, int c) const {
    typedef int v4 __attribute__((ext_vector_type(4)));
    const v4 x = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(t < T && c < hd ? (uint32_t)t * st2 + (uint32_t)c * 2u : 0x80000000u), 0, 0);
    return make_uint4((uint32_t)x.x, (uint32_t)x.y, (uint32_t)x.z, (uint32_t)x.w);
  }
};

// Two whole [T][hd] operands of one head on their way to LDS, [rows][HD + 8] each (rows past T and hd chunks past hd are
// zero); NT threads.  Nothing else runs on a compute unit whose LDS one head fills, so a workgroup's loads go out
// together, up to the largest head of eight wavefronts in one batch, next to those of the rows that a wavefront keeps in
// registers: 257 tokens x 384 heads of 64 30.1 -> 28.6 us, 65 tokens x 256 heads 6.5 -> 5.7, in two batches behind the rows -> this.
template <int HD, int NT> struct HeadPair {
  static constexpr int VPR = HD / 8, LD = HD + 8, U = NT == 512 ? (HD == 64 ? 5 : 7) : (HD == 64 ? 4 : 6);
  uint4 vx[U], vy[U];
  __device__ __forceinline__ void issue(const HeadRows& x, const HeadRows& y, int rows, int tid, int e0 = 0) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int e = e0 + i * NT + tid;
      if (e0 + i * NT < rows * VPR) {
        vx[i] = x.load(e / VPR, (e % VPR) * 8);
        vy[i] = y.load(e / VPR, (e % VPR) * 8);
      }
    }
  }
  __device__ __forceinline__ void store(uint16_t* sx, uint16_t* sy, int n, int tid, int e0 = 0) const {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int e = e0 + i * NT + tid;
      if (e < n) {
        *(uint4*)(sx + (e / VPR) * LD + (e % VPR) * 8) = vx[i];
        *(uint4*)(sy + (e / VPR) * LD + (e % VPR) * 8) = vy[i];
      }
    }
  }
  // the first batch, issued before, and whatever it did not hold
  __device__ __forceinline__ void finish(const HeadRows& x, const HeadRows& y, uint16_t* sx, uint16_t* sy, int rows, int tid) {
    const int n = rows * VPR;
    store(sx, sy, n, tid);
    for (int e0 = NT * U; e0 < n; e0 += NT * U) {
      issue(x, y, rows, tid, e0);
      store(sx, sy, n, tid, e0);
    }
  }
};

// forward: workgroup = NT / 2 queries of one (batch, head) at a time, wavefront = 32 of them; keys in
// steps of 32.  NT = 512 (eight wavefronts): ONE workgroup covers a whole head, so that the head's K and V are fetched
// once instead of once per 128 queries.  With `share` its ninth tile (257 to 288 tokens) is everybody's: each wavefront sweeps an
// eighth of the keys, and the eight partial results meet in LDS, where one wavefront would sweep all keys with the other
// seven gone.  257 tokens x 384 heads of 64: 32.2 -> 30.1 us, backward 89 -> 78; x 16 heads of 88 17.7 -> 16.9.
// NT = 256: a wavefront whose tile lies past what the grid covers at once takes it in a second pass.
template <int DT, int HD, int NT>
__global__ __launch_bounds__(NT) void attn_fwd_short_kernel(const AttnArgs a, int rows, int share) {
  constexpr int NC = HD / 16, NO = HD / 32, LD = HD + 8;
  extern __shared__ __align__(16) uint16_t smem[];
  uint16_t* sK = smem;
  uint16_t* sV = smem + rows * LD;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = blockIdx.y, b = bh / a.H, h = bh % a.H;
  const int q_step = (int)gridDim.x * (NT / 2);
  int q0 = blockIdx.x * (NT / 2) + wave * 32;
  const uint16_t* Q = a.q + b * a.q_sb + h * a.q_sh;
  const float sc = a.scale * LOG2E;
  const int shift = a.Tk - a.Tq;

  const HeadRows rq(Q, a.q_st, a.Tq, a.hd);
  const HeadRows rk(a.k + b * a.k_sb + h * a.k_sh, a.k_st, a.Tk, a.hd), rv(a.v + b * a.v_sb + h * a.v_sh, a.v_st, a.Tk, a.hd);
  uint4 qf[NC];
  auto load_q = [&](int qs) {
#pragma unroll
    for (int c = 0; c < NC; ++c) qf[c] = rq.load(qs + (lane & 31), c * 16 + (lane >> 5) * 8);
  };
  {
    HeadPair<HD, NT> kv;
    kv.issue(rk, rv, rows, tid);
    load_q(q0);
    kv.finish(rk, rv, sK, sV, rows, tid);
  }
  __syncthreads();
  // no barrier follows but for a shared tile: a wavefront without a query tile leaves, one with several loops
  constexpr int SHARED = NT / 2;             // the tile from here on is shared by all wavefronts where they share one
  const bool sharing = NT == 512 && share;
  for (; q0 < a.Tq; q0 = sharing ? (q0 < SHARED ? SHARED : a.Tq) : q0 + q_step) {
  const bool shared = sharing && q0 >= SHARED;
  const int k_first = shared ? wave * 32 : 0, k_step = shared ? NT / 2 : 32;
  const int qi = q0 + (lane & 31);
  float16_t oacc[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[o][r] = 0.f;
  float m = -INFINITY, l = 0.f;
  const int k_end = a.causal ? min(a.Tk, min(q0 + 31, a.Tq - 1) + shift + 1) : a.Tk;
  for (int k0 = k_first; k0 < k_end; k0 += k_step) {
    float16_t s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const uint4 kf = *(const uint4*)(sK + (k0 + (lane & 31)) * LD + c * 16 + (lane >> 5) * 8);
      s = M32<DT>::run(kf, qf[c], s);
    }
    const bool masked = (k0 + 32 > a.Tk) || (a.causal && k0 + 31 > q0 + shift);
    float mx = m;
    if (masked) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kj = k0 + acc_row(r, lane);
        const bool ok = kj < a.Tk && (!a.causal || kj <= qi + shift);
        s[r] = ok ? s[r] : -INFINITY;
        mx = fmaxf(mx, s[r]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const bool dead = (mx == -INFINITY);
    const float moff = dead ? 0.f : -mx * sc;
    const float alpha = dead ? 1.f : __builtin_amdgcn_exp2f((m - mx) * sc);
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = __builtin_amdgcn_exp2f(fmaf(s[r], sc, moff));
      s[r] = p;
      psum += p;
    }
    l = l * alpha + psum;
    m = mx;
    if (__any(alpha != 1.f)) {
#pragma unroll
      for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[o][r] *= alpha;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint4 pf = pack8<DT>(s, 8 * j);
#pragma unroll
      for (int o = 0; o < NO; ++o) oacc[o] = M32<DT>::run(frag_tr<LD>(sV, k0 + 16 * j, o * 32, lane), pf, oacc[o]);
    }
  }
  l += __shfl_xor(l, 32, 64);
  if (!shared) {
    const int qn = sharing ? SHARED : q0 + q_step;
    if (qn < a.Tq) load_q(qn);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    if (qi < a.Tq) {
      uint16_t* O = a.out + b * a.o_sb + h * a.o_sh + (int64_t)qi * a.o_st;
#pragma unroll
      for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int h0 = o * 32 + 8 * g + 4 * (lane >> 5);
          if (h0 < a.hd)
            *(uint2*)(O + h0) = make_uint2(M32<DT>::pack(oacc[o][4 * g] * inv, oacc[o][4 * g + 1] * inv),
                                           M32<DT>::pack(oacc[o][4 * g + 2] * inv, oacc[o][4 * g + 3] * inv));
        }
      if ((lane >> 5) == 0) a.lse[((int64_t)bh) * a.Tq + qi] = (l > 0.f) ? (m * sc + log2f(l)) / LOG2E : -INFINITY;
    }
  } else if constexpr (NT == 512) {
    // each wavefront's maxima meet first, then its sums on the scale of the largest; wavefront w finishes registers
    // 2 w and 2 w + 1 of every tile of the head dimension
    float* xm = (float*)smem;             // [8][32]
    float* xl = xm + 256;                 // [8][32]
    float* xo = xl + 256;                 // [8][NO][16][64]
    __syncthreads();                      // K and V are no longer read
    if (lane < 32) xm[wave * 32 + lane] = m;
    __syncthreads();
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < 8; ++w) top = fmaxf(top, xm[w * 32 + (lane & 31)]);
    const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - top) * sc);
    if (lane < 32) xl[wave * 32 + lane] = l * f;
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
      for (int r = 0; r < 16; ++r) xo[((wave * NO + o) * 16 + r) * 64 + lane] = oacc[o][r] * f;
    __syncthreads();
    l = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) l += xl[w * 32 + (lane & 31)];
    const float inv = l > 0.f ? 1.f / l : 0.f;
    float x[2 * NO];
#pragma unroll
    for (int e = 0; e < 2 * NO; ++e) x[e] = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w)
#pragma unroll
      for (int e = 0; e < 2 * NO; ++e) x[e] += xo[((w * NO + e / 2) * 16 + 2 * wave + e % 2) * 64 + lane];
    if (qi < a.Tq) {
      uint16_t* O = a.out + b * a.o_sb + h * a.o_sh + (int64_t)qi * a.o_st;
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        const int h0 = o * 32 + acc_row(2 * wave, lane);
        if (h0 < a.hd) *(uint32_t*)(O + h0) = M32<DT>::pack(x[2 * o] * inv, x[2 * o + 1] * inv);
      }
      if (wave == 0 && lane < 32) a.lse[((int64_t)bh) * a.Tq + qi] = (l > 0.f) ? (top * sc + log2f(l)) / LOG2E : -INFINITY;
    }
  }
  }
}

// The sum over eight wavefronts of a tile's accumulators: wavefront w gets registers 2 w and 2 w + 1 of each of the
// NO tiles.  (All wavefronts call; `red` may hold what they have read until now.)
template <int NO>
__device__ __forceinline__ void sum_waves(const float16_t (&acc)[NO], float* red, int wave, int lane, float (&x)[2 * NO]) {
  __syncthreads();
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[((wave * NO + o) * 16 + r) * 64 + lane] = acc[o][r];
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 2 * NO; ++e) x[e] = 0.f;
#pragma unroll
  for (int w = 0; w < 8; ++w)
#pragma unroll
    for (int e = 0; e < 2 * NO; ++e) x[e] += red[((w * NO + e / 2) * 16 + 2 * wave + e % 2) * 64 + lane];
}

// dQ (and delta = rowsum(dO * O), which the dK/dV kernel launched after this one reads)
template <int DT, int HD, int NT>
__global__ __launch_bounds__(NT) void attn_dq_short_kernel(const AttnArgs a, float* delta_out, int rows, int share) {
  constexpr int NC = HD / 16, NO = HD / 32, LD = HD + 8;
  extern __shared__ __align__(16) uint16_t smem[];
  uint16_t* sK = smem;
  uint16_t* sV = smem + rows * LD;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = blockIdx.y, b = bh / a.H, h = bh % a.H;
  const int q_step = (int)gridDim.x * (NT / 2);
  int q0 = blockIdx.x * (NT / 2) + wave * 32;
  const uint16_t* Q = a.q + b * a.q_sb + h * a.q_sh;
  const uint16_t* DO = a.d_o + b * a.do_sb + h * a.do_sh;
  const uint16_t* OO = a.o + b * a.o_sb + h * a.o_sh;
  const float sc = a.scale * LOG2E;
  const int shift = a.Tk - a.Tq;

  constexpr int SHARED = NT / 2;             // the tile from here on is shared by all wavefronts where they share one
  const bool sharing = NT == 512 && share;
  const HeadRows rq(Q, a.q_st, a.Tq, a.hd), rdo(DO, a.do_st, a.Tq, a.hd), ro(OO, a.o_st, a.Tq, a.hd);
  const HeadRows rk(a.k + b * a.k_sb + h * a.k_sh, a.k_st, a.Tk, a.hd), rv(a.v + b * a.v_sb + h * a.v_sh, a.v_st, a.Tk, a.hd);
  uint4 qf[NC], dof[NC], of[NC];
  float dlt, lse2;
  // this lane's query row of the tile at `qs`: Q, dO, O and the row's lse
  auto load_rows = [&](int qs) {
    const int qr = qs + (lane & 31);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int h0 = c * 16 + (lane >> 5) * 8;
      qf[c] = rq.load(qr, h0);
      dof[c] = rdo.load(qr, h0);
      of[c] = ro.load(qr, h0);
    }
    lse2 = qr < a.Tq ? a.lse[(int64_t)bh * a.Tq + qr] * LOG2E : INFINITY;
  };
  // ... and its delta (also written out)
  auto row_delta = [&](int qs) {
    const int qr = qs + (lane & 31);
    dlt = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float x[8], y[8];
      unpack8<DT>(dof[c], x);
      unpack8<DT>(of[c], y);
#pragma unroll
      for (int k = 0; k < 8; ++k) dlt += x[k] * y[k];
    }
    dlt += __shfl_xor(dlt, 32, 64);
    if (qr < a.Tq && (lane >> 5) == 0 && (wave == 0 || !sharing || qs < SHARED)) delta_out[(int64_t)bh * a.Tq + qr] = dlt;
  };
  {
    HeadPair<HD, NT> kv;
    load_rows(q0);
    kv.issue(rk, rv, rows, tid);
    row_delta(q0);
    kv.finish(rk, rv, sK, sV, rows, tid);
  }
  __syncthreads();
  // no barrier follows but for a shared tile: a wavefront without a query tile leaves, one with several loops
  for (; q0 < a.Tq; q0 = sharing ? (q0 < SHARED ? SHARED : a.Tq) : q0 + q_step) {
  const bool shared = sharing && q0 >= SHARED;
  const int k_first = shared ? wave * 32 : 0, k_step = shared ? NT / 2 : 32;
  const int qi = q0 + (lane & 31);
  const bool qok = qi < a.Tq;
  float16_t acc[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[o][r] = 0.f;
  const int k_end = a.causal ? min(a.Tk, min(q0 + 31, a.Tq - 1) + shift + 1) : a.Tk;
  for (int k0 = k_first; k0 < k_end; k0 += k_step) {
    float16_t s, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int off = (k0 + (lane & 31)) * LD + c * 16 + (lane >> 5) * 8;
      s = M32<DT>::run(*(const uint4*)(sK + off), qf[c], s);
      dp = M32<DT>::run(*(const uint4*)(sV + off), dof[c], dp);
    }
    const bool masked = (k0 + 32 > a.Tk) || (a.causal && k0 + 31 > q0 + shift);
    if (masked) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kj = k0 + acc_row(r, lane);
        const bool ok = kj < a.Tk && (!a.causal || kj <= qi + shift);
        const float p = ok ? __builtin_amdgcn_exp2f(s[r] * sc - lse2) : 0.f;
        s[r] = p * (dp[r] - dlt);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(s[r] * sc - lse2) * (dp[r] - dlt);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint4 dsf = pack8<DT>(s, 8 * j);
#pragma unroll
      for (int o = 0; o < NO; ++o) acc[o] = M32<DT>::run(frag_tr<LD>(sK, k0 + 16 * j, o * 32, lane), dsf, acc[o]);
    }
  }
  if (!shared) {
    const int qn = sharing ? SHARED : q0 + q_step;
    if (qn < a.Tq) {
      load_rows(qn);
      row_delta(qn);
    }
    if (qok) {
      uint16_t* DQ = a.dq + b * a.dq_sb + h * a.dq_sh + (int64_t)qi * a.dq_st;
#pragma unroll
      for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int h0 = o * 32 + 8 * g + 4 * (lane >> 5);
          if (h0 < a.hd)
            *(uint2*)(DQ + h0) = make_uint2(M32<DT>::pack(acc[o][4 * g] * a.scale, acc[o][4 * g + 1] * a.scale),
                                            M32<DT>::pack(acc[o][4 * g + 2] * a.scale, acc[o][4 * g + 3] * a.scale));
        }
    }
  } else if constexpr (NT == 512) {
    float x[2 * NO];
    sum_waves<NO>(acc, (float*)smem, wave, lane, x);
    if (qok) {
      uint16_t* DQ = a.dq + b * a.dq_sb + h * a.dq_sh + (int64_t)qi * a.dq_st;
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        const int h0 = o * 32 + acc_row(2 * wave, lane);
        if (h0 < a.hd) *(uint32_t*)(DQ + h0) = M32<DT>::pack(x[2 * o] * a.scale, x[2 * o + 1] * a.scale);
      }
    }
  }
  }
}

// A tile of scores and of dP, [query][key], into P and dS / scale = P * (dP - delta) (the scale is applied to dK at the
// end).  lse (times log2 e), delta: this lane's first query's (a lane's are 8 (r / 4) + r % 4 rows on); rows before
// `first` do not see this lane's key.  The row of a register is a constant beside a lane's threshold, and lse and delta come four at a time:
// 281 -> 241 instructions per step of 32 x 32 x 96, 197 tokens x 1024 heads of 64 100 -> 94 us (whole backward).
__device__ __forceinline__ void p_and_ds(float16_t& s, float16_t& dp, const float* lse, const float* delta, float sc, int first) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const float4_t l = *(const float4_t*)(lse + 8 * g), d = *(const float4_t*)(delta + 8 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 4 * g + e;
      const float p = __builtin_amdgcn_exp2f(s[r] * sc - l[e]);
      s[r] = 8 * g + e < first ? 0.f : p;
      dp[r] = s[r] * (dp[r] - d[e]);
    }
  }
}

// dK/dV: workgroup = NT / 2 keys, wavefront = 32 of them; queries in steps of 32
template <int DT, int HD, int NT>
__global__ __launch_bounds__(NT) void attn_dkv_short_kernel(const AttnArgs a, int rows, int share) {
  constexpr int NC = HD / 16, NO = HD / 32, LD = HD + 8;
  extern __shared__ __align__(16) uint16_t smem[];
  uint16_t* sQ = smem;
  uint16_t* sDO = smem + rows * LD;
  float* sLse = (float*)(smem + 2 * rows * LD);
  float* sDelta = sLse + rows;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = blockIdx.y, b = bh / a.H, h = bh % a.H;
  const int k_step = (int)gridDim.x * (NT / 2);
  int kw0 = blockIdx.x * (NT / 2) + wave * 32;
  const uint16_t* K = a.k + b * a.k_sb + h * a.k_sh;
  const uint16_t* V = a.v + b * a.v_sb + h * a.v_sh;
  const float sc = a.scale * LOG2E;
  const int shift = a.Tk - a.Tq;

  const HeadRows rk(K, a.k_st, a.Tk, a.hd), rv(V, a.v_st, a.Tk, a.hd);
  const HeadRows rq(a.q + b * a.q_sb + h * a.q_sh, a.q_st, a.Tq, a.hd), rdo(a.d_o + b * a.do_sb + h * a.do_sh, a.do_st, a.Tq, a.hd);
  uint4 kf[NC], vf[NC];
  auto load_rows = [&](int ks) {   // this lane's key row of the tile at `ks`
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      kf[c] = rk.load(ks + (lane & 31), c * 16 + (lane >> 5) * 8);
      vf[c] = rv.load(ks + (lane & 31), c * 16 + (lane >> 5) * 8);
    }
  };
  {
    HeadPair<HD, NT> qd;
    qd.issue(rq, rdo, rows, tid);
    load_rows(kw0);
    for (int i = tid; i < rows; i += NT) {
      // rows past the end: Q and dO rows are zero, lse = +inf makes their P exactly zero
      sLse[i] = i < a.Tq ? a.lse[(int64_t)bh * a.Tq + i] * LOG2E : INFINITY;
      sDelta[i] = i < a.Tq ? a.delta[(int64_t)bh * a.Tq + i] : 0.f;
    }
    qd.finish(rq, rdo, sQ, sDO, rows, tid);
  }
  __syncthreads();
  // no barrier follows but for a shared tile: a wavefront without a key tile leaves, one with several loops
  constexpr int SHARED = NT / 2;             // the tile from here on is shared by all wavefronts where they share one
  const bool sharing = NT == 512 && share;
  for (; kw0 < a.Tk; kw0 = sharing ? (kw0 < SHARED ? SHARED : a.Tk) : kw0 + k_step) {
  const bool shared = sharing && kw0 >= SHARED;
  const int q_step = shared ? NT / 2 : 32;
  const int kj = kw0 + (lane & 31);
  const bool kok = kj < a.Tk;
  float16_t dk[NO], dv[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int r = 0; r < 16; ++r) dk[o][r] = dv[o][r] = 0.f;
  int q_begin = 0;
  if (a.causal) q_begin = max(0, kw0 - shift) / 32 * 32;   // queries i with i + shift >= kw0 see this wavefront's keys
  for (int q0 = q_begin + (shared ? wave * 32 : 0); q0 < a.Tq; q0 += q_step) {
    float16_t s, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int off = (q0 + (lane & 31)) * LD + c * 16 + (lane >> 5) * 8;
      s = M32<DT>::run(*(const uint4*)(sQ + off), kf[c], s);
      dp = M32<DT>::run(*(const uint4*)(sDO + off), vf[c], dp);
    }
    const int ql = q0 + 4 * (lane >> 5);
    p_and_ds(s, dp, sLse + ql, sDelta + ql, sc, a.causal ? kj - (ql + shift) : 0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint4 pf = pack8<DT>(s, 8 * j);
      const uint4 dsf = pack8<DT>(dp, 8 * j);
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        dv[o] = M32<DT>::run(frag_tr<LD>(sDO, q0 + 16 * j, o * 32, lane), pf, dv[o]);
        dk[o] = M32<DT>::run(frag_tr<LD>(sQ, q0 + 16 * j, o * 32, lane), dsf, dk[o]);
      }
    }
  }
  if (!shared) {
    const int kn = sharing ? SHARED : kw0 + k_step;
    if (kn < a.Tk) load_rows(kn);
    if (kok) {
      uint16_t* DK = a.dk + b * a.dk_sb + h * a.dk_sh + (int64_t)kj * a.dk_st;
      uint16_t* DV = a.dv + b * a.dv_sb + h * a.dv_sh + (int64_t)kj * a.dv_st;
#pragma unroll
      for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int h0 = o * 32 + 8 * g + 4 * (lane >> 5);
          if (h0 < a.hd) {
            *(uint2*)(DK + h0) = make_uint2(M32<DT>::pack(dk[o][4 * g] * a.scale, dk[o][4 * g + 1] * a.scale),
                                            M32<DT>::pack(dk[o][4 * g + 2] * a.scale, dk[o][4 * g + 3] * a.scale));
            *(uint2*)(DV + h0) = make_uint2(M32<DT>::pack(dv[o][4 * g], dv[o][4 * g + 1]),
                                            M32<DT>::pack(dv[o][4 * g + 2], dv[o][4 * g + 3]));
          }
        }
    }
  } else if constexpr (NT == 512) {
    float xk[2 * NO], xv[2 * NO];
    sum_waves<NO>(dk, (float*)smem, wave, lane, xk);
    sum_waves<NO>(dv, (float*)smem, wave, lane, xv);
    if (kok) {
      uint16_t* DK = a.dk + b * a.dk_sb + h * a.dk_sh + (int64_t)kj * a.dk_st;
      uint16_t* DV = a.dv + b * a.dv_sb + h * a.dv_sh + (int64_t)kj * a.dv_st;
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        const int h0 = o * 32 + acc_row(2 * wave, lane);
        if (h0 < a.hd) {
          *(uint32_t*)(DK + h0) = M32<DT>::pack(xk[2 * o] * a.scale, xk[2 * o + 1] * a.scale);
          *(uint32_t*)(DV + h0) = M32<DT>::pack(xv[2 * o], xv[2 * o + 1]);
        }
      }
    }
  }
  }
}

// dQ, dK and dV of one head in ONE workgroup of eight wavefronts (heads of up to 256 queries and 256
// keys, head dim <= 64): Q, dO, K and V are loaded into LDS once (4 x 32 KB at 197 tokens), every
// wavefront first forms delta and dQ for its 32 queries (sweeping the keys), then, after one barrier,
// dK and dV for its 32 keys (sweeping the queries); against the two-kernel form this saves a launch and
// one load of the head.  Same arithmetic, in the same order, as attn_dq_short_kernel and
// attn_dkv_short_kernel.  Heads from `whole` on have two workgroups each: there four wavefronts form dQ of half of the queries
// beside four that form dK and dV of half of the keys.
template <int DT, int HD>
__global__ __launch_bounds__(512) void attn_bwd_short_fused_kernel(const AttnArgs a, float* delta_out, int rows_q, int rows_k, int whole) {
  constexpr int NC = HD / 16, NO = HD / 32, LD = HD + 8, NT = 512;
  extern __shared__ __align__(16) uint16_t smem[];
  uint16_t* sK = smem;
  uint16_t* sV = sK + rows_k * LD;
  uint16_t* sQ = sV + rows_k * LD;
  uint16_t* sDO = sQ + rows_q * LD;
  float* sLse = (float*)(sDO + rows_q * LD);
  float* sDelta = sLse + rows_q;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // heads from `whole` on: two workgroups each
  const int part = (int)blockIdx.y - whole, bh = part < 0 ? (int)blockIdx.y : whole + part / 2, b = bh / a.H, h = bh % a.H;
  const uint16_t* OO = a.o + b * a.o_sb + h * a.o_sh;
  const float sc = a.scale * LOG2E;
  const int shift = a.Tk - a.Tq;

  // delta = rowsum(dO * O) and lse of this lane's query row
  int q0 = wave * 32, qi = q0 + (lane & 31);
  bool qok = qi < a.Tq;
  const HeadRows rdo(a.d_o + b * a.do_sb + h * a.do_sh, a.do_st, a.Tq, a.hd), ro(OO, a.o_st, a.Tq, a.hd);
  const HeadRows rq(a.q + b * a.q_sb + h * a.q_sh, a.q_st, a.Tq, a.hd);
  const HeadRows rk(a.k + b * a.k_sb + h * a.k_sh, a.k_st, a.Tk, a.hd), rv(a.v + b * a.v_sb + h * a.v_sh, a.v_st, a.Tk, a.hd);
  float dlt = 0.f;
  float lse2 = qok ? a.lse[(int64_t)bh * a.Tq + qi] * LOG2E : INFINITY;
  {
    HeadPair<HD, NT> kv, qd;
    uint4 dof[NC], of[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      dof[c] = rdo.load(qi, c * 16 + (lane >> 5) * 8);
      of[c] = ro.load(qi, c * 16 + (lane >> 5) * 8);
    }
    kv.issue(rk, rv, rows_k, tid);
    qd.issue(rq, rdo, rows_q, tid);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float x[8], y[8];
      unpack8<DT>(dof[c], x);
      unpack8<DT>(of[c], y);
#pragma unroll
      for (int k = 0; k < 8; ++k) dlt += x[k] * y[k];
    }
    dlt += __shfl_xor(dlt, 32, 64);
    kv.finish(rk, rv, sK, sV, rows_k, tid);
    qd.finish(rq, rdo, sQ, sDO, rows_q, tid);
  }
  if (q0 < rows_q && (lane >> 5) == 0) {
    // rows past the end: Q and dO rows are zero, lse = +inf makes their P exactly zero
    sLse[qi] = lse2;
    sDelta[qi] = qok ? dlt : 0.f;
    if (qok) delta_out[(int64_t)bh * a.Tq + qi] = dlt;
  }
  __syncthreads();

  // ---- dQ for queries q0 .. q0+31
  int kw0 = q0;
  if (part >= 0) {
    // half of the head: dQ by the first four wavefronts and dK, dV by the others, at the same time
    const int hq = (rows_q / 32 + 1) / 2, hk = (rows_k / 32 + 1) / 2;
    q0 = wave < hq && wave < 4 ? ((part & 1) * hq + wave) * 32 : a.Tq;
    kw0 = wave >= 4 && wave - 4 < hk ? ((part & 1) * hk + wave - 4) * 32 : a.Tk;
    qi = q0 + (lane & 31);
    qok = qi < a.Tq;
    if (q0 < a.Tq) {
      lse2 = sLse[qi];
      dlt = sDelta[qi];
    }
  }
  if (q0 < a.Tq) {
    uint4 qf[NC], dof[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int off = qi * LD + c * 16 + (lane >> 5) * 8;
      qf[c] = *(const uint4*)(sQ + off);
      dof[c] = *(const uint4*)(sDO + off);
    }
    float16_t acc[NO];
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[o][r] = 0.f;
    const int k_end = a.causal ? min(a.Tk, min(q0 + 31, a.Tq - 1) + shift + 1) : a.Tk;
    for (int k0 = 0; k0 < k_end; k0 += 32) {
      float16_t s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int off = (k0 + (lane & 31)) * LD + c * 16 + (lane >> 5) * 8;
        s = M32<DT>::run(*(const uint4*)(sK + off), qf[c], s);
        dp = M32<DT>::run(*(const uint4*)(sV + off), dof[c], dp);
      }
      const bool masked = (k0 + 32 > a.Tk) || (a.causal && k0 + 31 > q0 + shift);
      if (masked) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kj = k0 + acc_row(r, lane);
          const bool ok = kj < a.Tk && (!a.causal || kj <= qi + shift);
          const float p = ok ? __builtin_amdgcn_exp2f(s[r] * sc - lse2) : 0.f;
          s[r] = p * (dp[r] - dlt);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(s[r] * sc - lse2) * (dp[r] - dlt);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint4 dsf = pack8<DT>(s, 8 * j);
#pragma unroll
        for (int o = 0; o < NO; ++o) acc[o] = M32<DT>::run(frag_tr<LD>(sK, k0 + 16 * j, o * 32, lane), dsf, acc[o]);
      }
    }
    if (qok) {
      uint16_t* DQ = a.dq + b * a.dq_sb + h * a.dq_sh + (int64_t)qi * a.dq_st;
#pragma unroll
      for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int h0 = o * 32 + 8 * g + 4 * (lane >> 5);
          if (h0 < a.hd)
            *(uint2*)(DQ + h0) = make_uint2(M32<DT>::pack(acc[o][4 * g] * a.scale, acc[o][4 * g + 1] * a.scale),
                                            M32<DT>::pack(acc[o][4 * g + 2] * a.scale, acc[o][4 * g + 3] * a.scale));
        }
    }
  }

  // ---- dK, dV for keys kw0 .. kw0+31 (sLse / sDelta were complete at the barrier above)
  const int kj = kw0 + (lane & 31);
  if (kw0 >= a.Tk) return;
  const bool kok = kj < a.Tk;
  uint4 kf[NC], vf[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int off = kj * LD + c * 16 + (lane >> 5) * 8;   // rows up to rows_k are in LDS (zero past Tk)
    kf[c] = *(const uint4*)(sK + off);
    vf[c] = *(const uint4*)(sV + off);
  }
  float16_t dk[NO], dv[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o)
#pragma unroll
    for (int r = 0; r < 16; ++r) dk[o][r] = dv[o][r] = 0.f;
  int q_begin = 0;
  if (a.causal) q_begin = max(0, kw0 - shift) / 32 * 32;
  for (int qs = q_begin; qs < a.Tq; qs += 32) {
    float16_t s, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int off = (qs + (lane & 31)) * LD + c * 16 + (lane >> 5) * 8;
      s = M32<DT>::run(*(const uint4*)(sQ + off), kf[c], s);
      dp = M32<DT>::run(*(const uint4*)(sDO + off), vf[c], dp);
    }
    const int ql = qs + 4 * (lane >> 5);
    p_and_ds(s, dp, sLse + ql, sDelta + ql, sc, a.causal ? kj - (ql + shift) : 0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint4 pf = pack8<DT>(s, 8 * j);
      const uint4 dsf = pack8<DT>(dp, 8 * j);
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        dv[o] = M32<DT>::run(frag_tr<LD>(sDO, qs + 16 * j, o * 32, lane), pf, dv[o]);
        dk[o] = M32<DT>::run(frag_tr<LD>(sQ, qs + 16 * j, o * 32, lane), dsf, dk[o]);
      }
    }
  }
  if (kok) {
    uint16_t* DK = a.dk + b * a.dk_sb + h * a.dk_sh + (int64_t)kj * a.dk_st;
    uint16_t* DV = a.dv + b * a.dv_sb + h * a.dv_sh + (int64_t)kj * a.dv_st;
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int h0 = o * 32 + 8 * g + 4 * (lane >> 5);
        if (h0 < a.hd) {
          *(uint2*)(DK + h0) = make_uint2(M32<DT>::pack(dk[o][4 * g] * a.scale, dk[o][4 * g + 1] * a.scale),
                                          M32<DT>::pack(dk[o][4 * g + 2] * a.scale, dk[o][4 * g + 3] * a.scale));
          *(uint2*)(DV + h0) = make_uint2(M32<DT>::pack(dv[o][4 * g], dv[o][4 * g + 1]),
                                          M32<DT>::pack(dv[o][4 * g + 2], dv[o][4 * g + 3]));
        }
      }
  }
}

bool strides_ok(const void* p, int64_t sb, int64_t sh, int64_t st) {
  return pf_aligned(p, 16) && sb % 8 == 0 && sh % 8 == 0 && st % 8 == 0;
}

int check_common(const pf_attn_desc* d, const char* name) {
  PF_REQUIRE(d != nullptr, "%s: null descriptor", name);
  PF_REQUIRE(d->dtype == PF_F16 || d->dtype == PF_BF16, "%s: dtype must be fp16 or bf16", name);
  PF_REQUIRE(d->B > 0 && d->H > 0 && d->Tq > 0 && d->Tk > 0 && d->hd > 0, "%s: bad shape", name);
  if (d->hd % 8 != 0 || d->hd > 128) {
    pf_set_error("%s: head dim %d is not supported by the fused kernels (multiple of 8, <= 128)", name, d->hd);
    return PF_ERR_UNSUPPORTED;
  }
  PF_REQUIRE((int64_t)d->B * d->H <= 65535, "%s: B*H exceeds 65535", name);
  PF_REQUIRE(d->q && d->k && d->v && d->lse, "%s: null operand", name);
  PF_REQUIRE(strides_ok(d->q, d->q_sb, d->q_sh, d->q_st) && strides_ok(d->k, d->k_sb, d->k_sh, d->k_st) &&
                 strides_ok(d->v, d->v_sb, d->v_sh, d->v_st),
             "%s: q/k/v must be 16-byte aligned with strides that are multiples of 8", name);
  if (d->o_lo) PF_REQUIRE(d->hd > 96 && pf_aligned(d->o_lo, 16), "%s: o_lo needs a head dim above 96 and 16-byte alignment", name);
  if (d->causal) PF_REQUIRE(d->Tk >= d->Tq, "%s: causal attention needs Tk >= Tq", name);
  return PF_OK;
}

// whole operands in LDS: two of them (and their padding) fit for head dims up to 96
// Do `rows` token rows of each operand that is loaded lie within 2 GiB, so that 32-bit byte offsets reach them?
bool rows_near(const pf_attn_desc* d, bool bwd, int rows) {
  auto near = [rows](int64_t st) { return st >= 0 && st < (1 << 30) / rows; };
  return near(d->q_st) && near(d->k_st) && near(d->v_st) && (!bwd || (near(d->o_st) && near(d->do_st)));
}
bool short_ok(const pf_attn_desc* d, bool bwd) {
  return d->Tq <= SHORT_T && d->Tk <= SHORT_T && d->hd <= 96 && rows_near(d, bwd, SHORT_T);
}

AttnArgs make_args(const pf_attn_desc* d) {
  AttnArgs a;
  a.q = (const uint16_t*)d->q; a.k = (const uint16_t*)d->k; a.v = (const uint16_t*)d->v;
  a.o = (const uint16_t*)d->o; a.d_o = (const uint16_t*)d->d_o; a.out = (uint16_t*)d->o;
  a.dq = (uint16_t*)d->dq; a.dk = (uint16_t*)d->dk; a.dv = (uint16_t*)d->dv;
  a.o_lo = (uint16_t*)d->o_lo; a.lse = d->lse; a.delta = d->delta;
  a.q_sb = d->q_sb; a.q_sh = d->q_sh; a.q_st = d->q_st; a.k_sb = d->k_sb; a.k_sh = d->k_sh; a.k_st = d->k_st;
  a.v_sb = d->v_sb; a.v_sh = d->v_sh; a.v_st = d->v_st; a.o_sb = d->o_sb; a.o_sh = d->o_sh; a.o_st = d->o_st;
  a.do_sb = d->do_sb; a.do_sh = d->do_sh; a.do_st = d->do_st; a.dq_sb = d->dq_sb; a.dq_sh = d->dq_sh;
  a.dq_st = d->dq_st; a.dk_sb = d->dk_sb; a.dk_sh = d->dk_sh; a.dk_st = d->dk_st; a.dv_sb = d->dv_sb;
  a.dv_sh = d->dv_sh; a.dv_st = d->dv_st;
  a.B = d->B; a.H = d->H; a.Tq = d->Tq; a.Tk = d->Tk; a.hd = d->hd; a.causal = d->causal ? 1 : 0;
  a.scale = d->scale;
  return a;
}

}  // namespace

// Launch of a short-sequence kernel with `lds` bytes of dynamic LDS.
template <typename K, typename... Args>
int launch_short(K kern, dim3 grid, int threads, size_t lds, hipStream_t st, Args... args) {
  const int rc = pf_allow_lds((const void*)kern, lds > 64 * 1024 ? 160 * 1024 : lds, "pf_attention");
  if (rc != PF_OK) return rc;
  hipLaunchKernelGGL(kern, grid, dim3((unsigned)threads), lds, st, args...);
  return PF_OK;
}

// Does a workgroup of eight wavefronts share the ninth tile of the T tokens along its axis?  Not under a mask
// (the wavefronts' own tiles differ in work, and all have to wait for the last: 275 causal tokens x 128 heads of 88 16.5 ->
// 18.1 us, backward 45.6 -> 50.5), and not over a sweep of few tiles, which costs less than the exchange (288 queries of
// 77 keys, backward 36.9 -> 45.6; 257 of 257 57 -> 49).
bool shares_tile(const pf_attn_desc* d, int64_t T, int64_t sweep) { return !d->causal && T > 256 && sweep > 192; }

// LDS of a short-sequence kernel whose operands take `operands` bytes; the partial results of a shared tile (eight
// accumulator tiles, and maxima and sums) take their place.
inline size_t lds_with_shared_tile(size_t operands, int share, int HD) {
  const size_t partial = 2048 + (size_t)8 * (HD / 32) * 16 * 64 * 4;
  return share && partial > operands ? partial : operands;
}

// T: tokens along the axis the workgroups divide (queries, or keys for dK/dV), in tiles of 32 per
// wavefront.  A head of more than 128 tokens takes ONE workgroup of eight wavefronts, its two LDS
// operands are fetched once.  WIDE96 false, at head dims above 64: workgroups of four; each takes four
// tiles and a remainder of one or two tiles becomes a second pass instead of a workgroup (and a
// load of the whole head) of its own.
#define PF_ATTN_SHORT(KERNEL, WIDE96, rc, T, BH, lds, st, dt, hd, ...)                                          \
  do {                                                                                                         \
    const int tiles_ = ((T) + 31) / 32;                                                                        \
    const bool w64_ = (hd) <= 64 && (T) > 128, w96_ = (hd) > 64 && (WIDE96) && (T) > 128;                       \
    const int gx_ = (w64_ || w96_) ? 1 : ((tiles_ + 1) / 4 > 1 ? (tiles_ + 1) / 4 : 1);                         \
    const dim3 grid_((unsigned)gx_, (unsigned)(BH));                                                           \
    if (dt == PF_F16) {                                                                                        \
      if (w64_) rc = launch_short(KERNEL<PF_F16, 64, 512>, grid_, 512, (lds)(64), st, __VA_ARGS__);             \
      else if (hd <= 64) rc = launch_short(KERNEL<PF_F16, 64, 256>, grid_, 256, (lds)(64), st, __VA_ARGS__);    \
      else if (w96_) rc = launch_short(KERNEL<PF_F16, 96, 512>, grid_, 512, (lds)(96), st, __VA_ARGS__);        \
      else rc = launch_short(KERNEL<PF_F16, 96, 256>, grid_, 256, (lds)(96), st, __VA_ARGS__);                  \
    } else {                                                                                                   \
      if (w64_) rc = launch_short(KERNEL<PF_BF16, 64, 512>, grid_, 512, (lds)(64), st, __VA_ARGS__);            \
      else if (hd <= 64) rc = launch_short(KERNEL<PF_BF16, 64, 256>, grid_, 256, (lds)(64), st, __VA_ARGS__);   \
      else if (w96_) rc = launch_short(KERNEL<PF_BF16, 96, 512>, grid_, 512, (lds)(96), st, __VA_ARGS__);       \
      else rc = launch_short(KERNEL<PF_BF16, 96, 256>, grid_, 256, (lds)(96), st, __VA_ARGS__);                 \
    }                                                                                                          \
  } while (0)

// (...: the kernel's template arguments after type and head dim)
#define PF_ATTN_DISPATCH(KERNEL, grid, st, a, dt, hd, ...)                                                    \
  do {                                                                                                       \
    if (dt == PF_F16) {                                                                                      \
      if (hd <= 64) hipLaunchKernelGGL((KERNEL<PF_F16, 64, __VA_ARGS__>), grid, dim3(256), 0, st, a);         \
      else if (hd <= 96) hipLaunchKernelGGL((KERNEL<PF_F16, 96, __VA_ARGS__>), grid, dim3(256), 0, st, a);    \
      else hipLaunchKernelGGL((KERNEL<PF_F16, 128, __VA_ARGS__>), grid, dim3(256), 0, st, a);                 \
    } else {                                                                                                 \
      if (hd <= 64) hipLaunchKernelGGL((KERNEL<PF_BF16, 64, __VA_ARGS__>), grid, dim3(256), 0, st, a);        \
      else if (hd <= 96) hipLaunchKernelGGL((KERNEL<PF_BF16, 96, __VA_ARGS__>), grid, dim3(256), 0, st, a);   \
      else hipLaunchKernelGGL((KERNEL<PF_BF16, 128, __VA_ARGS__>), grid, dim3(256), 0, st, a);                \
    }                                                                                                        \
  } while (0)

extern "C" int pf_attention_fwd(const pf_attn_desc* d, void* stream) {
  int rc = check_common(d, "pf_attention_fwd");
  if (rc != PF_OK) return rc;
  PF_REQUIRE(d->o && strides_ok(d->o, d->o_sb, d->o_sh, d->o_st) && d->o_st % 4 == 0,
             "pf_attention_fwd: bad output operand");
  AttnArgs a = make_args(d);
  const dim3 grid((unsigned)((d->Tq + 127) / 128), (unsigned)(d->B * d->H));
  if (short_ok(d, false)) {
    const int rows = (d->Tk + 31) / 32 * 32;
    const int share = shares_tile(d, d->Tq, d->Tk);
    auto lds = [rows, share](int HD) { return lds_with_shared_tile((size_t)2 * rows * (HD + 8) * 2, share, HD); };
    PF_ATTN_SHORT(attn_fwd_short_kernel, true, rc, d->Tq, d->B * d->H, lds, (hipStream_t)stream, d->dtype, d->hd, a, rows, share);
    if (rc != PF_OK) return rc;
  } else {
    if (rows_near(d, false, 128)) PF_ATTN_DISPATCH(attn_fwd_kernel, grid, (hipStream_t)stream, a, d->dtype, d->hd, false);
    else PF_ATTN_DISPATCH(attn_fwd_kernel, grid, (hipStream_t)stream, a, d->dtype, d->hd, true);
  }
  PF_CHECK_LAUNCH("pf_attention_fwd");
  return PF_OK;
}

extern "C" int pf_attention_bwd(const pf_attn_desc* d, void* stream) {
  int rc = check_common(d, "pf_attention_bwd");
  if (rc != PF_OK) return rc;
  PF_REQUIRE(d->o && d->d_o && d->dq && d->dk && d->dv && d->delta, "pf_attention_bwd: null operand");
  PF_REQUIRE(strides_ok(d->o, d->o_sb, d->o_sh, d->o_st) && strides_ok(d->d_o, d->do_sb, d->do_sh, d->do_st),
             "pf_attention_bwd: o/dO must be 16-byte aligned with strides that are multiples of 8");
  PF_REQUIRE(pf_aligned(d->dq, 8) && pf_aligned(d->dk, 8) && pf_aligned(d->dv, 8) && d->dq_sb % 4 == 0 &&
                 d->dq_sh % 4 == 0 && d->dq_st % 4 == 0 && d->dk_sb % 4 == 0 && d->dk_sh % 4 == 0 &&
                 d->dk_st % 4 == 0 && d->dv_sb % 4 == 0 && d->dv_sh % 4 == 0 && d->dv_st % 4 == 0,
             "pf_attention_bwd: gradient operands must be 8-byte aligned with strides that are multiples of 4");
  AttnArgs a = make_args(d);
  hipStream_t st = (hipStream_t)stream;
  const dim3 gq((unsigned)((d->Tq + 127) / 128), (unsigned)(d->B * d->H));
  const dim3 gk((unsigned)((d->Tk + 127) / 128), (unsigned)(d->B * d->H));
  if (short_ok(d, true)) {
    const int rows_k = (d->Tk + 31) / 32 * 32, rows_q = (d->Tq + 31) / 32 * 32;
    if (d->hd <= 64 && d->Tq <= 256 && d->Tk <= 256 && (d->Tq > 128 || d->Tk > 128)) {
      // one workgroup per head forms dQ, dK and dV from a single load of the head
      const size_t lds = (size_t)2 * (rows_k + rows_q) * (64 + 8) * 2 + (size_t)rows_q * 8;
      // A CU has LDS for one of them.  Up to 128 heads that are left after rounds of 256 go to two workgroups each, half of the queries and
      // half of the keys to one (us, a workgroup / two, 197 tokens, head dim 64: 24 heads 17.6 / 13.3, 60 18.5 / 14.2, 120 20.0 / 16.7,
      // 258 40.0 / 35.0, 372 42.0 / 40.1).
      const int heads = d->B * d->H, rest = heads % 256, whole = rest <= 128 ? heads - rest : heads;
      const dim3 gf(1, (unsigned)(2 * heads - whole));
      if (d->dtype == PF_F16) rc = launch_short(attn_bwd_short_fused_kernel<PF_F16, 64>, gf, 512, lds, st, a, d->delta, rows_q, rows_k, whole);
      else rc = launch_short(attn_bwd_short_fused_kernel<PF_BF16, 64>, gf, 512, lds, st, a, d->delta, rows_q, rows_k, whole);
      if (rc != PF_OK) return rc;
      PF_CHECK_LAUNCH("pf_attention_bwd");
      return PF_OK;
    }
    // dQ first: it also leaves delta = rowsum(dO * O) for the dK/dV kernel
    const int share_q = shares_tile(d, d->Tq, d->Tk), share_k = shares_tile(d, d->Tk, d->Tq);
    auto lds_q = [rows_k, share_q](int HD) { return lds_with_shared_tile((size_t)2 * rows_k * (HD + 8) * 2, share_q, HD); };
    auto lds_k = [rows_q, share_k](int HD) {
      return lds_with_shared_tile((size_t)2 * rows_q * (HD + 8) * 2 + (size_t)rows_q * 8, share_k, HD);
    };
    PF_ATTN_SHORT(attn_dq_short_kernel, true, rc, d->Tq, d->B * d->H, lds_q, st, d->dtype, d->hd, a, d->delta, rows_k, share_q);
    if (rc != PF_OK) return rc;
    // dK/dV above head dim 64: one workgroup of eight wavefronts per head, or two of four, which fill more of the chip while
    // there are few heads (two -> one, us of backward: 197 tokens x 64 heads of 80 31.0 -> 33.8, x 128 of 88 37.6 -> 39.4, x 192
    // 53 -> 41, x 384 91 -> 82; 257 tokens x 768 261 -> 206).  Up to six tiles the second form is one workgroup too (145
    // tokens x 96 heads: 28.5 -> 25.9 on eight).
    const bool wide = d->B * d->H > 128 || d->Tk <= 192;
    PF_ATTN_SHORT(attn_dkv_short_kernel, wide, rc, d->Tk, d->B * d->H, lds_k, st, d->dtype, d->hd, a, rows_q, share_k);
    if (rc != PF_OK) return rc;
    PF_CHECK_LAUNCH("pf_attention_bwd");
    return PF_OK;
  }
  const bool near = rows_near(d, true, 128);
  // dQ first: it also leaves delta for the dK/dV kernel
  if (near) PF_ATTN_DISPATCH(attn_dq_kernel, gq, st, a, d->dtype, d->hd, false);
  else PF_ATTN_DISPATCH(attn_dq_kernel, gq, st, a, d->dtype, d->hd, true);
  // few keys, many queries (cross attention to a short context): split each key tile's query sweep
  // over the four wavefronts of a workgroup
  if (near && (int64_t)gk.x * gk.y < 200 && d->Tq >= 256 && d->hd <= 96) {   // (two 128-row tiles of more do not fit)
    const dim3 gs((unsigned)((d->Tk + 31) / 32), (unsigned)(d->B * d->H));
    if (d->dtype == PF_F16) {
      if (d->hd <= 64) hipLaunchKernelGGL((attn_dkv_kernel<PF_F16, 64, true>), gs, dim3(256), 0, st, a);
      else hipLaunchKernelGGL((attn_dkv_kernel<PF_F16, 96, true>), gs, dim3(256), 0, st, a);
    } else {
      if (d->hd <= 64) hipLaunchKernelGGL((attn_dkv_kernel<PF_BF16, 64, true>), gs, dim3(256), 0, st, a);
      else hipLaunchKernelGGL((attn_dkv_kernel<PF_BF16, 96, true>), gs, dim3(256), 0, st, a);
    }
  } else if (near) {
    PF_ATTN_DISPATCH(attn_dkv_kernel, gk, st, a, d->dtype, d->hd, false, false);
  } else {
    PF_ATTN_DISPATCH(attn_dkv_kernel, gk, st, a, d->dtype, d->hd, false, true);
  }
  PF_CHECK_LAUNCH("pf_attention_bwd");
  return PF_OK;
}
