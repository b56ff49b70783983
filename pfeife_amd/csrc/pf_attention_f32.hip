// Fused attention in fp32 (forward, dQ, dK/dV) on v_mfma_f32_16x16x4_f32: softmax(Q K^T * scale [+ causal]) V without score
// or probability matrices in memory.
//
// As in pf_attention.hip score tiles are computed transposed: a lane owns ONE column of a 16x16 tile (lane % 16) and its rows 4 g + r, g =
// lane / 16 and r = 0..3, in four registers.  A matrix instruction adds over any four reduction indices, one to each group of 16 lanes:
// register r of a score tile is the next product's right-hand operand as it stands (reduction indices r, 4 + r, 8 + r, 12 + r), and of the
// head dimension a lane takes four neighbouring elements with one 16-byte access (element e into instruction e of four).
//
// A workgroup has one tile of 16 columns of one head (queries in the forward pass and for dQ, keys for dK/dV); its four wavefronts take every
// fourth tile of 16 of the tokens on the other side and add their parts up through LDS at the end.  No two of them read the same token, so
// tokens go from memory (L2) to registers as operands: along a row (16 bytes a lane) for scores, across four rows (4 bytes a lane, 64-byte
// pieces) for what is summed over tokens.  The loads of a tile's second use are issued before its first, those of the next tile's first
// behind it: a score phase or more lies between a load and its use.
// What bounds it: the matrix pipes (34 cycles an instruction, beside which no vector instruction issues), NC * 8 / 12 / 16 instructions a
// tile: 96 / 84 TFLOP/s forward / backward over long sequences.  Short ones lose to tiles: 96 heads of 197 tokens are 1248 workgroups in one
// and two waves of the device.  Workgroups of 64 columns with the tokens staged in LDS had 384 (23.0 us forward and 66.9 backward there).
// us, products and softmax through memory / this, forward and backward:
//   96 heads, 197 tokens, head dim 64:            51 / 18    83 / 61        24 heads of them:          27 /  9    38 /  28
//   32 heads, 2048 tokens causal, 64:            815 / 163  1220 / 644      64 heads, 512 causal, 128: 139 / 58  241 / 224
//   80 heads, 1024 queries of 77 keys, 64:        95 / 33   150 / 105       16 heads, 5 tokens, 16:    9.6 / 3.3 15.5 / 7.2
// Relative error against 64 bits, through memory / this, O and dQ: 3.7e-7 / 2.2e-7 and 3.9e-7 / 2.5e-7 at 197 tokens (chains of sums a quarter
// as long), 8.7e-8 / 8.7e-8 and 1.3e-7 / 1.3e-7 at 5.
//
// Probabilities: exp2(x) / l with x = s * scale * log2(e) - R, an integer R near the row's largest x, and l kept beside R (one log-sum-exp
// would be rounded at its own size, and with it every probability of the row).
#include "pf_gemm_f32.h"

namespace {

struct Args {
  const float* q; const float* k; const float* v; const float* o; const float* d_o;
  float* out; float* dq; float* dk; float* dv;
  float* stats; float* delta;
  int64_t q_sb, q_sh, q_st, k_sb, k_sh, k_st, v_sb, v_sh, v_st, o_sb, o_sh, o_st;
  int64_t do_sb, do_sh, do_st, dq_sb, dq_sh, dq_st, dk_sb, dk_sh, dk_st, dv_sb, dv_sh, dv_st;
  int H, Tq, Tk, hd, causal;
  float scale, sc, sc_lo;      // sc + sc_lo = scale * log2(e)
};

__device__ __forceinline__ float el(const float4& x, int e) { return e == 0 ? x.x : e == 1 ? x.y : e == 2 ? x.z : x.w; }

// tokens of one head as operands of 16 at a time
template <int NC> struct Tokens {
  const float* X;
  int64_t st;
  int T, hd, g, c15;
  uint32_t row, last;      // byte offset of this lane's elements in a tile, and of those of the last 16 columns (none past hd)
  __device__ __forceinline__ Tokens(const float* x, int64_t st_, int T_, int hd_, int lane)
      : X(x), st(st_), T(T_), hd(hd_), g(lane >> 4), c15(lane & 15), row((uint32_t)((c15 * (int)st + 4 * g) * 4)),
        last(16 * (NC - 1) + 4 * g < hd ? row + 64 * (NC - 1) : 0x80000000u) {}
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t tile(int t0) const {      // (nothing to read in a tile past the end)
    const int rows = T - t0 < 16 ? T - t0 : 16;
    return make_rsrc(X + (int64_t)t0 * st, rows > 0 ? (uint32_t)(((rows - 1) * (int)st + hd) * 4) : 0u);
  }
  // token lane % 16, elements 16 c + 4 g ..: zeros past hd and past the last token
  __device__ __forceinline__ void rows(float4 (&x)[NC], int t0) const {
    const __amdgpu_buffer_rsrc_t rs = tile(t0);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const uint4 w = buf_load16(rs, c < NC - 1 ? row + 64 * c : last);
      x[c] = make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w));
    }
  }
  // tokens 4 g + r, element 16 o + lane % 16: zeros past the last token (what lies past hd ends in rows that are not stored)
  __device__ __forceinline__ void cols(float (&x)[4][NC], int t0) const {
    const __amdgpu_buffer_rsrc_t rs = tile(t0);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int o = 0; o < NC; ++o)
        x[r][o] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, (int)((((4 * g + r) * (int)st + c15) * 4) + 64 * o), 0, 0));
  }
};
// The 16 columns' own rows in LDS, [column][16 NC + 4]: all four wavefronts multiply by them, and registers hold what differs between them.
template <int NC>
__device__ __forceinline__ void stage_columns(float* lds, const float* X, int64_t st, int t0, int T, int hd, int tid) {
  for (int at = tid; at < 64 * NC; at += 256) {
    const int col = at / (4 * NC), d = at % (4 * NC) * 4;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (t0 + col < T && d < hd) x = *(const float4*)(X + (int64_t)(t0 + col) * st + d);
    *(float4*)(lds + col * (16 * NC + 4) + d) = x;
  }
}
// tile of 16 tokens (A) times the 16 columns (B) over the head dimension
template <int NC>
__device__ __forceinline__ float4_t scores(const float4 (&a)[NC], const float* lds, int lane) {
  int off = (lane & 15) * (16 * NC + 4) + 4 * (lane >> 4);
  asm volatile("" : "+v"(off));      // (read for every tile: hoisted out of the loop they would fill the registers)
  float4_t s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const float4 b = *(const float4*)(lds + off + 16 * c);
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(el(a[c], e), el(b, e), s[e & 1], 0, 0, 0);
  }
  return s[0] + s[1];
}
// acc[element][column] += tokens^T . tile s
template <int NC>
__device__ __forceinline__ void add_tokens(float4_t (&acc)[NC], const float (&x)[4][NC], const float4_t& s) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int o = 0; o < NC; ++o) acc[o] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[r][o], s[r], acc[o], 0, 0, 0);
}
// exp2(s * (sc + sc_lo) - R) to an ulp or so: the fraction is formed without rounding at the exponent's size.  FAR: also where s is -inf (which
// has no fraction) and where R + n would not be exact.
template <bool FAR>
__device__ __forceinline__ float power(const Args& a, float s, float R) {
  const float t = fmaf(s, a.sc, -R), n = !FAR || fabsf(R) < 4e6f ? rintf(t) : 0.f;
  const float p = ldexpf(__builtin_amdgcn_exp2f(fmaf(s, a.sc_lo, fmaf(s, a.sc, -(R + n)))), (int)n);
  return FAR && t < -150.f ? 0.f : p;
}
// over the four lanes that share a column
__device__ __forceinline__ float col_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16, 64));
  return fmaxf(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ float col_sum(float v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}
// The wavefronts' parts of [column][element] summed and stored by all four of them.
template <int NC>
__device__ __forceinline__ void store_sum(float* lds, const float4_t (&acc)[NC], float by, float* X, int64_t st, int t0, int T, int hd, int tid) {
  constexpr int LD = 16 * NC + 4;
  const int lane = tid & 63;
  float* mine = lds + ((tid >> 6) * 16 + (lane & 15)) * LD + 4 * (lane >> 4);
#pragma unroll
  for (int o = 0; o < NC; ++o) *(float4_t*)(mine + 16 * o) = acc[o];
  __syncthreads();
  for (int at = tid; at < 64 * NC; at += 256) {
    const int col = at / (4 * NC), d = at % (4 * NC) * 4;
    const float* p = lds + col * LD + d;
    const float4_t x = (*(const float4_t*)p + *(const float4_t*)(p + 16 * LD)) + (*(const float4_t*)(p + 32 * LD) + *(const float4_t*)(p + 48 * LD));
    if (t0 + col < T && d < hd) *(float4_t*)(X + (int64_t)(t0 + col) * st + d) = x * by;
  }
}

template <int NC>
__global__ __launch_bounds__(256, NC <= 4 ? 5 : NC <= 6 ? 4 : 3) void attn32_fwd_kernel(const Args a) {
  __shared__ __align__(16) float sQ[16 * (16 * NC + 4)], sO[64 * (16 * NC + 4)], sR[4][16], sL[4][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4;
  // under a causal mask the heaviest tiles of every head are started first
  const int bh = blockIdx.x, b = bh / a.H, h = bh % a.H, q0 = 16 * (a.causal ? gridDim.y - 1 - blockIdx.y : blockIdx.y);
  const int qi = q0 + (lane & 15), shift = a.Tk - a.Tq;
  const Tokens<NC> K(a.k + b * a.k_sb + h * a.k_sh, a.k_st, a.Tk, a.hd, lane), V(a.v + b * a.v_sb + h * a.v_sh, a.v_st, a.Tk, a.hd, lane);
  float4 kr[NC];
  float4_t acc[NC];
#pragma unroll
  for (int o = 0; o < NC; ++o) acc[o] = float4_t{0.f, 0.f, 0.f, 0.f};
  float R = -INFINITY, l = 0.f;      // (l: of this lane's rows)

  const int end = a.causal ? min(a.Tk, q0 + 16 + shift) : a.Tk;
  int k0 = 16 * ((wave + blockIdx.y) & 3);      // (the wavefront with a tile more is not the same one in every workgroup)
  K.rows(kr, k0);
  stage_columns<NC>(sQ, a.q + b * a.q_sb + h * a.q_sh, a.q_st, q0, a.Tq, a.hd, tid);
  __syncthreads();
  for (; k0 < end; k0 += 64) {
    float vc[4][NC];
    V.cols(vc, k0);
    float4_t s = scores<NC>(kr, sQ, lane);
    K.rows(kr, k0 + 64);
    if (k0 + 16 > a.Tk || (a.causal && k0 + 15 > q0 + shift)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kj = k0 + 4 * g + r;
        if (kj >= a.Tk || (a.causal && kj > qi + shift)) s[r] = -INFINITY;
      }
    }
    // (scale > 0: the largest score has the largest exponent)
    const float hi = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])) * a.sc - R, lo = fminf(fminf(s[0], s[1]), fminf(s[2], s[3])) * a.sc - R;
    if (__any(!(hi <= 16.f) || lo < -100.f || fabsf(R) >= 4e6f)) {
      // exponents out of the middle range: R follows the largest one seen (an integer, so that no part has to be scaled by more than a shift)
      const float mx = col_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))) * a.sc;
      const float up = fmaxf(R, mx < 1e30f ? rintf(mx) : mx);
      const float by = R == -INFINITY || up == R ? 1.f : __builtin_amdgcn_exp2f(R - up);
      R = up;
      l *= by;
#pragma unroll
      for (int o = 0; o < NC; ++o) acc[o] *= by;
      const float ref = R == -INFINITY ? 0.f : R;
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = power<true>(a, s[r], ref);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = power<false>(a, s[r], R);
    }
    l += (s[0] + s[1]) + (s[2] + s[3]);
    add_tokens<NC>(acc, vc, s);
  }
  l = col_sum(l);
  if (g == 0) {
    sR[wave][lane] = R;
    sL[wave][lane] = l;
  }
  __syncthreads();
  float top = -INFINITY, sum = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) top = fmaxf(top, sR[w][lane & 15]);
  const float ref = top == -INFINITY ? 0.f : top;
#pragma unroll
  for (int w = 0; w < 4; ++w) sum += sL[w][lane & 15] * __builtin_amdgcn_exp2f(sR[w][lane & 15] - ref);
  const float inv = sum > 0.f ? 1.f / sum : 0.f, by = __builtin_amdgcn_exp2f(R - ref) * inv;
#pragma unroll
  for (int o = 0; o < NC; ++o) acc[o] *= by;
  store_sum<NC>(sO, acc, 1.f, a.out + b * a.o_sb + h * a.o_sh, a.o_st, q0, a.Tq, a.hd, tid);
  if (tid < 16 && qi < a.Tq) {
    float* st = a.stats + (int64_t)bh * 2 * a.Tq + qi;
    st[0] = ref;
    st[a.Tq] = inv;
  }
}

// dQ, and delta = rowsum(dO * O) (at up to 64 keys rowsum(P * dP)), which the dK/dV kernel launched after this one reads
template <int NC>
__global__ __launch_bounds__(256, NC <= 4 ? 4 : NC <= 6 ? 3 : 2) void attn32_dq_kernel(const Args a) {
  __shared__ __align__(16) float sQ[16 * (16 * NC + 4)], sD[16 * (16 * NC + 4)], sX[64 * (16 * NC + 4)], sPart[4][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4;
  const int bh = blockIdx.x, b = bh / a.H, h = bh % a.H, q0 = 16 * (a.causal ? gridDim.y - 1 - blockIdx.y : blockIdx.y);
  const int qi = q0 + (lane & 15), shift = a.Tk - a.Tq;
  const Tokens<NC> K(a.k + b * a.k_sb + h * a.k_sh, a.k_st, a.Tk, a.hd, lane), V(a.v + b * a.v_sb + h * a.v_sh, a.v_st, a.Tk, a.hd, lane);
  const int end = a.causal ? min(a.Tk, q0 + 16 + shift) : a.Tk;
  int k0 = 16 * ((wave + blockIdx.y) & 3);
  float4 kr[NC], vr[NC];
  K.rows(kr, k0);
  V.rows(vr, k0);
  stage_columns<NC>(sQ, a.q + b * a.q_sb + h * a.q_sh, a.q_st, q0, a.Tq, a.hd, tid);
  stage_columns<NC>(sD, a.d_o + b * a.do_sb + h * a.do_sh, a.do_st, q0, a.Tq, a.hd, tid);
  stage_columns<NC>(sX, a.o + b * a.o_sb + h * a.o_sh, a.o_st, q0, a.Tq, a.hd, tid);
  __syncthreads();
  float delta = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int at = (lane & 15) * (16 * NC + 4) + 16 * c + 4 * g;
    const float4 x = *(const float4*)(sX + at), y = *(const float4*)(sD + at);
#pragma unroll
    for (int e = 0; e < 4; ++e) delta = fmaf(el(x, e), el(y, e), delta);
  }
  delta = col_sum(delta);
  const float* st = a.stats + (int64_t)bh * 2 * a.Tq;
  const float R = qi < a.Tq ? st[qi] : 0.f, inv = qi < a.Tq ? st[a.Tq + qi] : 0.f;
  float4_t acc[NC];
#pragma unroll
  for (int o = 0; o < NC; ++o) acc[o] = float4_t{0.f, 0.f, 0.f, 0.f};
  for (; k0 < (a.Tk <= 64 ? 64 : end); k0 += 64) {
    float kc[4][NC];
    K.cols(kc, k0);
    float4_t s = scores<NC>(kr, sQ, lane);
    K.rows(kr, k0 + 64);
    const float4_t dp = scores<NC>(vr, sD, lane);
    V.rows(vr, k0 + 64);
    if (k0 + 16 > a.Tk || (a.causal && k0 + 15 > q0 + shift)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kj = k0 + 4 * g + r;
        if (kj >= a.Tk || (a.causal && kj > qi + shift)) s[r] = -INFINITY;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) s[r] = power<true>(a, s[r], R) * inv;
    if (a.Tk <= 64) {
      // one tile to every wavefront: delta without the rounding of O, as sum of P dP
      float part = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) part = fmaf(s[r], dp[r], part);
      part = col_sum(part);
      if (g == 0) sPart[wave][lane] = part;
      __syncthreads();
      delta = (sPart[0][lane & 15] + sPart[1][lane & 15]) + (sPart[2][lane & 15] + sPart[3][lane & 15]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) s[r] *= dp[r] - delta;      // dS^T / scale (applied at the end)
    add_tokens<NC>(acc, kc, s);
  }
  if (tid < 16 && qi < a.Tq) a.delta[(int64_t)bh * a.Tq + qi] = delta;
  __syncthreads();       // (a wavefront without a tile of its own: the others may still read O)
  store_sum<NC>(sX, acc, a.scale, a.dq + b * a.dq_sb + h * a.dq_sh, a.dq_st, q0, a.Tq, a.hd, tid);
}

template <int NC>
__global__ __launch_bounds__(256, NC <= 4 ? 4 : NC <= 6 ? 2 : 1) void attn32_dkv_kernel(const Args a) {
  __shared__ __align__(16) float sK[16 * (16 * NC + 4)], sV[16 * (16 * NC + 4)], sX[64 * (16 * NC + 4)];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4;
  const int bh = blockIdx.x, b = bh / a.H, h = bh % a.H, k0 = 16 * blockIdx.y, kj = k0 + (lane & 15), shift = a.Tk - a.Tq;
  const Tokens<NC> Q(a.q + b * a.q_sb + h * a.q_sh, a.q_st, a.Tq, a.hd, lane), D(a.d_o + b * a.do_sb + h * a.do_sh, a.do_st, a.Tq, a.hd, lane);
  float4 qr[NC], dr[NC];
  const float* st = a.stats + (int64_t)bh * 2 * a.Tq;
  const float* dl = a.delta + (int64_t)bh * a.Tq;
  float4_t dk[NC], dv[NC];
#pragma unroll
  for (int o = 0; o < NC; ++o) dk[o] = dv[o] = float4_t{0.f, 0.f, 0.f, 0.f};
  // queries i with i + shift >= the tile's first key see it
  int q0 = (a.causal ? max(0, k0 - shift) / 16 * 16 : 0) + 16 * ((wave + blockIdx.y) & 3);
  Q.rows(qr, q0);
  D.rows(dr, q0);
  stage_columns<NC>(sK, a.k + b * a.k_sb + h * a.k_sh, a.k_st, k0, a.Tk, a.hd, tid);
  stage_columns<NC>(sV, a.v + b * a.v_sb + h * a.v_sh, a.v_st, k0, a.Tk, a.hd, tid);
  __syncthreads();
  for (; q0 < a.Tq; q0 += 64) {
    float qc[4][NC], dc[4][NC], R[4], inv[4], delta[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {      // (rows past the end: 1 / l = 0 makes their P zero)
      const int i = q0 + 4 * g + r;
      R[r] = i < a.Tq ? st[i] : 0.f;
      inv[r] = i < a.Tq ? st[a.Tq + i] : 0.f;
      delta[r] = i < a.Tq ? dl[i] : 0.f;
    }
    D.cols(dc, q0);
    float4_t s = scores<NC>(qr, sK, lane);
    Q.cols(qc, q0);
    float4_t dp = scores<NC>(dr, sV, lane);
    if (a.causal && k0 + 15 > q0 + shift) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (kj > q0 + 4 * g + r + shift) s[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = power<true>(a, s[r], R[r]) * inv[r];
      dp[r] = s[r] * (dp[r] - delta[r]);      // dS / scale (applied to dK at the end)
    }
    Q.rows(qr, q0 + 64);
    add_tokens<NC>(dv, dc, s);
    D.rows(dr, q0 + 64);
    add_tokens<NC>(dk, qc, dp);
  }
  store_sum<NC>(sX, dv, 1.f, a.dv + b * a.dv_sb + h * a.dv_sh, a.dv_st, k0, a.Tk, a.hd, tid);
  __syncthreads();
  store_sum<NC>(sX, dk, a.scale, a.dk + b * a.dk_sb + h * a.dk_sh, a.dk_st, k0, a.Tk, a.hd, tid);
}

bool operand_ok(const void* p, int64_t sb, int64_t sh, int64_t st, int hd) {
  return p != nullptr && pf_aligned(p, 16) && sb % 4 == 0 && sh % 4 == 0 && st % 4 == 0 && st >= hd && st < (1 << 23);
}

int check(const pf_attn_desc* d, const char* name) {
  PF_REQUIRE(d != nullptr, "%s: null descriptor", name);
  PF_REQUIRE(d->dtype == PF_F32, "%s: dtype must be fp32", name);
  PF_REQUIRE(d->B > 0 && d->H > 0 && d->Tq > 0 && d->Tk > 0 && d->hd > 0 && d->scale > 0.f, "%s: bad shape or scale", name);
  if (d->hd % 4 != 0 || d->hd > 128) {
    pf_set_error("%s: head dim %d is not supported by the fused kernels (multiple of 4, <= 128)", name, d->hd);
    return PF_ERR_UNSUPPORTED;
  }
  PF_REQUIRE((int64_t)d->B * d->H < (1 << 23) && d->Tq <= 65535 * 16 && d->Tk <= 65535 * 16, "%s: too many heads or tokens", name);
  PF_REQUIRE(d->lse && operand_ok(d->q, d->q_sb, d->q_sh, d->q_st, d->hd) && operand_ok(d->k, d->k_sb, d->k_sh, d->k_st, d->hd) &&
                 operand_ok(d->v, d->v_sb, d->v_sh, d->v_st, d->hd) && operand_ok(d->o, d->o_sb, d->o_sh, d->o_st, d->hd),
             "%s: operands must be 16-byte aligned with strides that are multiples of 4 and tokens apart by hd or more", name);
  if (d->causal) PF_REQUIRE(d->Tk >= d->Tq, "%s: causal attention needs Tk >= Tq", name);
  return PF_OK;
}

Args make_args(const pf_attn_desc* d) {
  Args a;
  a.q = (const float*)d->q; a.k = (const float*)d->k; a.v = (const float*)d->v; a.o = (const float*)d->o; a.d_o = (const float*)d->d_o;
  a.out = (float*)d->o; a.dq = (float*)d->dq; a.dk = (float*)d->dk; a.dv = (float*)d->dv; a.stats = d->lse; a.delta = d->delta;
  a.q_sb = d->q_sb; a.q_sh = d->q_sh; a.q_st = d->q_st; a.k_sb = d->k_sb; a.k_sh = d->k_sh; a.k_st = d->k_st;
  a.v_sb = d->v_sb; a.v_sh = d->v_sh; a.v_st = d->v_st; a.o_sb = d->o_sb; a.o_sh = d->o_sh; a.o_st = d->o_st;
  a.do_sb = d->do_sb; a.do_sh = d->do_sh; a.do_st = d->do_st; a.dq_sb = d->dq_sb; a.dq_sh = d->dq_sh; a.dq_st = d->dq_st;
  a.dk_sb = d->dk_sb; a.dk_sh = d->dk_sh; a.dk_st = d->dk_st; a.dv_sb = d->dv_sb; a.dv_sh = d->dv_sh; a.dv_st = d->dv_st;
  a.H = d->H; a.Tq = d->Tq; a.Tk = d->Tk; a.hd = d->hd; a.causal = d->causal ? 1 : 0;
  const double x = (double)d->scale * 1.4426950408889634;
  a.scale = d->scale; a.sc = (float)x; a.sc_lo = (float)(x - (double)a.sc);
  return a;
}

// one kernel to every 16 elements of head dimension
#define PF_ATTN32(KERNEL, T)                                                                                     \
  do {                                                                                                           \
    const dim3 grid_((unsigned)(d->B * d->H), (unsigned)(((T) + 15) / 16));                                      \
    switch ((d->hd + 15) / 16) {                                                                                 \
      case 1: hipLaunchKernelGGL(KERNEL<1>, grid_, dim3(256), 0, st, a); break;                                  \
      case 2: hipLaunchKernelGGL(KERNEL<2>, grid_, dim3(256), 0, st, a); break;                                  \
      case 3: hipLaunchKernelGGL(KERNEL<3>, grid_, dim3(256), 0, st, a); break;                                  \
      case 4: hipLaunchKernelGGL(KERNEL<4>, grid_, dim3(256), 0, st, a); break;                                  \
      case 5: hipLaunchKernelGGL(KERNEL<5>, grid_, dim3(256), 0, st, a); break;                                  \
      case 6: hipLaunchKernelGGL(KERNEL<6>, grid_, dim3(256), 0, st, a); break;                                  \
      case 7: hipLaunchKernelGGL(KERNEL<7>, grid_, dim3(256), 0, st, a); break;                                  \
      default: hipLaunchKernelGGL(KERNEL<8>, grid_, dim3(256), 0, st, a);                                        \
    }                                                                                                            \
  } while (0)

}  // namespace

extern "C" int pf_attention_f32_fwd(const pf_attn_desc* d, void* stream) {
  const int rc = check(d, "pf_attention_f32_fwd");
  if (rc != PF_OK) return rc;
  const Args a = make_args(d);
  hipStream_t st = (hipStream_t)stream;
  PF_ATTN32(attn32_fwd_kernel, d->Tq);
  PF_CHECK_LAUNCH("pf_attention_f32_fwd");
  return PF_OK;
}

extern "C" int pf_attention_f32_bwd(const pf_attn_desc* d, void* stream) {
  const int rc = check(d, "pf_attention_f32_bwd");
  if (rc != PF_OK) return rc;
  PF_REQUIRE(d->delta && operand_ok(d->d_o, d->do_sb, d->do_sh, d->do_st, d->hd) && operand_ok(d->dq, d->dq_sb, d->dq_sh, d->dq_st, d->hd) &&
                 operand_ok(d->dk, d->dk_sb, d->dk_sh, d->dk_st, d->hd) && operand_ok(d->dv, d->dv_sb, d->dv_sh, d->dv_st, d->hd),
             "pf_attention_f32_bwd: gradients must be 16-byte aligned with strides that are multiples of 4 and tokens apart by hd or more");
  const Args a = make_args(d);
  hipStream_t st = (hipStream_t)stream;
  PF_ATTN32(attn32_dq_kernel, d->Tq);
  PF_ATTN32(attn32_dkv_kernel, d->Tk);
  PF_CHECK_LAUNCH("pf_attention_f32_bwd");
  return PF_OK;
}
