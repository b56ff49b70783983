// The direct-to-LDS 16-bit MFMA kernel and its launchers.  Included by one translation unit per
// operand dtype and tile shape (the instantiations take minutes to compile; separate units build in parallel).
#pragma once
#include "pf_gemm_common.h"

namespace {

// ---------------------------------------------------------------------------
// 16-bit MFMA kernel, direct-to-LDS pipeline (the throughput path)
//
// Operand tiles go from global memory straight into LDS (buffer_load_dwordx4 ... lds:
// no staging registers, no LDS store instructions), ST tiles deep.  One such
// instruction fills 1024 consecutive LDS bytes, lane l supplying the 16-byte chunk at
// position l, but every lane fetches from an address of its own: the chunk order inside
// LDS is therefore free, and it is chosen (XOR swizzle) so that the MFMA fragment reads
// are bank-conflict free without padding:
//   reduction-contiguous operand  [row][k]: chunk c of a row sits at c ^ f(row), fragments
//                                           are single ds_read_b128;
//   reduction-strided operand     [k][row]: kept in that order (8-row chunk c of k-row k at
//                                           c ^ 4*(k%4)) and read with ds_read_b64_tr_b16,
//                                           the transposing LDS read, which hands a lane
//                                           four consecutive k of one row.
// Each wavefront owns a (BM/WGM) x (BN/WGN) block of accumulators, computed with v_mfma_f32_16x16x32.  That
// shape instead of 32x32x16 because of power: at the same peak rate (on zeros 2.4 PFLOP/s either way) the matrix pipes
// of the whole chip sustain 1.87 against 1.63 PFLOP/s (fp16, random data; bf16 1.99 / 1.76; pf_mfma_rate.hip), and a
// large product is bound by the board's power.  The price is twice as many instructions of half the length, so the K loop deals out its LDS reads and
// loads one at a time between them.  The K loop has ONE barrier per tile, before the tile's last MFMA group: by
// then the group's fragments are in registers, so the buffer can be refilled at once, and the first fragments
// of the next tile are read under that last group's MFMAs (no LDS latency exposed at the barrier).
// Measured against the 32x32x16 form with an epilogue through LDS (us): 8192^3 fp16 946 -> 852;
// [3152 x 1024] . [1024 x 1024] 11.9 -> 10.7, [3152 x 4096] . [4096 x 1024] 34.0 -> 30.1,
// [3152 x 1024] . [1024 x 4096] 33.7 -> 30.9; one workgroup's fixed cost at K = 64: 256x256 7.6 -> 6.3,
// 128x128 4.2 -> 3.4; weight gradient 4096x4096 over 4096 rows 128.5 -> 113.6.
// ---------------------------------------------------------------------------
#define PF_LDS(T) __attribute__((address_space(3))) T*
typedef int v2i_t __attribute__((ext_vector_type(2)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

typedef short short8_t __attribute__((ext_vector_type(8)));
// MFMA operand fragment as it comes out of LDS: one 16-byte read, or (transposing reads) two
// 8-byte halves that are only joined where the MFMA consumes them, so that nothing in the
// group that issues the reads depends on their data
template <bool TRANS> struct Frag;
template <> struct Frag<false> {
  short8_t v;
  __device__ __forceinline__ short8_t get() const { return v; }
};
template <> struct Frag<true> {
  short4_t lo, hi;
  __device__ __forceinline__ short8_t get() const { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }
};
// Keeps the registers of a fragment that inline assembly reads into allocated to it up to this
// point of the program: the compiler takes the output of such a read for complete where the read
// is issued, and once the value is dead it is free to put something else into the register, which
// the read, arriving later, would then overwrite.
__device__ __forceinline__ void frag_hold(Frag<false>&) {}
__device__ __forceinline__ void frag_hold(Frag<true>& f) { asm volatile("" : "+v"(f.lo), "+v"(f.hi)); }
template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// PW > 1 (right-hand operand of a row-major product): inside every 16*PW rows the tile holds row PW*i + t
// as row i of MFMA tile t, so that the accumulators a lane keeps of PW tiles are PW CONSECUTIVE columns
// of the result.
template <int R, int BK, int NW, bool TRANS, int PW> struct DTile {
  static constexpr int BYTES = R * BK * 2;
  static constexpr int NI = BYTES / 1024;  // wavefront-wide load instructions per tile
  static constexpr int IPW = (NI + NW - 1) / NW;   // ... per wavefront
  // (12 instructions over 8 wavefronts, the 192-row tile: the last two wavefronts repeat the last one, the
  // same bytes to the same place, so that every wavefront has the same number of loads in flight)
  static __device__ __forceinline__ int instr(int wave, int q) {
    return NI % NW == 0 || wave * IPW + q < NI ? wave * IPW + q : NI - 1;
  }
  static constexpr int CPR = BK / 8;       // [row][k]: 16-byte chunks per row
  static constexpr int RPI = 64 / CPR;     //           rows per instruction
  static constexpr int ROWB = TRANS ? R * 2 : BK * 2;  // bytes per LDS row
  static constexpr int CPK = R / 8;        // [k][row]: chunks per k-row
  static constexpr int KPI = 64 / CPK;     //           k-rows per instruction
  static_assert(!TRANS || R == 64 || R == 128 || R == 256, "transposed tiles are 64, 128 or 256 rows wide");
  static_assert(BK == 64 || BK == 32, "BK is 32 or 64");

  static __device__ __forceinline__ int swz_row(int row) { return BK == 64 ? ((row >> 1) & 7) : ((row >> 1) & 3); }
  // (the four k-rows and two neighbouring k-groups that transposing reads touch together land on different banks;
  // 64-row tiles have two k-rows per 256 bytes of banks)
  static __device__ __forceinline__ int swz_k(int k) {
    return R == 64 ? (((k >> 1) & 1) << 2) ^ (((k >> 3) & 1) << 1) : ((k & 3) << 2) ^ (((k >> 3) & 1) << 1);
  }

  static __device__ __forceinline__ uint32_t extent(int64_t R_total, int64_t K, int64_t ld) {
    return TRANS ? (uint32_t)(((K - 1) * ld + (R_total + 7) / 8 * 8) * 2)
                 : (uint32_t)(((R_total - 1) * ld + (K + 7) / 8 * 8) * 2);
  }
  // byte offset (inside K-tile 0) of the chunk this lane fetches in its q-th instruction
  // tail[q]: all ones if that chunk lies past the `left` reduction elements of the last K-tile (RAG kernels)
  static __device__ __forceinline__ void init(uint32_t (&off)[IPW], uint32_t (&tail)[IPW], int64_t ld, int64_t r0, int left, int wave,
                                              int lane) {
#pragma unroll
    for (int q = 0; q < IPW; ++q) {
      const int ii = instr(wave, q);
      if (!TRANS) {
        const int row = ii * RPI + lane / CPR;
        const int c = (lane % CPR) ^ swz_row(row);
        const int src = PW > 1 ? row / (16 * PW) * (16 * PW) + (row & 15) * PW + (row >> 4) % PW : row;
        off[q] = (uint32_t)(((r0 + src) * ld + c * 8) * 2);
        tail[q] = c * 8 >= left ? 0xffffffffu : 0u;
      } else {
        const int k = ii * KPI + lane / CPK;
        const int mc = (lane % CPK) ^ swz_k(k);
        off[q] = (uint32_t)((k * ld + r0 + mc * 8) * 2);
        tail[q] = 0u;   // (whole k-rows past K fall outside the buffer)
      }
    }
  }
  static __device__ __forceinline__ uint32_t tile_step(int64_t ld) { return TRANS ? (uint32_t)(BK * ld * 2) : (uint32_t)(BK * 2); }
  // lds: byte address of this operand's tile inside LDS (wave-uniform); issues the wavefront's
  // instructions Q0 <= q < Q1 (clipped to [0, IPW))
  // (RAG: sel = ~0 for the last K-tile sends the chunks past K out of the buffer's range, which reads zeros)
  template <int Q0, int Q1, bool RAG>
  static __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rs, const uint32_t (&off)[IPW], const uint32_t (&tail)[IPW],
                                               uint32_t adv, uint32_t sel, uint32_t lds, int wave) {
#pragma unroll
    for (int q = (Q0 < 0 ? 0 : Q0); q < (Q1 > IPW ? IPW : Q1); ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (PF_LDS(void))(uintptr_t)(lds + (uint32_t)instr(wave, q) * 1024u), 16,
                                               (int)(RAG ? (off[q] + adv) | (tail[q] & sel & 0x80000000u) : off[q] + adv), 0, 0, 0);
  }
  // Fragment addressing.  w0: first row of the wavefront's block inside the tile.
  //   [row][k]: foff[kk] = byte offset of (row w0 + lane%16, chunk 4*kk + lane/16); + i*16*ROWB per MFMA tile
  //   [k][row]: foff[0]  = byte offset for MFMA tile 0 at kk = 0, first half; + (32*kk + 4*h)*ROWB; tile i
  //             differs in address bits that only the swizzle touches, by exclusive or: ^ tile_xor(i)
  // kk0: first 32-deep MFMA group of a tile that this wavefront multiplies (wavefronts that split
  // a tile's reduction depth between them start at different groups)
  // (a wavefront's block starts at a multiple of its own width, a power of two times 16 rows)
  static constexpr uint32_t tile_xor(int i) { return (uint32_t)(i * 32); }
  template <int NF>
  static __device__ __forceinline__ void frag_init(uint32_t (&foff)[NF], int w0, int lane, int kk0) {
    if constexpr (!TRANS) {
      const int row = w0 + (lane & 15), quarter = lane >> 4;
#pragma unroll
      for (int kk = 0; kk < NF; ++kk) foff[kk] = (uint32_t)(row * ROWB + ((((kk0 + kk) * 4 + quarter) ^ swz_row(row)) * 16));
    } else {
      const int g = lane >> 4, j = lane & 15;
      const int k = g * 8 + (j >> 2);
      const int m = w0 + 4 * (j & 3);
#pragma unroll
      for (int i = 0; i < NF; ++i) foff[i] = (uint32_t)((k + kk0 * 32) * ROWB + (((m >> 3) ^ swz_k(k)) * 16) + (m & 7) * 2) ^ tile_xor(i);
    }
  }
  static constexpr int NRD = TRANS ? 2 : 1;   // LDS reads per fragment
  // read H of MFMA tile I's fragment of group KKI
  template <int NF, int I, int KKI, int H>
  static __device__ __forceinline__ void read(Frag<TRANS>& f, uint32_t lds, const uint32_t (&foff)[NF]) {
    if constexpr (!TRANS) {
      f.v = *(PF_LDS(const short8_t))(uintptr_t)(lds + foff[KKI] + (uint32_t)(I * 16 * ROWB));
    } else {
      // Inline assembly on purpose: the compiler makes an LDS read it cannot tell apart from the
      // destination of an earlier direct-to-LDS load wait for ALL outstanding loads, and it cannot
      // for this instruction, which would serialise the whole tile pipeline.  The price: it does
      // not know that these results arrive asynchronously either; the K loop waits for them by hand.
      const uint32_t a = lds + (NF > 1 ? foff[NF > 1 ? I : 0] : (foff[0] ^ tile_xor(I)));
      if constexpr (H == 0) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(f.lo) : "v"(a), "n"(KKI * 32 * ROWB) : "memory");
      else asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(f.hi) : "v"(a), "n"(KKI * 32 * ROWB + 4 * ROWB) : "memory");
    }
  }
  template <int NF, int I>
  static __device__ __forceinline__ void read_first(Frag<TRANS>& f, uint32_t lds, const uint32_t (&foff)[NF]) {
    static_for<NRD>([&](auto hc) { read<NF, I, 0, decltype(hc)::value>(f, lds, foff); });
  }
};

// reads among the events e = 0 .. ne-1 (nl of them loads, spread evenly) dealt to the slots 0 .. m of ns
constexpr int count_reads(int ne, int ns, int nl, int m) {
  int n = 0;
  for (int e = 0; e < ne; ++e)
    if (e * ns / ne <= m && (e + 1) * nl / ne == e * nl / ne) ++n;
  return n;
}

template <int DT> __device__ __forceinline__ float unpack1(uint32_t w, int hi) {
  if (DT == PF_BF16) return __uint_as_float(hi ? (w & 0xffff0000u) : (w << 16));
  return pf_f16_bits_to_f32((uint16_t)(hi ? (w >> 16) : (w & 0xffffu)));
}
template <int DT> __device__ __forceinline__ uint32_t pack2(float a, float b) {
  return DT == PF_BF16 ? pf_pack2_bf16(a, b) : pf_pack2_f16(a, b);
}
// N 32-bit words that travel in one buffer access (8 words: two)
template <int N> struct Words {
  int w[N];
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
    if constexpr (N == 1) {
      w[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0);
    } else if constexpr (N == 2) {
      const v2i_t t = __builtin_amdgcn_raw_buffer_load_b64(rs, (int)off, 0, 0);
      w[0] = t.x; w[1] = t.y;
    } else {
#pragma unroll
      for (int q = 0; q < N; q += 4) {
        const v4i_t t = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off + q * 4), 0, 0);
#pragma unroll
        for (int k = 0; k < 4; ++k) w[q + k] = t[k];
      }
    }
  }
  __device__ __forceinline__ void store(__amdgpu_buffer_rsrc_t rs, uint32_t off) const {
    if constexpr (N == 1) {
      __builtin_amdgcn_raw_buffer_store_b32(w[0], rs, (int)off, 0, 0);
    } else if constexpr (N == 2) {
      const v2i_t t = {w[0], w[1]};
      __builtin_amdgcn_raw_buffer_store_b64(t, rs, (int)off, 0, 0);
    } else {
#pragma unroll
      for (int q = 0; q < N; q += 4) {
        const v4i_t t = {w[q], w[q + 1], w[q + 2], w[q + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(t, rs, (int)(off + q * 4), 0, 0);
      }
    }
  }
};

// A 16-row block's accumulators for the epilogue; out of the accumulation registers by hand, where they are used (left
// to itself the compiler moves all of them at once, and spills)
template <bool AGPR, int TN> __device__ __forceinline__ void acc_read(float4_t (&x)[TN], const float4_t (&acc)[TN]) {
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    if constexpr (AGPR) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v;
        asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc[j][r]));
        x[j][r] = v;
      }
    } else {
      x[j] = acc[j];
    }
  }
}

// `pid`: index of this workgroup among the workgroups of its problem (the launch may hold several
// problems, see gemm16x_group_kernel)
template <int DT, int BM, int BN, int BK, int WGM, int WGN, int KS, int ST, bool AT, bool BT, int EC, bool RAG = false>
__device__ __forceinline__ void gemm16x_body(const pf_gemm_desc& p, const GemmGrid& g, const int pid) {
  // KS = 2: the wavefronts form two WGM x WGN grids; grid h multiplies the h-th half of every
  // tile's 16-deep MFMA groups, and the two partial accumulator blocks are added through LDS
  // before the epilogue.  Eight wavefronts (two per SIMD, so that one's LDS reads and waits run
  // under the other's MFMAs) then read no more fragment bytes from LDS than four do, and the
  // LDS port (128 B/clk per CU for fragment reads and arriving tiles together) is what bounds
  // these tiles.
  constexpr int NWMN = WGM * WGN;
  constexpr int NW = NWMN * KS;
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int TM = WM / 16, TN = WN / 16;
  constexpr int KK = BK / 32 / KS;     // 32-deep MFMA groups per tile and wavefront
  static_assert(KS == 1 || KS == 2, "the reduction depth of a tile is split over one or two wavefront grids");
  static_assert((BK / 32) % KS == 0 && KK >= 1, "MFMA groups do not divide over the wavefront grids");
  constexpr bool C32 = EC == EC_STORE32 || EC == EC_RES32 || EC == EC_ACC32;
  using TA = DTile<BM, BK, NW, AT, 1>;
  using TB = DTile<BN, BK, NW, BT, BT ? 1 : TN>;
  constexpr int STAGE = TA::BYTES + TB::BYTES;
  constexpr int LPW = TA::IPW + TB::IPW;  // load instructions per wavefront per tile
  static_assert((ST - 1) * LPW <= 63, "too many loads in flight for the 6-bit counter");
  // (transposing reads: an address per MFMA tile where the block leaves the registers for it; the small blocks
  // are bound by instruction issue)
  constexpr int NFA = AT ? (TM * TN <= 16 ? TM : 1) : KK, NFB = BT ? (TM * TN <= 16 ? TN : 1) : KK;
  static_assert((!AT || (WM & (WM - 1)) == 0) && (!BT || (WN & (WN - 1)) == 0), "tile_xor");
  // Two stages (three of the right-hand operand): four wavefronts with 128x128 blocks, one to a SIMD, see below
  constexpr bool TWO = ST == 2;
  static_assert(!TWO || (NW == 4 && TM * TN == 64 && KS == 1 && BK == 64 && !RAG), "the two-stage pipeline's tile");
  extern __shared__ __align__(16) uint16_t smem[];

  const int t = gemm_tile_id(pid, g.tiles_m * g.tiles_n, g.per_xcd);
  if (t < 0) return;
  int tm, tn;
  gemm_tile_rc(t, g.tiles_m, g.tiles_n, tm, tn);
  const int64_t M = p.M, N = p.N, K = p.K, lda = p.lda, ldb = p.ldb;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int64_t z = blockIdx.y, z1 = z / p.batch2, z2 = z % p.batch2;
  const uint16_t* A = (const uint16_t*)p.A + z1 * p.a_stride1 + z2 * p.a_stride2;
  const uint16_t* B = (const uint16_t*)p.B + z1 * p.b_stride1 + z2 * p.b_stride2;
  const int64_t c_base = z1 * p.c_stride1 + z2 * p.c_stride2;
  const Epi epi = make_epi(p);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_k = wave / NWMN, wave_mn = wave % NWMN;
  const int wm0 = (wave_mn / WGN) * WM, wn0 = (wave_mn % WGN) * WN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  const __amdgpu_buffer_rsrc_t rs_a = make_rsrc(A, TA::extent(M, K, lda));
  const __amdgpu_buffer_rsrc_t rs_b = make_rsrc(B, TB::extent(N, K, ldb));
  uint32_t offa[TA::IPW], offb[TB::IPW], taila[TA::IPW], tailb[TB::IPW];
  const int nk = (int)((K + BK - 1) / BK);
  TA::init(offa, taila, lda, m0, (int)(K - (int64_t)(nk - 1) * BK), wave, lane);
  TB::init(offb, tailb, ldb, n0, (int)(K - (int64_t)(nk - 1) * BK), wave, lane);
  const uint32_t step_a = TA::tile_step(lda), step_b = TB::tile_step(ldb);
  uint32_t foa[NFA], fob[NFB];
  TA::template frag_init<NFA>(foa, wm0, lane, wave_k * KK);
  TB::template frag_init<NFB>(fob, wn0, lane, wave_k * KK);

  // This lane's part of C: rows row0 + 16 i + r (r = 0..3); columns c0 .. c0 + TN - 1, one per MFMA tile, of a
  // row-major product (see DTile's PW), c0 + 16 j of a reduction-strided one (the transposing LDS reads fix
  // the order of its columns).  16 neighbouring lanes cover 16 * TN (or 16) consecutive columns of a row:
  // neighbouring lanes have to, the address coalescer joins the accesses of lanes 4 k .. 4 k + 3 only.
  // (The two-stage pipeline's transposed operands go to the MFMA tiles eight rows to a lane: rows row0 + 8 r + i, and
  // again TN consecutive columns.)
  constexpr bool RUNS = !BT || TWO;        // a lane keeps runs of TN columns
  const int64_t row0 = m0 + wm0 + (lane >> 4) * (AT && TWO ? 32 : 4);
  const int64_t c0 = n0 + wn0 + (lane & 15) * (RUNS ? TN : 1);
  auto row_in = [](uint32_t h, uint32_t r) { return AT && TWO ? 8 * r + h : 16 * h + r; };
  float bias[TN];
  // One branch on the dtype around all of the bias loads; a missing bias, and columns past N, read as zeros
  // through the buffer's extent.
  auto load_bias = [&]() {
    const bool b32 = epi.bias_dtype == PF_F32;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(epi.bias, epi.bias != nullptr ? (uint32_t)(N * (b32 ? 4 : 2)) : 0u);
    if (b32) {
#pragma unroll
      for (int j = 0; j < TN; ++j) bias[j] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)((c0 + j) * 4), 0, 0));
    } else {
      uint32_t raw[TN / 2];
#pragma unroll
      for (int j = 0; j < TN / 2; ++j) raw[j] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, (int)((c0 + 2 * j) * 2), 0, 0);
      const bool bf = epi.bias_dtype == PF_BF16;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const uint32_t h = (raw[j / 2] >> (16 * (j % 2))) & 0xffffu;
        bias[j] = bf ? __uint_as_float(h << 16) : pf_f16_bits_to_f32((uint16_t)h);
      }
    }
  };
  // Fetched before the K loop, which hides the latency; after it in the GELU' class, which hardly ever has a
  // bias and has no registers to spare for one.  (Weight-gradient products with a bias take the generic class.)
  constexpr bool HAS_BIAS = EC != EC_GENERIC && !AT;
  constexpr bool BIAS_EARLY = HAS_BIAS && EC != EC_DACT16;
  if constexpr (BIAS_EARLY) load_bias();

  // Tiles past the end of K are requested too, at an offset beyond the buffer extent: the hardware
  // range check drops them (no memory traffic), and every iteration of the K loop is the same
  // straight-line code with the same number of loads in flight.
  // The loads of one tile are dealt over the sub-groups of one MFMA group: a burst of them would fill the
  // memory pipeline's queue and stall the wavefront for as long as the tile takes to stream in.
  static_assert(ST >= 3 || TWO, "a stage is refilled while the next tile is multiplied");
  auto adv_of = [&](int kt, uint32_t step) { return kt < nk ? (uint32_t)kt * step : 0x80000000u; };
  auto sel_of = [&](int kt) { return RAG && kt == nk - 1 ? 0xffffffffu : 0u; };
  auto issue_all = [&](int kt, uint32_t sb) {
    TA::template issue<0, TA::IPW, RAG>(rs_a, offa, taila, adv_of(kt, step_a), sel_of(kt), sb, wave);
    TB::template issue<0, TB::IPW, RAG>(rs_b, offb, tailb, adv_of(kt, step_b), sel_of(kt), sb + TA::BYTES, wave);
  };
  // One 32-deep MFMA group ("phase") = NM matrix instructions on the fragments in register set `cur`, the
  // LDS reads that fill the other set for the next phase, and its share of the loads that refill the
  // stage that is free.  An MFMA occupies the matrix pipe for 16 cycles and the wavefront issues in order:
  // the reads and loads are dealt out ONE at a time between the MFMAs (each followed by a scheduling
  // barrier), evenly over the first 7/8 of the phase; two or three of them side by side leave the pipe idle.
  // (The phase that starts with a barrier waits for all of its predecessor's reads.)
  // Blocks of more than 128 accumulator registers (the four-wavefront 256x256 and 192x256 tiles), and those that exchange
  // half their sums with another wavefront, have no room for two sets of fragments: they read a phase's fragments at its start (SINGLE).
  constexpr int NM = TM * TN;
  constexpr bool SINGLE = !TWO && (NM > 32 || (KS == 2 && NM == 32));
  constexpr int NREADS = TM * TA::NRD + TN * TB::NRD;
  Frag<AT> fa[SINGLE ? 1 : 2][TM];
  Frag<BT> fb[SINGLE ? 1 : 2][TN];
  // kkn: MFMA group (of the tile in stage sbr) whose fragments are read into the other register set;
  // loads PART * LPW / PARTS .. (PART + 1) * LPW / PARTS - 1 of tile ktl go into stage sbl
  auto phase = [&](uint32_t sbr, auto kknc, auto curc, auto partc, auto partsc, int ktl, uint32_t sbl) {
    constexpr int kkn = decltype(kknc)::value, cur = SINGLE ? 0 : decltype(curc)::value, slot = cur ^ 1;
    constexpr int PART = decltype(partc)::value, PARTS = decltype(partsc)::value;
    constexpr int Q0 = PART * LPW / PARTS, NL = (PART + 1) * LPW / PARTS - Q0;
    constexpr int NRE = SINGLE ? 0 : NREADS;
    constexpr int NE = NRE + NL;                     // reads and loads, interleaved evenly
    if constexpr (SINGLE) {
      static_for<TN>([&](auto jc) {
        static_for<TB::NRD>([&](auto hc) { TB::template read<NFB, decltype(jc)::value, kkn, decltype(hc)::value>(fb[0][decltype(jc)::value], sbr + TA::BYTES, fob); });
      });
      static_for<TM>([&](auto ic) {
        static_for<TA::NRD>([&](auto hc) { TA::template read<NFA, decltype(ic)::value, kkn, decltype(hc)::value>(fa[0][decltype(ic)::value], sbr, foa); });
      });
    }
    constexpr int NS = NM > 8 ? NM * 7 / 8 : NM;
    const uint32_t adv_a = adv_of(ktl, step_a), adv_b = adv_of(ktl, step_b), sel = sel_of(ktl);
    if constexpr (AT && BT && SINGLE) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int i = 0; i < TM; ++i) frag_hold(fa[0][i]);   // (nothing that uses them may move above the wait)
#pragma unroll
      for (int j = 0; j < TN; ++j) frag_hold(fb[0][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    static_for<NM>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      static_for<NE>([&](auto ec) {
        constexpr int e = decltype(ec)::value;
        if constexpr (e * NS / NE == m) {
          // event e is a load where the running count of loads steps up, else a read
          constexpr int l0 = e * NL / NE, l1 = (e + 1) * NL / NE;
          if constexpr (l1 > l0) {
            constexpr int q = Q0 + l0;                   // index into A's then B's list of loads
            if constexpr (q < TA::IPW) TA::template issue<q, q + 1, RAG>(rs_a, offa, taila, adv_a, sel, sbl, wave);
            else TB::template issue<q - TA::IPW, q - TA::IPW + 1, RAG>(rs_b, offb, tailb, adv_b, sel, sbl + TA::BYTES, wave);
          } else {
            constexpr int r = e - l0;                    // B's fragments first, then A's
            if constexpr (r < TN * TB::NRD) TB::template read<NFB, r / TB::NRD, kkn, r % TB::NRD>(fb[slot][r / TB::NRD], sbr + TA::BYTES, fob);
            else {
              constexpr int ra = r - TN * TB::NRD;
              TA::template read<NFA, ra / TA::NRD, kkn, ra % TA::NRD>(fa[slot][ra / TA::NRD], sbr, foa);
            }
          }
        }
      });
      if constexpr (AT && BT && !SINGLE && m % TN == 0) {
        // This row of MFMAs takes fragments read by inline assembly during the previous phase, B's and A's up
        // to row m / TN.  LDS answers in order: they are there once no more reads are outstanding than came after.
        constexpr int need = TN * TB::NRD + (m / TN + 1) * TA::NRD;
        constexpr int issued = count_reads(NE, NS, NL, m);
        constexpr int later = NREADS - need + issued;
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(later < 15 ? later : 15) : "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
      constexpr int i = m / TN, j = (i & 1) ? TN - 1 - m % TN : m % TN;   // (serpentine: one operand changes at a time)
      acc[i][j] = Mfma<DT>::run16(fa[cur][i].get(), fb[cur][j].get(), acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  if constexpr (TWO) {
    // What bounds the tiles above is the way of the operands, not the matrix pipes: eight 128x64 blocks of a 256x256 tile
    // read 96 KB of fragments per 32 of depth and 32 KB arrive, together all that the LDS port moves while the MFMAs run, and a
    // tile step 32 deep takes half of every 128-byte line it requests.  Four wavefronts with 128x128 blocks read a
    // third less, steps 64 deep request whole lines (half the requests to the L2), and there is one barrier per 128
    // MFMAs.  One wavefront to a SIMD has the registers for it: 256 accumulators (AGPRs, named in the MFMAs by hand:
    // the compiler's own choice moves them about inside the loop) and two sets of fragments, so that a phase's reads
    // run under the phase before.  160 KB are two stages of A and THREE of B: B's tile kt + 2 is requested during
    // the first phase of tile kt, A's during the second, when the last fragments of tile kt are in registers; at even
    // spacing, as four wavefronts that all load at once stall each other.  Each load has a tile's time, 2048 cycles, to arrive.
    // 8192^3 926 -> 775 us (bf16; 1.42 PFLOP/s), [8192 x 5632] . [5632 x 2048] 160 -> 140, 4096 x 4096 over 32768 977 -> 766,
    // [12608 x 4096] . [4096 x 1024] 111 -> 97, over 1024 30 -> 28 (eight wavefronts -> four, one card).
    // A lone wavefront has no other to issue under its MFMAs: whatever stands between two of them beyond two or three
    // instructions is time.  So a tile's place in memory is in the descriptor, two scalar sums and a choice of its extent per tile in
    // place of an addition per load (past the end of K the extent is empty and the loads are dropped), four loads share one
    // LDS base, and loads and fragment reads take turns: 245 -> 202 instructions per 128 MFMAs beside them, 8192^3
    // 716 -> 698 us, 4096 x 4096 over 12608 281 -> 275, [8192 x 5632] . [5632 x 2048] 149 -> 145.
    static_assert(TA::IPW == 8 && TB::IPW == 8, "eight loads of 1 KB per wavefront and operand tile");
    constexpr int LEAD = 3072;      // four loads share an LDS base: their distance is in the instruction, which moves both addresses
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      offa[q] += LEAD - (q & 3) * 1024;
      offb[q] += LEAD - (q & 3) * 1024;
    }
    const uint32_t ext_a = TA::extent(M, K, lda), ext_b = TB::extent(N, K, ldb);
    // (A row-major operand's extent goes on past the end of its rows, so whether there is a tile kt is asked of kt: the two tiles
    // past K that it would let through were 25 % of a launch's read requests to the L2 at K = 384, 11 % at 1024, 9 % at 1280.  Alone
    // the times are the same, within 0.5 %.)
    auto tile_rsrc = [&](const uint16_t* base, uint32_t ext, int kt, uint32_t step) {
      const uint32_t adv = (uint32_t)kt * step;
      return make_rsrc((const char*)base - LEAD + adv, kt < nk ? ext + LEAD - adv : 0u);
    };
    auto fetch = [&](__amdgpu_buffer_rsrc_t rs, const uint32_t (&off)[8], uint32_t dst, auto qc) {
      constexpr int q = decltype(qc)::value;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (PF_LDS(void))(uintptr_t)(dst + (uint32_t)wave * 8192u + (q / 4) * 4096u), 16, (int)off[q], 0, (q & 3) * 1024, 0);
    };
    auto fetch_a = [&](int kt, uint32_t dst) { static_for<8>([&](auto qc) { fetch(tile_rsrc(A, ext_a, kt, step_a), offa, dst, qc); }); };
    auto fetch_b = [&](int kt, uint32_t dst) { static_for<8>([&](auto qc) { fetch(tile_rsrc(B, ext_b, kt, step_b), offb, dst, qc); }); };
    auto mm = [&](auto curc, auto lac, uint32_t ra, uint32_t rb, int ktl, uint32_t dst) {
      constexpr int cur = decltype(curc)::value, slot = cur ^ 1, kkn = cur ^ 1;
      constexpr bool LA = decltype(lac)::value;           // this phase requests A's tile (else B's)
      const __amdgpu_buffer_rsrc_t rs = LA ? tile_rsrc(A, ext_a, ktl, step_a) : tile_rsrc(B, ext_b, ktl, step_b);
      static_for<NM>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        static_for<8>([&](auto ec) {
          constexpr int l = decltype(ec)::value;
          if constexpr (7 * l + 2 == m) fetch(rs, LA ? offa : offb, dst, ec);
        });
        static_for<NREADS>([&](auto ec) {
          constexpr int r = decltype(ec)::value;
          if constexpr (r * 7 / 2 == m) {   // (never beside a load: each slot takes one more instruction or two)
            if constexpr (r < TN * TB::NRD) TB::template read<NFB, r / TB::NRD, kkn, r % TB::NRD>(fb[slot][r / TB::NRD], rb, fob);
            else {
              constexpr int q = r - TN * TB::NRD;
              TA::template read<NFA, q / TA::NRD, kkn, q % TA::NRD>(fa[slot][q / TA::NRD], ra, foa);
            }
          }
        });
        constexpr int i = m / TN, j = (i & 1) ? TN - 1 - m % TN : m % TN;
        Mfma<DT>::run16_agpr(fa[cur][i].get(), fb[cur][j].get(), acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    // Reduction-strided operands lie in LDS as they do in memory, [k][row].  ds_read_b64_tr_b16 moves 64 bytes a cycle, half of what
    // ds_read_b128 does, and bounds these products on the other tiles.  Here a lane reads eight whole 16-byte chunks, eight rows
    // of one k each, and puts its eight fragments together in registers, one byte permutation per pair of k: lane i's rows
    // 8 i + t are row i of MFMA tile t.  32 permutations per operand and phase run between the MFMAs: A's tile t + 1 while
    // tile t is multiplied, B's for the next phase as its chunks arrive, none beside two others.  bf16, eight wavefronts
    // with transposing reads / this: 4096 x 4096 over 12608 323 / 312 us, over 3152 104 / 100, 4096 x 1024 over 12608 239 / 226,
    // 2048 x 5632 over 32768 655 / 637, 32000 x 2048 over 788 184 / 175 (the permutations keep it 5 % behind row-major
    // products of these sizes).
    short8_t rwa[AT ? 2 : 1][8], rwb[8];
    u32x4_t fpa[2], fpb[2][8];
    uint32_t fta[4], ftb[4];
    if constexpr (AT && BT) {
      const int g8 = (lane >> 4) * 8, c = (lane & 15) ^ (((lane >> 4) & 1) << 1);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        fta[q] = (uint32_t)(g8 * TA::ROWB + (wm0 / 8 + (c ^ (q << 2))) * 16);
        ftb[q] = (uint32_t)(g8 * TB::ROWB + (wn0 / 8 + (c ^ (q << 2))) * 16);
      }
    }
    auto raw_a = [&](short8_t& f, uint32_t lds, auto ec, auto kkc) {
      constexpr int e = decltype(ec)::value, kk = decltype(kkc)::value;
      f = *(PF_LDS(const short8_t))(uintptr_t)(lds + fta[e & 3] + (uint32_t)((kk * 32 + e) * TA::ROWB));
    };
    auto raw_b = [&](short8_t& f, uint32_t lds, auto ec, auto kkc) {
      constexpr int e = decltype(ec)::value, kk = decltype(kkc)::value;
      f = *(PF_LDS(const short8_t))(uintptr_t)(lds + ftb[e & 3] + (uint32_t)((kk * 32 + e) * TB::ROWB));
    };
    // dword P of tile T's fragment: k 2 P and 2 P + 1 of row T of the lane's eight
    auto join = [](u32x4_t& f, const short8_t (&raw)[8], auto tc, auto pc) {
      constexpr int T = decltype(tc)::value, P = decltype(pc)::value;
      const u32x4_t lo = __builtin_bit_cast(u32x4_t, raw[2 * P]), hi = __builtin_bit_cast(u32x4_t, raw[2 * P + 1]);
      f[P] = __builtin_amdgcn_perm(hi[T / 2], lo[T / 2], T % 2 ? 0x07060302u : 0x05040100u);
    };
    auto mt = [&](auto curc, auto lac, uint32_t ra, uint32_t rb, int ktl, uint32_t dst) {
      constexpr int cur = decltype(curc)::value, kkn = cur ^ 1;
      constexpr bool LA = decltype(lac)::value;
      constexpr std::integral_constant<int, kkn> kknc{};
      const __amdgpu_buffer_rsrc_t rs = LA ? tile_rsrc(A, ext_a, ktl, step_a) : tile_rsrc(B, ext_b, ktl, step_b);
      static_for<NM>([&](auto mc) {
        constexpr int m = decltype(mc)::value, i = m / TN, j = (i & 1) ? TN - 1 - m % TN : m % TN;
        static_for<8>([&](auto ec) {
          constexpr int l = decltype(ec)::value;
          if constexpr (7 * l + 2 == m) fetch(rs, LA ? offa : offb, dst, ec);
        });
        // the next phase's chunks: B's first
        if constexpr (m < 16 && m % 2 == 1) raw_b(rwb[m / 2], rb, std::integral_constant<int, m / 2>{}, kknc);
        if constexpr (m >= 16 && m < 48 && m % 4 == 0) raw_a(rwa[cur ^ 1][m / 4 - 4], ra, std::integral_constant<int, m / 4 - 4>{}, kknc);
        // A's next fragment (after the last row of MFMAs, the next phase's first); its last part two MFMAs before its first
        // use, the distance that the matrix instructions ask of a register written by another
        if constexpr (m % 2 == 0) {
          constexpr std::integral_constant<int, (i + 1) & 7> tc{};
          constexpr std::integral_constant<int, (m % TN) / 2> pc{};
          join(fpa[(i + 1) & 1], rwa[i == TM - 1 ? (cur ^ 1) : cur], tc, pc);
        }
        // B's for the next phase, in the order in which its chunks arrive
        static_for<32>([&](auto nc) {
          constexpr int n = decltype(nc)::value;
          if constexpr ((n < 26 ? 13 + 2 * n : 34 + 4 * (n - 26)) == m)
            join(fpb[cur ^ 1][n % 8], rwb, std::integral_constant<int, n % 8>{}, std::integral_constant<int, n / 8>{});
        });
        Mfma<DT>::run16_agpr(__builtin_bit_cast(short8_t, fpa[i & 1]), __builtin_bit_cast(short8_t, fpb[cur][j]), acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    uint32_t a0 = lds0, a1 = lds0 + TA::BYTES, b0 = lds0 + 2 * TA::BYTES, b1 = b0 + TB::BYTES, b2 = b1 + TB::BYTES;
    fetch_a(0, a0);
    fetch_b(0, b0);
    fetch_b(1, b1);
    fetch_a(1, a1);
    wait_vm<LPW>();
    lds_barrier();
    if constexpr (AT && BT) {
      static_for<8>([&](auto ec) { raw_b(rwb[decltype(ec)::value], b0, ec, std::integral_constant<int, 0>{}); });
      static_for<8>([&](auto ec) { raw_a(rwa[0][decltype(ec)::value], a0, ec, std::integral_constant<int, 0>{}); });
      static_for<8>([&](auto tc) { static_for<4>([&](auto pc) { join(fpb[0][decltype(tc)::value], rwb, tc, pc); }); });
      static_for<4>([&](auto pc) { join(fpa[0], rwa[0], std::integral_constant<int, 0>{}, pc); });
    } else {
      static_for<TN>([&](auto jc) { TB::template read_first<NFB, decltype(jc)::value>(fb[0][decltype(jc)::value], b0, fob); });
      static_for<TM>([&](auto ic) { TA::template read_first<NFA, decltype(ic)::value>(fa[0][decltype(ic)::value], a0, foa); });
    }
    asm volatile("s_nop 7" ::: "memory");   // (the compiler sees no MFMA: the distance to the zeros written to AGPRs is kept by hand)
    __builtin_amdgcn_sched_barrier(0);
    int kt = 0;
    do {
      if constexpr (AT && BT) mt(std::integral_constant<int, 0>{}, std::false_type{}, a0, b0, kt + 2, b2);
      else mm(std::integral_constant<int, 0>{}, std::false_type{}, a0, b0, kt + 2, b2);
      wait_vm<TB::IPW>();
      lds_barrier();       // tile kt + 1 landed everywhere, stage a0 and (since the barrier before) b2 no longer read
      if constexpr (AT && BT) mt(std::integral_constant<int, 1>{}, std::true_type{}, a1, b1, kt + 2, a0);
      else mm(std::integral_constant<int, 1>{}, std::true_type{}, a1, b1, kt + 2, a0);
      const uint32_t ta = a0, tb = b0;
      a0 = a1; a1 = ta;
      b0 = b1; b1 = b2; b2 = tb;
    } while (++kt < nk);
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // (and the distance from the last MFMA to the first read of its result)
  } else {
  // A tile's fragments are in registers at the barrier that opens its last phase: from there on its stage is
  // refilled with the tile ST further on, the first part in that phase, the others in the next tile's
  // phases but its last (one part per phase keeps the stream of loads even).  With one phase per tile the
  // register sets alternate by tile.  (SINGLE reads a phase's fragments inside it: its stage is free one
  // barrier later.)
  // prologue: fill the stages, wait for tile 0
#pragma unroll
  for (int s = 0; s < ST - 1; ++s) issue_all(s, lds0 + (uint32_t)s * STAGE);
  constexpr int P0 = SINGLE ? 0 : LPW / KK;    // loads of tile ST - 1 that go out here
  {
    const uint32_t sbl = lds0 + (uint32_t)(ST - 1) * STAGE, adv_a = adv_of(ST - 1, step_a), adv_b = adv_of(ST - 1, step_b);
    TA::template issue<0, P0, RAG>(rs_a, offa, taila, adv_a, sel_of(ST - 1), sbl, wave);
    TB::template issue<0, P0 - TA::IPW, RAG>(rs_b, offb, tailb, adv_b, sel_of(ST - 1), sbl + TA::BYTES, wave);
  }
  wait_vm<(ST - 2) * LPW + P0>();
  lds_barrier();
  if constexpr (!SINGLE) {
    // (B's first: the phases count on that order when they wait for part of the reads)
    static_for<TN>([&](auto jc) { TB::template read_first<NFB, decltype(jc)::value>(fb[0][decltype(jc)::value], lds0 + TA::BYTES, fob); });
    static_for<TM>([&](auto ic) { TA::template read_first<NFA, decltype(ic)::value>(fa[0][decltype(ic)::value], lds0, foa); });
  }
  __builtin_amdgcn_sched_barrier(0);

  uint32_t sb = lds0;                                   // stage of tile kt
  uint32_t sb_prev = lds0 + (uint32_t)(ST - 1) * STAGE; // stage of tile kt-1
  // one tile; `par`: register set its first phase multiplies
  auto tile = [&](int kt, auto parc) {
    constexpr int par = decltype(parc)::value;
    const uint32_t sb_next = (sb + STAGE == lds0 + (uint32_t)ST * STAGE) ? lds0 : sb + STAGE;
    static_for<KK>([&](auto kkc) {
      constexpr int kk = decltype(kkc)::value;
      constexpr std::integral_constant<int, (par + kk) & 1> cur{};
      constexpr std::integral_constant<int, KK> parts{};
      if constexpr (SINGLE) {
        if (kk == 0 && kt > 0) {
          wait_vm<(ST - 2) * LPW>();
          lds_barrier();                            // tile kt landed everywhere, stage of tile kt-1 no longer read
        }
        phase(sb, kkc, cur, kkc, parts, kt + ST - 1, sb_prev);
      } else if constexpr (kk + 1 < KK) {
        phase(sb, std::integral_constant<int, kk + 1>{}, cur, std::integral_constant<int, kk + 1>{}, parts, kt + ST - 1, sb_prev);
      } else {
        wait_vm<(ST - 2) * LPW>();
        lds_barrier();                              // tile kt+1 landed everywhere, stage sb no longer read
        phase(sb_next, std::integral_constant<int, 0>{}, cur, std::integral_constant<int, 0>{}, parts, kt + ST, sb);
      }
    });
    sb_prev = sb;
    sb = sb_next;
  };
  if constexpr (KK % 2 == 0 || SINGLE) {
    for (int kt = 0; kt < nk; ++kt) tile(kt, std::integral_constant<int, 0>{});
  } else {
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
      tile(kt, std::integral_constant<int, 0>{});
      tile(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < nk) tile(kt, std::integral_constant<int, 0>{});
  }
  }
  // The last tile's last phase has read fragments of a tile that does not exist, and nothing
  // consumes them: the reads issued by inline assembly may still be in flight here, and the
  // compiler, which knows nothing of that, would hand their registers to the epilogue's first
  // values (seen: the lane's row inside the block, overwritten with a fragment of zeros whenever
  // other kernels on the same compute unit delayed the LDS: every lane then took itself for a
  // lane of row 0 and 15 rows in 16 of the wavefront's block were never written).
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int sl = 0; sl < (SINGLE ? 1 : 2); ++sl) {
#pragma unroll
    for (int i = 0; i < TM; ++i) if constexpr (!(AT && TWO)) frag_hold(fa[sl][i]);
#pragma unroll
    for (int j = 0; j < TN; ++j) if constexpr (!(BT && TWO)) frag_hold(fb[sl][j]);
  }
  // (the dropped requests past K are counted too)  The builtin, not inline assembly: the compiler
  // tracks the LDS-writing loads itself and, unless it sees them retired here, makes every LDS
  // read of the epilogue wait for ALL vector memory operations, i.e. for the epilogue's own
  // stores to drain, once per row pass.
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)

  // Epilogue.  D layout of v_mfma_f32_16x16x*: lane l holds column l % 16 and rows 4*(l/16) + r, r = 0..3, and
  // with the order of the columns chosen for it (above) every access goes straight from the accumulators'
  // layout to whole runs of a row: no trip through LDS, no barrier.
  lds_barrier();  // every wavefront is done with the operand tiles
  if constexpr (KS == 2) {
    // the second grid hands its partial sums over (16 bytes per lane, lanes side by side: no bank
    // conflicts) and leaves; a barrier only counts the wavefronts that are still running
    float4_t* xch = (float4_t*)smem + wave_mn * (TM * TN * 64) + lane;
    if (wave_k == 1) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) xch[(i * TN + j) * 64] = acc[i][j];
    }
    lds_barrier();
    if (wave_k == 1) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += xch[(i * TN + j) * 64];
    lds_barrier();  // all partial sums are read before the epilogue uses the LDS (column sums)
  }
  if constexpr (HAS_BIAS && !BIAS_EARLY) load_bias();
  static_assert(BT || TN == 2 || TN == 4 || TN == 8, "whole vectors per lane and row");
  if constexpr (EC == EC_GENERIC) {
    // one rolled loop over 16-row blocks (unrolled, the run-time switches of this class fill the instruction cache)
    float worst = 0.f;   // sum of v * 0 over the values written: 0 if all are finite, NaN otherwise
#pragma nounroll
    for (int h = 0; h < TM; ++h) {
      float4_t x[TN];
      static_for<TM>([&](auto hc) {
        constexpr int c = decltype(hc)::value;
        if (h == c) acc_read<TWO>(x, acc[c]);
      });
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = row0 + row_in((uint32_t)h, (uint32_t)r);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int64_t col = c0 + (RUNS ? 1 : 16) * j;
          if (row < M && col < N) worst = fmaf(epilogue_scalar(epi, c_base, row, col, x[j][r]), 0.f, worst);
        }
      }
    }
    if (epi.nonfinite != nullptr && worst != 0.f) *epi.nonfinite = 1.f;
    return;
  } else {
    // Straight-line classes.  All global accesses are raw buffer operations whose range check drops rows
    // past M (lanes past N get an out-of-range offset): no branch, so no join at which the compiler would
    // wait for every outstanding memory operation.  The one operand a class reads (residual, old C or
    // aux_in) is requested DEPTH row blocks ahead, into the registers the operand fragments have left.
    constexpr bool LOADS = EC == EC_RES32 || EC == EC_ACC32 || EC == EC_DACT16 || EC == EC_ACC16 || EC == EC_RES16;
    constexpr int ESC = C32 ? 4 : 2;       // (the operand read has the element size of C in every class)
    constexpr int NG = RUNS ? 1 : TN;      // runs of columns per lane and row
    constexpr int GW = RUNS ? TN : 1;      // columns per run
    constexpr int NV = GW * ESC / 4;       // 32-bit words per run
    static_assert(!BT || C32, "reduction-strided products have fp32 results");
    constexpr int DEPTH = !LOADS ? 1 : (TM * NG * NV <= 16 ? TM : (16 / (NG * NV) > 0 ? 16 / (NG * NV) : 1));
    const uint32_t OOB = 0x80000000u;
    const __amdgpu_buffer_rsrc_t rs_c = make_rsrc((const char*)epi.C + c_base * ESC, (uint32_t)(((M - 1) * epi.ldc + N) * ESC));
    const void* lp = (EC == EC_RES32 || EC == EC_RES16) ? epi.residual
                                                        : (EC == EC_DACT16 ? epi.aux_in : (const void*)((const char*)epi.C + c_base * ESC));
    const int64_t ld_l = (EC == EC_RES32 || EC == EC_RES16) ? epi.ld_res : (EC == EC_DACT16 ? epi.ld_aux_in : epi.ldc);
    // (a product that stores, beta = 0, inside a launch of the accumulate class, i.e. one member of a
    // grouped weight-gradient launch, reads its old C through a descriptor of extent 0: all zeros)
    const bool loads_on = LOADS && !(EC == EC_ACC32 && epi.beta == 0);
    const __amdgpu_buffer_rsrc_t rs_l = make_rsrc(LOADS ? lp : epi.C, loads_on ? (uint32_t)(((M - 1) * ld_l + N) * ESC) : 0u);
    const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(EC == EC_ACT16 ? epi.aux_out : epi.C,
                                                  EC == EC_ACT16 ? (uint32_t)(((M - 1) * epi.ld_aux_out + N) * 2) : 0u);
    uint32_t off_c[NG], off_l[NG], off_x[NG];
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const bool ok = c0 + j * 16 < N;
      off_c[j] = ok ? (uint32_t)((row0 * epi.ldc + c0 + j * 16) * ESC) : OOB;
      off_l[j] = ok ? (uint32_t)((row0 * ld_l + c0 + j * 16) * ESC) : OOB;
      off_x[j] = ok ? (uint32_t)((row0 * epi.ld_aux_out + c0 + j * 16) * 2) : OOB;
    }
    const uint32_t step_c = (uint32_t)(epi.ldc * ESC), step_l = (uint32_t)(ld_l * ESC), step_x = (uint32_t)(epi.ld_aux_out * 2);
    const float alpha = epi.alpha;
    const bool round_mid = epi.round_mid != 0;
    float csum[TN];      // EC_DACT16: column sums of the stored values
    float worst = 0.f;   // fp32 classes: sum of v * 0 over the values written: 0 if all are finite, NaN otherwise
#pragma unroll
    for (int j = 0; j < TN; ++j) csum[j] = 0.f;

    // one 16-row block: x = its accumulators, old = the operand read
    auto block = [&](uint32_t h, const float4_t (&x)[TN], const Words<NV> (&old)[4][NG]) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool row_ok = row0 + (int64_t)row_in(h, (uint32_t)r) < M;
        float bad = 0.f;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          float v[GW];
#pragma unroll
          for (int k = 0; k < GW; ++k) {
            v[k] = x[RUNS ? k : g][r] * alpha;
            if constexpr (HAS_BIAS) v[k] += bias[k];
          }
          // (the plain 16-bit store rounds once, when it packs: rounding to the same format before
          // that changes nothing.  The GELU class rounds by packing what it keeps, below.)
          if constexpr (EC != EC_STORE16 && EC != EC_ACT16 && !BT) {
            if (round_mid) {
#pragma unroll
              for (int k = 0; k < GW; k += 2) {
                const uint32_t w = pack2<DT>(v[k], v[k + 1]);
                v[k] = unpack1<DT>(w, 0);
                v[k + 1] = unpack1<DT>(w, 1);
              }
            }
          }
          const uint32_t oc = off_c[g] + row_in(h, (uint32_t)r) * step_c;
          Words<NV> o;
          if constexpr (C32) {
            if constexpr (LOADS) {
#pragma unroll
              for (int k = 0; k < GW; ++k) v[k] += __int_as_float(old[r][g].w[k]);
            }
            if constexpr (EC == EC_STORE32 || EC == EC_ACC32) {
#pragma unroll
              for (int k = 0; k < GW; ++k) bad = fmaf(v[k], 0.f, bad);
            }
#pragma unroll
            for (int k = 0; k < GW; ++k) o.w[k] = __float_as_int(v[k]);
          } else {
            if constexpr (EC == EC_ACT16) {   // GELU only (other activations take the generic class)
#pragma unroll
              for (int k = 0; k < NV; ++k) o.w[k] = (int)pack2<DT>(v[2 * k], v[2 * k + 1]);
              o.store(rs_x, off_x[g] + row_in(h, (uint32_t)r) * step_x);
              if (round_mid) {
#pragma unroll
                for (int k = 0; k < GW; ++k) v[k] = unpack1<DT>((uint32_t)o.w[k / 2], k % 2);
              }
#pragma unroll
              for (int k = 0; k < GW; ++k) v[k] = pf_gelu_erf(v[k]);
            }
            if constexpr (LOADS) {
#pragma unroll
              for (int k = 0; k < GW; ++k) {
                const float t = unpack1<DT>((uint32_t)old[r][g].w[k / 2], k % 2);
                if constexpr (EC == EC_DACT16) v[k] *= pf_gelu_erf_grad(t);
                else v[k] += t;
              }
            }
#pragma unroll
            for (int k = 0; k < NV; ++k) o.w[k] = (int)pack2<DT>(v[2 * k], v[2 * k + 1]);
            if constexpr (EC == EC_DACT16) {   // sums run over the ROUNDED values, rows past M excluded
              const float keep = row_ok ? 1.f : 0.f;
#pragma unroll
              for (int k = 0; k < GW; ++k) csum[k] += unpack1<DT>((uint32_t)o.w[k / 2], k % 2) * keep;
            }
          }
          o.store(rs_c, oc);
        }
        if constexpr (EC == EC_STORE32 || EC == EC_ACC32) worst += row_ok ? bad : 0.f;
      }
    };
    auto fetch = [&](uint32_t h, Words<NV> (&old)[4][NG]) {
      if constexpr (LOADS) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int g = 0; g < NG; ++g) old[r][g].load(rs_l, off_l[g] + row_in(h, (uint32_t)r) * step_l);
      }
    };
    if constexpr (EC == EC_ACT16 || EC == EC_DACT16) {
      // the arithmetic exists once, in a rolled loop: unrolled, its code would stream through an instruction
      // cache that is cold at every launch
      Words<NV> old[4][NG], next[4][NG];
      fetch(0u, old);
#pragma nounroll
      for (int h = 0; h < TM; ++h) {
        fetch((uint32_t)(h + 1), next);   // (of the block past the last one nobody reads anything)
        float4_t x[TN];
        static_for<TM>([&](auto cc) {
          constexpr int c = decltype(cc)::value;
          if (h == c) acc_read<TWO>(x, acc[c]);
        });
        block((uint32_t)h, x, old);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int g = 0; g < NG; ++g) old[r][g] = next[r][g];
      }
    } else {
      Words<NV> old[DEPTH][4][NG];
      static_for<DEPTH>([&](auto hc) { fetch((uint32_t)decltype(hc)::value, old[decltype(hc)::value]); });
      static_for<TM>([&](auto hc) {
        constexpr int h = decltype(hc)::value;
        float4_t x[TN];
        acc_read<TWO>(x, acc[h]);
        block((uint32_t)h, x, old[h % DEPTH]);
        if constexpr (LOADS && h + DEPTH < TM) fetch((uint32_t)(h + DEPTH), old[h % DEPTH]);
        __builtin_amdgcn_sched_barrier(0);   // (left alone, the scheduler starts every block at once and spills)
      });
    }
    if constexpr (EC == EC_STORE32 || EC == EC_ACC32) {
      // every writer writes the same value: no atomic needed
      if (epi.nonfinite != nullptr && worst != 0.f) *epi.nonfinite = 1.f;
    }
    if constexpr (EC == EC_DACT16) {
      if (epi.colsum_ws != nullptr) {   // uniform over the grid
        // lanes with the same lane % 16 hold the same columns (different rows)
#pragma unroll
        for (int off = 16; off < 64; off <<= 1)
#pragma unroll
          for (int k = 0; k < TN; ++k) csum[k] += __shfl_xor(csum[k], off, 64);
        // wavefronts of one block column add up in wavefront-row order through LDS
        float* red = (float*)smem;
        lds_barrier();
        if (lane < 16) {
#pragma unroll
          for (int k = 0; k < TN; ++k) red[wave * WN + lane * TN + k] = csum[k];
        }
        lds_barrier();
        if (wave / WGN == 0) {
          for (int c = lane * 4; c < WN; c += 256) {
            if (n0 + wn0 + c >= N) continue;
            float4_t t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < WGM; ++w) t += *(const float4_t*)(red + (w * WGN + wave % WGN) * WN + c);
            *(float4_t*)(epi.colsum_ws + (int64_t)tm * N + n0 + wn0 + c) = t;
          }
        }
      }
    }
  }
}

#define PF_X_BOUNDS __launch_bounds__(64 * WGM * WGN * KS, (ST * (BM + BN) * BK * 2 <= 80 * 1024 && 64 * WGM * WGN * KS <= 256) ? 2 : 1)
template <int DT, int BM, int BN, int BK, int WGM, int WGN, int KS, int ST, bool AT, bool BT, int EC>
__global__ PF_X_BOUNDS void gemm16x_kernel(const pf_gemm_desc p, const GemmGrid g) {
  gemm16x_body<DT, BM, BN, BK, WGM, WGN, KS, ST, AT, BT, EC>(p, g, (int)blockIdx.x);
}

// Row-major products whose reduction length is a multiple of 8 but not of the stage depth (head dimensions 80 and
// 88 give such widths): a kernel of its own, the mask costs an instruction and a register per load.
template <int DT, int BM, int BN, int BK, int WGM, int WGN, int KS, int ST, bool AT, bool BT, int EC>
__global__ PF_X_BOUNDS void gemm16x_ragged_kernel(const pf_gemm_desc p, const GemmGrid g) {
  gemm16x_body<DT, BM, BN, BK, WGM, WGN, KS, ST, AT, BT, EC, true>(p, g, (int)blockIdx.x);
}

// Several independent problems of the same kind in one launch: problem i owns the workgroups
// [start[i], start[i+1]).  Weight-gradient products are independent of everything that follows
// them in a backward job; small ones (64 tiles for a 1024x1024 weight) are launched together so
// that they fill the 256 CUs.
constexpr int GEMM_GROUP_MAX = PF_GEMM_GROUP_MAX;   // 8 problems: 2.3 KB of kernel arguments
struct GemmGroup {
  pf_gemm_desc p[GEMM_GROUP_MAX];
  GemmGrid g[GEMM_GROUP_MAX];
  int start[GEMM_GROUP_MAX];
  int n;
};
template <int DT, int BM, int BN, int BK, int WGM, int WGN, int KS, int ST, bool AT, bool BT, int EC>
__global__ PF_X_BOUNDS void gemm16x_group_kernel(const GemmGroup ga) {
  int i = 0;
#pragma unroll
  for (int k = 1; k < GEMM_GROUP_MAX; ++k)
    if (k < ga.n && (int)blockIdx.x >= ga.start[k]) i = k;
  i = __builtin_amdgcn_readfirstlane(i);
  gemm16x_body<DT, BM, BN, BK, WGM, WGN, KS, ST, AT, BT, EC>(ga.p[i], ga.g[i], (int)blockIdx.x - ga.start[i]);
}

template <int DT, int BM, int BN, int BK, int WGM, int WGN, int KS, int ST, bool AT, bool BT, int EC, bool RAG>
int launch16x_t(const pf_gemm_desc& d, const GemmGrid& g, hipStream_t st) {
  constexpr int NT = 64 * WGM * WGN * KS;
  constexpr size_t lds_xch = KS == 2 ? (size_t)BM * BN * 4 : 0;   // one grid's partial sums on their way to the other
  constexpr size_t lds_main = ((size_t)ST * (BM + BN) * BK * 2 > lds_xch) ? (size_t)ST * (BM + BN) * BK * 2 : lds_xch;
  constexpr size_t lds = lds_main + (ST == 2 ? (size_t)BN * BK * 2 : 0);   // (the third stage of B)
  static_assert(lds <= 160 * 1024, "tile pipeline exceeds the 160 KB of LDS");
  void (*kern)(const pf_gemm_desc, const GemmGrid);
  if constexpr (RAG) kern = gemm16x_ragged_kernel<DT, BM, BN, BK, WGM, WGN, KS, ST, AT, BT, EC>;
  else kern = gemm16x_kernel<DT, BM, BN, BK, WGM, WGN, KS, ST, AT, BT, EC>;
  const int rc = pf_allow_lds((const void*)kern, lds, "pf_gemm");
  if (rc != PF_OK) return rc;
  const dim3 grid((unsigned)(g.per_xcd * 8), (unsigned)(d.batch1 * d.batch2), 1);
  hipLaunchKernelGGL(kern, grid, dim3(NT), lds, st, d, g);
  PF_CHECK_LAUNCH("pf_gemm");
  return PF_OK;
}

template <int DT, int BM, int BN, int BK, int WGM, int WGN, int KS, int ST>
int launch16x(const pf_gemm_desc& d, hipStream_t st) {
  GemmGrid g;
  g.tiles_m = (int)((d.M + BM - 1) / BM);
  g.tiles_n = (int)((d.N + BN - 1) / BN);
  const int64_t total = (int64_t)g.tiles_m * g.tiles_n;
  g.per_xcd = (int)((total + 7) / 8);
  g.vec_epi = epi_vec_ok(d);
  // A ragged reduction tail is zero-filled by the hardware range check only when whole k-rows
  // fall outside the operand, i.e. when both operands are stored [k][row].
  const bool ragged = d.K % BK != 0 && !(d.a_trans && d.b_trans);
  constexpr bool HAS_RAGGED = x_tile_ragged(BM, BN, WGM * WGN);
  if (ragged && !(HAS_RAGGED && d.K % 8 == 0)) {
    pf_set_error("pf_gemm: this variant needs K %% %d == 0 unless both operands are transposed", BK);
    return PF_ERR_INVALID;
  }
  const int ec = x_epi_class(d, g.vec_epi, BM);
#define PF_X(AT, BT, EC) launch16x_t<DT, BM, BN, BK, WGM, WGN, KS, ST, AT, BT, EC, false>(d, g, st)
#define PF_XR(EC) launch16x_t<DT, BM, BN, BK, WGM, WGN, KS, ST, false, false, EC, HAS_RAGGED>(d, g, st)
  if constexpr (HAS_RAGGED) {
    if (ragged) {
      if (d.a_trans || d.b_trans) return PF_ERR_INVALID;
      switch (ec) {
        case EC_STORE16: return PF_XR(EC_STORE16);
        case EC_STORE32: return PF_XR(EC_STORE32);
        case EC_ACT16: return PF_XR(EC_ACT16);
        case EC_RES32: return PF_XR(EC_RES32);
        case EC_ACC32: return PF_XR(EC_ACC32);
        case EC_DACT16: return PF_XR(EC_DACT16);
        case EC_ACC16: return PF_XR(EC_ACC16);
        case EC_RES16: return PF_XR(EC_RES16);
        default: return PF_XR(EC_GENERIC);
      }
    }
  }
  if (!d.a_trans && !d.b_trans) {   // forward and input-gradient products
    switch (ec) {
      case EC_STORE16: return PF_X(false, false, EC_STORE16);
      case EC_STORE32: return PF_X(false, false, EC_STORE32);
      case EC_ACT16: return PF_X(false, false, EC_ACT16);
      case EC_RES32: return PF_X(false, false, EC_RES32);
      case EC_ACC32: return PF_X(false, false, EC_ACC32);
      case EC_DACT16: return PF_X(false, false, EC_DACT16);
      case EC_ACC16: return PF_X(false, false, EC_ACC16);
      case EC_RES16: return PF_X(false, false, EC_RES16);
      default: return PF_X(false, false, EC_GENERIC);
    }
  }
  // transposed (reduction-strided) tiles exist for 128 and 256 rows only
  if constexpr (BM != 192) {
    if (d.a_trans && d.b_trans) {   // weight-gradient products
      if (ec == EC_ACC32) return PF_X(true, true, EC_ACC32);
      if (ec == EC_STORE32) return PF_X(true, true, EC_STORE32);
      return PF_X(true, true, EC_GENERIC);
    }
  }
#undef PF_X
#undef PF_XR
  pf_set_error("pf_gemm: tile %dx%d has no variant for a_trans=%d b_trans=%d", BM, BN, d.a_trans, d.b_trans);
  return PF_ERR_INVALID;
}

// Several weight-gradient products (both operands reduction-strided, fp32 C accumulated) in one
// launch; the caller has checked that they all take tile BMxBN and the EC_ACC32 epilogue.
template <int DT, int BM, int BN, int BK, int WGM, int WGN, int KS, int ST>
int launch16x_group(const pf_gemm_desc* d, int n, hipStream_t st) {
  if constexpr (BM != 192) {
    constexpr int NT = 64 * WGM * WGN * KS;
    constexpr size_t lds_xch = KS == 2 ? (size_t)BM * BN * 4 : 0;
    constexpr size_t lds_main = ((size_t)ST * (BM + BN) * BK * 2 > lds_xch) ? (size_t)ST * (BM + BN) * BK * 2 : lds_xch;
    constexpr size_t lds = lds_main + (ST == 2 ? (size_t)BN * BK * 2 : 0);
    GemmGroup ga;
    int blocks = 0;
    for (int i = 0; i < n; ++i) {
      ga.p[i] = d[i];
      ga.g[i].tiles_m = (int)((d[i].M + BM - 1) / BM);
      ga.g[i].tiles_n = (int)((d[i].N + BN - 1) / BN);
      ga.g[i].per_xcd = (int)(((int64_t)ga.g[i].tiles_m * ga.g[i].tiles_n + 7) / 8);
      ga.g[i].vec_epi = epi_vec_ok(d[i]);
      ga.start[i] = blocks;          // a multiple of 8: the workgroup -> XCD dealing stays aligned
      blocks += ga.g[i].per_xcd * 8;
    }
    for (int i = n; i < GEMM_GROUP_MAX; ++i) {
      ga.p[i] = d[0];
      ga.g[i] = ga.g[0];
      ga.start[i] = blocks;
    }
    ga.n = n;
    auto kern = gemm16x_group_kernel<DT, BM, BN, BK, WGM, WGN, KS, ST, true, true, EC_ACC32>;
    const int rc = pf_allow_lds((const void*)kern, lds, "pf_gemm_grouped");
    if (rc != PF_OK) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks, 1, 1), dim3(NT), lds, st, ga);
    PF_CHECK_LAUNCH("pf_gemm_grouped");
    return PF_OK;
  }
  pf_set_error("pf_gemm_grouped: tile %dx%d has no transposed variant", BM, BN);
  return PF_ERR_INVALID;
}

// one tile shape per translation unit (see pf_gemm_x_inst.hip)
template <int DT, int XT>
int gemm_x_group_launch(const pf_gemm_desc* d, int n, hipStream_t st) {
  using T = XTile<XT>;
  return launch16x_group<DT, T::BM, T::BN, T::BK, T::WGM, T::WGN, T::KS, T::ST>(d, n, st);
}
template <int DT, int XT>
int gemm_x_launch(const pf_gemm_desc& d, hipStream_t st) {
  using T = XTile<XT>;
  static_assert(x_tile_bm(XT) == T::BM, "x_tile_bm");
  return launch16x<DT, T::BM, T::BN, T::BK, T::WGM, T::WGN, T::KS, T::ST>(d, st);
}

}  // namespace
