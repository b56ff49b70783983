// fp32 matrix products whose wavefronts split the depth of the reduction (pf_gemm_f32.hip: those that split the tile).
#include "pf_gemm_f32.h"

namespace {

// ---------------------------------------------------------------------------
// fp32 MFMA kernel, depth split over the wavefronts
//
// The fp32 matrix rate is 1/16 of the 16-bit one (157 TFLOP/s), so operand traffic hardly matters; what bounds these products is
// how evenly they spread over 256 CUs and how well loads, LDS reads and barriers hide behind the matrix instructions (nothing else
// does: vector instructions do not run beside v_mfma_f32_16x16x4_f32).  Hence four wavefronts that split the DEPTH of a stage, 16 of 64 each, and
// all compute the whole tile: a tile may then have any number of 16x16 blocks (3152 x 384 is 250 tiles of 64x80 for 256 CUs, 384 x 1536
// 256 of 48x48), a wavefront has up to 20 independent accumulators, and an LDS read feeds 4 matrix instructions per block of the other
// operand.  The four partial sums meet in LDS once, at the end; they are shorter than one sum, too: the error against 64 bits at K = 1536 is
// 3.5e-7 where one chain had 7.0e-7.  Tiles travel by buffer_load ... lds (no staging registers, no LDS stores), up to ST stages ahead.
//
// A stage is 64 deep.  A lane's fragment of one operand is 16 bytes: of its wavefront's 16 of depth the reduction indices 4*(lane/16) .. +3 of
// row lane%16; element e of both operands goes into matrix instruction e (which adds over any four reduction indices, here e, 4+e, 8+e, 12+e).
//   reduction-contiguous operand [row][k]: 16-byte chunk c of a row sits at c ^ row%16: single ds_read_b128,
//     no bank conflicts.  Chunks past K (K no multiple of 64) are zeroed in registers, in the last stage only.
//   reduction-strided operand [k][row]: k-row 16h + 4g + e sits at LDS row 16h + 4e + g; the four k-rows that a read touches
//     together (g = 0..3) have to lie on different banks, which an odd number of blocks per row sees to by itself, and else 64-byte groups of
//     a row that are swapped by g.  k-rows past K are outside the buffer and read as zeros.
// Buffer descriptors are rebuilt for each stage (scalar instructions), so operands may exceed 4 GiB.
//
// Against wavefronts that split the tile, 32 deep (us): 3152 x 384 x 1536 52.5 -> 36.5, 3152 x 1536 x 384 41.5 -> 37.7, 3152 x 384 x 384 17.6 -> 12.8,
// 788 x 384 x 1536 20.8 -> 14.9, 4096 x 4096 x 1024 265 -> 256 (134 TFLOP/s); weight gradients over 3152 rows: 384 x 1536 60 -> 34, 384 x 384 25 -> 20.
// ---------------------------------------------------------------------------
constexpr int FK = 64, FNW = 4;   // depth of a stage, wavefronts: 16 of it to each

// one operand's part of a stage: T times 16 rows
template <int T, bool TRANS> struct FTile {
  static constexpr int R = 16 * T, BYTES = R * FK * 4;
  static constexpr int IPW = T;                       // wavefront-wide load instructions (1 KB each) per wavefront
  static constexpr int ROWB = TRANS ? R * 4 : FK * 4;   // bytes per LDS row
  static constexpr int CPR = ROWB / 16;               // 16-byte chunks per LDS row
  static_assert(BYTES == IPW * FNW * 1024, "loads");

  static __device__ __forceinline__ int swz(int row) {
    return !TRANS ? row & 15 : T % 4 == 0 ? (row & 3) << 2 : T % 4 == 2 ? ((row >> 1) & 1) << 2 : 0;
  }
  // byte offset from the tile's first element of the chunk this lane fetches in its q-th instruction
  static __device__ __forceinline__ void init(uint32_t (&off)[IPW], int64_t ld, int wave, int lane) {
#pragma unroll
    for (int q = 0; q < IPW; ++q) {
      const int at = (wave * IPW + q) * 64 + lane, pos = at / CPR;
      const int c = (at % CPR) ^ swz(pos);
      const int row = TRANS ? (pos & ~15) | ((pos & 3) << 2) | ((pos >> 2) & 3) : pos;
      off[q] = (uint32_t)((row * ld + c * 4) * 4);
    }
  }
  // The buffer of a tile holds exactly what of it lies inside the operand; past the last tile nothing.  (Rows are
  // padded to 16 bytes: ld is a multiple of 4.)  edge: bytes of the tile's rows but the last / of its last row's part
  static __device__ __forceinline__ int edge(int64_t ld, int64_t r0, int64_t R_total) {
    const int rows = (int)(R_total - r0 < R ? R_total - r0 : R);
    return TRANS ? (rows + 3) / 4 * 16 : (rows - 1) * (int)ld * 4;
  }
  static __device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const float* X, int64_t ld, int edge_bytes, int kt, int K) {
    const int k = K - kt * FK, kc = k < FK ? k : FK;
    const int bytes = edge_bytes + (TRANS ? (kc - 1) * (int)ld * 4 : (kc + 3) / 4 * 16);
    return make_rsrc(X + (int64_t)kt * (TRANS ? FK * ld : FK), k > 0 ? (uint32_t)bytes : 0u);
  }
  template <int Q> static __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rs, const uint32_t (&off)[IPW], uint32_t lds, int wave) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (PF_LDS(void))(uintptr_t)(lds + (uint32_t)(wave * IPW + Q) * 1024u), 16, (int)off[Q], 0, 0, 0);
  }
  // LDS byte offsets of this lane's fragments in its wavefront's 16 of depth: [row][k] one (MFMA tile i is 16 i rows on),
  // [k][row] one per MFMA tile
  static constexpr int NF = TRANS ? T : 1;
  static __device__ __forceinline__ void frag_init(uint32_t (&foff)[NF], int wave, int lane) {
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < NF; ++i)
      foff[i] = !TRANS ? (uint32_t)(r * ROWB + ((4 * wave + g) ^ swz(r)) * 16)
                       : (uint32_t)((16 * wave + g) * ROWB + (((r + 16 * i) >> 2) ^ swz(g)) * 16 + (r & 3) * 4);
  }
  template <int I> static __device__ __forceinline__ void read(FragF<TRANS>& f, uint32_t lds, const uint32_t (&foff)[NF]) {
    if constexpr (!TRANS) {
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.v) : "v"(lds + foff[0]), "n"(I * 16 * ROWB) : "memory");
    } else {   // (offsets in units of 64 elements)
      asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(f.lo) : "v"(lds + foff[I]), "n"(0), "n"(T) : "memory");
      asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(f.hi) : "v"(lds + foff[I]), "n"(2 * T), "n"(3 * T) : "memory");
    }
  }
};

template <int TM, int TN, int ST, bool AT, bool BT>
__global__ __launch_bounds__(64 * FNW) __attribute__((amdgpu_waves_per_eu(TM * TN >= 9 ? 2 : 4, TM * TN >= 9 ? 2 : 4))) void gemm32k_kernel(const pf_gemm_desc p, const GemmGrid g) {
  constexpr int BM = 16 * TM, BN = 16 * TN, NB = TM * TN;
  using TA = FTile<TM, AT>;
  using TB = FTile<TN, BT>;
  constexpr int STAGE = TA::BYTES + TB::BYTES, LPW = TM + TN;
  static_assert(ST * LPW <= 63, "too many loads in flight for the wait counter");
  extern __shared__ __align__(1024) float smem[];

  const int t = gemm_tile_id((int)blockIdx.x, g.tiles_m * g.tiles_n, g.per_xcd);
  if (t < 0) return;
  int tm, tn;
  gemm_tile_rc(t, g.tiles_m, g.tiles_n, tm, tn);
  const int64_t M = p.M, N = p.N, K = p.K;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int64_t z = blockIdx.y, z1 = z / p.batch2, z2 = z % p.batch2;
  const float* A = (const float*)p.A + z1 * p.a_stride1 + z2 * p.a_stride2;
  const float* B = (const float*)p.B + z1 * p.b_stride1 + z2 * p.b_stride2;
  const int64_t c_base = z1 * p.c_stride1 + z2 * p.c_stride2;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

  uint32_t offa[TM], offb[TN];
  TA::init(offa, p.lda, wave, lane);
  TB::init(offb, p.ldb, wave, lane);
  uint32_t foa[TA::NF], fob[TB::NF];
  TA::frag_init(foa, wave, lane);
  TB::frag_init(fob, wave, lane);

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  const int nk = (int)((K + FK - 1) / FK), left = (int)(K - (int64_t)(nk - 1) * FK);
  A += AT ? m0 : m0 * p.lda;
  B += BT ? n0 : n0 * p.ldb;
  const int edge_a = TA::edge(p.lda, m0, M), edge_b = TB::edge(p.ldb, n0, N);
  auto issue = [&](int kt, uint32_t sb) {
    const __amdgpu_buffer_rsrc_t ra = TA::buffer(A, p.lda, edge_a, kt, (int)K), rb = TB::buffer(B, p.ldb, edge_b, kt, (int)K);
    static_for<TM>([&](auto qc) { TA::template issue<decltype(qc)::value>(ra, offa, sb, wave); });
    static_for<TN>([&](auto qc) { TB::template issue<decltype(qc)::value>(rb, offb, sb + TA::BYTES, wave); });
  };
  // A stage's fragments are read while the one before it is multiplied: at the barrier between two nothing is left to
  // wait for but the other wavefronts.  Two sets of fragments, by parity of the stage.
  FragF<AT> fa[2][TM];
  FragF<BT> fb[2][TN];
  auto arrived = [&](auto setc) {
    constexpr int S = decltype(setc)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[S][i].arrived();
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[S][j].arrived();
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};

#pragma unroll
  for (int s = 0; s < ST; ++s) issue(s, lds0 + (uint32_t)s * STAGE);
  wait_vm<(ST - 1) * LPW>();
  asm volatile("s_barrier" ::: "memory");
  static_for<TM>([&](auto ic) { TA::template read<decltype(ic)::value>(fa[0][decltype(ic)::value], lds0, foa); });
  static_for<TN>([&](auto jc) { TB::template read<decltype(jc)::value>(fb[0][decltype(jc)::value], lds0 + TA::BYTES, fob); });
  uint32_t sb = lds0;   // stage of tile kt
  auto tile = [&](int kt, auto setc) {
    constexpr int S = decltype(setc)::value;
    const uint32_t sb_next = sb + STAGE == lds0 + (uint32_t)ST * STAGE ? lds0 : sb + STAGE;
    wait_vm<(ST - 2) * LPW>();
    wait_lds<0>();
    arrived(setc);
    asm volatile("s_barrier" ::: "memory");   // tile kt + 1 is in LDS, tile kt in everybody's registers
    if (!(AT && BT) && left < FK && kt == nk - 1) {
      const int k = 16 * wave + 4 * (lane >> 4);
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[S][i].mask(k, left);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[S][j].mask(k, left);
    }
    const __amdgpu_buffer_rsrc_t ra = TA::buffer(A, p.lda, edge_a, kt + ST, (int)K), rb = TB::buffer(B, p.ldb, edge_b, kt + ST, (int)K);
    __builtin_amdgcn_sched_barrier(0);
    // 4 NB matrix instructions; between them the next stage's reads, then the loads that refill this stage
    constexpr int NE = 2 * LPW;
    static_for<NE>([&](auto ec) {
      constexpr int q = decltype(ec)::value, first = q * 4 * NB / NE, last = (q + 1) * 4 * NB / NE;
      if constexpr (q < TN) TB::template read<q>(fb[1 - S][q], sb_next + TA::BYTES, fob);
      else if constexpr (q < LPW) TA::template read<q - TN>(fa[1 - S][q - TN], sb_next, foa);
      else if constexpr (q < LPW + TM) TA::template issue<q - LPW>(ra, offa, sb, wave);
      else TB::template issue<q - LPW - TM>(rb, offb, sb + TA::BYTES, wave);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = first; m < last; ++m) {
        const int e = m / NB, i = m % NB / TN, j = m % TN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[S][i].get(e), fb[S][j].get(e), acc[i][j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    sb = sb_next;
  };
  int kt = 0;
#pragma nounroll
  for (; kt + 1 < nk; kt += 2) {
    tile(kt, c0);
    tile(kt + 1, c1);
  }
  if (kt < nk) tile(kt, c0);
  // (fragments of a tile past the end may still be on their way into their registers)
  wait_lds<0>();
  arrived(c0);
  arrived(c1);
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the dropped requests past K
  asm volatile("s_barrier" ::: "memory");

  // The wavefronts' sums meet in LDS.  D layout of v_mfma_f32_16x16x*: lane l holds column l % 16 and rows 4*(l/16) + r; wavefront w goes
  // on with r = w: its own, then those of the wavefronts w + 1, w + 2, w + 3 (modulo 4).
  float1_t v[TM][TN];
  static_for<FNW>([&](auto wc) {
    constexpr int W = decltype(wc)::value;
    if (wave == W) {
#pragma unroll
      for (int h = 0; h < NB; ++h) {
#pragma unroll
        for (int s = 1; s < FNW; ++s)      // to wavefront W - s, which reads it as its s-th
          smem[(((W + FNW - s) % FNW * (FNW - 1) + s - 1) * NB + h) * 64 + lane] = acc[h / TN][h % TN][(W + FNW - s) % FNW];
        v[h / TN][h % TN][0] = acc[h / TN][h % TN][W];
      }
    }
  });
  __syncthreads();
#pragma unroll
  for (int h = 0; h < NB; ++h)
#pragma unroll
    for (int s = 1; s < FNW; ++s) v[h / TN][h % TN][0] += smem[((wave * (FNW - 1) + s - 1) * NB + h) * 64 + lane];

  epilogue_f32<BM>(p, g, v, m0, 4 * (lane >> 4) + wave, n0 + (lane & 15), c_base);
}

template <int TM, int TN, int ST, bool AT, bool BT>
int launch_one(const pf_gemm_desc& d, const GemmGrid& g, dim3 grid, hipStream_t st) {
  constexpr size_t lds = (size_t)ST * (TM + TN) * 16 * FK * 4;
  static_assert(lds >= (size_t)(FNW - 1) * TM * TN * 1024 && lds <= 160 * 1024, "the wavefronts' sums meet where the operands were");
  auto kern = gemm32k_kernel<TM, TN, ST, AT, BT>;
  const int rc = pf_allow_lds((const void*)kern, lds, "pf_gemm(f32)");
  if (rc != PF_OK) return rc;
  hipLaunchKernelGGL(kern, grid, dim3(64 * FNW), lds, st, d, g);
  PF_CHECK_LAUNCH("pf_gemm(f32)");
  return PF_OK;
}

template <int TM, int TN, int ST>
int launch(const pf_gemm_desc& d, hipStream_t st) {
  constexpr int BM = 16 * TM, BN = 16 * TN;
  GemmGrid g;
  g.tiles_m = (int)((d.M + BM - 1) / BM);
  g.tiles_n = (int)((d.N + BN - 1) / BN);
  g.per_xcd = (int)(((int64_t)g.tiles_m * g.tiles_n + 7) / 8);
  g.vec_epi = epi_f32_vec_ok(d, BM);
  const dim3 grid((unsigned)(g.per_xcd * 8), (unsigned)(d.batch1 * d.batch2), 1);
  if (d.a_trans && d.b_trans) return launch_one<TM, TN, ST, true, true>(d, g, grid, st);
  if (d.a_trans) return launch_one<TM, TN, ST, true, false>(d, g, grid, st);
  if (d.b_trans) return launch_one<TM, TN, ST, false, true>(d, g, grid, st);
  return launch_one<TM, TN, ST, false, false>(d, g, grid, st);
}

// Tiles: 16-row blocks, stages (two workgroups fit a CU's LDS but for the 64x80 tile with four stages, which is for one round), and
// the time of a launch in microseconds, fitted to 110 products of 16 .. 12000 by 16 .. 6000 over 32 .. 6000 (rms 3 to 8 %): fixed, and
// per stage t0 in an empty device, t0 + t1 with a tile on every CU; from the second round on, where two tiles share a CU, per round and stage
// `sat`, and `over` per round.  On these products the choice is on average 0.6 % off the fastest tile, 10 % at most, and takes
// 0.84 of what the wavefronts that split the tile took (0.65 .. 1.04 over depths from 131 on).
struct Tile {
  int bm, bn;
  double fixed, t0, t1, sat, over;
  const char* shape;
};
constexpr Tile TILES[] = {{16, 32, 3.17, 0.203, 0.043, 0.175, 0.97, "1, 2, 6"}, {32, 32, 3.28, 0.307, 0.048, 0.275, 0.98, "2, 2, 4"},
                          {32, 48, 3.54, 0.421, 0.087, 0.387, 1.14, "2, 3, 4"}, {48, 48, 3.73, 0.578, 0.096, 0.546, 1.21, "3, 3, 3"},
                          {48, 64, 3.68, 0.795, 0.293, 0.709, 1.36, "3, 4, 2"}, {64, 64, 3.96, 1.009, 0.339, 0.914, 1.55, "4, 4, 2"},
                          {64, 80, 4.99, 1.176, 0.161, 1.182, 3.35, "4, 5, 4"}, {64, 80, 4.35, 1.231, 0.266, 1.112, 1.85, "4, 5, 2"}};

int choose(const pf_gemm_desc& d) {
  const int64_t nb = (d.batch1 > 0 ? d.batch1 : 1) * (d.batch2 > 0 ? d.batch2 : 1);
  const double nk = (double)((d.K + FK - 1) / FK);
  int best = 0;
  double t_best = 0;
  for (int i = 0; i < (int)(sizeof(TILES) / sizeof(TILES[0])); ++i) {
    const Tile& t = TILES[i];
    const int64_t tiles = ((d.M + t.bm - 1) / t.bm) * ((d.N + t.bn - 1) / t.bn) * nb, rounds = (tiles + 255) / 256;
    const double c = t.fixed + (rounds <= 1 ? nk * (t.t0 + t.t1 * (double)tiles / 256) : (double)rounds * (nk * t.sat + t.over));
    if (i == 0 || c < t_best) best = i, t_best = c;
  }
  return best;
}
}  // namespace

const char* pf_gemm_f32_depth_shape(const pf_gemm_desc& d) { return TILES[choose(d)].shape; }

int pf_gemm_f32_depth(const pf_gemm_desc& d, hipStream_t st) {
  switch (choose(d)) {
    case 0: return launch<1, 2, 6>(d, st);
    case 1: return launch<2, 2, 4>(d, st);
    case 2: return launch<2, 3, 4>(d, st);
    case 3: return launch<3, 3, 3>(d, st);
    case 4: return launch<3, 4, 2>(d, st);
    case 5: return launch<4, 4, 2>(d, st);
    case 6: return launch<4, 5, 4>(d, st);
    default: return launch<4, 5, 2>(d, st);
  }
}
