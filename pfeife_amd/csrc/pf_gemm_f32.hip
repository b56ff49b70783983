// fp32 matrix products on v_mfma_f32_16x16x4_f32, operands straight from global memory into LDS: shallow ones, and the choice.
#include "pf_gemm_f32.h"

namespace {

// ---------------------------------------------------------------------------
// fp32 MFMA kernel, direct-to-LDS pipeline
//
// The fp32 matrix rate is 1/16 of the 16-bit one (157 TFLOP/s), so operand traffic hardly matters; what bounds
// these products is how many CUs get work and how well loads, LDS reads and barriers hide behind the matrix
// instructions.  Hence: tiles down to 32x32, tiles that travel by buffer_load ... lds (no staging registers, no
// LDS stores) ST-1 ahead, and two or more wavefronts per SIMD.
//
// A tile is 32 deep: 128-byte rows, the same bytes as 64 16-bit elements.  A lane's fragment of one operand is
// 16 bytes: reduction indices 4*(lane/16) .. +3 of row lane%16; element e of both operands goes into matrix
// instruction e (which adds over any four reduction indices, here e, 4+e, 8+e, 12+e).
//   reduction-contiguous operand [row][k]: 16-byte chunk c of a row sits at c ^ (row/2)%8: single ds_read_b128,
//     no bank conflicts.  Chunks past K (K no multiple of 32) are zeroed in registers, in the last tile only.
//   reduction-strided operand [k][row]: k-row 16h + 4g + e sits at LDS row 16h + 4e + g, and 64-byte groups of a
//     row are swapped by g: the four k-rows that a read touches together (g = 0..3) lie on different banks.
//     k-rows past K are outside the buffer and read as zeros.
// Buffer descriptors are rebuilt for each tile (scalar instructions), so operands may exceed 4 GiB.
//
// Against 64x64 tiles staged through registers for 32x32x2 instructions (us): 788 x 384 x 384 16.8 -> 7.8,
// 788 x 384 x 1536 55.2 -> 20.3, 788 x 1536 x 384 27.2 -> 17.3, 3152 x 1536 x 384 64.1 -> 37.9, 4096 x 4096 x 1024
// 307 -> 261 (131 TFLOP/s); weight gradients over 3152 rows: 384 x 384 83 -> 24, 1536 x 384 84 -> 57.
// ---------------------------------------------------------------------------
constexpr int FK = 32;   // depth of a tile

template <int R, int NW, bool TRANS> struct FTile {
  static constexpr int BYTES = R * FK * 4;
  static constexpr int NI = BYTES / 1024;            // wavefront-wide load instructions per tile
  static constexpr int IPW = (NI + NW - 1) / NW;     // ... per wavefront
  static constexpr int ROWB = TRANS ? R * 4 : FK * 4;   // bytes per LDS row
  static constexpr int CPR = ROWB / 16;              // 16-byte chunks per LDS row
  static constexpr int NRD = TRANS ? 2 : 1;          // LDS reads per fragment
  static_assert(R == 32 || R == 64 || R == 128, "tiles are 32, 64 or 128 rows wide");

  // (where there are fewer instructions than wavefronts the last ones repeat the last instruction: every
  // wavefront has the same number of loads in flight)
  static __device__ __forceinline__ int instr(int wave, int q) { return NI % NW == 0 ? wave * IPW + q : (wave < NI ? wave : NI - 1); }
  static_assert(NI % NW == 0 || NI < NW, "instr");
  static __device__ __forceinline__ int swz(int row) {
    return !TRANS ? (row >> 1) & 7 : (R == 32 ? ((row >> 1) & 1) << 2 : (row & 3) << 2);
  }
  // byte offset from the tile's first element of the chunk this lane fetches in its q-th instruction
  static __device__ __forceinline__ void init(uint32_t (&off)[IPW], int64_t ld, int wave, int lane) {
#pragma unroll
    for (int q = 0; q < IPW; ++q) {
      const int pos = instr(wave, q) * (64 / CPR) + lane / CPR;
      const int c = (lane % CPR) ^ swz(pos);
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
  static __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rs, const uint32_t (&off)[IPW], uint32_t lds, int wave) {
#pragma unroll
    for (int q = 0; q < IPW; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (PF_LDS(void))(uintptr_t)(lds + (uint32_t)instr(wave, q) * 1024u), 16, (int)off[q], 0, 0, 0);
  }
  // LDS byte offsets of this lane's fragments: [row][k] one per half h of the tile (MFMA tile i is 16 i rows on),
  // [k][row] one per MFMA tile (half h is 16 h rows on).  w0: first row of the wavefront's block, which starts at a
  // multiple of its own width.
  template <int NF> static __device__ __forceinline__ void frag_init(uint32_t (&foff)[NF], int w0, int lane) {
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const int r = w0 + (lane & 15), g = lane >> 4;
      foff[i] = !TRANS ? (uint32_t)(r * ROWB + ((4 * i + g) ^ swz(r)) * 16)
                       : (uint32_t)(g * ROWB + (((r + 16 * i) >> 2) ^ swz(g)) * 16 + (r & 3) * 4);
    }
  }
  template <int NF, int I, int H> static __device__ __forceinline__ void read(FragF<TRANS>& f, uint32_t lds, const uint32_t (&foff)[NF]) {
    if constexpr (!TRANS) {
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.v) : "v"(lds + foff[H]), "n"(I * 16 * ROWB) : "memory");
    } else {
      constexpr int S = 4 * ROWB / 256, H0 = H * 16 * ROWB / 256;   // (offsets in units of 64 elements)
      asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(f.lo) : "v"(lds + foff[I]), "n"(H0), "n"(H0 + S) : "memory");
      asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(f.hi) : "v"(lds + foff[I]), "n"(H0 + 2 * S), "n"(H0 + 3 * S) : "memory");
    }
  }
};

template <int BM, int BN, int WGM, int WGN, int ST, bool AT, bool BT>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm32d_kernel(const pf_gemm_desc p, const GemmGrid g) {
  constexpr int NW = WGM * WGN, WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
  using TA = FTile<BM, NW, AT>;
  using TB = FTile<BN, NW, BT>;
  constexpr int STAGE = TA::BYTES + TB::BYTES, LPW = TA::IPW + TB::IPW;
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
  const int wm0 = (wave / WGN) * WM, wn0 = (wave % WGN) * WN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

  uint32_t offa[TA::IPW], offb[TB::IPW];
  TA::init(offa, p.lda, wave, lane);
  TB::init(offb, p.ldb, wave, lane);
  constexpr int NFA = AT ? TM : 2, NFB = BT ? TN : 2;
  uint32_t foa[NFA], fob[NFB];
  TA::template frag_init<NFA>(foa, wm0, lane);
  TB::template frag_init<NFB>(fob, wn0, lane);

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
    TA::issue(TA::buffer(A, p.lda, edge_a, kt, (int)K), offa, sb, wave);
    TB::issue(TB::buffer(B, p.ldb, edge_b, kt, (int)K), offb, sb + TA::BYTES, wave);
  };
  // A tile's fragments are read, both halves of its depth, while the tile before it is multiplied: at the barrier
  // between two tiles nothing is left to wait for but the other wavefronts.  Two sets of fragments, by parity of the tile.
  FragF<AT> fa[2][2][TM];
  FragF<BT> fb[2][2][TN];
  auto read = [&](auto setc, auto hc, uint32_t sb) {
    constexpr int S = decltype(setc)::value, H = decltype(hc)::value;
    static_for<TM>([&](auto ic) { TA::template read<NFA, decltype(ic)::value, H>(fa[S][H][decltype(ic)::value], sb, foa); });
    static_for<TN>([&](auto jc) { TB::template read<NFB, decltype(jc)::value, H>(fb[S][H][decltype(jc)::value], sb + TA::BYTES, fob); });
  };
  auto arrived = [&](auto setc) {
    constexpr int S = decltype(setc)::value;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[S][h][i].arrived();
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[S][h][j].arrived();
    }
  };
  auto multiply = [&](auto setc, auto hc, auto ec) {
    constexpr int S = decltype(setc)::value, H = decltype(hc)::value, E = decltype(ec)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[S][H][i].get(E), fb[S][H][j].get(E), acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  constexpr std::integral_constant<int, 2> c2{};
  constexpr std::integral_constant<int, 3> c3{};

#pragma unroll
  for (int s = 0; s < ST; ++s) issue(s, lds0 + (uint32_t)s * STAGE);
  wait_vm<(ST - 1) * LPW>();
  asm volatile("s_barrier" ::: "memory");
  read(c0, c0, lds0);
  read(c0, c1, lds0);
  uint32_t sb = lds0;   // stage of tile kt
  auto tile = [&](int kt, auto setc) {
    constexpr std::integral_constant<int, 1 - decltype(setc)::value> other{};
    const uint32_t sb_next = sb + STAGE == lds0 + (uint32_t)ST * STAGE ? lds0 : sb + STAGE;
    wait_vm<(ST - 2) * LPW>();
    wait_lds<0>();
    arrived(setc);
    asm volatile("s_barrier" ::: "memory");   // tile kt + 1 is in LDS, tile kt in everybody's registers
    if (!(AT && BT) && left < FK && kt == nk - 1) {
      constexpr int S = decltype(setc)::value;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = 16 * h + 4 * (lane >> 4);
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[S][h][i].mask(k, left);
#pragma unroll
        for (int j = 0; j < TN; ++j) fb[S][h][j].mask(k, left);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    multiply(setc, c0, c0);
    read(other, c0, sb_next);
    multiply(setc, c0, c1);
    read(other, c1, sb_next);
    multiply(setc, c0, c2);
    issue(kt + ST, sb);
    __builtin_amdgcn_sched_barrier(0);
    multiply(setc, c0, c3);
    multiply(setc, c1, c0);
    multiply(setc, c1, c1);
    multiply(setc, c1, c2);
    multiply(setc, c1, c3);
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

  // D layout of v_mfma_f32_16x16x*: lane l holds column l % 16 and rows 4*(l/16) + r
  epilogue_f32<BM>(p, g, acc, m0, wm0 + 4 * (lane >> 4), n0 + wn0 + (lane & 15), c_base);
}

template <int BM, int BN, int WGM, int WGN, int ST, bool AT, bool BT>
int launch_one(const pf_gemm_desc& d, const GemmGrid& g, dim3 grid, hipStream_t st) {
  constexpr size_t lds = (size_t)ST * (BM + BN) * FK * 4;
  auto kern = gemm32d_kernel<BM, BN, WGM, WGN, ST, AT, BT>;
  const int rc = pf_allow_lds((const void*)kern, lds, "pf_gemm(f32)");
  if (rc != PF_OK) return rc;
  hipLaunchKernelGGL(kern, grid, dim3(64 * WGM * WGN), lds, st, d, g);
  PF_CHECK_LAUNCH("pf_gemm(f32)");
  return PF_OK;
}

template <int BM, int BN, int WGM, int WGN, int ST>
int launch(const pf_gemm_desc& d, hipStream_t st) {
  GemmGrid g;
  g.tiles_m = (int)((d.M + BM - 1) / BM);
  g.tiles_n = (int)((d.N + BN - 1) / BN);
  g.per_xcd = (int)(((int64_t)g.tiles_m * g.tiles_n + 7) / 8);
  g.vec_epi = epi_f32_vec_ok(d, BM);
  const dim3 grid((unsigned)(g.per_xcd * 8), (unsigned)(d.batch1 * d.batch2), 1);
  if (d.a_trans && d.b_trans) return launch_one<BM, BN, WGM, WGN, ST, true, true>(d, g, grid, st);
  if (d.a_trans) return launch_one<BM, BN, WGM, WGN, ST, true, false>(d, g, grid, st);
  if (d.b_trans) return launch_one<BM, BN, WGM, WGN, ST, false, true>(d, g, grid, st);
  return launch_one<BM, BN, WGM, WGN, ST, false, false>(d, g, grid, st);
}

// Tiles.  ST so that a microsecond or more of loads is in flight and (but for the largest) two or more workgroups fit
// a CU.  cost: time per output element and unit of depth relative to the largest tile's, from K = 384 .. 1536 (a
// 128x128 tile takes 58 ns per unit of depth, 64x64 17.1, 32x64 8.8 .. 10.7, 32x32 5.5; the matrix instructions
// alone 53, 13.3, 6.7, 3.3), and about 3.5 us per launch whatever the tile.
struct Tile {
  int bm, bn;
  double cost;   // time per output element relative to the largest tile's
  const char* shape;
};
constexpr Tile TILES[] = {
    {128, 128, 1.0, "128, 128, 2, 4, 4"}, {64, 64, 1.12, "64, 64, 4, 2, 4"}, {32, 64, 1.3, "32, 64, 2, 4, 6"}, {32, 32, 1.45, "32, 32, 2, 2, 8"}};

// What counts is the busiest CU, which takes ceil(tiles / 256) of them; as a launch rarely has the chip to itself
// (another stage's runs beside it), what its last round leaves idle is only half lost.
int choose(const pf_gemm_desc& d) {
  const int64_t nb = (d.batch1 > 0 ? d.batch1 : 1) * (d.batch2 > 0 ? d.batch2 : 1);
  int best = 0;
  double t_best = 0;
  for (int i = 0; i < 4; ++i) {
    const Tile& t = TILES[i];
    const int64_t tiles = ((d.M + t.bm - 1) / t.bm) * ((d.N + t.bn - 1) / t.bn) * nb;
    const double full = (double)((tiles + 255) / 256), even = (double)tiles / 256;
    const double c = (tiles <= 256 ? 1.0 : (full + even) / 2) * t.bm * t.bn * t.cost;
    if (i == 0 || c < t_best) best = i, t_best = c;
  }
  return best;
}
}  // namespace

// 16-byte loads need aligned operands and rows, byte offsets inside a tile 31 bits
bool pf_gemm_f32_direct_ok(const pf_gemm_desc& d) {
  const int64_t lim = (1ll << 31) / (4 * 128) - 1;
  return d.K >= 1 && pf_aligned(d.A, 16) && pf_aligned(d.B, 16) && d.lda % 4 == 0 && d.ldb % 4 == 0 && d.a_stride1 % 4 == 0 &&
         d.a_stride2 % 4 == 0 && d.b_stride1 % 4 == 0 && d.b_stride2 % 4 == 0 && d.lda < lim && d.ldb < lim && d.K < (1ll << 31) &&
         d.N < (1ll << 29);
}

// Depths from 129 on go to the wavefronts that split the depth, unless its stages of 64 would be a fifth empty.  us here / there: 3152 x 384 over 384
// 17.6 / 12.8, 788 x 384 over 1536 20.8 / 14.9, 442 x 1476 over 176 8.6 / 7.2, 4877 x 80 over 281 7.1 / 7.3; 96 products of 197 x 64 over 197 16.9 / 18.2,
// 8675 x 364 over 69 12.6 / 16.7, 7967 x 4996 over 126 122 / 128, 96 products of 197 x 197 over 64 19.3 / 20.0
static bool by_depth(const pf_gemm_desc& d) { return d.K > 128 && (d.K + 63) / 64 * 64 * 4 <= d.K * 5; }

void pf_gemm_f32_direct_name(const pf_gemm_desc& d, char* out, size_t cap) {
  const char* layouts = d.a_trans ? (d.b_trans ? "true, true" : "true, false") : (d.b_trans ? "false, true" : "false, false");
  if (by_depth(d)) snprintf(out, cap, "gemm32k_kernel<%s, %s>", pf_gemm_f32_depth_shape(d), layouts);
  else snprintf(out, cap, "gemm32d_kernel<%s, %s>", TILES[choose(d)].shape, layouts);
}

int pf_gemm_f32_direct(const pf_gemm_desc& d, hipStream_t st) {
  if (by_depth(d)) return pf_gemm_f32_depth(d, st);
  switch (choose(d)) {
    case 0: return launch<128, 128, 2, 4, 4>(d, st);
    case 1: return launch<64, 64, 4, 2, 4>(d, st);
    case 2: return launch<32, 64, 2, 4, 6>(d, st);
    default: return launch<32, 32, 2, 2, 8>(d, st);
  }
}
