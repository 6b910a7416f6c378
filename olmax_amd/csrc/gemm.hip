// bf16 MFMA GEMM for gfx950 (MI355X): C[M,N] = A[M,K] * B[N,K]^T (+ R), fp32 accumulate.
//
// Replaces the cuBLASLt calls XLA issues for olmax.nn.functional.linear
// (reference src/olmax/nn/functional.py:14-27) and for the two transposed
// products its autodiff derives (dX = dY W, dW = dY^T X).
//
// One kernel template covers the three operand storage combinations:
//   A "KC": A[m*lda + k]   (reduction dim contiguous)   A "MC": A[k*lda + m]
//   B "KC": B[n*ldb + k]                                 B "NC": B[k*ldb + n]
// forward  Y = X W^T      : A=X  (KC), B=W  (KC)
// dX = dY W               : A=dY (KC), B=W  (NC)   (reduction over out-features)
// dW = dY^T X             : A=dY (MC), B=X  (NC)   (reduction over tokens)
//
// Tiling: BM x BN x 64 block tile, 64-lane waves each owning a WM x WN sub-tile as
// (WM/16) x (WN/16) v_mfma_f32_16x16x32_bf16 accumulators. Operand tiles stream from
// global memory straight into LDS (global_load_lds_dwordx4, no VGPR staging, no LDS-write
// phase) into what has been consumed of two stages. K-contiguous tiles live in LDS as [rows][64]; M/N-contiguous
// tiles live as [64][rows] and are read with ds_read_b64_tr_b16, the gfx950 transposing
// LDS load, which hands each lane 4 consecutive reduction-dim elements of its column.
//
// LDS bank geometry (measured on gfx950 with SQ_LDS_BANK_CONFLICT): 64 banks x 4 B, i.e.
// 256 B per clock.  ds_read_b128 serves 16 lanes per clock in the fixed groups
// {0-3,12-15,20-23,24-27}, {4-7,8-11,16-19,28-31} (+32 for the upper half); ds_read_b64
// serves lanes 0-31, then 32-63.  The 16-byte chunk index of every tile is XOR-swizzled so
// that each such group touches 16 distinct chunks modulo 256 B:
//   [rows][64]  (128 B rows, two rows per bank line): chunk ^= (row >> 1) & 7
//   [64][rows]  (a transposing read of 32 lanes covers k-rows {k..k+3} and {k+8..k+11},
//               32 B each): chunk ^= ((k & 3) << 2) | ((k >> 2) & 2)
//
// Workgroup -> tile mapping is XCD aware: hardware deals consecutive workgroup ids
// round-robin over the 8 XCDs, so id i is remapped to (i % 8) * (grid/8) + i / 8, giving
// every XCD one contiguous run of tiles; runs walk the tile grid in column groups so that
// the A row-panels and B column-panels a single L2 sees are re-used.
#include "common.h"
#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>
#include <vector>

namespace {

constexpr int BK = 64;
constexpr int THIN_TILE = 256 + 128;  // 256 rows x 128 columns
typedef u32x4 __attribute__((aligned(2))) u32x4_u;  // 16 bytes at any element (ragged column edges)
typedef f32x4 __attribute__((aligned(4))) f32x4_u;

#ifndef GEMM_VGPR_CAP
#define GEMM_VGPR_CAP
#endif

// Optional per-launch timing (HIP events recorded on the launch stream around every GEMM),
// switched on by olmax_gemm_profile_begin(); used by the benchmark's roofline report.
struct ProfRec {
  hipEvent_t e0, e1;
  double flops;
  double bytes;  // algorithmic: every operand and the result moved once
  int key;  // tile | a_kc<<12 | b_kc<<13 | has_res<<14 | out_f32<<15
  int M, N, K;
};
std::atomic<bool> g_prof_on{false};  // diagnostic switch, process-wide
std::vector<ProfRec> g_prof;
std::mutex g_prof_mu;

// GLU != 0 (1 silu, 2 tanh-gelu) turns the kernel into the fused gate/up projection of a gated
// MLP: B is [Wgate; Wup] ([2F, K]), a block covers 128 features and loads their 128 gate rows
// and 128 up rows, arranged in LDS so that every wave owns the gate AND the up columns of the
// same 32 features; the epilogue writes act = f(gate) * up ([M, F], leading dimension ldr) and,
// when Cv is given, gate|up ([M, 2F]) as the plain GEMM would.  N is F in that mode.
//
// EPI == 4 / 5 (silu / tanh-gelu) is the same projection run in the BACKWARD pass of a block whose
// forward kept nothing: gate and up are recomputed in the accumulators and, with the gradient of
// the activation output (dact [M, F], passed through the cos_t pointer with its row stride in
// seq_len), leave the kernel as act = f(gate) * up (R, for the down projection's weight gradient)
// and d gate | d up (Cv [M, 2F]) -- gate | up never reach memory and no separate GLU backward
// kernel runs.  Same roundings as olmax_gemm_glu_bf16 followed by olmax_glu_bwd.
//
// EPI == 3 is the fused q|k|v projection + rotary embedding: columns below rope_cols are heads of
// 128 that leave the kernel rotated (out = x cos + rotate_half(x) sin in fp32 on the bf16-rounded
// projection, as the separate RoPE kernel computes it); a wave's 64 columns are one half of a
// head and its neighbour (wave ^ 1) holds the other, so the rotation reads both from the LDS
// staging of the epilogue.  The position of a row is row % seq_len; cos/sin are [seq_len, 64] fp32.
//
// EPI == 6 is one part of a reduction that several workgroups share (see olmax_gemm_padded): blockIdx.y
// takes k in [y * seq_len, (y + 1) * seq_len), the last one the rest, and the accumulators leave as they
// are, 1 KB per instruction, to Cv[part][tile][wave][i][j][lane] for gemm_split_sum_kernel.  With `sums` (both gradients in one launch) the
// operands are already those of a part, and its accumulators go there.
//
// RAG: 1 where M or N, 2 where K is not a multiple of the tile.  The last tile of a row or column is
// moved back so that it ends with the matrix (the loop then reads nothing outside it and is the same
// code) and stores only what no other tile stores.  The partial k-tile at the end of K is taken FIRST, ahead of
// the loop, which then sees whole k-tiles only: it is fetched with per-lane addresses, and the wave
// that fetched a chunk past the end overwrites it with zeros in LDS once its own fetches have landed,
// before the barrier that publishes the stage.  Wants M >= BM, N >= BN, K >= 64 and 16-byte chunks that do not cross the end of a row (see olmax_gemm_padded).
//
// The tile that workgroup `pid` of `nwg` takes; the residual of a HAS_RES form may be null.  BLOCKS: the sums of every `block` k-tiles (an
// even number) are added up by themselves, for shorter chains of fp32 additions: 1 in registers, 2 (256 tiles, which have none left) parked
// in `park`, 256 KB a tile and block.  us in a block's backward pass, both gradients with one chain -> with blocks: 3000 x 1024 x 3072 44.6 -> 46.6,
// 4096 x 1024 x 3072 59.8 -> 60.4, 512 x 2816 x 1024 16.8 -> 17.6; 2048 x 4096 x 12288 302 -> 308, x 22016 540 -> 555.
template <int BM, int BN, int WM, int WN, bool A_KC, bool B_KC, bool HAS_RES, bool OUT_F32, int EPI, int RAG, int BLOCKS = 0>
__device__ __forceinline__ void gemm_tile(
    const bf16* __restrict__ A, const bf16* __restrict__ B, void* __restrict__ Cv,
    const bf16* __restrict__ R, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
    int64_t ldr, int tiles_m, int tiles_n, int c_vec, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, int seq_len, int rope_cols, int order, int pid, const int nwg, unsigned char* smem, int block = 0, float* park = nullptr,
    float* sums = nullptr) {
  constexpr int GLU = (EPI == 1 || EPI == 2) ? EPI : (EPI == 4 ? 1 : (EPI == 5 ? 2 : 0));
  constexpr bool GLU_BWD = EPI == 4 || EPI == 5;
  constexpr bool ROPE = EPI == 3;
  constexpr bool SPLIT = EPI == 6;
  static_assert(EPI == 0 || SPLIT || (BN == 256 && WN == 64 && B_KC && !HAS_RES && !OUT_F32), "fused epilogues: 256-wide NT tiles only");
  constexpr int NW = (BM / WM) * (BN / WN);
  constexpr int TM = WM / 16, TN = WN / 16;  // accumulators of 16x16 per wave
  constexpr int WAVES_N = BN / WN;
  constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2;
  constexpr int A_INS = A_BYTES / 1024 / NW;  // DMA instructions (1 KB each) per wave per k-tile
  constexpr int B_INS = B_BYTES / 1024 / NW;
  static_assert(A_INS >= 1 && B_INS >= 1, "tile too small for the wave count");
  constexpr int NINS = A_INS + B_INS;
  constexpr bool THIN = BM == 256 && BN == 128;
  constexpr int STAGES = THIN ? 3 : 2;  // of LDS

  // LDS: [A stage 0 | A stage 1 | .. | B stage 0 | B stage 1 | ..]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;

  // ---- XCD-aware tile assignment ----
  int tile_m, tile_n;
  if (order > 0) {
    // Windows of 8 x 4 tiles (what the 32 CUs of an XCD hold at a time: 12 operand panels for
    // 32 tiles in that XCD's L2), dealt to the XCDs so that the 8 windows in flight together
    // form one block of `order` 8-row strips by 32 / order columns (order 2: 16 x 16 tiles, 32
    // distinct panels per round for the whole chip; order 4: 32 x 8; order 8: 64 x 4).  Groups of
    // `order` strips sweep all columns before the next group starts, so B is read once per group
    // and a group's A panels are re-read from the memory-side cache on every step of the sweep.
    // The tile grid is padded to whole windows and the launch to whole rounds; workgroups that
    // fall into the padding leave at once.
    const int xcd = pid & 7, slot = pid >> 3;
    const int c = (slot >> 5) * 8 + xcd, w = slot & 31;  // window, tile inside the window
    const int strips = (tiles_m + 7) >> 3, wpr = (tiles_n + 3) >> 2;  // 8-row strips, windows per strip
    if (c >= strips * wpr) return;
    const int full = (strips / order) * order * wpr;      // windows in whole groups of strips
    int sg, v, S;
    if (c < full) { sg = c / (order * wpr); v = c % (order * wpr); S = order; }
    else { sg = strips / order; v = c - full; S = strips % order; }
    tile_m = ((order * sg + v % S) << 3) + (w & 7);
    tile_n = ((v / S) << 2) + (w >> 3);
    if (tile_m >= tiles_m || tile_n >= tiles_n) return;
  } else {
    {
      const int per = nwg >> 3;
      if ((nwg & 7) == 0) pid = (pid & 7) * per + (pid >> 3);
    }
    // column-grouped walk: groups of GM row-tiles, sweep N inside a group
    constexpr int GM = 8;
    const int group_sz = GM * tiles_n;
    const int gid = pid / group_sz;
    const int first_m = gid * GM;
    const int gm = min(tiles_m - first_m, GM);
    tile_m = first_m + (pid % group_sz) % gm;
    tile_n = (pid % group_sz) / gm;
  }
  if (SPLIT) {
    const int k_lo = blockIdx.y * seq_len;
    A += A_KC ? (int64_t)k_lo : (int64_t)k_lo * lda;
    B += B_KC ? (int64_t)k_lo : (int64_t)k_lo * ldb;
    K = blockIdx.y + 1 == gridDim.y ? K - k_lo : seq_len;
  }
  constexpr bool KRAG = RAG == 2;
  constexpr int BNC = GLU ? BN / 2 : BN;  // output columns of a block (GLU: features)
  int m0 = tile_m * BM, n0 = tile_n * BNC;
  // rows / columns of the block that this tile stores: all, or (RAG) those behind the previous tile's
  int row_lo = 0, row_hi = BM, col_lo = 0;
  if (RAG) {
    m0 = min(m0, (A_KC ? M : (M + 7) & ~7) - BM);
    n0 = min(n0, N - BNC);
    row_lo = tile_m * BM - m0;
    row_hi = M - m0;
    col_lo = tile_n * BNC - n0;
  }
  // 8 output columns from column c of the block; c and the block's end are whole chunks except where
  // N is not a multiple of 8 (then the chunk shared with the previous tile is stored by elements)
  auto store8 = [&](bf16* dst, int c, const u32x4& v) {
    if (!RAG) {
      *reinterpret_cast<u32x4*>(dst) = v;
    } else if (c >= col_lo) {
      *reinterpret_cast<u32x4_u*>(dst) = v;
    } else if (c + 8 > col_lo) {
      Pack8 t;
      t.u = v;
#pragma unroll
      for (int e = 1; e < 8; e++)
        if (c + e >= col_lo) dst[e] = t.e[e];
    }
  };
  auto stores_row = [&](int row) { return !RAG || (row >= row_lo && row < row_hi); };

  // swizzles (see the bank-geometry note at the top of the file)
  auto kswz = [](int row) { return (row >> 1) & 7; };                         // [rows][64] tiles
  auto tswz = [](int kr) { return ((kr & 3) << 2) | ((kr >> 2) & 2); };        // [64][rows] tiles

  // ---- DMA sources: instruction i of this wave fills LDS block (i*NW + wave) of 1 KB, i.e.
  // 16-byte chunks p = block*64 + lane of the tile; the lane fetches whichever global chunk the
  // swizzle places there.  Consecutive instructions of a wave are a whole number of swizzle
  // periods (16 rows) apart, so a lane's byte offset inside the operand panel is one VGPR for all
  // of them; instruction and k-tile only move the wave-uniform base (SGPRs), and the loop spends
  // no vector instruction and one register per operand on DMA addresses.
  unsigned a_off, b_off;
  constexpr int A_IROWS = A_KC ? NW * 8 : NW * 64 / (BM / 8);  // tile rows between two instructions
  constexpr int B_IROWS = B_KC ? NW * 8 : NW * 64 / (BN / 8);
  static_assert(A_IROWS % 16 == 0 && B_IROWS % 16 == 0, "instructions of a wave must share the swizzle");
  static_assert(GLU == 0 || B_IROWS == 64, "GLU row mapping: one instruction per wave tile of 64 rows");
  {
    const int p = wave * 64 + lane;
    if (A_KC) {
      const int row = p >> 3, ph = p & 7;
      a_off = (unsigned)(((int64_t)row * lda + ((ph ^ kswz(row)) << 3)) * 2);
    } else {
      constexpr int CPR = BM / 8;  // chunks per k-row
      const int kr = p / CPR, ph = p % CPR;
      a_off = (unsigned)(((int64_t)kr * lda + ((ph ^ tswz(kr)) << 3)) * 2);
    }
    if (B_KC) {
      const int row = p >> 3, ph = p & 7;
      // GLU: LDS row (wave w: 64w .. 64w+63) = gate rows of features 32w .. 32w+31, then their up
      // rows; instruction i covers LDS rows 64i .. 64i+63, i.e. 32 features further on per step
      const int64_t grow = GLU ? (int64_t)((row >> 5) & 1) * N + (row & 31) : row;
      b_off = (unsigned)((grow * ldb + ((ph ^ kswz(row)) << 3)) * 2);
    } else {
      constexpr int CPR = BN / 8;
      const int kr = p / CPR, ph = p % CPR;
      b_off = (unsigned)(((int64_t)kr * ldb + ((ph ^ tswz(kr)) << 3)) * 2);
    }
  }
  const int64_t a_istep = (int64_t)A_IROWS * lda;  // elements between two instructions' sources
  const int64_t b_istep = (int64_t)(GLU ? 32 : B_IROWS) * ldb;
  const int64_t a_step = A_KC ? (int64_t)BK : (int64_t)BK * lda;
  const int64_t b_step = B_KC ? (int64_t)BK : (int64_t)BK * ldb;
  // k-tile 0 of this block's rows (KRAG: of the loop's numbering, in which 1 is the first whole one)
  const bf16* a_panel = (A_KC ? A + (int64_t)m0 * lda : A + m0) - (KRAG ? a_step : 0);
  const bf16* b_panel = (B_KC ? B + (int64_t)n0 * ldb : B + n0) - (KRAG ? b_step : 0);

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[i][j][r] = 0.f;

  const int KTF = K / BK;             // whole k-tiles
  const int KT = KTF + (KRAG ? 1 : 0);
  const unsigned lds_base = lds_addr_of(smem);
  // issue DMA instructions [lo, hi) of the combined A+B list of k-tile kt into `stage`
  auto dma = [&](int kt, int stage, int lo, int hi) {
    const unsigned sa = lds_base + stage * A_BYTES;
    const unsigned sb = lds_base + STAGES * A_BYTES + stage * B_BYTES;
#pragma unroll
    for (int i = 0; i < NINS; i++) {
      if (i < lo || i >= hi) continue;
      if (i < A_INS) {
        dma16_s(a_panel + (int64_t)kt * a_step + i * a_istep, a_off, sa + (i * NW + wave) * 1024);
      } else {
        const int j = i - A_INS;
        dma16_s(b_panel + (int64_t)kt * b_step + j * b_istep, b_off, sb + (j * NW + wave) * 1024);
      }
    }
  };

  // KRAG: source of DMA instruction i (of A, then of B) of the partial k-tile for this lane; chunks past
  // the end are fetched from the row's start (k-contiguous) or from the last k-row and zeroed later
  auto tail_src = [&](int i, bool& valid) -> const bf16* {
    const int p = wave * 64 + lane;
    if (i < A_INS) {
      if (A_KC) {
        const int row = i * A_IROWS + (p >> 3), k = KTF * BK + (((p & 7) ^ kswz(row)) << 3);
        valid = k < K;
        return A + (int64_t)(m0 + row) * lda + (valid ? k : 0);
      }
      constexpr int CPR = BM / 8;
      const int kr = i * A_IROWS + p / CPR, k = KTF * BK + kr;
      valid = k < K;
      return A + (int64_t)(valid ? k : K - 1) * lda + m0 + (((p % CPR) ^ tswz(kr)) << 3);
    }
    const int j = i - A_INS;
    if (B_KC) {
      const int row = j * B_IROWS + (p >> 3), k = KTF * BK + (((p & 7) ^ kswz(row)) << 3);
      valid = k < K;
      return B + (int64_t)(n0 + row) * ldb + (valid ? k : 0);
    }
    constexpr int CPR = BN / 8;
    const int kr = j * B_IROWS + p / CPR, k = KTF * BK + kr;
    valid = k < K;
    return B + (int64_t)(valid ? k : K - 1) * ldb + n0 + (((p % CPR) ^ tswz(kr)) << 3);
  };
  auto tail_lds = [&](int i, int stage) -> unsigned {
    return i < A_INS ? lds_base + stage * A_BYTES + (i * NW + wave) * 1024
                     : lds_base + STAGES * A_BYTES + stage * B_BYTES + ((i - A_INS) * NW + wave) * 1024;
  };
  auto dma_tail = [&](int stage) {
#pragma unroll 1
    for (int i = 0; i < NINS; i++) {
      bool valid;
      const bf16* src = tail_src(i, valid);
      dma16(src, tail_lds(i, stage));
    }
  };
  auto zero_tail = [&](int stage) {  // only after this wave's own fetches have landed
#pragma unroll 1
    for (int i = 0; i < NINS; i++) {
      bool valid;
      (void)tail_src(i, valid);
      if (!valid)
        *reinterpret_cast<__attribute__((address_space(3))) u32x4*>((uintptr_t)(tail_lds(i, stage) + lane * 16)) = u32x4{0u, 0u, 0u, 0u};
    }
  };

  // v_mfma_f32_16x16x32_bf16 operand geometry: lane -> row/column (lane % 16) of the 16-wide
  // tile, k-group lane / 16 (8 consecutive k each); accumulator lane -> column lane % 16,
  // rows 4*(lane/16) + r.  It sustains ~7 % more FLOP/s than the 32x32x16 form under the
  // board's power limit (less accumulator traffic per FLOP).
  const int l16 = lane & 15, g16 = lane >> 4;

  // Per-lane LDS byte addresses of the operand fragments, computed once.  LDS holds the A tiles
  // of both stages first, then the B tiles ([A0 | A1 | B0 | B1]), so that one base register
  // reaches a fragment of either stage with an immediate below 64 KB: for k-contiguous tiles one
  // base per k-step with stage and tile row (i*16 rows = i*2048 B) as immediate; for transposed
  // tiles one base per tile row -- the XOR swizzle permutes the chunk differently in every lane
  // -- with stage, k-step and half ((kk*32 + h*4) k-rows) as immediate.  The bases pass through
  // an empty asm so that the compiler keeps exactly these registers instead of re-deriving (and
  // spilling) one address per read; the loop then holds no address arithmetic at all.
  // (Adding whole 16-row tiles leaves kswz, which looks at row bits 1-3, unchanged; adding
  // multiples of 4 k-rows leaves tswz unchanged as long as bit 3 of the k-row comes from the
  // lane, which it does: k-row = 32*kk + 8*(lane/16) + 4*h + lane%16/4.)
  constexpr int NA_BASE = A_KC ? 2 : TM, NB_BASE = B_KC ? 2 : TN;
  static_assert(A_BYTES + 36 * (BM > BN ? BM : BN) * 2 < 65536, "fragment immediates must fit 16 bits");
  unsigned a_base[NA_BASE], b_base[NB_BASE], a_base2[THIN ? NA_BASE : 1];  // (A's third stage is out of the immediates' reach)
#pragma unroll
  for (int x = 0; x < NA_BASE; x++) {
    unsigned v;
    if (A_KC) {  // x = k-step
      const int row = wm * WM + l16;
      v = row * 128 + (((x * 4 + g16) ^ kswz(row)) << 4);
    } else {     // x = tile row i
      const int col = wm * WM + x * 16 + ((l16 & 3) << 2);
      const int kr = g16 * 8 + (l16 >> 2);
      v = kr * (BM * 2) + (((col >> 3) ^ tswz(kr)) << 4) + ((col & 7) << 1);
    }
    v += lds_base;
    asm volatile("" : "+v"(v));
    a_base[x] = v;
    if (THIN) {
      v += 2 * A_BYTES;
      asm volatile("" : "+v"(v));
      a_base2[THIN ? x : 0] = v;
    }
  }
#pragma unroll
  for (int x = 0; x < NB_BASE; x++) {
    unsigned v;
    if (B_KC) {
      const int row = wn * WN + l16;
      v = row * 128 + (((x * 4 + g16) ^ kswz(row)) << 4);
    } else {
      const int col = wn * WN + x * 16 + ((l16 & 3) << 2);
      const int kr = g16 * 8 + (l16 >> 2);
      v = kr * (BN * 2) + (((col >> 3) ^ tswz(kr)) << 4) + ((col & 7) << 1);
    }
    v += lds_base + STAGES * A_BYTES;
    asm volatile("" : "+v"(v));
    b_base[x] = v;
  }
  auto lds_b128 = [](unsigned addr) -> bf16x8 {
    return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>((uintptr_t)addr);
  };
  auto lds_tr64 = [](unsigned addr) -> u32x2 {
    s16x4 t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(uintptr_t)addr);
    return (u32x2&)t;
  };
  // one operand fragment (16 rows x 32 k) of k-step kk (0 or 1) of stage st (all compile-time)
  auto load_a1 = [&](int st, int kk, int i) -> bf16x8 {
    if (A_KC) {
      return lds_b128(THIN && st == 2 ? a_base2[THIN ? kk : 0] + i * 2048 : a_base[kk] + st * A_BYTES + i * 2048);
    } else {
      // transposing read: the 16-lane group g16 fetches k-rows kk*32 + 8*g16 + {0..3, 4..7}
      Pack8 p;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const u32x2 t = lds_tr64((THIN && st == 2 ? a_base2[THIN ? i : 0] : a_base[i] + st * A_BYTES) + (kk * 32 + h * 4) * (BM * 2));
        p.u[h * 2 + 0] = t[0];
        p.u[h * 2 + 1] = t[1];
      }
      return p.v;
    }
  };
  auto load_b1 = [&](int st, int kk, int j) -> bf16x8 {
    if (B_KC) {
      return lds_b128(b_base[kk] + st * B_BYTES + j * 2048);
    } else {
      Pack8 p;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const u32x2 t = lds_tr64(b_base[j] + st * B_BYTES + (kk * 32 + h * 4) * (BN * 2));
        p.u[h * 2 + 0] = t[0];
        p.u[h * 2 + 1] = t[1];
      }
      return p.v;
    }
  };

  constexpr int NM = TM * TN, NF = TM + TN;
  constexpr bool PINGPONG = BM == 256;
  // ---- main loop of the 256 x 256 tiles: the two waves of a SIMD (w and w + 4) take turns.  A k-tile is two phases; in each a wave
  // first fetches the fragments and issues DMA (memory part), then runs 32 MFMAs with nothing between them (matrix part), and a
  // barrier after every part keeps waves 4-7 exactly one part behind waves 0-3: while one wave of the SIMD owns the matrix pipe, the
  // other waits for its LDS reads, for the DMA queue and for the landing of the next k-tile, where it costs no MFMA time.  (Before, all
  // eight waves issued reads and DMA between their own MFMAs and met at one barrier per k-tile: a full DMA queue or a late line stopped
  // all of them, 61 % of the MFMA rate on operands of zeros, which leave the power limit out; now 80-86 %.)  us on random operands, before -> now:
  //   NT 8192 x 12288 x 4096 558 -> 545, 8192 x 22016 x 4096 1067 -> 1004, 8192 x 4096 x 11008 514 -> 475, 8192 x 100352 x 4096 4895 -> 4529
  //   NN 8192 x 4096 x 12288 565 -> 532, 8192 x 4096 x 22016 1028 -> 951;  TN 12288 x 4096 x 8192 581 -> 536, 22016 x 4096 x 8192 1096 -> 1011
  // Bound by the board's power on such operands (zeros run 30 % faster).  Four phases of 16 MFMAs: NT 0 to -1 %, NN and TN +2 to +4 %;
  // a higher wave priority in the matrix part +0.5 %; DMA ahead of the reads +0.3 to +2.5 %.
  //   phases: by k-step where A is [64][rows] (a DMA instruction covers whole k-rows, so k-steps are what becomes free), else by half
  //     of the wave's rows.  B's fragments of both k-steps are fetched in phase 0 and kept, but where both go by k-step;
  //   DMA: in the memory part after the one that read it last a region is refilled for two k-tiles on: what phase 0 reads (d0)
  //     in phase 1 of k-tile t for t + 2, what phase 1 reads (d1) in phase 0 of t + 1 for t + 2.  Past the end the last k-tile is fetched
  //     again into a region nobody reads any more;
  //   waits: every wave's LDS reads are complete before the barrier that ends its memory part, so no refill can overtake a read, and
  //     vmcnt(8) there leaves only what was issued behind the d0 / d1 that the next phase of this kind reads.
  //
  // 256 x 128 tiles (THIN): as above, but a k-tile is one phase (64 registers of fragments, 32 MFMAs) and LDS has three stages, so that k-tile t + 2 is fetched
  // into the stage of t - 1 while t is worked on.  They move 25 % less than four waves' 128 x 128 tiles, two of which share a CU (see thin_takes).
  //
  // ---- main loop of the 128 x 128 tiles: software pipeline, all of it in registers and the two LDS stages:
  //   * fragments are double-buffered (fa/fb[0] = k-step 0, [1] = k-step 1 of a k-tile), and
  //     every LDS read is issued half a k-tile before the MFMAs that consume it;
  //   * the DMA of k-tile kt+2 goes into the stage k-tile kt occupied, right after the barrier
  //     that retires it, so it has a whole k-tile of MFMAs to land;
  //   * reads and DMA issues are slotted one per MFMA (pinned with sched_barrier), so that a
  //     wave never leaves the matrix pipe without work for longer than one MFMA;
  //   * the steady state has no branches: past the end the DMA re-fetches the last k-tile and
  //     the reads fetch a stage nobody uses any more.
  static_assert(PINGPONG || (2 * NINS <= NM && NF + 1 <= NM && NINS + NF <= NM), "not enough MFMA slots for the loads");
  static_assert(!PINGPONG || THIN || (NW == 8 && TM == 8 && TN == 4 && A_INS == 4 && B_INS == 4), "phases are laid out for 8 waves of 128 x 64");
  static_assert(!THIN || (NW == 8 && TM == 4 && TN == 4), "8 waves of 64 x 64");
  constexpr bool BY_K = !A_KC, B_WHOLE = A_KC || B_KC;  // PINGPONG: phases by k-step; all of B is read in phase 0
  constexpr int ND0 = B_WHOLE ? 6 : 4;                  // DMA instructions of d0
  bf16x8 fa[2][PINGPONG ? 4 : TM], fb[2][TN];
  // k-tiles t + 1 (PINGPONG) and t + 2 while they exist, then the last one
  const bf16 *ap1 = a_panel + (int64_t)min(1, KT - 1) * a_step, *bp1 = b_panel + (int64_t)min(1, KT - 1) * b_step;
  const bf16 *ap = a_panel + (int64_t)min(2, KT - 1) * a_step, *bp = b_panel + (int64_t)min(2, KT - 1) * b_step;
  auto dma_a = [&](const bf16* p, int stage, int i) { dma16_s(p + i * a_istep, a_off, lds_base + stage * A_BYTES + (i * NW + wave) * 1024); };
  auto dma_b = [&](const bf16* p, int stage, int i) { dma16_s(p + i * b_istep, b_off, lds_base + STAGES * A_BYTES + stage * B_BYTES + (i * NW + wave) * 1024); };
  // (instruction i holds rows 64i .. 64i+63 of a k-contiguous tile: i even, the first half of the rows of waves 0-3 / 4-7; k-rows 16i .. 16i+15 of the others)
  auto d0 = [&](const bf16* pa, const bf16* pb, int stage) {
    dma_a(pa, stage, 0);
    dma_b(pb, stage, 0);
    if (B_WHOLE) dma_b(pb, stage, 1);
    dma_a(pa, stage, BY_K ? 1 : 2);
    dma_b(pb, stage, B_WHOLE ? 2 : 1);
    if (B_WHOLE) dma_b(pb, stage, 3);
  };
  auto d1 = [&](const bf16* pa, const bf16* pb, int stage) {
    dma_a(pa, stage, BY_K ? 2 : 1);
    if (!B_WHOLE) dma_b(pb, stage, 2);
    dma_a(pa, stage, 3);
    if (!B_WHOLE) dma_b(pb, stage, 3);
  };
  auto d_all = [&](const bf16* pa, const bf16* pb, int stage) {
#pragma unroll
    for (int i = 0; i < A_INS; i++) dma_a(pa, stage, i);
#pragma unroll
    for (int i = 0; i < B_INS; i++) dma_b(pb, stage, i);
  };
  if (KRAG) dma_tail(0);
  else dma(0, 0, 0, NINS);
  if constexpr (PINGPONG) {
    if (KRAG) {
      dma_wait_all();
      zero_tail(0);
    }
    if (THIN) d_all(ap1, bp1, 1);
    else d0(ap1, bp1, 1);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(THIN ? NINS : ND0) : "memory");  // k-tile 0 has landed
    __builtin_amdgcn_s_barrier();
    if (wave >= 4) __builtin_amdgcn_s_barrier();  // one part behind (waves 0-3 make up for it after the loop)
  } else {
    if (KT > 1) {
      dma(1, 1, 0, NINS);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NINS) : "memory");  // k-tile 0 has landed
    } else {
      dma_wait_all();
    }
    if (KRAG) zero_tail(0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; i++) fa[0][i] = load_a1(0, 0, i);
#pragma unroll
    for (int j = 0; j < TN; j++) fb[0][j] = load_b1(0, 0, j);
  }
  // One phase of a k-tile (PINGPONG); stage and phase are compile-time constants (the loop below is unrolled by two k-tiles), so every LDS address
  // is a loop-invariant per-lane register plus an immediate: no address arithmetic is left in the loop.
  auto phase = [&](auto cur_tag, auto ph_tag) {
    constexpr int cur = decltype(cur_tag)::value, ph = decltype(ph_tag)::value;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < 8; x++)
      if (B_WHOLE ? ph == 0 : x < 4) fb[x >> 2][x & 3] = load_b1(cur, B_WHOLE ? x >> 2 : ph, x & 3);
#pragma unroll
    for (int x = 0; x < 8; x++) fa[x >> 2][x & 3] = BY_K ? load_a1(cur, ph, x) : load_a1(cur, x >> 2, ph * 4 + (x & 3));
    __builtin_amdgcn_sched_barrier(0);
    if (ph == 0) d1(ap1, bp1, cur ^ 1);
    else d0(ap, bp, cur);
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < 8; x++) {  // fragment x of A with all of B's that go with it
      const int i = BY_K ? x : ph * 4 + (x & 3);
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[!B_WHOLE ? 0 : BY_K ? ph : x >> 2][j], fa[x >> 2][x & 3], acc[i][j], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto k_tile = [&](int kt, auto cur_tag) {
    constexpr int cur = decltype(cur_tag)::value;
    constexpr int nxt = cur ^ 1;
    if constexpr (THIN) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 8; x++) fb[x >> 2][x & 3] = load_b1(cur, x >> 2, x & 3);
#pragma unroll
      for (int x = 0; x < 8; x++) fa[x >> 2][x & 3] = load_a1(cur, x >> 2, x & 3);
      __builtin_amdgcn_sched_barrier(0);
      d_all(ap, bp, (cur + 2) % 3);
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NINS) : "memory");  // k-tile kt+1 has landed
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 8; x++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[x & 3][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[x >> 2][j], fa[x >> 2][x & 3], acc[x & 3][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    } else if constexpr (PINGPONG) {
      phase(cur_tag, std::integral_constant<int, 0>());
      phase(cur_tag, std::integral_constant<int, 1>());
      ap1 = ap;
      bp1 = bp;
    } else {
      // ---- first half: k-step 0 from registers; the fragments of k-step 1 are fetched meanwhile
      // (no fetch in slot 0: hoisted above the first MFMA it would make that MFMA's operand wait,
      // an in-order counter, cover the new read's latency as well)
#pragma unroll
      for (int m = 0; m < NM; m++) {
        const int i = m / TN, j = m % TN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[0][j], fa[0][i], acc[i][j], 0, 0, 0);
        if (m >= 1 && m <= TN) fb[1][m - 1] = load_b1(cur, 1, m - 1);
        if (m > TN && m <= NF) fa[1][m - TN - 1] = load_a1(cur, 1, m - TN - 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      // k-tile kt+1 has landed (issued one k-tile ago); every wave is done reading k-tile kt
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __syncthreads();
      // ---- second half: k-step 1 from registers; the slots issue the DMA of k-tile kt+2 into the
      // retired stage and fetch k-step 0 of k-tile kt+1; the first MFMA goes out right behind the barrier
#pragma unroll
      for (int m = 0; m < NM; m++) {
        const int i = m / TN, j = m % TN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[1][j], fa[1][i], acc[i][j], 0, 0, 0);
        int q = -1, f = -1;  // DMA instruction / fragment of this slot
        // DMA issues and fragment reads alternate while both last, from slot 1 when they fit
        constexpr int FIRST = (NINS + NF <= NM - 1) ? 1 : 0;
        constexpr int BOTH = NINS < NF ? NINS : NF;
        const int k = m - FIRST;
        if (k >= 0 && k < 2 * BOTH) { if (k & 1) f = k >> 1; else q = k >> 1; }
        else if (k >= 2 * BOTH && k < NINS + NF) { if (NINS > NF) q = k - BOTH; else f = k - BOTH; }
        if (q >= 0) {
          if (q < A_INS) dma_a(ap, cur, q);
          else dma_b(bp, cur, q - A_INS);
        }
        if (f >= 0) {
          if (f < TN) fb[0][f] = load_b1(nxt, 0, f);
          else fa[0][f - TN] = load_a1(nxt, 0, f - TN);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (kt + 3 < KT) {
      ap += a_step;
      bp += b_step;
    }
  };
  f32x4 sum[BLOCKS == 1 ? TM : 1][TN];
  if (BLOCKS == 1) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) sum[BLOCKS == 1 ? i : 0][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  int ends = block, parked = 0;  // of the block; blocks before it
  auto parking = [&](int b) { return park + ((((int64_t)b * tiles_m + tile_m) * tiles_n + tile_n) * NW + wave) * (NM * 256); };  // of this wave
  // (a copy of the lane id that the compiler cannot see through: no address of the rare accesses lives through the loop)
  auto hidden_lane = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l * 4;
  };
  int kt = 0;
  for (; kt + STAGES <= KT; kt += STAGES) {
    k_tile(kt, std::integral_constant<int, 0>());
    k_tile(kt + 1, std::integral_constant<int, 1>());
    if constexpr (THIN) k_tile(kt + 2, std::integral_constant<int, 2>());
    if (BLOCKS && kt + STAGES == ends && ends < KT) {
      ends += block;
      float* q = parking(parked++);
      const int at = hidden_lane();
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
          if (BLOCKS == 1) sum[BLOCKS == 1 ? i : 0][j] += acc[i][j];
          else *reinterpret_cast<f32x4*>(q + (i * TN + j) * 256 + at) = acc[i][j];
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  if (kt < KT) k_tile(kt, std::integral_constant<int, 0>());
  if constexpr (THIN)
    if (kt + 1 < KT) k_tile(kt + 1, std::integral_constant<int, 1>());
  if (PINGPONG && wave < 4) __builtin_amdgcn_s_barrier();
  if (BLOCKS == 1) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) acc[i][j] += sum[BLOCKS == 1 ? i : 0][j];
  }
  dma_wait_all();  // the redundant tail DMAs must not outlive the workgroup's LDS allocation
  if (BLOCKS == 2) {  // (all that was parked has been written)
    for (int b = 0; b < parked; b++) {
      const float* q = parking(b);
      const int at = hidden_lane();
#pragma unroll
      for (int i = 0; i < TM; i++) {
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] += *reinterpret_cast<const f32x4*>(q + (i * TN + j) * 256 + at);
        __builtin_amdgcn_sched_barrier(0);  // (the loads of all rows at once do not fit the registers)
      }
    }
  }
  // The epilogue derives its addresses from a copy of the lane id that the compiler cannot see
  // through, so none of them is computed ahead of the loop and kept in registers across it.
  int lane_e = lane;
  asm volatile("" : "+v"(lane_e));
  const int l16e = lane_e & 15, g16e = lane_e >> 4;

  if (SPLIT || sums) {
    float* part = SPLIT ? reinterpret_cast<float*>(Cv) + (int64_t)blockIdx.y * tiles_m * tiles_n * (NW * NM * 256) : sums;
    part += (((int64_t)tile_m * tiles_n + tile_n) * NW + wave) * (NM * 256);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) *reinterpret_cast<f32x4*>(part + ((i * TN + j) * 64 + lane_e) * 4) = acc[i][j];
    return;
  }

  // ---- epilogue.  The MFMAs ran with their operands swapped (B fragment as the instruction's A),
  // so each accumulator is a transposed 16x16 tile: lane -> row l16e, columns 4*g16e + r, i.e. four
  // consecutive columns of one row of C per lane.
  if (GLU) {
    bf16* act = const_cast<bf16*>(R);
    bf16* gu = reinterpret_cast<bf16*>(Cv);
    if (c_vec == 2) {
      // Whole-line stores through LDS.  A wave's 128 x 32 features are half a line per row, so the
      // block's 256 x 128 output is staged wave by wave (64-byte rows, 16-byte chunks XOR-swizzled
      // by (row >> 2) & 3) and written out by rows: wave w takes rows 32w .. 32w+31, four rows of
      // 256 B per instruction.  First act, then (when kept for the backward pass) gate and up, or,
      // in the backward form, d gate and d up.
      constexpr int REG = WM * 64;  // bytes of one wave's staging region
      // backward form: this lane's gradients of the activation output, in accumulator layout
      // (8 bytes = its 4 features of one row), requested before the barrier that they ride out
      Pack4 dd[GLU_BWD ? TM : 1][2];
      if (GLU_BWD) {
        const bf16* dact = reinterpret_cast<const bf16*>(cos_t);
        const int64_t lddact = seq_len;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < 2; j++)
            dd[i][j].u = *reinterpret_cast<const u32x2*>(dact + (int64_t)(m0 + wm * WM + i * 16 + l16e) * lddact + n0 + wn * 32 + j * 16 + g16e * 4);
      }
      __syncthreads();              // every wave is done reading the operand stages
#pragma unroll 1
      for (int pass = 0; pass < ((gu || GLU_BWD) ? 2 : 1); pass++) {
        if (pass) __syncthreads();  // the previous pass has been read back
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) {
            const int row = i * 16 + l16e;
            unsigned char* dst = smem + wave * REG + row * 64 + ((((j << 1) | (g16e >> 1)) ^ ((row >> 2) & 3)) << 4) + ((g16e & 1) << 3);
            Pack4 pa, pg, pu;
#pragma unroll
            for (int r = 0; r < 4; r++) {
              // same roundings as the unfused path: gate and up are bf16 arrays, so is f(gate)
              pg.e[r] = f2bf(acc[i][j][r]);
              pu.e[r] = f2bf(acc[i][j + 2][r]);
              const float gf = bf2f(pg.e[r]);
              const float fg = GLU == 2 ? act_gelu(gf) : act_silu(gf);
              pa.e[r] = f2bf(bf2f(f2bf(fg)) * bf2f(pu.e[r]));
              if (GLU_BWD) {  // d gate = dact * up * f'(gate), d up = dact * f(gate)
                const float df = bf2f(dd[GLU_BWD ? i : 0][j].e[r]);
                pg.e[r] = f2bf(df * bf2f(pu.e[r]) * (GLU == 2 ? act_gelu_grad(gf) : act_silu_grad(gf)));
                pu.e[r] = f2bf(df * fg);
              }
            }
            if (pass == 0) {
              *reinterpret_cast<u32x2*>(dst) = pa.u;
            } else {
              *reinterpret_cast<u32x2*>(dst) = pg.u;
              *reinterpret_cast<u32x2*>(dst + 8 * REG) = pu.u;
            }
          }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 8; t++) {
          const int row = wave * 32 + t * 4 + (lane_e >> 4), c = lane_e & 15;
          if (!stores_row(row)) continue;
          const int lrow = row & (WM - 1);
          const unsigned char* src = smem + ((row / WM) * WAVES_N + (c >> 2)) * REG + lrow * 64 + (((c & 3) ^ ((lrow >> 2) & 3)) << 4);
          if (pass == 0) {
            store8(act + (int64_t)(m0 + row) * ldr + n0 + c * 8, c * 8, *reinterpret_cast<const u32x4*>(src));
          } else {
            store8(gu + (int64_t)(m0 + row) * ldc + n0 + c * 8, c * 8, *reinterpret_cast<const u32x4*>(src));
            store8(gu + (int64_t)(m0 + row) * ldc + N + n0 + c * 8, c * 8, *reinterpret_cast<const u32x4*>(src + 8 * REG));
          }
        }
      }
      return;
    }
    if (GLU_BWD || RAG) return;  // the backward form and ragged sizes are only launched with whole-line stores
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int64_t row = m0 + wm * WM + i * 16 + l16e;
        const int col = n0 + wn * 32 + j * 16 + g16e * 4;  // first of this lane's 4 features
        Pack4 pa, pg, pu;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          // same roundings as the unfused path: gate and up are bf16 arrays, so is f(gate)
          pg.e[r] = f2bf(acc[i][j][r]);
          pu.e[r] = f2bf(acc[i][j + 2][r]);
          const float gf = bf2f(pg.e[r]);
          const float a = bf2f(f2bf(GLU == 2 ? act_gelu(gf) : act_silu(gf)));
          pa.e[r] = f2bf(a * bf2f(pu.e[r]));
        }
        if (c_vec) {
          *reinterpret_cast<u32x2*>(act + row * ldr + col) = pa.u;
          if (gu) {
            *reinterpret_cast<u32x2*>(gu + row * ldc + col) = pg.u;
            *reinterpret_cast<u32x2*>(gu + row * ldc + N + col) = pu.u;
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            act[row * ldr + col + r] = pa.e[r];
            if (gu) {
              gu[row * ldc + col + r] = pg.e[r];
              gu[row * ldc + N + col + r] = pu.e[r];
            }
          }
        }
      }
    return;
  }
  if (!OUT_F32 && c_vec) {
    // Through LDS (free now), so that C leaves in whole 128-byte lines: each wave parks its
    // WM x 64 tile as bf16 rows of 128 B (16-byte chunks swizzled like the operand tiles), reads
    // it back 16 B per lane -- 8 lanes per row -- and stores 8 full lines per instruction.  A
    // residual joins on the way out, read in the same whole-line pattern: y = bf16(bf16(A B^T) + r),
    // the two roundings of the reference's `x + linear(...)` on bf16 arrays.
    static_assert(WN == 64, "the staging layout assumes 64-column wave tiles");
    __syncthreads();  // every wave is done reading the operand stages
    unsigned char* ws = smem + wave * (WM * 128);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int row = i * 16 + l16e;
        const int chunk = j * 2 + (g16e >> 1);
        Pack4 pk;
#pragma unroll
        for (int r = 0; r < 4; r++) pk.e[r] = f2bf(acc[i][j][r]);
        *reinterpret_cast<u32x2*>(ws + row * 128 + ((chunk ^ kswz(row)) << 4) + ((g16e & 1) << 3)) = pk.u;
      }
    bf16* C = reinterpret_cast<bf16*>(Cv);
    if (ROPE && n0 < rope_cols) {  // uniform over the block: rope_cols is a multiple of 256
      // Rotation on the way out.  Every wave has staged its half-heads; now wave w takes rows
      // 32w .. 32w+31 of the whole 256-column block, two rows (2 x 512 B) per instruction, so
      // that the four lanes of a row that need the same cos/sin entry (two heads x two halves)
      // sit in one instruction and share one request: the tables cost 128 KB per block, not 512.
      __syncthreads();
#pragma unroll 4
      for (int t = 0; t < 16; t++) {
        const int row = wave * 32 + t * 2 + (lane_e >> 5);      // row of the block
        const int c32 = lane_e & 31, chunk = c32 & 7;            // 16-byte chunk of the 512-byte row
        if (!stores_row(row)) continue;
        const int lrow = row & (WM - 1);                         // row inside the staging region
        const unsigned char* own = smem + ((row / WM) * WAVES_N + (c32 >> 3)) * (WM * 128) + lrow * 128 + ((chunk ^ kswz(lrow)) << 4);
        const unsigned char* oth = smem + ((row / WM) * WAVES_N + ((c32 >> 3) ^ 1)) * (WM * 128) + lrow * 128 + ((chunk ^ kswz(lrow)) << 4);
        Pack8 xo, xp, o;
        xo.u = *reinterpret_cast<const u32x4*>(own);
        xp.u = *reinterpret_cast<const u32x4*>(oth);
        const int pos = (m0 + row) % seq_len;
        const float* cp = cos_t + (int64_t)pos * 64 + chunk * 8;
        const float* sp = sin_t + (int64_t)pos * 64 + chunk * 8;
        const f32x4 c0 = *reinterpret_cast<const f32x4*>(cp), c1 = *reinterpret_cast<const f32x4*>(cp + 4);
        const f32x4 s0 = *reinterpret_cast<const f32x4*>(sp), s1 = *reinterpret_cast<const f32x4*>(sp + 4);
        const float sign = (c32 & 8) ? 1.f : -1.f;  // first half: x1 cos - x2 sin; second: x2 cos + x1 sin
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float cs = e < 4 ? c0[e & 3] : c1[e & 3], sn = e < 4 ? s0[e & 3] : s1[e & 3];
          o.e[e] = f2bf(bf2f(xo.e[e]) * cs + sign * bf2f(xp.e[e]) * sn);
        }
        *reinterpret_cast<u32x4*>(C + (int64_t)(m0 + row) * ldc + n0 + c32 * 8) = o.u;
      }
      return;
    }
    if (HAS_RES && R) {
      Pack8 rr[WM / 8];
#pragma unroll
      for (int t = 0; t < WM / 8; t++) {  // all residual lines requested before the first is needed
        const int row = t * 8 + (lane_e >> 3), chunk = lane_e & 7;
        if (!stores_row(wm * WM + row)) continue;
        rr[t].u = *reinterpret_cast<const u32x4_u*>(R + (int64_t)(m0 + wm * WM + row) * ldr + n0 + wn * WN + chunk * 8);
      }
#pragma unroll
      for (int t = 0; t < WM / 8; t++) {
        const int row = t * 8 + (lane_e >> 3), chunk = lane_e & 7;
        if (!stores_row(wm * WM + row)) continue;
        Pack8 line, o;
        line.u = *reinterpret_cast<const u32x4*>(ws + row * 128 + ((chunk ^ kswz(row)) << 4));
#pragma unroll
        for (int e = 0; e < 8; e++) o.e[e] = f2bf(bf2f(line.e[e]) + bf2f(rr[t].e[e]));
        store8(C + (int64_t)(m0 + wm * WM + row) * ldc + n0 + wn * WN + chunk * 8, wn * WN + chunk * 8, o.u);
      }
      return;
    }
#pragma unroll
    for (int t = 0; t < WM / 8; t++) {
      const int row = t * 8 + (lane_e >> 3), chunk = lane_e & 7;
      const u32x4 line = *reinterpret_cast<const u32x4*>(ws + row * 128 + ((chunk ^ kswz(row)) << 4));
      if (stores_row(wm * WM + row)) store8(C + (int64_t)(m0 + wm * WM + row) * ldc + n0 + wn * WN + chunk * 8, wn * WN + chunk * 8, line);
    }
    return;
  }
  // element-wise stores: fp32 output, or a C / R whose alignment rules out vector accesses
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int64_t row = m0 + wm * WM + i * 16 + l16e;
      if (!stores_row(wm * WM + i * 16 + l16e)) continue;
      if (RAG && OUT_F32 && wn * WN + j * 16 + g16e * 4 >= col_lo) {  // (element by element a 2816 x 3200 x 512 takes 46 us, so 24)
        const int col = n0 + wn * WN + j * 16 + g16e * 4;
        f32x4 v = acc[i][j];
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (HAS_RES && R) v[r] += bf2f(R[row * ldr + col + r]);
        *reinterpret_cast<f32x4_u*>(reinterpret_cast<float*>(Cv) + row * ldc + col) = v;
        continue;
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int col = n0 + wn * WN + j * 16 + g16e * 4 + r;
        if (RAG && col < n0 + col_lo) continue;
        float v = acc[i][j][r];
        if (HAS_RES && R) v = (OUT_F32 ? v : bf2f(f2bf(v))) + bf2f(R[row * ldr + col]);  // bf16 output: round, add, round
        if (OUT_F32)
          reinterpret_cast<float*>(Cv)[row * ldc + col] = v;
        else
          reinterpret_cast<bf16*>(Cv)[row * ldc + col] = f2bf(v);
      }
    }
}

template <int BM, int BN, int WM, int WN, bool A_KC, bool B_KC, bool HAS_RES, bool OUT_F32, int EPI = 0, int RAG = 0>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) GEMM_VGPR_CAP void gemm_bf16_kernel(
    const bf16* __restrict__ A, const bf16* __restrict__ B, void* __restrict__ Cv,
    const bf16* __restrict__ R, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
    int64_t ldr, int tiles_m, int tiles_n, int c_vec, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, int seq_len, int rope_cols, int order) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  gemm_tile<BM, BN, WM, WN, A_KC, B_KC, HAS_RES, OUT_F32, EPI, RAG>(A, B, Cv, R, M, N, K, lda, ldb, ldc, ldr, tiles_m, tiles_n, c_vec, cos_t,
                                                                    sin_t, seq_len, rope_cols, order, blockIdx.x, gridDim.x, smem);
}

// dX = dY W (+ R) and dW = dY^T X in one launch of T x T tiles: the second starts on the CUs that the first's last round of tiles
// leaves idle.  Workgroups [0, n_first) are the product with the longer reduction (and padding up to a whole number of XCDs).
// us in a block's backward pass, two calls -> one, T x in x out: tiles of 128: 3000 x 1024 x 3072 76 -> 47, 3000 x 2816 x 1024 65 -> 42, 4096 x 1024 x 3072 92 -> 60;
// tiles of 256: 2048 x 4096 x 12288 339 -> 308, 1500 x 4096 x 28672 706 -> 601, 8192 x 1024 x 5632 199 -> 178, 8192 x 11008 x 4096 1066 -> 1008; no longer 2048 x 4096 x 22016 549 -> 555.
// 240 registers (the cap counts pairs): as in the single kernels a wave of the overlapped update fits beside two of these.
struct PairSide {
  const bf16 *A, *B, *R;
  bf16* C;
  int M, N, K;
  int64_t lda, ldb, ldc, ldr;
  int tiles_m, tiles_n, order, nwg, block;  // nwg: of one part
  int parts = 1, chunk;                     // parts of dW's reduction in 256 tiles, k of all but the last
  float* park;                              // parked blocks, or the sums of the parts
};
template <int T, int W, int RAGX, int RAGW, int BLOCKS>
__global__ __launch_bounds__((T / W) * (T / 64) * 64) __attribute__((amdgpu_num_vgpr(120))) void gemm_pair_kernel(const PairSide x, const PairSide w, int x_first, int n_first) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const bool second = (int)blockIdx.x >= n_first;
  const int pid = second ? blockIdx.x - n_first : blockIdx.x;
  if (second != (x_first != 0)) {
    if (pid >= x.nwg) return;
    gemm_tile<T, T, W, 64, true, false, true, false, 0, RAGX, BLOCKS>(x.A, x.B, x.C, x.R, x.M, x.N, x.K, x.lda, x.ldb, x.ldc, x.ldr, x.tiles_m, x.tiles_n, 1,
                                                                      nullptr, nullptr, 1, 0, x.order, pid, x.nwg, smem, x.block, x.park);
  } else {
    if (pid >= w.nwg * w.parts) return;
    const int part = T == 256 ? pid / w.nwg : 0, k = part * w.chunk;
    float* sums = T == 256 && w.parts > 1 ? w.park + (int64_t)part * w.tiles_m * w.tiles_n * 65536 : nullptr;
    gemm_tile<T, T, W, 64, false, false, false, false, 0, RAGW, BLOCKS>(w.A + k * w.lda, w.B + k * w.ldb, w.C, nullptr, w.M, w.N, part + 1 < w.parts ? w.chunk : w.K - k,
                                                                        w.lda, w.ldb, w.ldc, 0, w.tiles_m, w.tiles_n, 1, nullptr, nullptr, 1, 0, w.order,
                                                                        pid - part * w.nwg, w.nwg, smem, w.block, w.park, sums);
  }
}

std::atomic<int> g_order{0};  // diagnostic override of the tile order, process-wide: 0 automatic, -1 run order, > 0 that many strips
// How many 8-row strips of tiles the 8 XCDs' windows cover together (see the kernel), 0: the
// run order.  Measured inside the 7B train step (same box, alternating settings, per shape):
//   forward (both operands k-contiguous), weights that fit the memory-side cache: 1 strip
//     (all XCDs share the same 8 activation row panels and stream the weights): q|k|v -4.7 %;
//     a weight matrix beyond the cache (the LM head) wants every row in flight instead;
//   input gradients (dX = dY W): 2 strips, -2 % at K = 4096, -3.5 % on the LM head, else neutral;
//   weight gradients (dW = dY^T X): 4 strips, -3 % to -5 % on every shape.
// Grids that would need padded windows keep the run order (the padding costs more than it gains), and so do those whose windows the
// XCDs cannot share evenly, up to three rounds of them (4 windows keep half of the GPU from the operands: 2048 x 4096 x 4096 108 us, run
// order 100, 6144 x 4096 x 2048 as a weight gradient 108, 100; a second product in the same launch waits for the XCDs that have too many;
// 196 windows, 100352 x 4096 x 8192 as a weight gradient: 4902 us, run order 5266).
int tile_order(int tm, int tn, bool a_kc, bool b_kc, int N, int K) {
  const int o = g_order.load(std::memory_order_relaxed);
  if (o < 0) return 0;
  if (o > 0) return o;
  const int windows = tm / 8 * (tn / 4);
  if (tm % 8 || tn % 4 || (windows < 24 && windows % 8)) return 0;
  const int strips = tm / 8;
  if (a_kc && b_kc) return (int64_t)N * K * 2 <= (128ll << 20) ? 1 : (strips < 8 ? strips : 8);
  if (a_kc) return strips < 2 ? strips : 2;
  return strips < 4 ? strips : 4;
}
unsigned order_grid(int order, int tm, int tn) {
  if (order <= 0) return (unsigned)(tm * tn);
  const int nwin = ((tm + 7) / 8) * ((tn + 3) / 4);
  return (unsigned)((nwin + 7) / 8 * 256);
}

template <int BM, int BN, int WM, int WN, bool A_KC, bool B_KC, bool HAS_RES, bool OUT_F32, int RAG>
int launch_tile(hipStream_t s, const bf16* A, const bf16* B, void* C, const bf16* R, int M, int N,
                int K, int64_t lda, int64_t ldb, int64_t ldc, int64_t ldr) {
  constexpr int NT = (BM / WM) * (BN / WN) * 64;
  constexpr int SMEM = (BM != BN ? 3 : 2) * (BM + BN) * BK * 2;
  auto kern = gemm_bf16_kernel<BM, BN, WM, WN, A_KC, B_KC, HAS_RES, OUT_F32, 0, RAG>;
  static std::once_flag attr_once;  // per instantiation
  std::call_once(attr_once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM); });
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  ProfRec rec{};
  if (g_prof_on) {
    (void)hipEventCreate(&rec.e0);
    (void)hipEventCreate(&rec.e1);
    (void)hipEventRecord(rec.e0, s);
  }
  // vector epilogue: 16-byte stores to C, 16-byte loads from R
  const int c_vec = RAG || (aligned16(C) && ldc % 8 == 0 && (!R || (aligned16(R) && ldr % 8 == 0)));
  const int order = tile_order(tm, tn, A_KC, B_KC, N, K);
  hipLaunchKernelGGL(kern, dim3(order_grid(order, tm, tn)), dim3(NT), SMEM, s, A, B, C, R, M, N, K, lda, ldb, ldc,
                     ldr, tm, tn, c_vec, (const float*)nullptr, (const float*)nullptr, 1, 0, order);
  if (g_prof_on) {
    (void)hipEventRecord(rec.e1, s);
    rec.flops = 2.0 * M * N * K;
    rec.bytes = 2.0 * ((double)M * K + (double)N * K + (double)M * N * (HAS_RES ? 2 : 1) * (OUT_F32 ? 2 : 1));
    rec.key = (BM != BN ? BM + BN : BM) | (A_KC << 12) | (B_KC << 13) | (HAS_RES << 14) | (OUT_F32 << 15);
    rec.M = M; rec.N = N; rec.K = K;
    std::lock_guard<std::mutex> lk(g_prof_mu);
    g_prof.push_back(rec);
  }
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

// EPI 1 / 2: forward form (gu optional); 4 / 5: backward form (dact given, gu = d gate | d up)
template <int EPI, int RAG>
int launch_glu(hipStream_t s, const bf16* A, const bf16* B, bf16* gu, bf16* act, int M, int F, int K, int64_t lda,
               int64_t ldb, int64_t ldgu, int64_t ldact, const bf16* dact = nullptr, int64_t lddact = 0) {
  constexpr int SMEM = 2 * (256 + 256) * BK * 2;
  auto kern = gemm_bf16_kernel<256, 256, 128, 64, true, true, false, false, EPI, RAG>;
  static std::once_flag attr_once;  // per instantiation
  std::call_once(attr_once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM); });
  const int tm = (M + 255) / 256, tn = (F + 127) / 128;
  ProfRec rec{};
  if (g_prof_on) {
    (void)hipEventCreate(&rec.e0);
    (void)hipEventCreate(&rec.e1);
    (void)hipEventRecord(rec.e0, s);
  }
  // 2: 16-byte stores of whole lines through LDS; 1: 8-byte stores straight from the accumulators
  const int c_vec = (aligned16(act) && ldact % 8 == 0 && (!gu || (aligned16(gu) && ldgu % 8 == 0 && F % 8 == 0))) ? 2
                    : ((((uintptr_t)act) & 7) == 0 && ldact % 4 == 0 && (!gu || ((((uintptr_t)gu) & 7) == 0 && ldgu % 4 == 0 && F % 4 == 0)));
  const int order = tile_order(tm, tn, true, true, 2 * F, K);
  hipLaunchKernelGGL(kern, dim3(order_grid(order, tm, tn)), dim3(512), SMEM, s, A, B, (void*)gu, (const bf16*)act, M, F, K, lda, ldb,
                     ldgu, ldact, tm, tn, c_vec, reinterpret_cast<const float*>(dact), (const float*)nullptr, (int)lddact, 0, order);
  if (g_prof_on) {
    (void)hipEventRecord(rec.e1, s);
    rec.flops = 4.0 * M * F * K;
    rec.bytes = 2.0 * ((double)M * K + 2.0 * F * K + (double)M * F * ((gu ? 3 : 1) + (dact ? 1 : 0)));
    rec.key = 256 | (1 << 12) | (1 << 13) | (1 << 16);
    rec.M = M; rec.N = 2 * F; rec.K = K;
    std::lock_guard<std::mutex> lk(g_prof_mu);
    g_prof.push_back(rec);
  }
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

template <int T, int W, int RAGX, int RAGW, int BLOCKS>
void launch_pair(hipStream_t s, PairSide x, PairSide w) {
  auto kern = gemm_pair_kernel<T, W, RAGX, RAGW, BLOCKS>;
  constexpr int SMEM = 4 * T * BK * 2;
  static std::once_flag attr_once;  // per instantiation
  std::call_once(attr_once, [&] { (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM); });
  for (auto p : {&x, &w}) {
    p->tiles_m = (p->M + T - 1) / T;
    p->tiles_n = (p->N + T - 1) / T;
    p->order = p->parts > 1 ? 0 : tile_order(p->tiles_m, p->tiles_n, p == &x, false, p->N, p->K);
    p->nwg = (int)order_grid(p->order, p->tiles_m, p->tiles_n);
  }
  const bool x_first = x.K > (w.parts > 1 ? w.chunk : w.K);
  const int nx = x.nwg, nw = w.nwg * w.parts, n_first = ((x_first ? nx : nw) + 7) & ~7;
  hipLaunchKernelGGL(kern, dim3((unsigned)(n_first + (x_first ? nw : nx))), dim3((T / W) * (T / 64) * 64), SMEM, s, x, w, (int)x_first, n_first);
}

template <bool A_KC, bool B_KC, bool HAS_RES, bool OUT_F32>
int dispatch_tile(hipStream_t s, const bf16* A, const bf16* B, void* C, const bf16* R, int M, int N,
                  int K, int64_t lda, int64_t ldb, int64_t ldc, int64_t ldr, int tile) {
  if constexpr (A_KC && B_KC && !OUT_F32) {
    if (tile == THIN_TILE) {
#define TILE(RAG) launch_tile<256, 128, 64, 64, A_KC, B_KC, HAS_RES, OUT_F32, RAG>(s, A, B, C, R, M, N, K, lda, ldb, ldc, ldr)
      return K % BK ? TILE(2) : M % 256 || N % 128 ? TILE(1) : TILE(0);
#undef TILE
    }
  }
  const bool rag = M % tile || N % tile;
#define TILE(T, W, RAG) launch_tile<T, T, W, 64, A_KC, B_KC, HAS_RES, OUT_F32, RAG>(s, A, B, C, R, M, N, K, lda, ldb, ldc, ldr)
  if (tile == 256) return K % BK ? TILE(256, 128, 2) : rag ? TILE(256, 128, 1) : TILE(256, 128, 0);
  return K % BK ? TILE(128, 64, 2) : rag ? TILE(128, 64, 1) : TILE(128, 64, 0);
#undef TILE
}

std::atomic<int> g_force_tile{0};  // diagnostic override, process-wide

// C = sum of the parts, in their order (+ R), with the roundings of the kernels above.  A wave takes one
// 16 x 64 strip of a wave tile; its loads are the 1 KB runs the accumulators were stored as.  Bound by
// the reads of the parts (at most 64 MB a round of workgroups, out of the memory-side cache).
__global__ __launch_bounds__(256) void gemm_split_sum_kernel(const float* __restrict__ parts, int nparts, void* __restrict__ Cv,
                                                             const bf16* __restrict__ R, int M, int N, int64_t ldc, int64_t ldr,
                                                             int m_edge, int tiles_n, int ntiles, int out_f32, int vec) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g16 = lane >> 4;
  const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);  // (tile, wave of it, i): 64 per tile
  const int tile = unit >> 6, wave = (unit >> 3) & 7, i = unit & 7;
  const int tile_m = tile / tiles_n, tile_n = tile % tiles_n;
  const int64_t stride = (int64_t)ntiles * 65536;
  const float* src = parts + (int64_t)unit * 1024 + lane * 4;
  f32x4 v[4];
#pragma unroll
  for (int j = 0; j < 4; j++) v[j] = *reinterpret_cast<const f32x4*>(src + j * 256);
#pragma unroll 4
  for (int p = 1; p < nparts; p++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(src + p * stride + j * 256);
#pragma unroll
      for (int r = 0; r < 4; r++) v[j][r] += x[r];
    }
  // a tile moved back to end with the matrix stores only what the one before it does not
  const int64_t row = min(tile_m * 256, m_edge - 256) + (wave >> 2) * 128 + i * 16 + l16;
  if (row < tile_m * 256 || row >= M) return;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int col = min(tile_n * 256, N - 256) + (wave & 3) * 64 + j * 16 + g16 * 4, lo = tile_n * 256 - col;
    const bool whole = vec && lo <= 0;
    Pack4 rr;
    if (R && whole) rr.u = *reinterpret_cast<const u32x2*>(R + row * ldr + col);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      if (r < lo) continue;
      if (R) v[j][r] = (out_f32 ? v[j][r] : bf2f(f2bf(v[j][r]))) + bf2f(whole ? rr.e[r] : R[row * ldr + col + r]);
      if (whole) continue;
      if (out_f32) reinterpret_cast<float*>(Cv)[row * ldc + col + r] = v[j][r];
      else reinterpret_cast<bf16*>(Cv)[row * ldc + col + r] = f2bf(v[j][r]);
    }
    if (!whole) continue;
    if (out_f32) {
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(Cv) + row * ldc + col) = v[j];
    } else {
      Pack4 o;
#pragma unroll
      for (int r = 0; r < 4; r++) o.e[r] = f2bf(v[j][r]);
      *reinterpret_cast<u32x2*>(reinterpret_cast<bf16*>(Cv) + row * ldc + col) = o.u;
    }
  }
}

void launch_split_sum(hipStream_t s, const float* sums, int parts, void* C, const bf16* R, int M, int N, int64_t ldc, int64_t ldr, bool a_kc, bool out_f32) {
  const int tm = (M + 255) / 256, tn = (N + 255) / 256;
  const int vec = N % 4 == 0 && ldc % 4 == 0 && !((uintptr_t)C & (out_f32 ? 15 : 7)) && (!R || (ldr % 4 == 0 && !((uintptr_t)R & 7)));
  hipLaunchKernelGGL(gemm_split_sum_kernel, dim3((unsigned)(tm * tn * 16)), dim3(256), 0, s, sums, parts, C, R, M, N, ldc, ldr, a_kc ? M : (M + 7) & ~7, tn,
                     tm * tn, (int)out_f32, vec);
}

template <bool A_KC, bool B_KC>
int launch_split(hipStream_t s, const bf16* A, const bf16* B, void* C, const bf16* R, int M, int N, int K, int64_t lda, int64_t ldb,
                 int64_t ldc, int64_t ldr, bool out_f32, int parts, float* scratch) {
  constexpr int SMEM = 2 * (256 + 256) * BK * 2;
  auto whole = gemm_bf16_kernel<256, 256, 128, 64, A_KC, B_KC, false, true, 6, 0>;
  auto ragged = gemm_bf16_kernel<256, 256, 128, 64, A_KC, B_KC, false, true, 6, 1>;
  auto kragged = gemm_bf16_kernel<256, 256, 128, 64, A_KC, B_KC, false, true, 6, 2>;
  static std::once_flag attr_once;
  std::call_once(attr_once, [&] {
    for (auto k : {whole, ragged, kragged}) (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
  });
  auto kern = K % BK ? kragged : (M % 256 || N % 256) ? ragged : whole;
  const int tm = (M + 255) / 256, tn = (N + 255) / 256;
  const int chunk = (K / BK + parts - 1) / parts;  // whole k-tiles of a part; every part has at least one
  parts = (K / BK + chunk - 1) / chunk;
  ProfRec rec{};
  if (g_prof_on) {
    (void)hipEventCreate(&rec.e0);
    (void)hipEventCreate(&rec.e1);
    (void)hipEventRecord(rec.e0, s);
  }
  // (run order: a round of windows is 256 tiles, and here there are fewer)
  hipLaunchKernelGGL(kern, dim3(tm * tn, parts), dim3(512), SMEM, s, A, B, (void*)scratch, (const bf16*)nullptr, M, N, K, lda,
                     ldb, (int64_t)0, (int64_t)0, tm, tn, 1, (const float*)nullptr, (const float*)nullptr, chunk * BK, 0, 0);
  launch_split_sum(s, scratch, parts, C, R, M, N, ldc, ldr, A_KC, out_f32);
  if (g_prof_on) {
    (void)hipEventRecord(rec.e1, s);
    rec.flops = 2.0 * M * N * K;
    rec.bytes = 2.0 * ((double)M * K + (double)N * K + (double)M * N * (R ? 2 : 1) * (out_f32 ? 2 : 1));
    rec.key = 256 | (A_KC << 12) | (B_KC << 13) | ((R != nullptr) << 14) | (out_f32 << 15) | (1 << 18);
    rec.M = M; rec.N = N; rec.K = K;
    std::lock_guard<std::mutex> lk(g_prof_mu);
    g_prof.push_back(rec);
  }
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

}  // namespace

extern "C" void olmax_gemm_set_tile(int tile) { g_force_tile = tile; }
extern "C" void olmax_gemm_set_order(int order) { g_order = order; }

// Start recording a HIP-event pair around every MFMA GEMM launch (diagnostic; allocates events).
extern "C" void olmax_gemm_profile_begin(void) {
  std::lock_guard<std::mutex> lk(g_prof_mu);
  g_prof.clear();
  g_prof_on = true;
}
// Stop recording, wait for the recorded events and aggregate per kernel instantiation.
// keys/ms/flops/launches: host arrays of `cap` entries; returns the number of distinct keys.
// key = tile (64: gemm_small_kernel) | a_layout<<12 | b_layout<<13 | has_residual<<14 | out_f32<<15 | glu_epilogue<<16 | rope_epilogue<<17 |
// shared_reduction<<18 | both_gradients<<19 (M, N, K: T, in, out), with a_layout / b_layout bit SET when the operand is reduction-contiguous.  flops / bytes:
// algorithmic totals (2MNK; every operand and the result moved once).
extern "C" int32_t olmax_gemm_profile_end(int32_t* keys, double* ms, double* flops, double* bytes, int64_t* launches,
                                          int32_t cap) {
  std::lock_guard<std::mutex> lk(g_prof_mu);
  g_prof_on = false;
  int n = 0;
  for (auto& r : g_prof) {
    (void)hipEventSynchronize(r.e1);
    float t = 0.f;
    (void)hipEventElapsedTime(&t, r.e0, r.e1);
    int i = 0;
    for (; i < n; i++)
      if (keys[i] == r.key) break;
    if (i == n) {
      if (n >= cap) continue;
      keys[n] = r.key; ms[n] = 0; flops[n] = 0; bytes[n] = 0; launches[n] = 0;
      n++;
    }
    ms[i] += t; flops[i] += r.flops; bytes[i] += r.bytes; launches[i] += 1;
    (void)hipEventDestroy(r.e0);
    (void)hipEventDestroy(r.e1);
  }
  g_prof.clear();
  return n;
}

// As olmax_gemm_profile_end, aggregated per (key, M, N, K): mnk receives 3 ints per entry.
extern "C" int32_t olmax_gemm_profile_end_shapes(int32_t* keys, int32_t* mnk, double* ms, int64_t* launches, int32_t cap) {
  std::lock_guard<std::mutex> lk(g_prof_mu);
  g_prof_on = false;
  int n = 0;
  for (auto& r : g_prof) {
    (void)hipEventSynchronize(r.e1);
    float t = 0.f;
    (void)hipEventElapsedTime(&t, r.e0, r.e1);
    int i = 0;
    for (; i < n; i++)
      if (keys[i] == r.key && mnk[3 * i] == r.M && mnk[3 * i + 1] == r.N && mnk[3 * i + 2] == r.K) break;
    if (i == n) {
      if (n >= cap) continue;
      keys[n] = r.key; mnk[3 * n] = r.M; mnk[3 * n + 1] = r.N; mnk[3 * n + 2] = r.K; ms[n] = 0; launches[n] = 0;
      n++;
    }
    ms[i] += t; launches[i] += 1;
    (void)hipEventDestroy(r.e0);
    (void)hipEventDestroy(r.e1);
  }
  g_prof.clear();
  return n;
}

static int device_cu_count() {
  static std::atomic<int> n{0};  // every thread that finds 0 computes the same value
  int v = n.load(std::memory_order_relaxed);
  if (!v) {
    int dev = 0;
    if (!(hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)) v = 256;
    n.store(v, std::memory_order_relaxed);
  }
  return v;
}

// Estimated time (us) of each kernel on a problem of kt k-tiles, from measurements at 16 to 8192 rows
// and 256 to 11008 columns (every layout; within about 15 %) on the 256 CUs of this GPU, on warm operands: with operands from HBM and behind another product all
// of them take a quarter to a half more.  What counts is how they compare.  A k-tile costs a 256 tile 1.05 us with few tiles in flight and 1.52 us with one on every CU, and a
// round 6 us beside: the figures of the loop before its waves took turns, which every choice below was compared with.  Now it is 1.27 to 1.35 and 9.5, so that
// long reductions take up to 12 % less than priced (8192 x 22016 x 4096 1130, 1004 measured) and short ones more.  A 128 tile costs
// 0.57 us alone, 0.83 us with one on every CU and 1.08 us with the two that fit, a 64 tile 0.22 us
// per round.  Up to 32 k-tiles and one 128 tile per CU the operands of a whole product stay near: 0.40 us up to 8 k-tiles, rising to 0.6,
// sooner where B is [K, N].  us of 128 tiles | 64 tiles: 384 x 2816 x 512 6.8 | 7.6, 512 x 4096 x 1024 10.3 | 11.5 ([K, N]: 10.6 | 11.3), 256 x 5632 x 1024
// 9.9 | 10.8 (10.7 | 10.8), 2048 x 1024 x 1024 11.6 | 10.8 (12.2 | 11.2), 512 x 2816 x 2048 18.0 | 16.6 (21.6 | 16.6).  Beyond, the rates of
// whole rounds are taken: 512 x 4096 x 4096 39.8 | 28.7, 1024 x 4096 x 4096 42.9 | 50.3.
static float cost_128(int64_t n, int kt, bool b_kc) {
  auto part = [&](int64_t r) {
    float f = r <= 64 ? 0.57f : r <= 256 ? 0.57f + 0.26f * (r - 64) / 192.f : 0.83f + 0.25f * (r - 256) / 256.f;
    if (kt <= 32 && r <= 256) f = kt <= 8 ? 0.4f : std::min(0.6f, 0.4f + (b_kc ? 0.0075f : 0.014f) * (kt - 8));
    return f * kt + 4.f;
  };
  return (n / 512) * (1.08f * kt + 4.f) + (n % 512 ? part(n % 512) : 0.f);
}
// n tiles of 256, their reductions shared by s workgroups each; a part costs 256 KB written and read again
static float cost_split(int64_t n, int kt, int s) {
  const int64_t w = n * s, r = w % 256;
  const int k = (kt + s - 1) / s;
  return (w / 256) * (1.52f * k + 6.f) + (r ? (1.05f + 0.47f * r / 256.f) * k + 6.f : 0.f) + 6.f + 0.1f * w;
}
// The cheapest number of parts (1: whole reductions) that `bytes` of scratch hold.  A part has 8 k-tiles or more.
static int pick_parts(int64_t n, int kt, int64_t bytes, float* cost) {
  int best = 1;
  for (int s = 2; s <= 64 && s * 8 <= kt && n * s <= 512 && n * s * 262144 <= bytes; s++)
    if (const float c = cost_split(n, kt, s); c < *cost) *cost = c, best = s;
  return best;
}
// n tiles of 256, the last round's at what it costs as a round
static float cost_rounds(int64_t n, int kt) {
  const int64_t r = n % 256;
  return (n / 256) * (1.52f * kt + 6.f) + (r ? (1.05f + 0.47f * r / 256.f) * kt + 6.f : 0.f);
}
static float cost_256(int64_t n, int kt, int64_t bytes, bool b_kc) {
  const int64_t r = n % 256;
  // (a last round that fills less than half of the CUs is cut off and runs as 128 tiles or shared reductions)
  if (n <= 256 || r == 0 || r >= 128) return cost_rounds(n, kt);
  float last = std::min(cost_rounds(r, kt), cost_128(4 * r, kt, b_kc));
  (void)pick_parts(r, kt, bytes, &last);
  return cost_rounds(n - r, kt) + last;
}
static float cost_64(int64_t n, int kt) { return ((n + 255) / 256) * (0.22f * kt + 1.2f) + 2.4f; }
// 32 tiles: 0.165 us per k-tile while each has a CU, 0.235 (0.30 where A is [K, M], whose lines are then 64 bytes) with two on every CU; from 1024 on
// 0.8 us for each further 512, so that larger tiles take many short ones (us in 32 tiles, and so: 8191 x 4099 x 64 54, 24; 2048 x
// 1024 x 16 6.7, 5.6; but 1024 x 1024 x 16 4.4, 4.9).
static float cost_32(int64_t n, int kt, bool a_kc) {
  const float two = a_kc ? 0.235f : 0.30f;
  if (n <= 512) return 3.6f + kt * (n <= 256 ? 0.165f : 0.165f + (two - 0.165f) * (n - 256) / 256.f);
  return 3.6f + two * kt * n / 512.f + (n > 1024 ? 0.8f * (n - 1024) / 512.f : 0.f);
}
static int64_t tiles_of(int M, int N, int t) { return (int64_t)((M + t - 1) / t) * ((N + t - 1) / t); }
static float cost_small(int M, int N, int kt, bool a_kc) { return std::min(cost_64(tiles_of(M, N, 64), kt), cost_32(tiles_of(M, N, 32), kt, a_kc)); }

// Which kernel takes a problem.  0: gemm_small (any size and alignment), else the edge of the
// direct-to-LDS kernel's tiles; *parts > 1: 256 tiles with that many workgroups to a reduction.  *cost: what it is expected to take.
static int pick_tile(int M, int N, int K, bool a_kc, bool b_kc, bool direct_ok, int64_t bytes, int* parts, float* cost) {
  *parts = 1;
  const int kt = (K + BK - 1) / BK;
  float& best = *cost;
  best = cost_small(M, N, kt, a_kc);
  if (!direct_ok || M < 128 || N < 128 || K < BK) return 0;
  auto tiles = [&](int t) { return tiles_of(M, N, t); };
  int tile = 0;
  if (const float c = cost_128(tiles(128), kt, b_kc); c < best) best = c, tile = 128;
  if (M < 256 || N < 256) return tile;
  if (const float c = cost_256(tiles(256), kt, bytes, b_kc); c < best) best = c, tile = 256;
  *parts = pick_parts(tiles(256), K / BK, bytes, &best);
  return *parts > 1 ? 256 : tile;
}
// What gemm_small runs a problem in: the edge of its tiles and the waves that share a tile's reduction.
struct SmallForm {
  int edge, groups;
};
static SmallForm small_form(int M, int N, int K, bool a_kc, bool b_kc, bool forced) {
  const int64_t n64 = tiles_of(M, N, 64), n32 = tiles_of(M, N, 32);
  const int kt = (K + BK - 1) / BK;
  // (the 0.6 us: one round of 64 tiles, measured at 4 to 128 k-tiles; pick_tile's boundaries were measured without)
  // Part of one k-tile, 64 tiles that two workgroups a CU take in one round: 900 x 1800 x 16 5.8 us in 32 tiles, 5.1 in 64, 1200 x 1200 x 56 5.5 and 4.9.
  // (With more or fewer of them 32 tiles win, 1500 x 1500 x 16 7.2 and 7.9, 1024 x 1024 x 16 3.8 and 4.4, and where chunks cross the end of a line,
  // 1100 x 1100 x 56 with B [K, N] 6.6 and 7.6.)
  const bool one_round = K < BK && n64 > 256 && n64 <= 512 && (a_kc || M % 8 == 0) && (b_kc || N % 8 == 0);
  const int edge = !forced && !one_round && cost_32(n32, kt, a_kc) < cost_64(n64, kt) + 0.6f ? 32 : 64;
  // eight waves share a tile while there are not more 64 tiles than CUs, else two workgroups fit a CU.  (A 32 tile does as well with four, 300 x 1024 x 2816
  // 11.0 us against 11.6, but a chain of fp32 additions twice as long is 7 to 29 % further from the exact sum; up to four k-tiles there is none.)
  return {edge, n64 <= 256 && (edge == 64 || kt > 4) ? 8 : 4};
}
// Whether the direct-to-LDS kernels can take the operands: whole 16-byte chunks everywhere, i.e. aligned rows, and a chunk never crosses the end
// of a row (a_padded: see olmax_gemm_padded).
static bool direct(const bf16* a, const bf16* b, int M, int N, int K, int64_t lda, int64_t ldb, bool a_kc, bool b_kc, bool a_padded) {
  return aligned16(a) && aligned16(b) && lda % 8 == 0 && ldb % 8 == 0 && (a_padded || (a_kc ? K : M) % 8 == 0) && (b_kc ? K : N) % 8 == 0;
}

// Wave quantisation: with one 256x256 tile per CU per round, a last round that fills less
// than half of the CUs (e.g. 1376 tiles = 5.375 rounds on 256 CUs) costs a whole round.
// Such a problem is cut along M or N into a part whose tile count is a whole number of
// rounds and a remainder that is dispatched again (and gets smaller tiles).
struct Cut {
  int rm = 0, cn = 0;  // largest row-tile / column-tile counts giving whole rounds, 0: none
};
static Cut find_cut(int tm, int tn) {
  Cut c;
  const int ncu = device_cu_count();
  const int64_t tiles = (int64_t)tm * tn;
  const int rem = (int)(tiles % ncu);
  if (!(tiles > ncu && rem > 0 && rem * 2 < ncu)) return c;
  for (int x = tm - 1; x > 0; x--) if (((int64_t)x * tn) % ncu == 0) { c.rm = x; break; }
  for (int x = tn - 1; x > 0; x--) if (((int64_t)x * tm) % ncu == 0) { c.cn = x; break; }
  return c;
}

// Whether a fused form, which runs in 256 tiles and is never cut, is worth more than the plain product X [M, K] W [N, K]^T followed by
// elementwise passes of `passes` us; its epilogue costs `per_round` us more than the plain one's.  On whole tiles it is.  Ragged rows
// leave up to half of a row of tiles unused, and there the plain product may have the better tiles.  us, fused | two steps, of a gated projection
// with gate|up kept: 384 x 8192 x 2048 (M, F, K) 46 | 33, 896 x 9216 x 2304 109 | 74, 1300 x 5632 x 2048 98 | 67, 2176 x 8192 x 2048 158 | 136; 1500 x 14336 x 4096
// 317 | 318, 5000 x 8192 x 2048 281 | 303.  Over 133 measured sizes the time lost against the better of the two, in calls: 6.5 always fused, 0.5
// with this rule (without gate|up 4.0 and 0.4, backward form 3.0 and 0.4; rotary projection, 70 sizes, 2.1 and 0.03).
static bool fused_wins(int M, int N, int K, float per_round, float passes) {
  if (M % 256 == 0) return true;
  const int kt = K / BK, tm = (M + 255) / 256, tn = N / 256;
  const int64_t n = (int64_t)tm * tn;
  auto tiles = [&](int t) { return (int64_t)((M + t - 1) / t) * (N / t); };
  const Cut cut = find_cut(tm, tn);
  float plain = std::min(cost_small(M, N, kt, true), cost_128(tiles(128), kt, true));
  plain = std::min(plain, cut.rm || cut.cn ? cost_256(n, kt, 0, true) : cost_rounds(n, kt));
  return cost_rounds(n, kt) + per_round * ((n + 255) / 256) <= plain + passes;
}
// Fp32 additions behind one another in a result, an MFMA counted as one: of n chains of `steps` k-tiles each that are added up,
static int chain_of_parts(int n, int steps) { return 2 * steps + (n > 1 ? n : 0); }
// of olmax_gemm_padded (the shortest of its parts where it cuts a problem),
static int chain_of_product(int M, int N, int K, bool a_kc, bool b_kc, bool direct_ok, int64_t bytes) {
  const int kt = (K + BK - 1) / BK;
  int parts;
  float cost;
  const int tile = pick_tile(M, N, K, a_kc, b_kc, direct_ok, bytes, &parts, &cost);
  if (parts > 1) return chain_of_parts(parts, (kt + parts - 1) / parts);
  if (tile == 0) {
    const int g = std::min(kt, small_form(M, N, K, a_kc, b_kc, false).groups);
    return chain_of_parts(g, (kt + g - 1) / g);
  }
  if (tile == 256) {
    const int tm = (M + 255) / 256, tn = (N + 255) / 256;
    const Cut cut = find_cut(tm, tn);
    auto part = [&](int m, int n) { return chain_of_product(m, n, K, a_kc, b_kc, direct_ok, bytes); };
    if (cut.rm || cut.cn) {
      const int m1 = cut.rm * 256, n1 = cut.cn * 256;
      return (int64_t)cut.rm * tn >= (int64_t)cut.cn * tm ? std::min(part(m1, N), part(M - m1, N)) : std::min(part(M, n1), part(M, N - n1));
    }
  }
  return chain_of_parts(1, kt);
}
// and of the small tiles in the one launch of both gradients (see olmax_gemm_small_pair).
static int chain_of_small_pair(int M, int N, int K) {
  const int kt = (K + BK - 1) / BK;
  const int g = std::min(kt, tiles_of(M, N, 64) <= 256 ? 8 : 4);
  return chain_of_parts(g, (kt + g - 1) / g);
}

// Blocks of k-tiles (gemm_tile) that keep a chain to `most` additions: as few and large as that allows, of an even number of k-tiles; 0: none do.
static int block_of(int kt, int most) {
  for (int n = 1;; n++) {
    const int b = ((kt + n - 1) / n + 1) & ~1;
    if (chain_of_parts((kt + b - 1) / b, std::min(kt, b)) <= most) return b;
    if (b == 2) return 0;
  }
}

// Whether a forward product that pick_tile gave to 128 tiles runs in 256 x 128 ones instead, while each of these has a CU of its own (the chains of additions are
// the same).  Both are bound by operand delivery.  us, 128 tiles -> so, behind another product and with operands from HBM, where some CUs get two tiles of 128: 8192 x 1024 x
// 2816 59.5 -> 48.6, 1000 x 6144 x 4096 76 -> 58, 1500 x 4096 x 4096 64 -> 58, 4096 x 1280 x 4096 62 -> 59, 448 x 9152 x 9152 240 -> 196; of 650 such measurements, K 2048 to 16384,
// the mean is 8 % less, 17 are 3 to 6 % more and one 14 % (2500 x 2304 x 16384 225 -> 262).  Where each has one, half of the CUs are left with
// nothing, and only a wide product, whose weights are then read half as often, is worth that: N >= 2 M and 96 such tiles or more 1000 x 4096 x 4096 59.7 -> 56.6, 768 x 5248 x 6336 105
// -> 91, 300 sizes 5 % less on average, 5 % more at most; others 2048 x 2048 x 2816 43.6 -> 45.0, 8192 x 512 x 11008 157 -> 166, 2048 x 2048 x 4096 59.1 -> 57.2, 2 % more on average.  A partial
// k-tile costs more here: 1500 x 4096 x 4104 84.5 -> 89.7, x 2056 47.9 -> 50.0, narrow products 8 % on average, wide ones with up to 288 tiles of 128 3 %; beyond they still gain 9 %
// (1064 x 5504 x 9144 213 -> 195).  Of short reductions 3000 x 1024 x 1024 14.0 -> 14.2.  (B stored [K, N]: 8 % at best; both operands so: up to 20 % slower, as the transposing reads
// fill LDS.)
static bool thin_takes(int M, int N, int K, int tile) {
  const int64_t n = (int64_t)((M + 255) / 256) * ((N + 127) / 128), n128 = tiles_of(M, N, 128);
  if (tile != 128 || M < 256 || K < 32 * BK || n > 256) return false;
  const bool wide = N >= 2 * (int64_t)M;
  return K % BK ? wide && n128 > 288 : n128 > 256 || (wide && n >= 96);
}

enum GluForm { GLU_SAVE, GLU_ONLY, GLU_BWD };
static bool glu_fused_wins(int M, int F, int K, GluForm form) {
  const float e = (float)M * F;  // the elementwise passes move 6 (backward: 16) bytes an element at 5 TB/s
  return fused_wins(M, 2 * F, K, form == GLU_SAVE ? 6.5f : form == GLU_ONLY ? 2.5f : 9.f, form == GLU_BWD ? 5.f + e * 3e-6f : 2.5f + e * 1.2e-6f);
}

// olmax_gemm_bf16 behind its argument checks.  a_padded: rows of A may be read up to the next multiple
// of 8 elements (row stride permitting), and for a k-contiguous A those elements are zeros: what
// lets an operand whose row length is not a multiple of 8 use 16-byte fetches.
int olmax_gemm_padded(hipStream_t stream, const bf16* a, const bf16* b, void* C, const bf16* r, int M, int N, int K,
                      int64_t lda, int64_t ldb, int64_t ldc, int64_t ldr, bool a_kc, bool b_kc, bool out_f32, bool a_padded,
                      GemmScratch scratch) {
  const bool direct_ok = direct(a, b, M, N, K, lda, ldb, a_kc, b_kc, a_padded);
  const int force_tile = g_force_tile.load(std::memory_order_relaxed);
  int parts;
  float cost;
  if ((b_kc && !a_kc) || force_tile || !aligned16(scratch.p)) scratch = GemmScratch();  // (no caller has that layout)
  int tile = pick_tile(M, N, K, a_kc, b_kc, direct_ok, scratch.bytes, &parts, &cost);
  if (a_kc && b_kc && !out_f32 && !force_tile && thin_takes(M, N, K, tile)) tile = THIN_TILE;
  if (parts > 1) {
    auto go = !a_kc ? launch_split<false, false> : b_kc ? launch_split<true, true> : launch_split<true, false>;
    return go(stream, a, b, C, r, M, N, K, lda, ldb, ldc, ldr, out_f32, parts, (float*)scratch.p);
  }
  if (force_tile && direct_ok && K >= BK) {  // whatever the rule chose, if the problem has a tile of that size
    if (force_tile == 256 && M >= 256 && N >= 256) tile = 256;
    if (force_tile == 128 && M >= 128 && N >= 128) tile = 128;
    if (force_tile == THIN_TILE && M >= 256 && N >= 128 && a_kc && b_kc && !out_f32) tile = THIN_TILE;
  }
  if (tile == 256 && !force_tile) {
    const Cut cut = find_cut((M + 255) / 256, (N + 255) / 256);
    if (cut.rm || cut.cn) {
      const int64_t rows = (int64_t)cut.rm * ((N + 255) / 256), cols = (int64_t)cut.cn * ((M + 255) / 256);
      const size_t esz = out_f32 ? 4 : 2;
      if (rows >= cols) {
        const int m1 = cut.rm * 256;
        int rc = olmax_gemm_padded(stream, a, b, C, r, m1, N, K, lda, ldb, ldc, ldr, a_kc, b_kc, out_f32, a_padded, scratch);
        if (rc) return rc;
        const bf16* a2 = a_kc ? a + (int64_t)m1 * lda : a + m1;
        return olmax_gemm_padded(stream, a2, b, (char*)C + (int64_t)m1 * ldc * esz, r ? r + (int64_t)m1 * ldr : nullptr,
                                 M - m1, N, K, lda, ldb, ldc, ldr, a_kc, b_kc, out_f32, a_padded, scratch);
      }
      const int n1 = cut.cn * 256;
      int rc = olmax_gemm_padded(stream, a, b, C, r, M, n1, K, lda, ldb, ldc, ldr, a_kc, b_kc, out_f32, a_padded, scratch);
      if (rc) return rc;
      const bf16* b2 = b_kc ? b + (int64_t)n1 * ldb : b + n1;
      return olmax_gemm_padded(stream, a, b2, (char*)C + (int64_t)n1 * esz, r ? r + n1 : nullptr, M, N - n1, K, lda,
                               ldb, ldc, ldr, a_kc, b_kc, out_f32, a_padded, scratch);
    }
  }
  if (tile == 0) {
    ProfRec rec{};
    if (g_prof_on) {
      (void)hipEventCreate(&rec.e0);
      (void)hipEventCreate(&rec.e1);
      (void)hipEventRecord(rec.e0, stream);
    }
    const SmallForm f = small_form(M, N, K, a_kc, b_kc, force_tile != 0);
    olmax_gemm_small(stream, a, b, C, r, M, N, K, lda, ldb, ldc, ldr, a_kc, b_kc, out_f32, f.edge, f.groups);
    if (g_prof_on) {
      (void)hipEventRecord(rec.e1, stream);
      rec.flops = 2.0 * M * N * K;
      rec.bytes = 2.0 * ((double)M * K + (double)N * K + (double)M * N * (r ? 2 : 1) * (out_f32 ? 2 : 1));
      rec.key = 64 | (a_kc << 12) | (b_kc << 13) | ((r != nullptr) << 14) | (out_f32 << 15);
      rec.M = M; rec.N = N; rec.K = K;
      std::lock_guard<std::mutex> lk(g_prof_mu);
      g_prof.push_back(rec);
    }
    OLMAX_LAUNCH_CHECK();
    return OLMAX_OK;
  }
#define GO(AK, BKC)                                                                              \
  do {                                                                                           \
    if (r) {                                                                                     \
      if (out_f32) return dispatch_tile<AK, BKC, true, true>(stream, a, b, C, r, M, N, K, lda, ldb, ldc, ldr, tile); \
      return dispatch_tile<AK, BKC, true, false>(stream, a, b, C, r, M, N, K, lda, ldb, ldc, ldr, tile);             \
    } else {                                                                                     \
      if (out_f32) return dispatch_tile<AK, BKC, false, true>(stream, a, b, C, r, M, N, K, lda, ldb, ldc, ldr, tile); \
      return dispatch_tile<AK, BKC, false, false>(stream, a, b, C, r, M, N, K, lda, ldb, ldc, ldr, tile);            \
    }                                                                                            \
  } while (0)
  if (a_kc && b_kc) GO(true, true);
  if (a_kc) GO(true, false);
  if (b_kc) GO(false, true);
  GO(false, false);
#undef GO
}

// The two products of olmax_gemm_grads as one launch: what it costs in each kernel that can run it.  Measured, with the two calls, on 312
// sizes (T 130 to 8192, widths 256 to 28672): the least of these estimates and of the calls' takes 11 % less than the calls, the best 13 %;
// what it loses where the calls were better is 4 % at most.
// With chains as short as the calls' and with 64 MB of scratch memory or none (T 64 to 8192, widths 256 to 73728): the 534 that take it are 20 % faster
// on average, seven are slower, by 5.5 % at most (1000 x 5376 x 5376 125 us, 119).
struct Work {
  int64_t n;  // tiles
  int kt;
};
// 64 and 32 tiles in 4-wave workgroups, two of which fit a CU: their k-tiles with every CU busy, or the longer of the two chains; 64 tiles alone
// that need a few more than one round of them end unevenly (1700 x 1024 x 1024, 688 of them: 22.7 us, two calls 21.6)
static float pair_small(int T, int in, int out) {
  int64_t n64 = 0;
  auto part = [&](int M, int N, int K, float* chain) {
    const int kt = (K + BK - 1) / BK;
    const int64_t n32 = tiles_of(M, N, 32), n = n32 <= 256 ? n32 : tiles_of(M, N, 64);
    n64 += n32 <= 256 ? 1024 : n;
    *chain = std::max(*chain, n32 <= 256 ? 3.6f + 0.165f * kt : 4.2f + 0.22f * kt);
    return n * ((n32 <= 256 ? 0.00046f : 0.00086f) * kt + 0.0047f);
  };
  float chain = 0.f;
  const float work = part(T, in, out, &chain) + part(out, in, T, &chain) + 3.5f;
  return std::max(work, chain) / (n64 > 512 && n64 < 800 ? 0.82f : 0.9f);
}
// 128 tiles, 512 at a time: 1 us per k-tile of each, 17 % more where they end unevenly; or the long chains, beside the others and then alone
static float pair_128(Work l, Work s) {
  const int64_t n = l.n + s.n;
  const float work = (float)(l.n * l.kt + s.n * s.kt) / 512 * (n < 800 ? 1.17f : 1.f) + 4.f * n / 512 + 2.f;
  const float both = std::min((float)l.kt, s.n * (s.kt + 4.f) / std::max<int64_t>(1, 512 - l.n));
  const float alone = l.n <= 128 ? 0.62f : l.n <= 256 ? 0.62f + 0.25f * (l.n - 128) / 128 : 0.87f;
  return std::max(work, 1.08f * both + alone * (l.kt - both) + 4.f) / 0.96f;
}
// 256 tiles, one on a CU: the long ones in rounds, the short ones on the CUs that the last of these leaves, then on all
static float pair_256(Work l, Work s) {
  const int64_t n = l.n + s.n, r = l.n % 256;
  const float f = n >= 256 ? 1.52f : 1.05f + 0.47f * n / 256, a = f * l.kt + 6.f, b = f * s.kt + 6.f;
  const float t0 = (l.n / 256) * a, t1 = r ? t0 + a : t0;  // the first and the last CU is free for short ones
  auto early = [&](float t) { return t <= t0 ? 0 : (int64_t)((t - t0) / b + 1e-3f); };  // short ones that a CU has ended by t
  auto late = [&](float t) { return t <= t1 ? 0 : (int64_t)((t - t1) / b + 1e-3f); };
  auto done = [&](float t) { return (256 - r) * early(t) + r * late(t); };
  float t = t1;
  while (done(t) < s.n) t = std::min(t0 + (early(t) + 1) * b, t1 + (late(t) + 1) * b);
  if (n >= 256) {  // the last ones have less company
    const float busy = std::min(1.f, (s.n - done(t - b) + (r && t - b < t1 ? r : 0)) / 256.f);
    t = std::max(t1, t - b + (1.05f + 0.47f * busy) * s.kt + 6.f);
  }
  return t / 0.97f;
}

// Both products in 256 tiles.  The few tiles of a narrow layer's dW have long chains, which the calls share among workgroups: here dW's reduction comes in
// `parts` (workgroups of their own, the sums added by a second kernel), or is whole and parks the sums of its blocks.  What costs the least among
// those whose chains are as short as the calls' and whose sums fit.  us in a training step, the better of two calls and 128 tiles -> so: 8192 x 1024 x 5632 195 ->
// 172 (parked), 8192 x 1024 x 3072 115 -> 104, 8192 x 2816 x 1024 117 -> 109 (five parts), 8192 x 1024 x 1024 61 -> 45 (eight).  dW of more tiles than CUs
// fills the GPU by itself: parked, 8192 x 4096 x 22016 takes 2070 us, two calls 1930.  The 0.89 is the present loop against the one that pair_256 prices (see cost_128): it
// is here, where the forms with sums were fitted, and not in the price of the form without, which was compared as it is.  Against 128 tiles in one launch, 230 products of drawn blocks (width
// 512 to 2560, 2000 to 8300 tokens) that take 256 tiles: 16 % less time on average, 208 faster, 15 slower by 2 to 14 %, half of them T x 2816 x 1024 of 5100 to 7800 tokens (6272: 79 -> 84).  T x 512 x
// 4096 varies with where the buffers lie (8027: 128 tiles 88 to 92, this 91 to 107, once 150).
struct PairPlan {
  int parts = 1;
  float cost = 1e30f;
};
static int64_t parked_of(Work v, int block) { return block >= v.kt ? 0 : ((v.kt + block - 1) / block - 1) * v.n; }  // of 256 KB
static PairPlan plan_256(Work x, Work w, int whole_w, int chain_w, int block_x, int block_w, int64_t bytes) {
  PairPlan best;
  for (int p = 1; block_x && (p == 1 || (p <= 8 && w.n * p <= 256)); p++) {
    const int chunk = (whole_w + p - 1) / p;  // whole k-tiles of a part, eight or more; the last one takes what is left, one at least, and a partial one
    const int longest = (w.kt + p - 1) / p;   // that partial one counted: chunk, or one more where the parts come out even
    if (p == 1 ? !block_w || (block_w < w.kt && w.n > 256) : p * 8 > whole_w || (whole_w + chunk - 1) / chunk != p || chain_of_parts(p, longest) > chain_w) continue;
    const int64_t sums = p > 1 ? w.n * p : parked_of(w, block_w);
    if ((sums + parked_of(x, block_x)) * 262144 > bytes) continue;
    const Work part = {w.n * p, longest};
    float c = x.kt > part.kt ? pair_256(x, part) : pair_256(part, x);
    if (sums) c = 0.89f * c + 0.1f * sums + (p > 1 ? 6.f : 0.f);
    if (c < best.cost) best = {p, c};
  }
  return best;
}

int olmax_gemm_grads(hipStream_t s, const bf16* dy, const bf16* w, const bf16* x, bf16* dx, const bf16* r, void* dw, int T, int in, int out,
                     int64_t lddy, int64_t ldw, int64_t ldx, int64_t lddx, int64_t ldr, int64_t lddw, bool dw_f32, bool dy_padded, GemmScratch scratch) {
  // what the kernels that take the operands need one after the other
  const int64_t bytes = aligned16(scratch.p) ? scratch.bytes : 0;
  const bool direct_x = direct(dy, w, T, in, out, lddy, ldw, true, false, dy_padded), direct_w = direct(dy, x, out, in, T, lddy, ldx, false, false, dy_padded);
  int parts;
  float best, best_w;
  (void)pick_tile(T, in, out, true, false, direct_x, bytes, &parts, &best);
  (void)pick_tile(out, in, T, false, false, direct_w, bytes, &parts, &best_w);
  best += best_w;
  // One launch may not be less precise: no chain of additions longer than the calls', which may have several waves or workgroups to a reduction.
  const int chain_x = chain_of_product(T, in, out, true, false, direct_x, bytes), chain_w = chain_of_product(out, in, T, false, false, direct_w, bytes);
  const int ktx = (out + BK - 1) / BK, ktw = (T + BK - 1) / BK, block_x = block_of(ktx, chain_x), block_w = block_of(ktw, chain_w);
  const bool whole = block_x >= ktx && block_w >= ktw;
  int tile = 0;  // of the one launch, 0: two calls
  // (the one form of the small kernel that is built: whole chunks, 32-bit line offsets and at least a tile of rows)
  const bool small = !dw_f32 && out % 8 == 0 && in % 8 == 0 && T >= 64 && lddy < (1 << 25) && ldw < (1 << 25) && ldx < (1 << 25);
  if (const float c = pair_small(T, in, out); small && c < best && chain_of_small_pair(T, in, out) <= chain_x && chain_of_small_pair(out, in, T) <= chain_w)
    best = c, tile = 64;
  // vector stores, whole k-tiles in the first product
  const bool large = !dw_f32 && direct_x && direct_w && out % BK == 0 && lddx % 8 == 0 && lddw % 8 == 0 && (!r || (ldr % 8 == 0 && aligned16(r))) &&
                     aligned16(dx) && aligned16(dw);
  PairPlan plan;
  if (large && T >= 128 && in >= 128 && out >= 128 && block_x && block_w) {
    const Work wx = {tiles_of(T, in, 128), ktx}, ww = {tiles_of(out, in, 128), ktw};
    if (const float c = wx.kt > ww.kt ? pair_128(wx, ww) : pair_128(ww, wx); c < best) best = c, tile = 128;
  }
  if (large && T >= 256 && in >= 256 && out >= 256) {
    plan = plan_256({tiles_of(T, in, 256), ktx}, {tiles_of(out, in, 256), ktw}, T / BK, chain_w, block_x, block_w, bytes);
    if (plan.cost < best) best = plan.cost, tile = 256;
  }
  // dW may take the place of W or of the residual, which the first product alone reads: not beside it
  auto meet = [](const void* p, int64_t n, const void* q, int64_t m) { return p && q && (uintptr_t)p < (uintptr_t)q + m && (uintptr_t)q < (uintptr_t)p + n; };
  const int64_t dw_bytes = ((out - 1) * lddw + in) * (dw_f32 ? 4 : 2);
  if (meet(dw, dw_bytes, w, ((out - 1) * ldw + in) * 2) || meet(dw, dw_bytes, r, ((T - 1) * ldr + in) * 2)) tile = 0;
  if (tile && !g_force_tile.load(std::memory_order_relaxed)) {
    ProfRec rec{};
    if (g_prof_on) {
      (void)hipEventCreate(&rec.e0);
      (void)hipEventCreate(&rec.e1);
      (void)hipEventRecord(rec.e0, s);
    }
    if (tile != 256) plan.parts = 1;
    if (tile == 64) {
      olmax_gemm_small_pair(s, dy, w, x, dx, r, (bf16*)dw, T, in, out, lddy, ldw, ldx, lddx, ldr, lddw);
    } else {
      PairSide px = {dy, w, r, dx, T, in, out, lddy, ldw, lddx, ldr}, pw = {dy, x, nullptr, (bf16*)dw, out, in, T, lddy, ldx, lddw, 0};
      px.block = block_x;
      pw.parts = plan.parts;  // (one in 128 tiles)
      pw.chunk = (T / BK + pw.parts - 1) / pw.parts * BK;  // the last part takes what is left, at least a whole k-tile
      pw.block = pw.parts > 1 ? ktw : block_w;
      px.park = (float*)scratch.p;
      pw.park = px.park + parked_of({tiles_of(T, in, 256), ktx}, block_x) * 65536;
      const bool rx = T % tile || in % tile;
      const int rw = T % BK ? 2 : out % tile || in % tile;
#define PAIR(E, W, B)                                                                                                           \
  do {                                                                                                                          \
    if (rx) rw == 2 ? launch_pair<E, W, 1, 2, B>(s, px, pw) : rw ? launch_pair<E, W, 1, 1, B>(s, px, pw) : launch_pair<E, W, 1, 0, B>(s, px, pw); \
    else rw == 2 ? launch_pair<E, W, 0, 2, B>(s, px, pw) : rw ? launch_pair<E, W, 0, 1, B>(s, px, pw) : launch_pair<E, W, 0, 0, B>(s, px, pw);    \
  } while (0)
      if (tile == 128 && !whole) PAIR(128, 64, 1);
      else if (tile == 128) PAIR(128, 64, 0);
      else if (block_x >= ktx && pw.block >= ktw) PAIR(256, 128, 0);
      else PAIR(256, 128, 2);
#undef PAIR
      if (pw.parts > 1) launch_split_sum(s, pw.park, pw.parts, dw, nullptr, out, in, lddw, 0, false, false);
    }
    if (g_prof_on) {
      (void)hipEventRecord(rec.e1, s);
      rec.flops = 4.0 * T * in * out;
      rec.bytes = 2.0 * ((double)T * out + 2.0 * T * in + (r ? 1.0 * T * in : 0.0) + 2.0 * in * out);
      rec.key = tile | ((r != nullptr) << 14) | (1 << 19);
      rec.M = T; rec.N = in; rec.K = out;
      std::lock_guard<std::mutex> lk(g_prof_mu);
      g_prof.push_back(rec);
    }
    OLMAX_LAUNCH_CHECK();
    return OLMAX_OK;
  }
  const int rc = olmax_gemm_padded(s, dy, w, dx, r, T, in, out, lddy, ldw, lddx, ldr, true, false, false, dy_padded, scratch);
  return rc ? rc : olmax_gemm_padded(s, dy, x, dw, nullptr, out, in, T, lddy, ldx, lddw, 0, false, false, dw_f32, dy_padded, scratch);
}

extern "C" int32_t olmax_gemm_bf16(hipStream_t stream, const void* A, const void* B, void* C,
                                   const void* R, int32_t M, int32_t N, int32_t K, int64_t lda,
                                   int64_t ldb, int64_t ldc, int64_t ldr, int32_t a_layout,
                                   int32_t b_layout, int32_t out_f32) {
  OLMAX_CHECK(A && B && C, OLMAX_ERR_ARG, "olmax_gemm_bf16: null operand");
  OLMAX_CHECK(M > 0 && N > 0 && K > 0, OLMAX_ERR_SHAPE, "olmax_gemm_bf16: M,N,K must be positive (got %d,%d,%d)", M, N, K);
  OLMAX_CHECK((a_layout == 0 || a_layout == 1) && (b_layout == 0 || b_layout == 1), OLMAX_ERR_ARG,
              "olmax_gemm_bf16: layout flags must be 0 (reduction-contiguous) or 1");
  const bool a_kc = a_layout == 0, b_kc = b_layout == 0;
  OLMAX_CHECK(lda >= (a_kc ? K : M) && ldb >= (b_kc ? K : N) && ldc >= N && (!R || ldr >= N),
              OLMAX_ERR_SHAPE, "olmax_gemm_bf16: leading dimension smaller than row length");
  return olmax_gemm_padded(stream, (const bf16*)A, (const bf16*)B, C, (const bf16*)R, M, N, K, lda, ldb, ldc, ldr, a_kc, b_kc,
                           out_f32 != 0, false);
}

extern "C" int32_t olmax_qk_rope_fwd(hipStream_t stream, const void* x, void* y, const void* w, const float* cos_t,
                                     const float* sin_t, int64_t tokens, int32_t heads, int32_t head_dim, int32_t seq_len,
                                     int64_t ldx, int64_t ldy, float eps);

// q|k|v projection with the rotary embedding of the q and k heads in the GEMM epilogue:
// out[M, N] = X W^T, then columns [0, rope_heads * 128) are rotated head by head (head_dim 128,
// position of row r = r % seq_len, cos/sin [seq_len, 64] fp32).  Equals olmax_gemm_bf16 followed
// by olmax_qk_rope_fwd in place on those columns, which is also what it falls back to when the
// shape does not fit the fused kernel.
extern "C" int32_t olmax_gemm_rope_bf16(hipStream_t stream, const void* X, const void* W, void* out, int32_t M, int32_t N,
                                        int32_t K, int64_t ldx, int64_t ldw, int64_t ldo, const float* cos_t,
                                        const float* sin_t, int32_t seq_len, int32_t rope_heads) {
  OLMAX_CHECK(X && W && out && cos_t && sin_t, OLMAX_ERR_ARG, "olmax_gemm_rope_bf16: null operand");
  OLMAX_CHECK(M > 0 && N > 0 && K > 0 && seq_len > 0 && rope_heads >= 0 && (int64_t)rope_heads * 128 <= N, OLMAX_ERR_SHAPE,
              "olmax_gemm_rope_bf16: bad shape (M %d N %d K %d seq_len %d rope_heads %d)", M, N, K, seq_len, rope_heads);
  OLMAX_CHECK(ldx >= K && ldw >= K && ldo >= N, OLMAX_ERR_SHAPE, "olmax_gemm_rope_bf16: leading dimension smaller than row length");
  const bool fits = aligned16(X) && aligned16(W) && aligned16(out) && aligned16(cos_t) && aligned16(sin_t) && ldx % 8 == 0 &&
                    ldw % 8 == 0 && ldo % 8 == 0 && K % BK == 0 && M >= 256 && N % 256 == 0 && rope_heads % 2 == 0 &&
                    (int64_t)((M + 255) / 256) * (N / 256) >= 128 && !g_force_tile.load(std::memory_order_relaxed);
  if (fits && fused_wins(M, N, K, 4.f, 3.f + (float)M * rope_heads * 8.5e-5f)) {  // (the rotation moves 512 bytes a head at 6 TB/s)
    constexpr int SMEM = 2 * (256 + 256) * BK * 2;
    auto whole = gemm_bf16_kernel<256, 256, 128, 64, true, true, false, false, 3>;
    auto ragged = gemm_bf16_kernel<256, 256, 128, 64, true, true, false, false, 3, 1>;
    static std::once_flag attr_once;
    std::call_once(attr_once, [&] {
      (void)hipFuncSetAttribute((const void*)whole, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
      (void)hipFuncSetAttribute((const void*)ragged, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
    });
    auto kern = M % 256 ? ragged : whole;
    const int tm = (M + 255) / 256, tn = N / 256;
    ProfRec rec{};
    if (g_prof_on) {
      (void)hipEventCreate(&rec.e0);
      (void)hipEventCreate(&rec.e1);
      (void)hipEventRecord(rec.e0, stream);
    }
    const int order = tile_order(tm, tn, true, true, N, K);
    hipLaunchKernelGGL(kern, dim3(order_grid(order, tm, tn)), dim3(512), SMEM, stream, (const bf16*)X, (const bf16*)W, out, (const bf16*)nullptr, M,
                       N, K, ldx, ldw, ldo, (int64_t)0, tm, tn, 1, cos_t, sin_t, seq_len, rope_heads * 128, order);
    if (g_prof_on) {
      (void)hipEventRecord(rec.e1, stream);
      rec.flops = 2.0 * M * N * K;
      rec.bytes = 2.0 * ((double)M * K + (double)N * K + (double)M * N);
      rec.key = 256 | (1 << 12) | (1 << 13) | (1 << 17);
      rec.M = M; rec.N = N; rec.K = K;
      std::lock_guard<std::mutex> lk(g_prof_mu);
      g_prof.push_back(rec);
    }
    OLMAX_LAUNCH_CHECK();
    return OLMAX_OK;
  }
  int rc = olmax_gemm_bf16(stream, X, W, out, nullptr, M, N, K, ldx, ldw, ldo, 0, 0, 0, 0);
  if (rc || rope_heads == 0) return rc;
  return olmax_qk_rope_fwd(stream, out, out, nullptr, cos_t, sin_t, M, rope_heads, 128, seq_len, ldo, ldo, 0.f);
}

extern "C" int32_t olmax_glu_fwd(hipStream_t stream, const void* gate, const void* up, void* out, int64_t T, int32_t F,
                                 int64_t ldg, int64_t ldu, int64_t ldo, int32_t act);

extern "C" int32_t olmax_gemm_glu_fused(const void* X, const void* W, const void* act_out, int32_t M, int32_t F, int32_t K,
                                        int64_t ldx, int64_t ldw, int64_t ldact) {
  const bool fits = aligned16(X) && aligned16(W) && ldx % 8 == 0 && ldw % 8 == 0 && K % BK == 0 && M >= 256 && F % 128 == 0 &&
                    (int64_t)((M + 255) / 256) * (F / 128) >= 128 && !g_force_tile.load(std::memory_order_relaxed);
  if (!fits || (M % 256 && !(aligned16(act_out) && ldact % 8 == 0))) return 0;  // ragged rows leave through the whole-line stores only
  return glu_fused_wins(M, F, K, GLU_ONLY) ? 1 : 2;
}

// Gated-MLP input projection with the activation fused into the GEMM epilogue:
// act_out[M, F] = f(X Wgate^T) * (X Wup^T), W = [Wgate; Wup] ([2F, K], row stride ldw); gu_out
// ([M, 2F], optional) receives gate|up for the backward pass.  Falls back to the plain GEMM
// plus olmax_glu_fwd (through a caller-provided gu_out) when the shape does not fit the tile, or when these are faster.
extern "C" int32_t olmax_gemm_glu_bf16(hipStream_t stream, const void* X, const void* W, void* gu_out, void* act_out,
                                       int32_t M, int32_t F, int32_t K, int64_t ldx, int64_t ldw, int64_t ldgu,
                                       int64_t ldact, int32_t act) {
  OLMAX_CHECK(X && W && act_out, OLMAX_ERR_ARG, "olmax_gemm_glu_bf16: null operand");
  OLMAX_CHECK(M > 0 && F > 0 && K > 0, OLMAX_ERR_SHAPE, "olmax_gemm_glu_bf16: M,F,K must be positive (got %d,%d,%d)", M, F, K);
  OLMAX_CHECK(act == 0 || act == 1, OLMAX_ERR_ARG, "olmax_gemm_glu_bf16: act must be 0 (silu) or 1 (gelu-tanh)");
  OLMAX_CHECK(ldx >= K && ldw >= K && ldact >= F && (!gu_out || ldgu >= 2 * (int64_t)F), OLMAX_ERR_SHAPE,
              "olmax_gemm_glu_bf16: leading dimension smaller than row length");
  const bool gu_lines = M % 256 == 0 || !gu_out || (aligned16(gu_out) && ldgu % 8 == 0);
  if (gu_lines && olmax_gemm_glu_fused(X, W, act_out, M, F, K, ldx, ldw, ldact) && (!gu_out || glu_fused_wins(M, F, K, GLU_SAVE))) {
#define GLU(E, RAG) launch_glu<E, RAG>(stream, (const bf16*)X, (const bf16*)W, (bf16*)gu_out, (bf16*)act_out, M, F, K, ldx, ldw, ldgu, ldact)
    if (act == 0) return M % 256 ? GLU(1, 1) : GLU(1, 0);
    return M % 256 ? GLU(2, 1) : GLU(2, 0);
#undef GLU
  }
  OLMAX_CHECK(gu_out, OLMAX_ERR_ARG, "olmax_gemm_glu_bf16: this shape needs gu_out as scratch for the unfused path");
  int rc = olmax_gemm_bf16(stream, X, W, gu_out, nullptr, M, 2 * F, K, ldx, ldw, ldgu, 0, 0, 0, 0);
  if (rc) return rc;
  return olmax_glu_fwd(stream, gu_out, (const bf16*)gu_out + F, act_out, M, F, ldgu, ldgu, ldact, act);
}

extern "C" int32_t olmax_glu_bwd(hipStream_t stream, const void* gate, const void* up, const void* dh, void* dgate, void* dup,
                                 int64_t T, int32_t F, int64_t ldg, int64_t ldu, int64_t lddh, int64_t lddg, int64_t lddu,
                                 int32_t act);

// The gated-MLP input projection re-run inside the backward pass (full-block recompute): from X, W = [Wgate; Wup] and
// dact = d loss / d (act(gate) * up) it produces act_out [M, F] (what the down projection's weight gradient needs) and
// dgu_out [M, 2F] = d gate | d up, without gate | up ever being written.  Equals olmax_gemm_glu_bf16 followed by
// olmax_glu_bwd, which is also the path taken (through dgu_out as scratch for gate | up) when the shape does not
// fit the tile.
extern "C" int32_t olmax_gemm_glu_bwd_bf16(hipStream_t stream, const void* X, const void* W, const void* dact, void* act_out,
                                           void* dgu_out, int32_t M, int32_t F, int32_t K, int64_t ldx, int64_t ldw,
                                           int64_t lddact, int64_t ldact, int64_t lddgu, int32_t act) {
  OLMAX_CHECK(X && W && dact && act_out && dgu_out, OLMAX_ERR_ARG, "olmax_gemm_glu_bwd_bf16: null operand");
  OLMAX_CHECK(M > 0 && F > 0 && K > 0, OLMAX_ERR_SHAPE, "olmax_gemm_glu_bwd_bf16: M,F,K must be positive (got %d,%d,%d)", M, F, K);
  OLMAX_CHECK(act == 0 || act == 1, OLMAX_ERR_ARG, "olmax_gemm_glu_bwd_bf16: act must be 0 (silu) or 1 (gelu-tanh)");
  OLMAX_CHECK(ldx >= K && ldw >= K && ldact >= F && lddact >= F && lddgu >= 2 * (int64_t)F, OLMAX_ERR_SHAPE,
              "olmax_gemm_glu_bwd_bf16: leading dimension smaller than row length");
  const bool fits = aligned16(X) && aligned16(W) && ldx % 8 == 0 && ldw % 8 == 0 && K % BK == 0 && M >= 256 &&
                    F % 128 == 0 && (int64_t)((M + 255) / 256) * (F / 128) >= 128 && !g_force_tile.load(std::memory_order_relaxed) &&
                    aligned16(act_out) && ldact % 8 == 0 && aligned16(dgu_out) && lddgu % 8 == 0 &&
                    ((((uintptr_t)dact) & 7) == 0) && lddact % 4 == 0 && lddact < (1ll << 31);
  if (fits && glu_fused_wins(M, F, K, GLU_BWD)) {
#define GLU(E, RAG)                                                                                                               \
  launch_glu<E, RAG>(stream, (const bf16*)X, (const bf16*)W, (bf16*)dgu_out, (bf16*)act_out, M, F, K, ldx, ldw, lddgu, ldact,     \
                     (const bf16*)dact, lddact)
    if (act == 0) return M % 256 ? GLU(4, 1) : GLU(4, 0);
    return M % 256 ? GLU(5, 1) : GLU(5, 0);
#undef GLU
  }
  // unfused: gate | up into dgu_out, then the elementwise backward in place over it
  int rc = olmax_gemm_glu_bf16(stream, X, W, dgu_out, act_out, M, F, K, ldx, ldw, lddgu, ldact, act);
  if (rc) return rc;
  return olmax_glu_bwd(stream, dgu_out, (const bf16*)dgu_out + F, dact, dgu_out, (bf16*)dgu_out + F, M, F, lddgu, lddgu, lddact, lddgu,
                       lddgu, act);
}
