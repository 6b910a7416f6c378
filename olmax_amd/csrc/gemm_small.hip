// bf16 MFMA GEMM for problems that do not fill the GPU with large tiles, and for operands the
// direct-to-LDS kernel of gemm.hip cannot take (rows that are not 16-byte aligned, any M, N, K):
// C[M,N] = A B^T (+ R) with the operand layouts and roundings of olmax_gemm_bf16.
//
// What bounds such a problem is not arithmetic but the serial chain of k-tiles of one workgroup, so
// the workgroup splits the REDUCTION: its KG waves each compute the whole 64 x 64 (or 32 x 32) output tile over
// every KG-th k-tile (64 wide) and the partial tiles are added through LDS at the end, in wave order
// (bitwise reproducible, no scratch in memory).  A wave shares nothing with the others until then:
// no barrier in the loop, 16 KB of operand loads in flight per wave while it works on the previous
// 16 KB.  With every CU busy that is 128 KB per CU and turn at 1.8 us = 18 TB/s, what the L2s deliver
// (0.22 us per k-tile, 580 TFLOP/s at most; a second k-tile in flight per wave changed nothing); with
// few tiles 1.5 us per turn of latency.  8192-long weight gradients of 1024 x 1024: 94 us with 64
// 128 x 128 tiles, 32 us here; 300 x 1024 x 2816: 31 -> 12.7 us; the bounds-checked scalar kernel it
// also replaces ran at 5-20 TFLOP/s (77 x 2816 x 1024: 47 -> 7 us).
// Where not even 64 x 64 tiles find a CU each, 32 x 32 ones do: half the bytes per k-tile and wave, four times the CUs.
// us, 64 -> 32: 256 x 256 x 2048 11.5 -> 8.8, 16 x 4096 x 4096 17.9 -> 11.3, 512 x 256 x 768 7.2 -> 5.1.  (Two or four k-tiles in
// flight per wave instead of one: no change with either tile, so it is not the latency of one load that is waited for.)
// Operands travel as 8 rows of 128 B per instruction into registers (the next k-tile's while this one is
// multiplied), are parked in the wave's own LDS slabs and read back as MFMA fragments (k-contiguous:
// ds_read_b128; m/n-contiguous: transposed, ds_read_b64_tr_b16).  Loading fragments of a k-contiguous
// operand straight from memory (16 rows x 64 B) saves the LDS trip but halves the rate.
// Chunks of 8 elements are loaded with one instruction at any 2-byte alignment (gfx950 global
// memory); only a chunk that crosses the end of its row is gathered element by element.
#include "common.h"
#include <algorithm>
#include <mutex>

namespace {

constexpr int BKS = 64;                    // k-tile
constexpr int acc_ld(int TS) { return TS + 4; }  // fp32 row stride of a parked partial tile
// LDS of a wave: two operand slabs, or one partial tile (TS 64: 17408 B, 32: 8192 B)
constexpr int wave_lds(int TS) { return std::max(2 * TS * BKS * 2, TS * acc_ld(TS) * 4); }

typedef u32x4 __attribute__((aligned(2))) u32x4_u;
typedef f32x4 __attribute__((aligned(4))) f32x4_u;

// chunk swizzle of the [64 k][64] slab (128 B rows, two rows per line of the 64 banks): the 32 lanes
// of a transposing read touch 2 chunks in each of the rows {k..k+3, k+8..k+11}; the four rows of one
// parity get four different chunk pairs.  Looks at row bits 1 and 3 only.  [64 k][32]: four rows of 64 B per
// line, so only the rows k and k + 8 meet.
template <int TS>
__device__ __forceinline__ int sswz(int kr) {
  return TS == 64 ? (((kr >> 1) & 1) | (((kr >> 3) & 1) << 1)) << 1 : ((kr >> 3) & 1) << 1;
}

// the same for the [64 rows][64 k] slab of a k-contiguous operand, read 16 lanes = 16 rows at a time
__device__ __forceinline__ int kswz(int row) { return (row >> 1) & 7; }

// n elements starting at q, zeros behind them
__device__ __forceinline__ u32x4 gather(const bf16* q, int n) {
  Pack8 t;
  t.u = u32x4{0u, 0u, 0u, 0u};
  if (n >= 8) {
    t.u = *reinterpret_cast<const u32x4_u*>(q);
  } else if (n > 0) {
#pragma unroll
    for (int e = 0; e < 7; e++)
      if (e < n) t.e[e] = q[e];
  }
  return t.u;
}

// One operand of the wave: rows r0 .. r0+63 of the output tile (nrows exist), all of k.  A slab is 64
// lines of 128 B: a line is a row (KC) or a k (otherwise); a lane owns 16-byte chunk lane % 8 of lines
// lane / 8 + 8 s.
enum Mode {
  WHOLE,  // both operands have 64 rows or more (a k-contiguous one's last tile is moved back to end with
          // them) and whole chunks: no bounds in the loop
  FEW,    // fewer rows: those past the end re-read the last
  PART    // chunks may cross the end of a line, or line offsets exceed 32 bits
};
template <bool KC, Mode MODE, int TS>
struct SmallOperand {
  static constexpr int NV = TS / 8;            // 16-byte vectors per lane and k-tile
  static constexpr int CPL = KC ? 8 : TS / 8;  // vectors of a line
  static constexpr int LPS = 64 / CPL;         // lines per instruction
  const bf16* base;       // wave-uniform: first row (KC) / first column of the tile at k = 0
  unsigned off;           // bytes from there to this lane's chunk of line lane / 8
  int64_t ld;
  int lds_r[KC ? 2 : TS / 16];  // byte offset of this lane's fragment reads: k-step (KC) or 16-column group
  int left;               // KC: rows of the tile that exist; else elements of this lane's chunk that do (>= 8: all)
  int last;               // KC: group of 8 rows that the existing ones end in (wave-uniform)
  unsigned off_last;      // KC: `off` with the rows of that group clamped to its last

  __device__ __forceinline__ void init(const bf16* mat, int64_t ld_, int r0, int nrows, int lane) {
    ld = ld_;
    const int l16 = lane & 15, g16 = lane >> 4;
    int c = lane & (CPL - 1);
    base = KC ? mat + (int64_t)r0 * ld : mat + r0;
    if (KC) {
      left = nrows - r0;
      last = min(left - 1, TS - 1) >> 3;
      off_last = (unsigned)((min(lane >> 3, left - 1 - last * 8) * ld + c * 8) * 2);
#pragma unroll
      for (int kk = 0; kk < 2; kk++) lds_r[kk] = l16 * 128 + (((kk * 4 + g16) ^ kswz(l16)) << 4);
    } else {
      left = nrows - (r0 + c * 8);
      if (MODE != PART && left <= 0) c = 0;  // whole chunks only: those past the end re-read the line's first
#pragma unroll
      for (int x = 0; x < TS / 16; x++) {
        const int col = x * 16 + ((l16 & 3) << 2), k = g16 * 8 + (l16 >> 2);
        lds_r[x] = k * (TS * 2) + (((col >> 3) ^ sswz<TS>(k)) << 4) + ((col & 7) << 1);
      }
    }
    off = (unsigned)(((lane / CPL) * ld + c * 8) * 2);
  }
  // line s of this lane in the k-tile starting at k0, in full 64-bit arithmetic
  __device__ __forceinline__ const bf16* line_ptr(int64_t k0, int s, int lane) const {
    const int line = s * LPS + lane / CPL, c = lane & (CPL - 1);
    return base + (KC ? k0 + (int64_t)min(line, left - 1) * ld : (k0 + line) * ld) + c * 8;
  }
  // k-tile starting at k0, all 64 k valid
  __device__ __forceinline__ void load(u32x4 (&v)[NV], int64_t k0, int lane) const {
    const bf16* q = base + (KC ? k0 : k0 * ld);
    if (MODE == PART) {
#pragma unroll
      for (int s = 0; s < NV; s++) v[s] = gather(line_ptr(k0, s, lane), KC ? 8 : left);
    } else if (KC && MODE == FEW) {
      // groups of 8 rows: whole ones, then the one the rows end in, again and again (branch-free)
#pragma unroll
      for (int s = 0; s < NV; s++)
        v[s] = *reinterpret_cast<const u32x4_u*>(reinterpret_cast<const char*>(q + (int64_t)(min(s, last) * 8) * ld) + (s < last ? off : off_last));
    } else {
#pragma unroll
      for (int s = 0; s < NV; s++)
        v[s] = *reinterpret_cast<const u32x4_u*>(reinterpret_cast<const char*>(q + (int64_t)(s * LPS) * ld) + off);
    }
  }
  // the last k-tile: only k < kend exists
  __device__ __forceinline__ void load_tail(u32x4 (&v)[NV], int64_t k0, int kend, int lane) const {
#pragma unroll
    for (int s = 0; s < NV; s++)
      v[s] = gather(line_ptr(k0, s, lane), KC ? kend - (int)k0 - (lane & 7) * 8 : k0 + s * LPS + lane / CPL < kend ? left : 0);
  }
  __device__ __forceinline__ void park(const u32x4 (&v)[NV], unsigned char* slab, int lane) const {
#pragma unroll
    for (int s = 0; s < NV; s++) {
      const int line = s * LPS + lane / CPL;
      *reinterpret_cast<u32x4*>(slab + line * (CPL * 16) + (((lane & (CPL - 1)) ^ (KC ? kswz(line) : sswz<TS>(line))) << 4)) = v[s];
    }
  }
  __device__ __forceinline__ bf16x8 frag(const unsigned char* slab, int kk, int i) const {
    if (KC) return *reinterpret_cast<const bf16x8*>(slab + lds_r[kk] + i * 2048);
    Pack8 f;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      s16x4 t = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (s16x4 __attribute__((address_space(3)))*)(slab + lds_r[KC ? 0 : i] + (kk * 32 + h * 4) * (TS * 2)));
      f.u[h * 2] = ((u32x2&)t)[0];
      f.u[h * 2 + 1] = ((u32x2&)t)[1];
    }
    return f.v;
  }
};

// One product C[M,N] = A B^T (+ R).
struct Problem {
  const bf16 *A, *B;
  void* C;
  const bf16* R;
  int M, N, K;
  int64_t lda, ldb, ldc, ldr;
  int out_f32;
};
template <int TS>
int tiles(const Problem& p) {
  return (int)((int64_t)((p.M + TS - 1) / TS) * ((p.N + TS - 1) / TS));
}

// Tile `pid` of `nwg` by the KG waves of a workgroup.  TWO: the first half of a wave's k-tiles is added up by itself, so that four
// waves have the chains of fp32 additions of eight.  (Two accumulators in turn, the loop's code twice: 2 % more time over 64 pairs of gradients,
// 2048 x 256 x 768 9.66 us, 9.42 in halves, 512 x 1024 x 1024 9.42 and 8.91.)
template <int TS, int KG, bool A_KC, bool B_KC, Mode MODE, bool TWO = false>
__device__ __forceinline__ void small_tile(const Problem& P, int pid, int nwg, unsigned char* smem) {
  const bf16 *A = P.A, *B = P.B, *R = P.R;
  void* Cv = P.C;
  const int M = P.M, N = P.N, K = P.K, out_f32 = P.out_f32;
  const int64_t lda = P.lda, ldb = P.ldb, ldc = P.ldc, ldr = P.ldr;
  const int tiles_m = (M + TS - 1) / TS, tiles_n = (N + TS - 1) / TS;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g16 = lane >> 4;

  // XCD-contiguous runs of tiles, walked in groups of 8 tile rows (as the large-tile kernel's run order)
  if ((nwg & 7) == 0) pid = (pid & 7) * (nwg >> 3) + (pid >> 3);
  const int gid = pid / (8 * tiles_n), first = gid * 8, gm = min(tiles_m - first, 8), in = pid - gid * 8 * tiles_n;
  const int m_own = (first + in % gm) * TS, n_own = (in / gm) * TS;  // first row / column this tile stores
  const int m0 = MODE == WHOLE && A_KC ? min(m_own, M - TS) : m_own, n0 = MODE == WHOLE && B_KC ? min(n_own, N - TS) : n_own;

  constexpr int TF = TS / 16;  // fragments per operand
  constexpr int WAVE_LDS = wave_lds(TS), ACC_LD = acc_ld(TS);
  unsigned char* slab_a = smem + wave * WAVE_LDS;
  unsigned char* slab_b = slab_a + TS * BKS * 2;
  SmallOperand<A_KC, MODE, TS> oa;
  SmallOperand<B_KC, MODE, TS> ob;
  oa.init(A, lda, m0, M, lane);
  ob.init(B, ldb, n0, N, lane);

  f32x4 accs[1 + TWO][TF][TF];
#pragma unroll
  for (int s = 0; s <= TWO; s++)
#pragma unroll
    for (int i = 0; i < TF; i++)
#pragma unroll
      for (int j = 0; j < TF; j++) accs[s][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // operands swapped, as in the large-tile kernel: an accumulator holds row l16, columns 4 g16 .. +3
  auto multiply = [&](f32x4 (&acc)[TF][TF]) {
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
      bf16x8 fa[TF], fb[TF];
#pragma unroll
      for (int i = 0; i < TF; i++) fa[i] = oa.frag(slab_a, kk, i);
#pragma unroll
      for (int j = 0; j < TF; j++) fb[j] = ob.frag(slab_b, kk, j);
#pragma unroll
      for (int i = 0; i < TF; i++)
#pragma unroll
        for (int j = 0; j < TF; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
  };

  u32x4 va[SmallOperand<A_KC, MODE, TS>::NV], vb[SmallOperand<B_KC, MODE, TS>::NV];
  auto load = [&](int kt) {
    oa.load(va, (int64_t)kt * BKS, lane);
    ob.load(vb, (int64_t)kt * BKS, lane);
  };
  auto park = [&]() {
    oa.park(va, slab_a, lane);
    ob.park(vb, slab_b, lane);
  };
  const int ktf = K / BKS;  // whole k-tiles
  int kt = wave;
  if (kt < ktf) load(kt);
  const int half = TWO ? wave + (ktf - wave + 2 * KG - 1) / (2 * KG) * KG : 0;  // first k-tile of the second half
  for (; kt < ktf; kt += KG) {
    if (TWO && kt == half) {
#pragma unroll
      for (int i = 0; i < TF; i++)
#pragma unroll
        for (int j = 0; j < TF; j++) {
          accs[TWO][i][j] = accs[0][i][j];
          accs[0][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    park();
    if (kt + KG < ktf) load(kt + KG);
    multiply(accs[0]);
  }
  if (kt == ktf && ktf * BKS < K) {  // the ragged k-tile falls to the wave whose turn it is
    oa.load_tail(va, (int64_t)ktf * BKS, K, lane);
    ob.load_tail(vb, (int64_t)ktf * BKS, K, lane);
    park();
    multiply(accs[0]);
  }
  f32x4 (&acc)[TF][TF] = accs[0];
  if (TWO) {
#pragma unroll
    for (int i = 0; i < TF; i++)
#pragma unroll
      for (int j = 0; j < TF; j++) acc[i][j] += accs[TWO][i][j];
  }

  // partial tiles into the waves' own regions, then every thread adds 8 columns of a row in wave order
  float* mine = reinterpret_cast<float*>(smem + wave * WAVE_LDS);
#pragma unroll
  for (int i = 0; i < TF; i++)
#pragma unroll
    for (int j = 0; j < TF; j++) *reinterpret_cast<f32x4*>(mine + (i * 16 + l16) * ACC_LD + j * 16 + g16 * 4) = acc[i][j];
  __syncthreads();
#pragma unroll
  for (int it = 0; it < (TS * TS / 8 + KG * 64 - 1) / (KG * 64); it++) {
    const int item = it * KG * 64 + threadIdx.x;
    const int trow = item / (TS / 8), tcol = item % (TS / 8) * 8;
    const int row = m0 + trow, col = n0 + tcol;
    if (trow >= TS || row < m_own || row >= M || col + 8 <= n_own || col >= N) continue;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = 0.f;
#pragma unroll
    for (int g = 0; g < KG; g++) {
      const float* src = reinterpret_cast<const float*>(smem + g * WAVE_LDS) + trow * ACC_LD + tcol;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(src), hi = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
      for (int e = 0; e < 4; e++) { v[e] += lo[e]; v[4 + e] += hi[e]; }
    }
    const int lo = max(0, n_own - col), n = min(8, N - col);
    const bool all = lo == 0 && n == 8;
    if (R) {
      const Pack8 rr = {gather(R + (int64_t)row * ldr + col, n)};
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] = (out_f32 ? v[e] : bf2f(f2bf(v[e]))) + bf2f(rr.e[e]);
    }
    if (out_f32) {
      float* c = reinterpret_cast<float*>(Cv) + (int64_t)row * ldc + col;
      if (all) {
        *reinterpret_cast<f32x4_u*>(c) = f32x4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4_u*>(c + 4) = f32x4{v[4], v[5], v[6], v[7]};
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++)
          if (e >= lo && e < n) c[e] = v[e];
      }
    } else {
      bf16* c = reinterpret_cast<bf16*>(Cv) + (int64_t)row * ldc + col;
      Pack8 o;
#pragma unroll
      for (int e = 0; e < 8; e++) o.e[e] = f2bf(v[e]);
      if (all) {
        *reinterpret_cast<u32x4_u*>(c) = o.u;
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++)
          if (e >= lo && e < n) c[e] = o.e[e];
      }
    }
  }
}

template <int TS, int KG, bool A_KC, bool B_KC, Mode MODE>
__global__ __launch_bounds__(KG * 64, 2) void gemm_small_kernel(const Problem p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  small_tile<TS, KG, A_KC, B_KC, MODE>(p, blockIdx.x, gridDim.x, smem);
}

// dX = dY W (tiles of TSX) and dW = dY^T X (TSW) in one launch: neither fills the GPU, a launch alone is 3 us, and the second does not
// need the first.  Workgroups of the longer reduction come first.  us, two launches -> one, T x in x out: 2048 x 256 x 2048
// 22.4 -> 13.2, 2048 x 1024 x 256 17.1 -> 13.1, 2048 x 256 x 256 14.5 -> 6.7, 4096 x 256 x 768 24.9 -> 16.7, 130 x 1024 x 3072 15.0 -> 13.4.
template <int TSX, int TSW, int KG, bool TWOX, bool TWOW>
__global__ __launch_bounds__(KG * 64, 2) void gemm_small_pair_kernel(const Problem dx, const Problem dw, int n_dx, int n_dw, int dx_first) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int id = blockIdx.x;
  if (dx_first ? id < n_dx : id >= n_dw) small_tile<TSX, KG, true, false, WHOLE, TWOX>(dx, dx_first ? id : id - n_dw, n_dx, smem);
  else small_tile<TSW, KG, false, false, WHOLE, TWOW>(dw, dx_first ? id - n_dx : id, n_dw, smem);
}

template <typename K>
void allow_lds(K kern, int bytes) {
  (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

template <int TS, int KG, bool A_KC, bool B_KC, Mode MODE>
void launch(hipStream_t s, const Problem& p) {
  auto kern = gemm_small_kernel<TS, KG, A_KC, B_KC, MODE>;
  constexpr int SMEM = KG * wave_lds(TS);
  static std::once_flag once;  // per instantiation
  std::call_once(once, [&] { allow_lds(kern, SMEM); });
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles<TS>(p)), dim3(KG * 64), SMEM, s, p);
}

template <int TS, int KG, bool A_KC, bool B_KC>
void dispatch(hipStream_t s, const Problem& p) {
  // line offsets of a slab stay below 2^32 bytes for row strides below 2^25 elements
  const bool part = (!A_KC && p.M % 8) || (!B_KC && p.N % 8) || p.lda >= (1 << 25) || p.ldb >= (1 << 25);
  if (part) launch<TS, KG, A_KC, B_KC, PART>(s, p);
  else if ((A_KC && p.M < TS) || (B_KC && p.N < TS)) launch<TS, KG, A_KC, B_KC, FEW>(s, p);
  else launch<TS, KG, A_KC, B_KC, WHOLE>(s, p);
}
template <int TS, int KG>
void dispatch(hipStream_t s, const Problem& p, bool a_kc, bool b_kc) {
  auto go = a_kc ? (b_kc ? dispatch<TS, KG, true, true> : dispatch<TS, KG, true, false>)
                 : (b_kc ? dispatch<TS, KG, false, true> : dispatch<TS, KG, false, false>);
  go(s, p);
}

template <int TSX, int TSW, int KG, bool TWOX = false, bool TWOW = false>
void launch_pair(hipStream_t s, const Problem& dx, const Problem& dw) {
  auto kern = gemm_small_pair_kernel<TSX, TSW, KG, TWOX, TWOW>;
  constexpr int SMEM = KG * std::max(wave_lds(TSX), wave_lds(TSW));
  static std::once_flag once;
  std::call_once(once, [&] { allow_lds(kern, SMEM); });
  const int n_dx = tiles<TSX>(dx), n_dw = tiles<TSW>(dw);
  hipLaunchKernelGGL(kern, dim3((unsigned)(n_dx + n_dw)), dim3(KG * 64), SMEM, s, dx, dw, n_dx, n_dw, (int)(dx.K > dw.K));
}

}  // namespace

void olmax_gemm_small(hipStream_t s, const bf16* A, const bf16* B, void* C, const bf16* R, int M, int N, int K, int64_t lda,
                      int64_t ldb, int64_t ldc, int64_t ldr, bool a_kc, bool b_kc, bool out_f32, int tile, int groups) {
  const Problem p = {A, B, C, R, M, N, K, lda, ldb, ldc, ldr, out_f32};
  if (tile == 32) {
    if (groups == 8) dispatch<32, 8>(s, p, a_kc, b_kc);
    else dispatch<32, 4>(s, p, a_kc, b_kc);
  } else if (groups == 8) {
    dispatch<64, 8>(s, p, a_kc, b_kc);
  } else {
    dispatch<64, 4>(s, p, a_kc, b_kc);
  }
}

void olmax_gemm_small_pair(hipStream_t s, const bf16* dy, const bf16* w, const bf16* x, bf16* dx, const bf16* r, bf16* dw, int T, int in,
                           int out, int64_t lddy, int64_t ldw, int64_t ldx, int64_t lddx, int64_t ldr, int64_t lddw) {
  const Problem px = {dy, w, dx, r, T, in, out, lddy, ldw, lddx, ldr, 0};
  const Problem pw = {dy, x, dw, nullptr, out, in, T, lddy, ldx, lddw, 0, 0};
  // Tiles of 32 while they find a CU each.  Eight waves to a tile where all of them have a CU; else four, with two chains each where the
  // product alone would have eight (up to 256 tiles of 64, more than four k-tiles): no chain of additions is longer than in the two calls.
  // us, eight waves | four, one chain | two (in turn; halves 2 % less): 1500 x 256 x 2048 12.0 | 11.8 | 13.3, 512 x 256 x 2048 7.1 | 7.0 | 7.6, 2048 x 256 x 256 6.8 | 6.6 | 6.9;
  // more tiles than CUs, 2048 x 256 x 768 12.8 | 10.7 | 11.3, 1000 x 256 x 2048 13.6 | 11.8 | 12.2, 1500 x 512 x 512 11.4 | 9.1 | 9.6.
  const int x32 = tiles<32>(px), w32 = tiles<32>(pw);
  if ((x32 <= 256 ? x32 : tiles<64>(px)) + (w32 <= 256 ? w32 : tiles<64>(pw)) <= 256) {
    auto go = x32 <= 256 ? (w32 <= 256 ? launch_pair<32, 32, 8> : launch_pair<32, 64, 8>)
                         : (w32 <= 256 ? launch_pair<64, 32, 8> : launch_pair<64, 64, 8>);
    go(s, px, pw);
    return;
  }
  auto form = [](const Problem& p) { return tiles<32>(p) <= 256 ? 0 : tiles<64>(p) > 256 || p.K <= 4 * BKS ? 1 : 2; };
  switch (form(px) * 3 + form(pw)) {
    case 0: launch_pair<32, 32, 4, true, true>(s, px, pw); break;
    case 1: launch_pair<32, 64, 4, true, false>(s, px, pw); break;
    case 2: launch_pair<32, 64, 4, true, true>(s, px, pw); break;
    case 3: launch_pair<64, 32, 4, false, true>(s, px, pw); break;
    case 4: launch_pair<64, 64, 4, false, false>(s, px, pw); break;
    case 5: launch_pair<64, 64, 4, false, true>(s, px, pw); break;
    case 6: launch_pair<64, 32, 4, true, true>(s, px, pw); break;
    case 7: launch_pair<64, 64, 4, true, false>(s, px, pw); break;
    default: launch_pair<64, 64, 4, true, true>(s, px, pw);
  }
}
