// Causal GQA flash attention for gfx950, head_dim 128 or 64 (D), BSHD layout, bf16 in/out, fp32
// softmax statistics, optional sliding window and tanh logit soft-cap.
//
// Replaces the cuDNN fused-attention custom call that
// jax.nn.dot_product_attention(is_causal=True, local_window_size=w) lowers to
// (reference src/olmax/nn/attention.py:96-103) and its autodiff transpose.
// Mask: key j visible to query i iff j <= i and (w < 0 or j >= i - w).
//
// All three kernels keep the score tile TRANSPOSED in the MFMA accumulators so that each
// lane owns one query (forward, dQ) or one key (dK/dV) column: row statistics become
// per-lane scalars, and the exponentiated tile is already laid out as the B operand of the
// next v_mfma_f32_32x32x16_bf16 (k index = accumulator row pattern).  The operand that must
// be read against its storage order (V^T, K^T, Q^T, dO^T) comes from LDS through
// ds_read_b64_tr_b16.  K/V (or Q/dO) tiles are double buffered in LDS with a register-held
// prefetch of the next tile; 16-byte chunks are XOR-swizzled so that both ds_read_b128 and
// the transposing reads are bank-conflict free.
//
// Backward is split in two deterministic halves (no atomics): dK/dV with the key tile
// stationary, dQ with the query tile stationary; each recomputes P from the saved LSE.  They
// are two kernels, or one launch where neither fills the GPU.
#include "common.h"
#include <algorithm>
#include <mutex>
#include <type_traits>

extern "C" int32_t olmax_fill_zero(hipStream_t stream, void* p, int64_t nbytes);

namespace {

__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
// tanh(raw * scale / cap) from a raw score, with c1 = 2 * scale * log2(e) / cap formed once per
// kernel: tanh(x) = 1 - 2 / (exp(2x) + 1) as one multiply, exp2, add, reciprocal and fma.  (Dividing
// by cap per score, as the formula reads, costs a correctly rounded division per element.)
__device__ __forceinline__ float cap_tanh(float raw, float c1) {
  return __builtin_fmaf(-2.f, __builtin_amdgcn_rcpf(fexp2(raw * c1) + 1.f), 1.f);
}
// Its error is an ulp of 1 whatever the result, which the cap multiplies.  At head_dim 128 that drowns in LSE's own error (1e-3 at
// most: it sums rounded probabilities).  At head_dim 64 LSE is good to 8e-7 and it would be 3e-6 (cap 30) or 5e-6 (cap 50):
// there the formula is taken as it reads, as the one-wave-per-query kernels take it.
template <int D>
__device__ __forceinline__ float cap_tanh_of(float raw, float c1, float scale, float cap) {
  return D == 64 ? tanhf(raw * scale / cap) : cap_tanh(raw, c1);
}

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;

// 16-byte chunk swizzle of the [rows][D] tiles.  ds_read_b128 serves the lane groups
// {0-3,12-15,20-23,24-27} / {4-7,8-11,16-19,28-31} (one row per lane, same logical chunk) per clock
// and the transposing ds_read_b64 serves lanes 0-31 (4 consecutive rows x 4 chunks); these masks give
// 16 distinct chunks modulo the 256-byte line of the 64 banks in both cases.  D = 128: a row is a
// line; D = 64: two rows share one, so the row's lowest bit already separates them, and bit 1 moves
// the transposed read's other two rows to the other half of their own.
template <int D>
__device__ __forceinline__ int swz(int row) {
  return D == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : ((row & 2) << 1) | ((row >> 2) & 3);
}

// Per-lane byte offsets of the operand fragments inside a [rows][D] tile.  The swizzle only
// looks at row bits 0-3, so stepping rows by 16 or 32 is a plain immediate offset and the
// D/16 (k-contiguous) plus D/16 (transposed) lane-dependent offsets are loop invariant.
// LEAN: the k-contiguous offsets are formed at each read from the first one (kc[s] = kc[0] ^ 32 s:
// the k-step only enters the XOR-swizzled chunk index) instead of living in registers, for a
// kernel that would otherwise spill them.
template <int D, bool LEAN = false>
struct FragAddr {
  int kc[LEAN ? 1 : D / 16];  // row (lane % 32), k-step s
  int tr[D / 32][2];          // column tile dt, half h of the transposed read
  __device__ __forceinline__ void init(int lane) {
    const int l32 = lane & 31, lhi = lane >> 5;
#pragma unroll
    for (int s = 0; s < (LEAN ? 1 : D / 16); s++) kc[s] = l32 * (2 * D) + (((2 * s + lhi) ^ swz<D>(l32)) << 4);
    const int j16 = lane & 15, g16 = lane >> 4;
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int col = dt * 32 + ((g16 & 1) << 4) + ((j16 & 3) << 2);
        const int row = ((g16 >> 1) << 2) + (h << 3) + (j16 >> 2);
        tr[dt][h] = row * (2 * D) + (((col >> 3) ^ swz<D>(row)) << 4) + ((col & 7) << 1);
      }
  }
  // k-contiguous fragment: rows row0 + lane%32 (row0 multiple of 16), k-step s
  __device__ __forceinline__ bf16x8 load_kc(const unsigned char* tile, int row0, int s) const {
    int off = kc[LEAN ? 0 : s];
    if (LEAN) {
      asm volatile("" : "+v"(off));  // keeps the XOR at the read: hoisted out of the loop it is a register again
      off ^= s << 5;
    }
    return *reinterpret_cast<const bf16x8*>(tile + off + row0 * (2 * D));
  }
  // transposed fragment: MFMA rows = storage columns dt*32 + lane%32, k = storage rows r0 + {..}
  __device__ __forceinline__ bf16x8 load_tr(const unsigned char* tile, int r0, int dt) const {
    Pack8 p;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      s16x4 t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(tile + tr[dt][h] + r0 * (2 * D)));
      p.u[h * 2 + 0] = ((u32x2&)t)[0];
      p.u[h * 2 + 1] = ((u32x2&)t)[1];
    }
    return p.v;
  }
};

// Stream ROWS rows of D bf16 (global row r0 + i, clamped to S-1, row stride ld) into the
// swizzled LDS tile at lds_addr: DMA instructions of 1 KB (512/D rows) shared by 4 waves.
template <int ROWS, int D>
__device__ __forceinline__ void dma_tile(const bf16* base, int64_t ld, int r0, int S, unsigned lds_addr, int wave, int lane) {
#pragma unroll
  for (int i = 0; i < ROWS * D / 2048; i++) {
    const int blk = i * 4 + wave;
    const int p = blk * 64 + lane;
    const int row = p / (D / 8), ph = p % (D / 8);
    const int gr = min(r0 + row, S - 1);
    dma16(base + (int64_t)gr * ld + ((ph ^ swz<D>(row)) << 3), lds_addr + blk * 1024);
  }
}

// Workgroup id -> (tile rank, K/V group, head inside the group).  Hardware deals consecutive
// ids round-robin to the 8 XCDs and every XCD starts its ids in order, so the tile rank (the
// amount of causal work) is the SLOWEST index: each XCD gets the same mix of long and short
// tiles and starts the longest first (with the rank fastest, one XCD got 54 % more work than
// another and the CUs idled 39 % of the kernel).  When the group count divides by 8 the
// heads sharing a K/V head also land on one XCD, i.e. one L2.
struct WgCoord { int rank, group, r; };
__device__ __forceinline__ WgCoord decode_wg(int id, int ngroups, int rep) {
  const int level = ngroups * rep;
  WgCoord c;
  c.rank = id / level;
  const int u = id % level;
  if ((ngroups & 7) == 0) {
    const int blk = u / (8 * rep), rem = u % (8 * rep);
    c.r = rem >> 3;
    c.group = blk * 8 + (rem & 7);
  } else {
    c.group = u / rep;
    c.r = u % rep;
  }
  return c;
}

// The same tile transfer with everything lane-dependent hoisted out of the loop: a lane's byte
// offset (row * ld + swizzled chunk) inside the rows of one instruction of the four waves is computed
// once, and since the swizzle only looks at row bits 0-3 the DMA instructions of a transfer differ by
// a wave-uniform 2048/D rows, which go into the scalar base: one vector register per
// operand whatever the tile height.  Only for tiles that lie entirely inside the sequence (no
// row clamping).
template <int ROWS, int D>
struct TileDma {
  unsigned off;
  int64_t step;
  __device__ __forceinline__ void init(int64_t ld, int wave, int lane) {
    const int p = wave * 64 + lane;
    const int row = p / (D / 8), ph = p % (D / 8);
    off = (unsigned)((row * ld + ((ph ^ swz<D>(row)) << 3)) * 2);
    step = (2048 / D) * ld;
  }
  __device__ __forceinline__ void issue(const bf16* row0, unsigned lds_addr, int wave) const {
#pragma unroll
    for (int i = 0; i < ROWS * D / 2048; i++) dma16_s(row0 + i * step, off, lds_addr + (i * 4 + wave) * 1024);
  }
};

// acc + sum of the two bf16 values in dword w of a packed fragment
__device__ __forceinline__ float dot2_ones(const bf16x8& v, int w, float acc) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  const bf2 pair = {v[2 * w], v[2 * w + 1]};
  const bf2 ones = {(__bf16)1.0f, (__bf16)1.0f};
  return __builtin_amdgcn_fdot2_f32_bf16(pair, ones, acc, false);
}

__device__ __forceinline__ bf16x8 pack_bf16x8(const f32x16& a, int base) {
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; e++) r[e] = f2bf(a[base + e]);
  return r;
}


// Sum over the GROUPS waves that hold partial accumulators of the same 32 columns (column block c): every wave parks its D/8 units of 4 floats per lane in LDS, [c][group][unit][lane], and after a
// barrier adds its share of the units in group order and hands them to `out`.
template <int D, int GROUPS, typename Out>
__device__ __forceinline__ void add_partials(unsigned char* smem, const f32x16 (&acc)[D / 32], int c, int group, int lane, Out out) {
  constexpr int UNITS = D / 8, MINE = UNITS / GROUPS;
  static_assert(UNITS % GROUPS == 0, "units are dealt evenly to the groups");
  f32x4* park = reinterpret_cast<f32x4*>(smem) + c * (GROUPS * UNITS * 64) + lane;
#pragma unroll
  for (int u = 0; u < UNITS; u++)
    park[(group * UNITS + u) * 64] = f32x4{acc[u >> 2][(u & 3) * 4], acc[u >> 2][(u & 3) * 4 + 1], acc[u >> 2][(u & 3) * 4 + 2], acc[u >> 2][(u & 3) * 4 + 3]};
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MINE; i++) {
    const int u = group * MINE + i;
    f32x4 v = park[u * 64];
#pragma unroll
    for (int g = 1; g < GROUPS; g++) v += park[(g * UNITS + u) * 64];
    out(u, v);
  }
}

// ---------------------------------------------------------------------------------------
// Rows of head_dim 64 that come out infinite or NaN.  The tile products take hidden pairs along as zeros, and zero times an
// infinity or a NaN in a token that a row does not see (V and K of a later one, Q and dO of an earlier one) is NaN.  The
// one-wave-per-query kernels, which took all of this head_dim before, look at visible pairs only, so a wave that finds such
// values among those it has stored (one multiply-add each) does their rows over as those kernels do: lane l has key or query
// l of 64 for the scores, element l of the row for the sums.  Speed does not matter here.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ float dot64(const bf16* a, const bf16* b) {
  float s = 0.f;
#pragma unroll 1
  for (int c = 0; c < 64; c += 8) {
    Pack8 x, y;
    x.u = *reinterpret_cast<const u32x4*>(a + c);
    y.u = *reinterpret_cast<const u32x4*>(b + c);
#pragma unroll
    for (int e = 0; e < 8; e++) s += bf2f(x.e[e]) * bf2f(y.e[e]);
  }
  return s;
}
// score of a pair and d score / d product
template <bool CAP>
__device__ __forceinline__ float score64(const bf16* q, const bf16* k, float scale, float cap, float* chain) {
  const float s = dot64(q, k) * scale;
  if (!CAP) return s;
  const float th = tanhf(s / cap);
  if (chain) *chain = 1.f - th * th;
  return cap * th;
}
// calls row(r) for the rows r of a wave's 32 in which a lane's sum of zeros is not zero
template <typename Row>
__device__ __forceinline__ void redo_rows(float zeros, Row row) {
  const uint64_t bad = __builtin_amdgcn_ballot_w64(zeros != 0.f);
  if (bad) dma_wait_all();  // the wave's stores to the same rows, made by other lanes
  for (uint32_t rows = (uint32_t)bad | (uint32_t)(bad >> 32); rows; rows &= rows - 1) row(__builtin_ctz(rows));
}
// output row i of the sequence and head that q, k, v point to; lanes [lo, hi) store
template <bool CAP>
__device__ __forceinline__ void redo_fwd(const bf16* q, const bf16* K, int64_t ldk, const bf16* V, int64_t ldv, bf16* o, float* lse, int i,
                                         int window, float scale, float cap, int lane, int lo, int hi) {
  const int first = window >= 0 ? max(0, i - window) : 0;
  float mx = -INFINITY, sm = 0.f, acc = 0.f;
#pragma unroll 1
  for (int j = first + lane; j <= i; j += 64) mx = fmaxf(mx, score64<CAP>(q, K + j * ldk, scale, cap, nullptr));
  mx = wave_max(mx);
#pragma unroll 1
  for (int j = first + lane; j <= i; j += 64) sm += __expf(score64<CAP>(q, K + j * ldk, scale, cap, nullptr) - mx);
  const float l = mx + __logf(wave_sum(sm));
#pragma unroll 1
  for (int j0 = first; j0 <= i; j0 += 64) {
    const int n = min(64, i - j0 + 1);
    float p = 0.f;
    if (lane < n) p = bf2f(f2bf(__expf(score64<CAP>(q, K + (j0 + lane) * ldk, scale, cap, nullptr) - l)));
#pragma unroll 1
    for (int t = 0; t < n; t++) acc += __shfl(p, t, 64) * bf2f(V[(j0 + t) * ldv + lane]);
  }
  if (lane >= lo && lane < hi) o[lane] = f2bf(acc);
  if (lse && lane == 0) *lse = l;
}
template <bool CAP>
__device__ __forceinline__ void redo_dq(const bf16* q, const bf16* K, int64_t ldk, const bf16* V, int64_t ldv, const bf16* o, const bf16* d_o,
                                        float lse, bf16* dq, int i, int window, float scale, float cap, int lane, int lo, int hi) {
  const float delta = wave_sum(bf2f(o[lane]) * bf2f(d_o[lane]));
  float acc = 0.f;
#pragma unroll 1
  for (int j0 = window >= 0 ? max(0, i - window) : 0; j0 <= i; j0 += 64) {
    const int n = min(64, i - j0 + 1);
    float ds = 0.f;
    if (lane < n) {
      float chain = 1.f;
      const float p = __expf(score64<CAP>(q, K + (j0 + lane) * ldk, scale, cap, &chain) - lse);
      ds = bf2f(f2bf(p * (dot64(d_o, V + (j0 + lane) * ldv) - delta) * chain));
    }
#pragma unroll 1
    for (int t = 0; t < n; t++) acc += __shfl(ds, t, 64) * bf2f(K[(j0 + t) * ldk + lane]);
  }
  if (lane >= lo && lane < hi) dq[lane] = f2bf(acc * scale);
}
// key j; Q, dO, lse, ndelta (minus delta, nd_step to the next head's) of the first of its rep query heads
template <bool CAP>
__device__ __forceinline__ void redo_dkv(const bf16* Q, int64_t ldq, const bf16* dO, int64_t lddo, const float* lse, const float* ndelta, int nd_step,
                                         const bf16* k, const bf16* v, bf16* dk, bf16* dv, int j, int S, int rep, int window, float scale,
                                         float cap, int lane, int lo, int hi) {
  const int last = window >= 0 ? min(S - 1, j + window) : S - 1;
  float ak = 0.f, av = 0.f;
#pragma unroll 1
  for (int r = 0; r < rep; r++, Q += 64, dO += 64, lse += S, ndelta += nd_step)
#pragma unroll 1
    for (int i0 = j; i0 <= last; i0 += 64) {
      const int n = min(64, last - i0 + 1);
      float p = 0.f, ds = 0.f;
      if (lane < n) {
        const int i = i0 + lane;
        float chain = 1.f;
        p = __expf(score64<CAP>(Q + i * ldq, k, scale, cap, &chain) - lse[i]);
        ds = bf2f(f2bf(p * (dot64(dO + i * lddo, v) + ndelta[i]) * chain));
        p = bf2f(f2bf(p));
      }
#pragma unroll 1
      for (int t = 0; t < n; t++) {
        ak += __shfl(ds, t, 64) * bf2f(Q[(i0 + t) * ldq + lane]);
        av += __shfl(p, t, 64) * bf2f(dO[(i0 + t) * lddo + lane]);
      }
    }
  if (lane >= lo && lane < hi) {
    dk[lane] = f2bf(ak * scale);
    dv[lane] = f2bf(av);
  }
}

// ---------------------------------------------------------------------------------------
// Forward.  grid = ceil(S/(32 QW))*H*B workgroups (see decode_wg) of QW x KS waves; wave (qw, ks) owns queries
// i0+32qw .. +31 and every KS-th of their K/V tiles.
// KS = 1 (QW = 4): two workgroups per CU, no merge; what a grid that fills the GPU takes.
// KS > 1: one workgroup of eight waves per CU with 1/KS of the serial chain of tiles; the partial softmaxes
// are merged through LDS in key-group order.  See q_split.
// ---------------------------------------------------------------------------------------
template <int D, bool CAP, int QW, int KS>
__global__ __launch_bounds__(QW * KS * 64, 2) void attn_fwd_kernel(
    const bf16* __restrict__ Q, const bf16* __restrict__ K, const bf16* __restrict__ V,
    bf16* __restrict__ O, float* __restrict__ LSE, int S, int H, int KH, int64_t ldq, int64_t ldk,
    int64_t ldv, int64_t ldo, float scale, int window, float cap) {
  constexpr int TILE = 64 * D * 2;  // bytes of a K or V tile of 64 keys
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];  // [KS][2][K | V], then (KS > 1) the merge's statistics
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform for the compiler too
  const int l32 = lane & 31, lhi = lane >> 5;
  const int qw = wave % QW, ks = wave / QW;
  constexpr int QR = QW * 32;         // queries of the workgroup
  constexpr int TEAMS = QW * KS / 4;  // tiles are fetched by teams of 4 waves
  const int nqt = (S + QR - 1) / QR;
  const WgCoord wg = decode_wg(blockIdx.x, (int)(gridDim.x / (nqt * (H / KH))), H / KH);
  const int qt = nqt - 1 - wg.rank;  // longest rows first
  const int b = wg.group / KH, kh = wg.group % KH;
  const int h = kh * (H / KH) + wg.r;
  const int i0 = qt * QR;
  const int iw0 = i0 + qw * 32;  // first query of this wave
  const int qi = iw0 + l32;        // this lane's query
  const int qic = min(qi, S - 1);

  bf16x8 qf[D / 16];
  {
    const bf16* qp = Q + ((int64_t)b * S + qic) * ldq + h * D + lhi * 8;
#pragma unroll
    for (int s = 0; s < D / 16; s++) qf[s] = *reinterpret_cast<const bf16x8*>(qp + s * 16);
  }
  const int j_lo = window >= 0 ? max(0, i0 - window) : 0;
  const int t_lo = j_lo >> 6;
  const int t_hi = min(i0 + QR - 1, S - 1) >> 6;  // inclusive

  f32x16 o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[dt][r] = 0.f;
  float m = -INFINITY, lsum = 0.f;

  const bf16* kbase = K + (int64_t)b * S * ldk + kh * D;
  const bf16* vbase = V + (int64_t)b * S * ldv + kh * D;
  const unsigned lds0 = lds_addr_of(smem);
  const int wv = wave & 3, team = wave >> 2;
  TileDma<64, D> dk, dv;
  dk.init(ldk, wv, lane);
  dv.init(ldv, wv, lane);
  // K/V tiles of round r: tile t_lo + r KS + g for key group g
  auto load_kv = [&](int round, int stage) {
#pragma unroll
    for (int g0 = 0; g0 < KS / TEAMS; g0++) {
      const int g = g0 * TEAMS + team, t = t_lo + round * KS + g;
      if (KS > 1 && t > t_hi) break;
      const unsigned dst = lds0 + (g * 2 + stage) * (2 * TILE);
      if (t * 64 + 64 <= S) {
        dk.issue(kbase + (int64_t)t * 64 * ldk, dst, wv);
        dv.issue(vbase + (int64_t)t * 64 * ldv, dst + TILE, wv);
      } else {
        dma_tile<64, D>(kbase, ldk, t * 64, S, dst, wv, lane);
        dma_tile<64, D>(vbase, ldv, t * 64, S, dst + TILE, wv, lane);
      }
    }
  };
  const float sc2 = scale * LOG2E;
  const float cap_c1 = CAP ? 2.f * sc2 / cap : 0.f, cap_l2 = cap * LOG2E;  // soft-cap: see cap_tanh
  // Scores and their maximum are held in log2 units; at head_dim 64 as the products give them (CAP: capped), so that
  // no constant's rounding gets into LSE through the maximum (log2 units: a sixth more LSE error)
  constexpr bool LOG2_UNITS = D != 64;
  const float to_log2 = CAP ? LOG2E : sc2, to_ln = CAP ? 1.f : scale;  // of a difference, of a score (!LOG2_UNITS)
  auto exp_of = [&](float x, float ref) { return LOG2_UNITS ? fexp2(x - ref) : fexp2((x - ref) * to_log2); };
  FragAddr<D> fa;
  fa.init(lane);

  load_kv(0, 0);
  dma_wait_all();
  __syncthreads();
  const int rounds = (t_hi - t_lo + KS) / KS;
  for (int r0 = 0; r0 < rounds; r0++) {
    const int cur = r0 & 1;
    if (r0 + 1 < rounds) load_kv(r0 + 1, cur ^ 1);
    const int t = t_lo + r0 * KS + ks, j0 = t * 64;
    // skip tiles this wave cannot see at all
    const bool visible = (KS == 1 || t <= t_hi) && (j0 <= iw0 + 31) && (window < 0 || j0 + 63 >= iw0 - window);
    if (visible) {
      const unsigned char* sk = smem + (ks * 2 + cur) * (2 * TILE);
      const unsigned char* sv = sk + TILE;
      f32x16 st[2];
#pragma unroll
      for (int jt = 0; jt < 2; jt++)
#pragma unroll
        for (int r = 0; r < 16; r++) st[jt][r] = 0.f;
#pragma unroll
      for (int s = 0; s < D / 16; s++)
#pragma unroll
        for (int jt = 0; jt < 2; jt++)
          st[jt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.load_kc(sk, jt * 32, s), qf[s], st[jt], 0, 0, 0);
      if (CAP) {
#pragma unroll
        for (int jt = 0; jt < 2; jt++)
#pragma unroll
          for (int r = 0; r < 16; r++) st[jt][r] = (LOG2_UNITS ? cap_l2 : cap) * cap_tanh_of<D>(st[jt][r], cap_c1, scale, cap);
      }
      const bool need_mask = (j0 + 63 > iw0) || (window >= 0 && j0 < iw0 + 31 - window);
      if (need_mask) {
#pragma unroll
        for (int jt = 0; jt < 2; jt++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int j = j0 + jt * 32 + (r >> 2) * 8 + lhi * 4 + (r & 3);
            const bool ok = (j <= qi) && (window < 0 || j >= qi - window);
            st[jt][r] = ok ? st[jt][r] : -INFINITY;
          }
      }
      float mt = -INFINITY;
#pragma unroll
      for (int jt = 0; jt < 2; jt++)
#pragma unroll
        for (int r = 0; r < 16; r++) mt = fmaxf(mt, st[jt][r]);
      if (!CAP && LOG2_UNITS) mt *= sc2;  // sc2 > 0: the max commutes with the scaling
      mt = half_swap_max(mt);
      // Lazy rescaling: the running reference m only moves when some row's maximum grew by more
      // than 2^8; until then exp2(s - m) <= 256 stays well inside fp32/bf16 range and the
      // 64-register rescale of O is skipped (wave-uniform decision).
      // head_dim 64: by more than 2, or the largest terms carry the rounding of a large exponent (rms error of LSE over 50 shapes against the
      // one-wave kernels': 1.05 with 2^8, 1.003 with 2; 4 x 1024, 16 heads over 4: 21.7 -> 22.4 us).
      const bool grow = LOG2_UNITS ? mt > m + 8.f : (mt - m) * to_log2 > 1.f;
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        const float m_new = fmaxf(m, mt);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = exp_of(m, m_use);  // m = -inf -> 0
        lsum *= alpha;
        m = m_new;
#pragma unroll
        for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
          for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
      }
      const float m_use = (m == -INFINITY) ? 0.f : m;
#pragma unroll
      for (int jt = 0; jt < 2; jt++)
#pragma unroll
        for (int r = 0; r < 16; r++)
          st[jt][r] = CAP || !LOG2_UNITS ? exp_of(st[jt][r], m_use) : fexp2(__builtin_fmaf(st[jt][r], sc2, -m_use));
      bf16x8 pb[4];
#pragma unroll
      for (int u = 0; u < 4; u++) pb[u] = pack_bf16x8(st[u >> 1], (u & 1) * 8);
      // Row sum.  D = 128: of the probabilities AS THE P.V PRODUCT SEES THEM (bf16), two per instruction
      // (v_dot2c_f32_bf16 against a pair of ones, two accumulators): numerator and denominator
      // of the softmax then carry the same rounding.  D = 64: in fp32, as the one-wave-per-query kernel that
      // took this head_dim before sums them (LSE to 4e-8 instead of 3e-5; the kernel has registers and issue slots to spare).
      if constexpr (D == 64) {  // pairwise
        float ps[16];
#pragma unroll
        for (int r = 0; r < 16; r++) ps[r] = st[0][r] + st[1][r];
#pragma unroll
        for (int w = 8; w > 0; w >>= 1)
#pragma unroll
          for (int r = 0; r < w; r++) ps[r] += ps[r + w];
        lsum += ps[0];
      } else {
        float ps0 = 0.f, ps1 = 0.f;
#pragma unroll
        for (int u = 0; u < 4; u++) {
          ps0 = dot2_ones(pb[u], 0, ps0);
          ps1 = dot2_ones(pb[u], 1, ps1);
          ps0 = dot2_ones(pb[u], 2, ps0);
          ps1 = dot2_ones(pb[u], 3, ps1);
        }
        lsum += ps0 + ps1;
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int dt = 0; dt < D / 32; dt++)
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.load_tr(sv, u * 16, dt), pb[u], o[dt], 0, 0, 0);
    }
    dma_wait_all();
    __syncthreads();
  }
  float ltot = half_swap_sum(lsum);
  float zeros = 0.f;  // of what is stored: NaN if a value is not finite (see redo_rows)
  auto store4 = [&](int dt, int g, const f32x4& v, float mul) {
    bf16* op = O + ((int64_t)b * S + qic) * ldo + h * D;
    Pack4 pk;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float x = v[e] * mul;
      if (D == 64) zeros = __builtin_fmaf(x, 0.f, zeros);
      pk.e[e] = f2bf(x);
    }
    *reinterpret_cast<u32x2*>(op + dt * 32 + g * 8 + lhi * 4) = pk.u;
  };
  if constexpr (KS == 1) {
    const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
    if (qi < S) {
#pragma unroll
      for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
        for (int g = 0; g < 4; g++)
          store4(dt, g, f32x4{o[dt][g * 4], o[dt][g * 4 + 1], o[dt][g * 4 + 2], o[dt][g * 4 + 3]}, inv);
    }
  } else {
    // statistics of the key groups behind the stages, then the accumulators, scaled to the common maximum,
    // in their place (the last round ended in a barrier)
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    f32x2* stats = reinterpret_cast<f32x2*>(smem + KS * 4 * TILE) + qw * (KS * 32) + l32;
    if (lhi == 0) stats[ks * 32] = f32x2{m, ltot};
    __syncthreads();
    const float m_own = m;
#pragma unroll
    for (int g = 0; g < KS; g++) {
      const f32x2 st = stats[g * 32];
      m = g == 0 ? st[0] : fmaxf(m, st[0]);
    }
    const float m_use = (m == -INFINITY) ? 0.f : m;
    ltot = 0.f;
#pragma unroll
    for (int g = 0; g < KS; g++) {
      const f32x2 st = stats[g * 32];
      ltot += st[1] * exp_of(st[0], m_use);
    }
    const float alpha = exp_of(m_own, m_use), inv = ltot > 0.f ? 1.f / ltot : 0.f;
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
    add_partials<D, KS>(smem, o, qw, ks, lane, [&](int u, const f32x4& v) {
      if (qi < S) store4(u >> 2, u & 3, v, inv);
    });
  }
  // (every wave of the row looks at its LSE: a row whose scores are all -inf sums to zero, not to NaN, until it is done over)
  if (qi < S && lhi == 0 && (D == 64 || ks == 0)) {
    const float lse = LOG2_UNITS ? (m + log2f(ltot)) * LN2 : m * to_ln + __logf(ltot);
    if (D == 64) zeros = __builtin_fmaf(lse, 0.f, zeros);
    if (ks == 0) LSE[((int64_t)b * H + h) * S + qi] = lse;
  }
  if constexpr (D == 64)
    redo_rows(zeros, [&](int r) {
      const int64_t at = (int64_t)b * S + iw0 + r;
      redo_fwd<CAP>(Q + at * ldq + h * D, kbase, ldk, vbase, ldv, O + at * ldo + h * D, ks == 0 ? LSE + ((int64_t)b * H + h) * S + iw0 + r : nullptr,
                    iw0 + r, window, scale, cap, lane, ks * (D / KS), (ks + 1) * (D / KS));
    });
}

// ---------------------------------------------------------------------------------------
// dQ.  Same tiling and grid as the forward; K/V tiles stream through LDS.
// ---------------------------------------------------------------------------------------
template <int D, bool CAP, int QW, int KS>
__device__ __forceinline__ void attn_dq(
    const bf16* __restrict__ Q, const bf16* __restrict__ K, const bf16* __restrict__ V,
    const bf16* __restrict__ O, const bf16* __restrict__ dO, const float* __restrict__ LSE,
    float* __restrict__ DELTA, bf16* __restrict__ dQ, int S, int H, int KH, int64_t ldq, int64_t ldk,
    int64_t ldv, int64_t ldo, int64_t lddo, int64_t lddq, float scale, int window, float cap, unsigned id, unsigned nwg, unsigned char* smem) {
#include "attn_dq.h"
}

template <int D, bool CAP, int QW, int KS>
__global__ __launch_bounds__(QW * KS * 64, 2) void attn_bwd_dq_kernel(
    const bf16* __restrict__ Q, const bf16* __restrict__ K, const bf16* __restrict__ V,
    const bf16* __restrict__ O, const bf16* __restrict__ dO, const float* __restrict__ LSE,
    float* __restrict__ DELTA, bf16* __restrict__ dQ, int S, int H, int KH, int64_t ldq, int64_t ldk,
    int64_t ldv, int64_t ldo, int64_t lddo, int64_t lddq, float scale, int window, float cap) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const unsigned id = blockIdx.x, nwg = gridDim.x;
#include "attn_dq.h"
}

// ---------------------------------------------------------------------------------------
// dK/dV.  grid = ceil(S/(32 KW))*KH*B workgroups of KW x QS waves; wave (kw, qs) owns keys j0+32kw..+31
// (K fragments stay in registers) and every QS-th of the iterations over the query heads of its
// group and the 32-row Q/dO tiles from the diagonal downwards.  LDS: per query group 2 stages of
// (Q | dO | lse 128 B | delta 128 B), then the V tile of 32 KW keys.
// KW = 4, QS = 1: two workgroups per CU, no reduction; what a grid that fills the GPU takes.
// KW = 2, QS = 4: one workgroup of eight waves per CU, half the keys and a quarter of the serial chain; the
// four partial sums are added through LDS in group order.  See dkv_split.
// ---------------------------------------------------------------------------------------
// dK/dV's LDS: stages and V tile, or the parked partial sums
constexpr int smem_kv(int D, int KW, int QS) {
  const int run = QS * 2 * (2 * 32 * D * 2 + 256) + KW * 32 * D * 2, sums = QS > 1 ? KW * QS * 32 * D * 4 : 0;
  return run > sums ? run : sums;
}
// waves of the split forward and dQ kernels: what 160 KB of stages hold
template <int D> constexpr int SPLIT_QW = D == 128 ? 4 : 2;
template <int D> constexpr int SPLIT_KS = D == 128 ? 2 : 4;

// BOTH: dQ in the same launch.  dK/dV's workgroups come first, longest first, then dQ's, longest first, so that the long ones of the second kind start where
// the short ones of the first end.  Takes calls whose workgroups nearly all find room at once, where each kernel by itself waits for its longest chains (bwd_form).
// Nobody hands delta over then: the workgroup forms that of all query rows it will meet itself, as dQ does, behind the rest of its LDS.
template <int D, bool CAP, int KW, int QS, bool BOTH = false>
__global__ __launch_bounds__(KW * QS * 64, 2) void attn_bwd_dkv_kernel(
    const bf16* __restrict__ Q, const bf16* __restrict__ K, const bf16* __restrict__ V,
    const bf16* __restrict__ dO, const float* __restrict__ LSE, const float* __restrict__ DELTA,
    bf16* __restrict__ dK, bf16* __restrict__ dV, int S, int H, int KH, int64_t ldq, int64_t ldk,
    int64_t ldv, int64_t lddo, int64_t lddk, int64_t lddv, float scale, int window, float cap,
    const bf16* __restrict__ O, bf16* __restrict__ dQ, int64_t ldo, int64_t lddq, int nkv) {  // (BOTH)
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  if constexpr (BOTH) {
    if ((int)blockIdx.x >= nkv) {
      constexpr int QW = QS > 1 ? SPLIT_QW<D> : 4, KS = QS > 1 ? SPLIT_KS<D> : 1;
      const unsigned id = blockIdx.x - nkv, nwg = gridDim.x - nkv;
      float* const DELTA = nullptr;
      if constexpr (CAP && D == 128) {
        attn_dq<D, CAP, QW, KS>(Q, K, V, O, dO, LSE, DELTA, dQ, S, H, KH, ldq, ldk, ldv, ldo, lddo, lddq, scale, window, cap, id, nwg, smem);
      } else {
#include "attn_dq.h"
      }
      return;
    }
  }
  const unsigned nwg = BOTH ? nkv : gridDim.x;
  constexpr int QT = 32;                   // query rows per iteration
  constexpr int TILE = QT * D * 2;
  constexpr int STAGE = 2 * TILE + 256;  // Q | dO | lse, delta
  constexpr int KT = KW * 32;            // keys of the workgroup
  constexpr int TEAMS = KW * QS / 4;     // tiles are fetched by teams of 4 waves
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform for the compiler too
  const int l32 = lane & 31, lhi = lane >> 5;
  const int kw = wave % KW, qs = wave / KW;
  // key tile 0 is seen by every query: rank order is already longest first
  const WgCoord wg = decode_wg(blockIdx.x, (int)(nwg / ((S + KT - 1) / KT)), 1);
  const int kt = wg.rank;
  const int b = wg.group / KH, kh = wg.group % KH;
  const int rep = H / KH;
  const int j0 = kt * KT;
  const int jw0 = j0 + kw * 32;
  const int kj = jw0 + l32;  // this lane's key
  const int kjc = min(kj, S - 1);

  // K fragments of this wave's 32 keys stay in registers; the V tile of the whole workgroup
  // is parked in LDS behind the stages and re-read as B operand every iteration
  bf16x8 kf[D / 16];
  {
    const bf16* kp = K + ((int64_t)b * S + kjc) * ldk + kh * D + lhi * 8;
#pragma unroll
    for (int s = 0; s < D / 16; s++) kf[s] = *reinterpret_cast<const bf16x8*>(kp + s * 16);
  }
  f32x16 dk[D / 32], dv[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) { dk[dt][r] = 0.f; dv[dt][r] = 0.f; }

  const int i_hi = window >= 0 ? min(S - 1, j0 + KT - 1 + window) : S - 1;
  const int t_lo = j0 / QT;
  const int t_hi = i_hi / QT;  // inclusive
  const int ntile = t_hi - t_lo + 1;
  const int total = ntile * rep;  // flattened (head, tile) iteration space
  const float sc2 = scale * LOG2E;
  const float cap_c1 = CAP ? 2.f * sc2 / cap : 0.f, cap_l2 = cap * LOG2E;  // soft-cap: see cap_tanh
  const unsigned lds0 = lds_addr_of(smem);
  const int wv = wave & 3, team = wave >> 2;
  const unsigned char* sgrp = smem + qs * (2 * STAGE);  // this query group's stages

  float sreg = 0.f;
  TileDma<QT, D> tq, tdo;
  tq.init(ldq, wv, lane);
  tdo.init(lddo, wv, lane);
  // (head, tile) of the next iteration to load of each query group this team fetches for, and of this
  // wave's own group (its row statistics); heads of the K/V group outermost
  struct Iter { int h, t; };
  auto advance = [&](Iter& x, int n) {
    x.t += n;
    while (x.t > t_hi) {
      x.t -= ntile;
      ++x.h;
    }
  };
  Iter own{kh * rep, t_lo}, ld[QS / TEAMS];
  advance(own, qs);
#pragma unroll
  for (int g = 0; g < QS / TEAMS; g++) {
    ld[g] = Iter{kh * rep, t_lo};
    advance(ld[g], g * TEAMS + team);
  }
  auto load_tile = [&](int round, int stage) {
#pragma unroll
    for (int g = 0; g < QS / TEAMS; g++) {
      const int grp = g * TEAMS + team;
      if (QS > 1 && round * QS + grp >= total) break;
      const int hq = ld[g].h, t = ld[g].t;
      advance(ld[g], QS);
      const unsigned dst = lds0 + (grp * 2 + stage) * STAGE;
      if (t * QT + QT <= S) {
        tq.issue(Q + ((int64_t)b * S + t * QT) * ldq + hq * D, dst, wv);
        tdo.issue(dO + ((int64_t)b * S + t * QT) * lddo + hq * D, dst + TILE, wv);
      } else {
        dma_tile<QT, D>(Q + (int64_t)b * S * ldq + hq * D, ldq, t * QT, S, dst, wv, lane);
        dma_tile<QT, D>(dO + (int64_t)b * S * lddo + hq * D, lddo, t * QT, S, dst + TILE, wv, lane);
      }
    }
    if (kw == 0 && (QS == 1 || round * QS + qs < total)) {
      const int ii = min(own.t * QT + l32, S - 1);
      const float* src = BOTH || lane < QT ? LSE : DELTA;
      sreg = src[((int64_t)b * H + own.h) * S + ii];  // consumed by store_stats a whole iteration later
    }
  };
  // (the log2 scaling of LSE happens here, not at the load: touching the loaded value there
  // would make wave 0 wait out the memory latency at the top of every iteration)
  auto store_stats = [&](int stage) {
    if (kw == 0) reinterpret_cast<float*>(smem + (qs * 2 + stage) * STAGE + 2 * TILE)[lane] = lane < QT ? sreg * LOG2E : sreg;
  };

  FragAddr<D, BOTH && CAP && D == 128> fa;  // (short of registers)
  fa.init(lane);
  const unsigned char* svt = smem + QS * 2 * STAGE;  // [KT keys][D] V tile
  if (team == 0) dma_tile<KT, D>(V + (int64_t)b * S * ldv + kh * D, ldv, j0, S, lds0 + QS * 2 * STAGE, wv, lane);
  load_tile(0, 0);
  float* const own_delta = reinterpret_cast<float*>(smem + smem_kv(D, KW, QS));  // [head of the group][rows from t_lo QT]
  if constexpr (BOTH) {
    for (int u = wave; u < total; u += KW * QS) {
      const int hq = u / ntile;
      const int64_t row = (int64_t)b * S + min((t_lo + u - hq * ntile) * QT + l32, S - 1);
      const bf16* op = O + row * ldo + (kh * rep + hq) * D + lhi * 8;
      const bf16* dp = dO + row * lddo + (kh * rep + hq) * D + lhi * 8;
      float dlt = 0.f;
#pragma unroll
      for (int s = 0; s < D / 16; s++) {
        const bf16x8 of = *reinterpret_cast<const bf16x8*>(op + s * 16), df = *reinterpret_cast<const bf16x8*>(dp + s * 16);
#pragma unroll
        for (int e = 0; e < 8; e++) dlt += bf2f(of[e]) * bf2f(df[e]);
      }
      dlt = half_swap_sum(dlt);
      if (lhi == 0) own_delta[u * QT + l32] = -dlt;
    }
  }
  store_stats(0);
  dma_wait_all();
  __syncthreads();
  // One round on the tiles in stage CUR (a compile-time constant, so that every LDS address
  // below is a loop-invariant register plus an immediate); `t` is the query-tile index of this wave's.
  auto iteration = [&](auto cur_tag, int round, int t, bool more) {
    constexpr int CUR = decltype(cur_tag)::value;
    if (more) {
      advance(own, QS);
      load_tile(round + 1, CUR ^ 1);
    }
    const int ib = t * QT;  // first query of the tile
    // this wave sees the tile iff some i in [ib, ib+QT) has j <= i <= j + window for its keys
    const bool visible = (QS == 1 || round * QS + qs < total) && (ib + QT - 1 >= jw0) && (window < 0 || ib <= jw0 + 31 + window);
    if (visible) {
      const unsigned char* sq = sgrp + CUR * STAGE;
      const unsigned char* so = sq + TILE;
      const float* slse = reinterpret_cast<const float*>(sq + 2 * TILE);
      const float* sdel = BOTH ? own_delta + (round * QS + qs) * QT : slse + QT;
      // every (query, key) pair of the tile is visible unless the tile touches the diagonal, the
      // window edge or the end of the sequence
      const bool need_mask = (ib < jw0 + 31) || (ib + QT > S) || (window >= 0 && ib + QT - 1 > jw0 + window);
      f32x16 sa, dpa;
      // accumulator rows are queries i = ib + 8*(r/4) + 4*lhi + r%4; column = key kj.
      // dP starts from -delta of its query (what DELTA holds): the products then give dP - delta
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f32x4 d4 = *reinterpret_cast<const f32x4*>(sdel + g * 8 + lhi * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) { sa[g * 4 + e] = 0.f; dpa[g * 4 + e] = d4[e]; }
      }
#pragma unroll
      for (int s = 0; s < D / 16; s++) {
        sa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.load_kc(sq, 0, s), kf[s], sa, 0, 0, 0);
        dpa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.load_kc(so, 0, s), fa.load_kc(svt, kw * 32, s), dpa, 0, 0, 0);
      }
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int il = g * 8 + lhi * 4;
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(slse + il);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int r = g * 4 + e;
          const int i = ib + il + e;
          float s = sa[r], chain = 1.f, p;
          if (CAP) {
            const float th = cap_tanh_of<D>(s, cap_c1, scale, cap);
            p = fexp2(__builtin_fmaf(th, cap_l2, -l4[e]));
            chain = 1.f - th * th;
          } else {
            p = fexp2(__builtin_fmaf(s, sc2, -l4[e]));
          }
          if (need_mask) {
            const bool ok = (kj <= i) && (i < S) && (window < 0 || kj >= i - window);
            p = ok ? p : 0.f;
          }
          sa[r] = p;
          dpa[r] = p * dpa[r] * chain;
        }
      }
      bf16x8 pb[2], dsb[2];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        pb[u] = pack_bf16x8(sa, u * 8);
        dsb[u] = pack_bf16x8(dpa, u * 8);
      }
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int dt = 0; dt < D / 32; dt++) {
          dv[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.load_tr(so, u * 16, dt), pb[u], dv[dt], 0, 0, 0);
          dk[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.load_tr(sq, u * 16, dt), dsb[u], dk[dt], 0, 0, 0);
        }
    }
    if (more) store_stats(CUR ^ 1);
    dma_wait_all();
    __syncthreads();
  };
  {
    const int rounds = (total + QS - 1) / QS;
    Iter cur{0, t_lo};  // query tile being consumed
    advance(cur, qs);
    for (int it = 0; it < rounds; it += 2) {
      iteration(std::integral_constant<int, 0>(), it, cur.t, it + 1 < rounds);
      advance(cur, QS);
      if (it + 1 < rounds) {
        iteration(std::integral_constant<int, 1>(), it + 1, cur.t, it + 2 < rounds);
        advance(cur, QS);
      }
    }
  }
  bf16* kp = dK + ((int64_t)b * S + kjc) * lddk + kh * D;
  bf16* vp = dV + ((int64_t)b * S + kjc) * lddv + kh * D;
  float zeros = 0.f;  // see redo_rows
  auto store4 = [&](bf16* p, int dt, int g, const f32x4& v, float mul) {
    Pack4 pk;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float x = v[e] * mul;
      if (D == 64) zeros = __builtin_fmaf(x, 0.f, zeros);
      pk.e[e] = f2bf(x);
    }
    *reinterpret_cast<u32x2*>(p + dt * 32 + g * 8 + lhi * 4) = pk.u;
  };
  if constexpr (QS == 1) {
    // A row leaves in 16-byte pieces, one instruction after the other: the compiler's own order, which comes back to a
    // line after eight others, costs 4 sequences of 1024, 32 heads 14 us of 170 and 16 of 512 34 us of 290 (backward).
    if (kj < S) {
#pragma unroll
      for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          store4(kp, dt, g, f32x4{dk[dt][g * 4], dk[dt][g * 4 + 1], dk[dt][g * 4 + 2], dk[dt][g * 4 + 3]}, scale);
          store4(vp, dt, g, f32x4{dv[dt][g * 4], dv[dt][g * 4 + 1], dv[dt][g * 4 + 2], dv[dt][g * 4 + 3]}, 1.f);
          __builtin_amdgcn_sched_barrier(0);  // in this order: see above
        }
    }
  } else {
    // the stages are free: the last round ended in a barrier; dK first, then dV in the same space
    add_partials<D, QS>(smem, dk, kw, qs, lane, [&](int u, const f32x4& v) {
      if (kj < S) store4(kp, u >> 2, u & 3, v, scale);
    });
    __syncthreads();
    add_partials<D, QS>(smem, dv, kw, qs, lane, [&](int u, const f32x4& v) {
      if (kj < S) store4(vp, u >> 2, u & 3, v, 1.f);
    });
  }
  if constexpr (D == 64)
    redo_rows(zeros, [&](int r) {
      const int64_t seq = (int64_t)b * S, at = seq + jw0 + r, row = ((int64_t)b * H + kh * rep) * S;
      redo_dkv<CAP>(Q + seq * ldq + kh * rep * D, ldq, dO + seq * lddo + kh * rep * D, lddo, LSE + row, BOTH ? own_delta - t_lo * QT : DELTA + row,
                    BOTH ? ntile * QT : S, K + at * ldk + kh * D,
                    V + at * ldv + kh * D, dK + at * lddk + kh * D, dV + at * lddv + kh * D, jw0 + r, S, rep, window, scale, cap, lane,
                    qs * (D / QS), (qs + 1) * (D / QS));
    });
}

// ---------------------------------------------------------------------------------------
// Any head_dim (<= 256): one wave per (batch, head, query); scores staged in LDS.
// Takes what the MFMA kernels do not: other head_dims and unaligned views.
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(64) void attn_fwd_generic(
    const bf16* __restrict__ Q, const bf16* __restrict__ K, const bf16* __restrict__ V,
    bf16* __restrict__ O, float* __restrict__ LSE, int S, int H, int KH, int D, int64_t ldq,
    int64_t ldk, int64_t ldv, int64_t ldo, float scale, int window, float cap) {
  extern __shared__ float sc[];  // S floats
  const int i = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int kh = h / (H / KH);
  const int lane = threadIdx.x;
  const bf16* q = Q + ((int64_t)b * S + i) * ldq + h * D;
  const int lo = window >= 0 ? max(0, i - window) : 0;
  float mx = -INFINITY;
  for (int j = lo + lane; j <= i; j += 64) {
    const bf16* k = K + ((int64_t)b * S + j) * ldk + kh * D;
    float s = 0.f;
    for (int d = 0; d < D; d++) s += bf2f(q[d]) * bf2f(k[d]);
    s *= scale;
    if (cap > 0.f) s = cap * tanhf(s / cap);
    sc[j] = s;
    mx = fmaxf(mx, s);
  }
  mx = wave_max(mx);
  float sm = 0.f;
  for (int j = lo + lane; j <= i; j += 64) sm += __expf(sc[j] - mx);
  sm = wave_sum(sm);
  const float lse = mx + __logf(sm);
  __syncthreads();
  for (int d = lane; d < D; d += 64) {
    float acc = 0.f;
    for (int j = lo; j <= i; j++) {
      const float p = bf2f(f2bf(__expf(sc[j] - lse)));
      acc += p * bf2f(V[((int64_t)b * S + j) * ldv + kh * D + d]);
    }
    O[((int64_t)b * S + i) * ldo + h * D + d] = f2bf(acc);
  }
  if (lane == 0) LSE[((int64_t)b * H + h) * S + i] = lse;
}

// dQ directly; dK/dV accumulated with fp32 atomics into [B*S, KH*D] workspaces.
__global__ __launch_bounds__(64) void attn_bwd_generic(
    const bf16* __restrict__ Q, const bf16* __restrict__ K, const bf16* __restrict__ V,
    const bf16* __restrict__ O, const bf16* __restrict__ dO, const float* __restrict__ LSE,
    bf16* __restrict__ dQ, float* __restrict__ dKf, float* __restrict__ dVf, int S, int H, int KH,
    int D, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo, int64_t lddo, int64_t lddq,
    float scale, int window, float cap) {
  extern __shared__ float sh[];  // p[S], ds[S]
  float* sp = sh;
  float* sds = sh + S;
  const int i = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int kh = h / (H / KH);
  const int lane = threadIdx.x;
  const bf16* q = Q + ((int64_t)b * S + i) * ldq + h * D;
  const bf16* o = O + ((int64_t)b * S + i) * ldo + h * D;
  const bf16* go = dO + ((int64_t)b * S + i) * lddo + h * D;
  const float lse = LSE[((int64_t)b * H + h) * S + i];
  const int lo = window >= 0 ? max(0, i - window) : 0;
  float dl = 0.f;
  for (int d = lane; d < D; d += 64) dl += bf2f(o[d]) * bf2f(go[d]);
  dl = wave_sum(dl);
  for (int j = lo + lane; j <= i; j += 64) {
    const bf16* k = K + ((int64_t)b * S + j) * ldk + kh * D;
    const bf16* v = V + ((int64_t)b * S + j) * ldv + kh * D;
    float s = 0.f, dp = 0.f;
    for (int d = 0; d < D; d++) {
      s += bf2f(q[d]) * bf2f(k[d]);
      dp += bf2f(go[d]) * bf2f(v[d]);
    }
    s *= scale;
    float chain = 1.f;
    if (cap > 0.f) {
      const float th = tanhf(s / cap);
      s = cap * th;
      chain = 1.f - th * th;
    }
    const float p = __expf(s - lse);
    sp[j] = bf2f(f2bf(p));
    sds[j] = bf2f(f2bf(p * (dp - dl) * chain));
  }
  __syncthreads();
  for (int d = lane; d < D; d += 64) {
    float acc = 0.f;
    const float qd = bf2f(q[d]), god = bf2f(go[d]);
    for (int j = lo; j <= i; j++) {
      acc += sds[j] * bf2f(K[((int64_t)b * S + j) * ldk + kh * D + d]);
      atomicAdd(&dKf[((int64_t)b * S + j) * KH * D + kh * D + d], sds[j] * qd * scale);
      atomicAdd(&dVf[((int64_t)b * S + j) * KH * D + kh * D + d], sp[j] * god);
    }
    dQ[((int64_t)b * S + i) * lddq + h * D + d] = f2bf(acc * scale);
  }
}

__global__ void strided_cast_f32_bf16(const float* __restrict__ in, bf16* __restrict__ out,
                                      int64_t rows, int cols, int64_t ldo) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * cols) return;
  out[(i / cols) * ldo + i % cols] = f2bf(in[i]);
}

// What the MFMA kernels take: head_dim 128, or 64 at lengths the one-wave-per-query kernels take too (the two
// head_dims of the configurations that train; any other one, and unaligned views, stay on those kernels, which
// hold a row of scores in LDS), 16-byte aligned operands.  head_dim 64, 4 heads, 4 sequences of 512: forward 620 -> 19 us,
// backward 1850 -> 40 us; 8 heads over 2, 2 sequences of 2048: 6740 -> 36 us, 21100 -> 310 us.
bool fast_ok(int D, int S, int max_s, const void* q, const void* k, const void* v, const void* o, int64_t ldq,
             int64_t ldk, int64_t ldv, int64_t ldo) {
  return (D == 128 || (D == 64 && S <= max_s)) && aligned16(q) && aligned16(k) && aligned16(v) && aligned16(o) && ldq % 8 == 0 &&
         ldk % 8 == 0 && ldv % 8 == 0 && ldo % 8 == 0;
}
// A window that reaches past the first key from the last query hides nothing: global.  The kernels add the window to
// positions, and sums up to 2 S fit; from windows near 2^31 they would wrap, the last query tile of a key would come
// out before its first, and dK/dV's walk over the tiles would not end.
int32_t reach(int32_t window, int32_t S) { return window >= S ? -1 : window; }
constexpr int GENERIC_MAX_S_FWD = 16384, GENERIC_MAX_S_BWD = 8192;  // 64 KB of LDS: one, two floats per key

bool bwd_fast_ok(const void* q, const void* k, const void* v, const void* o, const void* d_o, const void* dq, const void* dk,
                 const void* dv, int S, int D, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo, int64_t lddo, int64_t lddq,
                 int64_t lddk, int64_t lddv) {
  return fast_ok(D, S, GENERIC_MAX_S_BWD, q, k, v, o, ldq, ldk, ldv, ldo) && aligned16(d_o) && aligned16(dq) && aligned16(dk) &&
         aligned16(dv) && lddo % 8 == 0 && lddq % 8 == 0 && lddk % 8 == 0 && lddv % 8 == 0;
}

// forward, dQ: stages (the parked partial sums fit in their place), statistics of the forward's merge
constexpr int smem_q(int D, int QW, int KS) { return KS * 2 * 2 * 64 * D * 2 + (KS > 1 ? QW * KS * 32 * 8 : 0); }
// both in one launch; rows: query rows that the longest workgroup of dK/dV meets
template <int D, int QW, int KS, int KW, int QS>
constexpr int smem_both(int rows) {
  const int q = smem_q(D, QW, KS), kv = smem_kv(D, KW, QS) + rows * 4;
  return q > kv ? q : kv;
}

// The most query rows that a workgroup of dK/dV meets where both run in one launch: their delta lies behind the 146 KB of its split form
constexpr int BOTH_ROWS = 2112;

// dynamic-LDS limits of the backward kernels, set once per process
template <int D, bool CAP>
void bwd_fast_attributes_of() {
  constexpr int QW = SPLIT_QW<D>, KS = SPLIT_KS<D>;
  constexpr auto ATTR = hipFuncAttributeMaxDynamicSharedMemorySize;
  (void)hipFuncSetAttribute((const void*)attn_bwd_dkv_kernel<D, CAP, 4, 1>, ATTR, smem_kv(D, 4, 1));
  (void)hipFuncSetAttribute((const void*)attn_bwd_dkv_kernel<D, CAP, 2, 4>, ATTR, smem_kv(D, 2, 4));
  (void)hipFuncSetAttribute((const void*)attn_bwd_dq_kernel<D, CAP, 4, 1>, ATTR, smem_q(D, 4, 1));
  (void)hipFuncSetAttribute((const void*)attn_bwd_dq_kernel<D, CAP, QW, KS>, ATTR, smem_q(D, QW, KS));
  (void)hipFuncSetAttribute((const void*)attn_bwd_dkv_kernel<D, CAP, 4, 1, true>, ATTR, smem_both<D, 4, 1, 4, 1>(BOTH_ROWS));
  (void)hipFuncSetAttribute((const void*)attn_bwd_dkv_kernel<D, CAP, 2, 4, true>, ATTR, smem_both<D, QW, KS, 2, 4>(BOTH_ROWS));
}
void bwd_fast_attributes() {
  static std::once_flag once;
  std::call_once(once, [] {
    bwd_fast_attributes_of<128, true>();
    bwd_fast_attributes_of<128, false>();
    bwd_fast_attributes_of<64, true>();
    bwd_fast_attributes_of<64, false>();
  });
}

// Whether the forward and dQ take their split kernels.  While few workgroups of 128 queries share a CU, a wave has a SIMD to itself and its
// chain of key tiles is what takes the time; a short chain is over before the split pays for its merge.  Forward | dQ, us a call,
// plain -> split, at n workgroups:
// head_dim 128 (split: eight waves per workgroup, one on a CU), n <= 256: 1 tile 6.4 -> 8.1 | 2.4 slower, 4 tiles 12.2 -> 12.7 | 0.4 slower,
// 8 tiles 17.4 -> 16.7 | 2.2 faster, 64 tiles 80.9 -> 65.5 | 37 faster.  Up to 512 the plain kernel has all of its workgroups on the GPU
// at once and the split one comes in two rounds: n = 320, 20 tiles 32.8 -> 27.7 | 12 faster, n = 384, 4 tiles 16.4 -> 22.6 | 10 slower,
// 16 tiles 29.2 -> 29.4 | 1.4 faster, n = 512, 16 tiles 31.2 -> 33.2 | 2.4 slower, 64 tiles 93.5 -> 79.5 | 31 faster.  From n = 513 on the plain
// kernels' two workgroups per CU keep the SIMDs busy by themselves: n = 640, 20 tiles 38 -> 50 | 15 slower.
// head_dim 64 (split: 64 queries to a workgroup, twice as many of them), n <= 128: 1 tile 5.0 -> 6.2 | 1.6 slower, 2 tiles 7.2 -> 6.9 | 0.2 faster,
// 8 tiles 12.3 -> 8.9 | 5.1 faster; n = 192: 3 tiles 7.2 -> 11.3 | 6 slower; n = 256: 8 tiles 1.5 slower | 1.5 slower, 16 tiles 19.0 -> 16.9 | 4.4
// faster; n = 320, 24 tiles 0.9 faster | 0.4 faster; n = 384, 32 tiles 0.5 slower | 3.9 faster; n = 480, 24 tiles 27.3 -> 36.5 | 9.7 slower.
// A window of half the sequence or less makes the chains equal, and with nothing short to start late a second round costs all of one: n = 312, 18
// tiles 32.7 -> 43.6 | 5 slower, n = 288, 34 tiles 56 -> 46 | 15 faster, n = 384, 34 tiles 63 -> 73; head_dim 64, n = 192, 18 tiles 23 -> 24, n = 224, 26 tiles 33 -> 28.
bool even_chains(int S, int window) { return window >= 0 && window <= S / 2; }
template <int D>
bool q_split(int B, int S, int H, int window) {
  const int64_t n = (int64_t)((S + 127) / 128) * H * B;
  const int tiles = (window >= 0 && window < S - 128 ? window + 128 : S + 63) / 64;
  const bool even = even_chains(S, window);
  if (D == 128) return n <= 256 ? tiles >= 6 : even ? n <= 300 && tiles >= 26 : n <= 512 && tiles >= 12 + 14 * (n - 256) / 256;
  return n <= 128 ? tiles >= 2 : n <= 256 ? tiles >= (even ? 26 : 12) : !even && n <= 384 && tiles >= n / 12;
}
// Whether dK/dV takes the split kernel.  One workgroup per key tile and K/V head is little parallel work when the
// heads are few: 224 workgroups for 2 x 1777 tokens of 8 K/V heads leave the GPU waiting for those of the first key tile,
// which walk the four query heads of 1777 tokens one 32-row tile at a time with one wave per SIMD.  Backward (dQ included), us, plain -> split,
// at n workgroups of 128 keys and chains of so many 32-row tiles:
// head_dim 128, n <= 128: 2 tiles 17.3 -> 18.1, 3 tiles 23.0 -> 21.1, 64 tiles 129 -> 66; n = 192, 4 tiles 30.5 -> 33.5; n = 256, 16 tiles 58.1 -> 51.7;
// n = 320: 16 tiles 82 -> 84, 160 tiles 323 -> 200; n = 384: 8 tiles 47.4 -> 56.5, 32 tiles 102 -> 95, 48 tiles 149 -> 135;
// n = 448: 4 tiles 45.8 -> 62.8, 8 tiles 49.6 -> 66.7; n = 512: 32 tiles 106 -> 112, 64 tiles 206 -> 204, 128 tiles 344 -> 309; beyond, the split kernel's
// halved reuse of Q and dO costs more: n = 640: 128 tiles 408 -> 421, 256 tiles 678 -> 655; n = 768: 256 tiles 741 -> 766.
// head_dim 64: n <= 128: 2 tiles as many, 3 tiles 16.4 -> 14.4, 4 tiles 19.1 -> 15.2; n = 192: 3 tiles 17 -> 19, 5 tiles 21 -> 20; n = 320: 8 tiles 33.0 -> 33.5,
// 16 tiles 53 -> 50; n = 448: 4 tiles 28.6 -> 36.8, 32 tiles as many; n = 512: 32 tiles 70.2 -> 71.4, 48 tiles 107 -> 102; n = 544: 128 tiles 241 -> 217; n = 640:
// 128 tiles 237 -> 235, 256 tiles 434 -> 410; n = 768: 256 tiles 459 -> 477.
// Equal chains (see above), head_dim 128: n = 192: 12 tiles 53 -> 54, 20 tiles 71 -> 70, 52 tiles 145 -> 134; n = 384: 36 tiles 130 -> 135, 72 tiles 237 -> 236, 97 tiles 271 -> 260;
// n = 448: 97 tiles 294 -> 306, 272 tiles 742 -> 755; head_dim 64: n = 288: 20 tiles 57 -> 58, 28 tiles 68 -> 66; n = 384: 36 tiles as many, 68 tiles 138 -> 135; n = 512: 97 tiles 196 -> 197.
template <int D>
bool dkv_split(int B, int S, int H, int KH, int window) {
  const int64_t n = (int64_t)((S + 127) / 128) * KH * B;
  const int64_t chain = (int64_t)(H / KH) * (((window >= 0 && window < S - 128 ? window + 128 : S) + 31) / 32);
  if (n <= 128) return chain >= 3;
  if (even_chains(S, window)) return n <= 384 && chain >= (D == 128 ? (n <= 256 ? 20 : 60) : n <= 256 ? 4 : 20 + (n - 256) / 4);
  if (n > 512) return n <= 640 && chain >= (D == 128 ? 200 : 128);
  const int base = D == 128 ? 8 : 4;
  return chain >= (n <= 256 ? base : base + (D == 128 ? 56 : 36) * (n - 256) / 256);
}

// Query rows (of all heads of a group) that a workgroup of dK/dV meets at most, in whole tiles of 32
int both_rows(int S, int rep, int keys, int window) {
  const int n = window >= 0 && window < S - keys ? window + keys : S;
  return (int)std::min<int64_t>((int64_t)rep * ((n + 31) / 32 + 1) * 32, 1 << 30);
}
// Whether an output shares memory with an input: dK/dV may then leave only when dQ is done, and the other way round.
bool meets_inputs(const bf16* const (&in)[5], const int64_t (&in_ld)[5], const int (&in_heads)[5], const bf16* const (&out)[3], const int64_t (&out_ld)[3],
                  const int (&out_heads)[3], int64_t rows, int D) {
  for (int i = 0; i < 5; i++)
    for (int o = 0; o < 3; o++) {
      const bf16 *ie = in[i] + (rows - 1) * in_ld[i] + in_heads[i] * D, *oe = out[o] + (rows - 1) * out_ld[o] + out_heads[o] * D;
      if (in[i] < oe && out[o] < ie) return true;
    }
  return false;
}
// How dQ and dK/dV run: each plain or split, in a launch of its own, or both in one, where both are split (eight waves) or both plain (four).
struct BwdForm {
  bool split_q, split_kv, one;
};
// Each kernel by itself waits for its longest chains while the rest of the GPU idles, and a launch costs 2 us; but dK/dV has to form delta itself, about 1 us for
// 256 query rows with eight waves.  us, two launches -> one (heads / K/V heads):
// split, by workgroups of both: 64 wide, 4 x 512 4/4 (256) 20.6 -> 14.9, 2 x 300 16/16 window 256 (320) 18.1 -> 14.2, 6 x 700 4/4 (528) 34 -> 25.7, 4 x 1024 4/4 (512) 31 -> 29.6;
// 128 wide, 1 x 130 32/32 (160) 23.8 -> 14.8, 2 x 1024 8/8 (384) 57.5 -> 45.3, 1 x 2000 8/8 soft-cap (384) 114 -> 80, 1 x 1024 32/16 (512) 77 -> 70; 3 x 1000 8/8 (576)
// 62.4 -> 64.3, 1 x 1000 32/32 (768) 70 -> 80, 8 x 1024 4/4 64 wide (1024) 44 -> 49; with equal chains (even_chains) 1 x 1024 16/16 window 256 (512) 19.6 -> 20.9.
// Rows to form delta of: 1 x 256 32/8 (1152) 40.6 -> 39.1, 1 x 400 40/8 (2240) 63 -> 72, 64 wide 2 x 500 16/4 (2176) 39.6 -> 43.9, 1 x 3000 8/8 135 -> 149.
// Up to 256 workgroups each has a CU of its own.  Beyond, the rest comes in a second round (and a third), which only long chains are worth.  By 32-row tiles of one
// query head's chain, 128 wide, one query head to a K/V head: 1 tile 4 x 30 48/48 (384) 13.9 -> 16.7, 11 x 31 24/24 (528) 16.9 -> 23.7; 2 tiles 8 x 55 24/24 (384) 17.6 -> 19.4;
// 3 tiles 8 x 86 16/16 (384) 22.1 -> 19.3, 11 x 68 16/16 (528) 22.9 -> 24.7; 14 tiles 3 x 437 16/16 (528) 42.2 -> 37.9.  Two to one: 2 tiles 9 x 34 32/16 (432) 21.8 -> 18.6;
// 4 tiles 8 x 113 32/16 (512) 27.5 -> 29.7; 10 tiles 3 x 312 32/16 (528) 40.3 -> 42.8; 16 tiles 2 x 492 32/16 soft-cap (512) 56.8 -> 53.9.  More: 1 tile
// 8 x 28 40/8 (384) 19.8 -> 16.0; 2 tiles 9 x 54 40/8 (432) 25.5 -> 26.7; 4 tiles 10 x 127 32/8 soft-cap (480) 40.9 -> 42.3; 5 tiles 10 x 156 16/4 (440) 36.1 -> 33.4.  64 wide:
// 1 tile 11 x 32 40/8 (528) 14.9 -> 17.3; 5 tiles 9 x 151 16/4 (540) 25.0 -> 20.6.  Equal chains: 2 x 1590 8/4 window 64 (408) 28.9 -> 31.9.
// plain, by workgroups of 128 queries: 64 wide, 4 x 500 16/16 (256) 35 -> 30.6; 128 wide, 3 x 512 32/32 (384) 67 -> 57, 3 x 1000 16/16 (384) 108 -> 84, 8 x 1024 8/8 (512)
// 112 -> 103, 5 x 1600 8/8 (520) 156 -> 137; 8 x 256 32/32 (512) 54 -> 59, 10 x 1024 8/8 (640) 120 -> 128, 1 x 2000 32/32 window 1024 (512) 129 -> 147, 2 x 1000 32/16 (512) 101 -> 136.
// (Also where dK/dV by itself would be split, 64 wide 4 x 709 16/16 soft-cap 92 -> 64, 3 x 282 32/32 28.4 -> 21.6: one fp32 chain in the place of four added up.  What P, dS and the
// results lose as bf16 hides that: the error of dK and dV against float64, 0.24 to 0.25 % over twenty such shapes, is 0.9995 to 1.0001 of the split form's.)
template <int D>
BwdForm bwd_form(int B, int S, int H, int KH, int window, bool apart) {
  const BwdForm two = {q_split<D>(B, S, H, window), dkv_split<D>(B, S, H, KH, window), false};
  if (apart) return two;
  const int rep = H / KH;
  const bool even = even_chains(S, window);
  const int tiles = ((window >= 0 && window < S - 64 ? window + 64 : S) + 31) / 32;
  int room = tiles < 5 ? 512 : 544;  // workgroups of both
  if (D == 128 && rep == 1 && tiles < 3) room = 256;
  if (D == 128 && rep == 2 && tiles < 16) room = tiles < 3 ? 480 : 400;
  if (D == 128 && rep > 2 && tiles < 5) room = tiles < 3 ? 400 : 448;
  if (even) room = std::min(room, D == 128 && rep == 2 ? 360 : 448);
  const int64_t split = (int64_t)((S + 32 * SPLIT_QW<D> - 1) / (32 * SPLIT_QW<D>)) * H * B + (int64_t)((S + 63) / 64) * KH * B;
  if (split <= room && both_rows(S, rep, 64, window) <= (rep <= 2 ? BOTH_ROWS : 1280)) return {true, true, true};
  const int64_t n = (int64_t)((S + 127) / 128) * H * B;
  if (rep == 1 && !even && !two.split_q && n >= 256 && n <= (S >= 512 ? 528 : 448) && both_rows(S, 1, 128, window) <= BOTH_ROWS) return {false, false, true};
  return two;
}

// The two MFMA kernels of the backward pass; delta: fp32 [B, H, S] scratch, fully
// written by the dQ kernel (each workgroup computes the entries of its own queries) before the
// dK/dV kernel, launched after it, reads them (one launch of both leaves it as it is).
template <int D>
void launch_bwd_fast(hipStream_t stream, const bf16* qp, const bf16* kp, const bf16* vp, const bf16* op, const float* lse,
                     const bf16* gop, bf16* dq, bf16* dk, bf16* dv, float* delta, int B, int S, int H, int KH, int64_t ldq,
                     int64_t ldk, int64_t ldv, int64_t ldo, int64_t lddo, int64_t lddq, int64_t lddk, int64_t lddv, int window,
                     float softcap) {
  const float scale = 1.f / sqrtf((float)D);
  bwd_fast_attributes();
  const bool apart = meets_inputs({qp, kp, vp, op, gop}, {ldq, ldk, ldv, ldo, lddo}, {H, KH, KH, H, H}, {dq, dk, dv}, {lddq, lddk, lddv}, {H, KH, KH}, (int64_t)B * S, D);
  const BwdForm form = bwd_form<D>(B, S, H, KH, window, apart);
  auto go = [&](auto cap) {
    constexpr bool CAP = decltype(cap)::value;
    auto one = [&](auto kern, int qr, int kr, int threads, int smem) {
      const int nkv = (S + kr - 1) / kr * KH * B;
      hipLaunchKernelGGL(kern, dim3((unsigned)(nkv + (S + qr - 1) / qr * H * B)), dim3(threads), smem, stream, qp, kp, vp, gop, lse, (const float*)nullptr, dk, dv, S, H, KH,
                         ldq, ldk, ldv, lddo, lddk, lddv, scale, window, softcap, op, dq, ldo, lddq, nkv);
    };
    constexpr int QW = SPLIT_QW<D>, KS = SPLIT_KS<D>;
    if (form.one && !form.split_q) return one(attn_bwd_dkv_kernel<D, CAP, 4, 1, true>, 128, 128, 256, smem_both<D, 4, 1, 4, 1>(both_rows(S, H / KH, 128, window)));
    if (form.one) return one(attn_bwd_dkv_kernel<D, CAP, 2, 4, true>, QW * 32, 64, 512, smem_both<D, QW, KS, 2, 4>(both_rows(S, H / KH, 64, window)));
    auto qk = [&](auto kern, int qw, int ks) {
      hipLaunchKernelGGL(kern, dim3((unsigned)(((S + 32 * qw - 1) / (32 * qw)) * H * B)), dim3(qw * ks * 64), smem_q(D, qw, ks), stream, qp, kp, vp, op, gop, lse, delta, dq, S, H, KH, ldq, ldk, ldv, ldo, lddo, lddq, scale, window, softcap);
    };
    if (form.split_q) qk(attn_bwd_dq_kernel<D, CAP, SPLIT_QW<D>, SPLIT_KS<D>>, SPLIT_QW<D>, SPLIT_KS<D>);
    else qk(attn_bwd_dq_kernel<D, CAP, 4, 1>, 4, 1);
    auto kv = [&](auto kern, int kw, int nqs) {
      hipLaunchKernelGGL(kern, dim3((unsigned)(((S + 32 * kw - 1) / (32 * kw)) * KH * B)), dim3(kw * nqs * 64), smem_kv(D, kw, nqs), stream, qp, kp, vp, gop, lse, delta, dk, dv, S, H, KH, ldq, ldk, ldv, lddo, lddk, lddv, scale, window, softcap, (const bf16*)nullptr, (bf16*)nullptr, (int64_t)0, (int64_t)0, 0);
    };
    if (form.split_kv) kv(attn_bwd_dkv_kernel<D, CAP, 2, 4>, 2, 4);
    else kv(attn_bwd_dkv_kernel<D, CAP, 4, 1>, 4, 1);
  };
  if (softcap > 0.f) go(std::true_type());
  else go(std::false_type());
}

template <int D>
void launch_fwd_fast(hipStream_t stream, const bf16* qp, const bf16* kp, const bf16* vp, bf16* o, float* lse, int B, int S, int H,
                     int KH, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo, int window, float softcap) {
  const float scale = 1.f / sqrtf((float)D);
  constexpr int QW = SPLIT_QW<D>, KS = SPLIT_KS<D>;
  static std::once_flag once;  // per head_dim
  std::call_once(once, [] {
    constexpr auto ATTR = hipFuncAttributeMaxDynamicSharedMemorySize;
    (void)hipFuncSetAttribute((const void*)attn_fwd_kernel<D, true, 4, 1>, ATTR, smem_q(D, 4, 1));
    (void)hipFuncSetAttribute((const void*)attn_fwd_kernel<D, false, 4, 1>, ATTR, smem_q(D, 4, 1));
    (void)hipFuncSetAttribute((const void*)attn_fwd_kernel<D, true, QW, KS>, ATTR, smem_q(D, QW, KS));
    (void)hipFuncSetAttribute((const void*)attn_fwd_kernel<D, false, QW, KS>, ATTR, smem_q(D, QW, KS));
  });
  const bool split = q_split<D>(B, S, H, window);
  auto go = [&](auto cap) {
    constexpr bool CAP = decltype(cap)::value;
    auto run = [&](auto kern, int qw, int ks) {
      hipLaunchKernelGGL(kern, dim3((unsigned)(((S + 32 * qw - 1) / (32 * qw)) * H * B)), dim3(qw * ks * 64), smem_q(D, qw, ks), stream, qp, kp, vp, o, lse, S, H, KH, ldq, ldk, ldv, ldo, scale, window, softcap);
    };
    if (split) run(attn_fwd_kernel<D, CAP, QW, KS>, QW, KS);
    else run(attn_fwd_kernel<D, CAP, 4, 1>, 4, 1);
  };
  if (softcap > 0.f) go(std::true_type());
  else go(std::false_type());
}

}  // namespace

// q [B*S, ldq] (head h at columns h*D..), k/v [B*S, ldk/ldv] (KH heads), o [B*S, ldo],
// lse [B, H, S] fp32 (natural log of the masked softmax normaliser of the scaled, capped scores).
// window < 0: global causal; window >= 0: keys i-window..i.  softcap <= 0: off.
extern "C" int32_t olmax_attn_fwd(hipStream_t stream, const void* q, const void* k, const void* v,
                                  void* o, float* lse, int32_t B, int32_t S, int32_t H, int32_t KH,
                                  int32_t D, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo,
                                  int32_t window, float softcap) {
  OLMAX_CHECK(q && k && v && o && lse, OLMAX_ERR_ARG, "olmax_attn_fwd: null pointer");
  OLMAX_CHECK(B > 0 && S > 0 && H > 0 && KH > 0 && D > 0 && H % KH == 0, OLMAX_ERR_SHAPE, "olmax_attn_fwd: bad shape B=%d S=%d H=%d KH=%d D=%d", B, S, H, KH, D);
  OLMAX_CHECK(ldq >= (int64_t)H * D && ldo >= (int64_t)H * D && ldk >= (int64_t)KH * D && ldv >= (int64_t)KH * D, OLMAX_ERR_SHAPE, "olmax_attn_fwd: row stride smaller than heads*head_dim");
  window = reach(window, S);
  const float scale = 1.f / sqrtf((float)D);
  const bf16 *qp = (const bf16*)q, *kp = (const bf16*)k, *vp = (const bf16*)v;
  if (fast_ok(D, S, GENERIC_MAX_S_FWD, q, k, v, o, ldq, ldk, ldv, ldo) && (D == 128 || o != q)) {
    auto go = D == 128 ? launch_fwd_fast<128> : launch_fwd_fast<64>;
    go(stream, qp, kp, vp, (bf16*)o, lse, B, S, H, KH, ldq, ldk, ldv, ldo, window, softcap);
  } else {
    OLMAX_CHECK(D <= 256 && S <= GENERIC_MAX_S_FWD, OLMAX_ERR_SHAPE, "olmax_attn_fwd: generic path supports head_dim <= 256 and seq_len <= 16384");
    hipLaunchKernelGGL(attn_fwd_generic, dim3(S, H, B), dim3(64), (size_t)S * 4, stream, qp, kp, vp, (bf16*)o, lse, S, H, KH, D, ldq, ldk, ldv, ldo, scale, window, softcap);
  }
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

// Workspace: delta [B,H,S] fp32, then two fp32 [B*S, KH*D] accumulators for the generic path.
// Which path runs depends on head_dim AND on the alignment of the operands (a head_dim-128 call
// on unaligned views takes the generic path), which this query cannot see: it always returns the
// size that covers both.
static int64_t attn_delta_bytes(int32_t B, int32_t S, int32_t H) { return ((int64_t)B * H * S * 4 + 255) / 256 * 256; }
static int64_t attn_acc_bytes(int32_t B, int32_t S, int32_t KH, int32_t D) { return ((int64_t)B * S * KH * D * 4 + 255) / 256 * 256; }
extern "C" int64_t olmax_attn_bwd_workspace_bytes(int32_t B, int32_t S, int32_t H, int32_t KH, int32_t D) {
  return attn_delta_bytes(B, S, H) + 2 * attn_acc_bytes(B, S, KH, D);
}
// What the MFMA path alone needs (delta only): for callers that KNOW head_dim is 128 and every
// operand is 16-byte aligned with row strides that are multiples of 8.
extern "C" int64_t olmax_attn_bwd_workspace_bytes_aligned(int32_t B, int32_t S, int32_t H) { return attn_delta_bytes(B, S, H); }

// Which kernels the backward takes for operands that need no others (aligned, outputs apart from inputs): see the header.
extern "C" int32_t olmax_attn_bwd_form(int32_t B, int32_t S, int32_t H, int32_t KH, int32_t D, int32_t window) {
  if (B <= 0 || S <= 0 || H <= 0 || KH <= 0 || H % KH || !(D == 128 || (D == 64 && S <= GENERIC_MAX_S_BWD))) return -1;
  const BwdForm f = (D == 128 ? bwd_form<128> : bwd_form<64>)(B, S, H, KH, reach(window, S), false);
  return (f.split_q ? 1 : 0) | (f.split_kv ? 2 : 0) | (f.one ? 4 : 0);
}

extern "C" int32_t olmax_attn_bwd(hipStream_t stream, const void* q, const void* k, const void* v,
                                  const void* o, const float* lse, const void* d_o, void* dq, void* dk,
                                  void* dv, void* workspace, int64_t workspace_bytes, int32_t B,
                                  int32_t S, int32_t H, int32_t KH, int32_t D, int64_t ldq, int64_t ldk,
                                  int64_t ldv, int64_t ldo, int64_t lddo, int64_t lddq, int64_t lddk,
                                  int64_t lddv, int32_t window, float softcap) {
  OLMAX_CHECK(q && k && v && o && lse && d_o && dq && dk && dv && workspace, OLMAX_ERR_ARG, "olmax_attn_bwd: null pointer");
  OLMAX_CHECK(B > 0 && S > 0 && H > 0 && KH > 0 && D > 0 && H % KH == 0, OLMAX_ERR_SHAPE, "olmax_attn_bwd: bad shape");
  OLMAX_CHECK(workspace_bytes >= attn_delta_bytes(B, S, H) && (((uintptr_t)workspace) & 255) == 0, OLMAX_ERR_WORKSPACE, "olmax_attn_bwd: workspace too small or not 256-byte aligned");
  OLMAX_CHECK(ldq >= (int64_t)H * D && ldo >= (int64_t)H * D && lddo >= (int64_t)H * D && lddq >= (int64_t)H * D && ldk >= (int64_t)KH * D && ldv >= (int64_t)KH * D && lddk >= (int64_t)KH * D && lddv >= (int64_t)KH * D, OLMAX_ERR_SHAPE, "olmax_attn_bwd: row stride smaller than heads*head_dim");
  window = reach(window, S);
  const float scale = 1.f / sqrtf((float)D);
  const bf16 *qp = (const bf16*)q, *kp = (const bf16*)k, *vp = (const bf16*)v, *op = (const bf16*)o, *gop = (const bf16*)d_o;
  float* delta = (float*)workspace;
  // In place: the one-wave-per-query kernels read a row before they write it and dK/dV leave last; the MFMA kernels read Q
  // and dO again after dQ is written.  head_dim 64 has always taken such calls, so they stay on the former.
  const void* const outs[] = {dq, dk, dv};
  const bool in_place = D != 128 && std::any_of(outs, outs + 3, [&](const void* p) { return p == q || p == k || p == v || p == o || p == d_o; });
  // (a workspace of delta alone is head_dim 128's: any other head_dim may meet an unaligned view)
  if (!in_place && bwd_fast_ok(q, k, v, o, d_o, dq, dk, dv, S, D, ldq, ldk, ldv, ldo, lddo, lddq, lddk, lddv) &&
      (D == 128 || workspace_bytes >= attn_delta_bytes(B, S, H) + 2 * attn_acc_bytes(B, S, KH, D))) {
    auto go = D == 128 ? launch_bwd_fast<128> : launch_bwd_fast<64>;
    go(stream, qp, kp, vp, op, lse, gop, (bf16*)dq, (bf16*)dk, (bf16*)dv, delta, B, S, H, KH, ldq, ldk, ldv, ldo, lddo,
       lddq, lddk, lddv, window, softcap);
  } else {
    OLMAX_CHECK(D <= 256 && S <= GENERIC_MAX_S_BWD, OLMAX_ERR_SHAPE, "olmax_attn_bwd: generic path supports head_dim <= 256 and seq_len <= 8192");
    const int64_t accb = attn_acc_bytes(B, S, KH, D);
    OLMAX_CHECK(workspace_bytes >= attn_delta_bytes(B, S, H) + 2 * accb, OLMAX_ERR_WORKSPACE,
                "olmax_attn_bwd: the generic path (head_dim not 128 or 64, or operands not 16-byte aligned) needs %ld workspace bytes",
                (long)(attn_delta_bytes(B, S, H) + 2 * accb));
    float* dkf = (float*)((char*)workspace + attn_delta_bytes(B, S, H));
    float* dvf = (float*)((char*)dkf + accb);
    { int rc = olmax_fill_zero(stream, dkf, 2 * accb); if (rc) return rc; }
    hipLaunchKernelGGL(attn_bwd_generic, dim3(S, H, B), dim3(64), (size_t)S * 8, stream, qp, kp, vp, op, gop, lse, (bf16*)dq, dkf, dvf, S, H, KH, D, ldq, ldk, ldv, ldo, lddo, lddq, scale, window, softcap);
    const int64_t n = (int64_t)B * S * KH * D;
    hipLaunchKernelGGL(strided_cast_f32_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, dkf, (bf16*)dk, (int64_t)B * S, KH * D, lddk);
    hipLaunchKernelGGL(strided_cast_f32_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, dvf, (bf16*)dv, (int64_t)B * S, KH * D, lddv);
  }
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

// ---------------------------------------------------------------------------------------
// olmax_attn_bwd for callers that cannot allocate (code under HIP graph capture, serving loops,
// harnesses that forbid hipMalloc): the delta scratch lives in a file-scope device array
// instead of a caller-provided workspace.  Each GPU the library runs on holds its own copy of the
// array (4 MiB) until the process ends; every call on a GPU shares it, so calls that overlap on
// one GPU (two streams, two threads) race on it.  Nothing in it has to start at zero: the first
// kernel of a call writes every delta entry the second one reads.
// ---------------------------------------------------------------------------------------
constexpr int64_t ATTN_SCRATCH_FLOATS = 1 << 20;  // B * H * S <= 1 Mi (4 MiB)
static __device__ __align__(256) float scratch[ATTN_SCRATCH_FLOATS];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[MAX_DEVICES];  // device address of `scratch` on each GPU, resolved on first use

// The array's name is only a host-side handle; its device address differs per GPU and comes
// from hipGetSymbolAddress with that GPU current.
// resolve == false: only look the address up (what a call under graph capture may do); the
// symbol query itself belongs to set-up, outside any capture.
int scratch_for_current_device(float** out, bool resolve) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES)
    return olmax_set_error(OLMAX_ERR_LAUNCH, "olmax_attn_bwd_noalloc: cannot identify the current device");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    if (!resolve)
      return olmax_set_error(OLMAX_ERR_ARG,
                             "olmax_attn_bwd_noalloc: first use on this device is under stream capture; call "
                             "olmax_attn_bwd_noalloc_init() (or the entry point once, eagerly) before recording");
    float* p = nullptr;
    const hipError_t e = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return olmax_set_error(OLMAX_ERR_LAUNCH, "olmax_attn_bwd_noalloc: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return OLMAX_OK;
}
}  // namespace

// Set-up for the current device: resolves the scratch address and sets the kernels' LDS limits.
// Call it once per device (with that device current) before recording olmax_attn_bwd_noalloc
// into a graph; an eager call of the entry point does the same.
extern "C" int32_t olmax_attn_bwd_noalloc_init(void) {
  float* p = nullptr;
  bwd_fast_attributes();
  return scratch_for_current_device(&p, true);
}

extern "C" int64_t olmax_attn_bwd_noalloc_max_rows(void) { return ATTN_SCRATCH_FLOATS; }

extern "C" int32_t olmax_attn_bwd_noalloc(hipStream_t stream, const void* q, const void* k, const void* v,
                                          const void* o, const float* lse, const void* d_o, void* dq, void* dk,
                                          void* dv, int32_t B, int32_t S, int32_t H, int32_t KH, int32_t D,
                                          int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo, int64_t lddo,
                                          int64_t lddq, int64_t lddk, int64_t lddv, int32_t window, float softcap) {
  OLMAX_CHECK(q && k && v && o && lse && d_o && dq && dk && dv, OLMAX_ERR_ARG, "olmax_attn_bwd_noalloc: null pointer");
  OLMAX_CHECK(B > 0 && S > 0 && H > 0 && KH > 0 && D > 0 && H % KH == 0, OLMAX_ERR_SHAPE, "olmax_attn_bwd_noalloc: bad shape");
  OLMAX_CHECK(ldq >= (int64_t)H * D && ldo >= (int64_t)H * D && lddo >= (int64_t)H * D && lddq >= (int64_t)H * D && ldk >= (int64_t)KH * D && ldv >= (int64_t)KH * D && lddk >= (int64_t)KH * D && lddv >= (int64_t)KH * D, OLMAX_ERR_SHAPE, "olmax_attn_bwd_noalloc: row stride smaller than heads*head_dim");
  window = reach(window, S);
  OLMAX_CHECK((int64_t)B * H * S <= ATTN_SCRATCH_FLOATS, OLMAX_ERR_WORKSPACE,
              "olmax_attn_bwd_noalloc: batch*heads*seq_len = %ld exceeds the built-in scratch of %ld rows; use olmax_attn_bwd with a workspace",
              (long)((int64_t)B * H * S), (long)ATTN_SCRATCH_FLOATS);
  OLMAX_CHECK(D == 128 && bwd_fast_ok(q, k, v, o, d_o, dq, dk, dv, S, D, ldq, ldk, ldv, ldo, lddo, lddq, lddk, lddv), OLMAX_ERR_ALIGN,
              "olmax_attn_bwd_noalloc: needs head_dim 128, 16-byte aligned pointers and row strides that are multiples of 8; use olmax_attn_bwd otherwise");
  float* delta = nullptr;
  {
    // under capture only a pointer resolved earlier may be used: the symbol query is set-up work
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    const bool capturing = stream && hipStreamIsCapturing(stream, &st) == hipSuccess && st == hipStreamCaptureStatusActive;
    int rc = scratch_for_current_device(&delta, !capturing);
    if (rc) return rc;
  }
  launch_bwd_fast<128>(stream, (const bf16*)q, (const bf16*)k, (const bf16*)v, (const bf16*)o, lse, (const bf16*)d_o, (bf16*)dq, (bf16*)dk,
                  (bf16*)dv, delta, B, S, H, KH, ldq, ldk, ldv, ldo, lddo, lddq, lddk, lddv, window, softcap);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}
