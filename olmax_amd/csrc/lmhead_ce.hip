// Cross-entropy over the full vocabulary and the fused LM-head + CE forward/backward.
//
// Reference semantics: cross_entropy_loss, src/olmax/nn/functional.py:70-91 (reduction
// "mean" over labels != ignore_index; an out-of-range label contributes zero loss and zero
// gradient but still counts in the denominator), fed by LMHead.forward,
// src/olmax/nn/lm_head.py:59-61 (logits = bf16 GEMM output widened to fp32).
//
// One block owns one row of logits.  bf16 rows of up to 163840 entries are loaded ONCE into the
// block's registers (128-bit loads), reduced to max and sum-exp, and written back as
// d logits = (softmax - onehot) * dloss / n_counted from the registers; longer ones keep 131072 entries
// there and read the rest again; soft-capped longer and fp32 rows take
// the streaming form (online max / sum-exp in pass 1, a second read of the row in pass 2).
// Optional final-logit soft-cap z = c*tanh(x/c) is applied on the fly in both passes.
#include "common.h"
#include <type_traits>

namespace {

// Sum of f(0) .. f(n - 1) over one workgroup of 1024; four loads of a thread are in flight at a time (a single
// workgroup walks all rows, so latency is its time: 8192 labels 14.8 -> 4.5 us).
template <typename F>
__device__ __forceinline__ float sum_rows(int64_t n, float* red, F f) {
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  int64_t i = threadIdx.x;
  for (; i + 3 * 1024 < n; i += 4 * 1024)
#pragma unroll
    for (int u = 0; u < 4; u++) s[u] += f(i + u * 1024);
  for (; i < n; i += 1024) s[0] += f(i);
  return block_sum<16>((s[0] + s[1]) + (s[2] + s[3]), red);
}

__global__ __launch_bounds__(1024) void ce_count_kernel(const int32_t* __restrict__ labels, int64_t T,
                                                        int32_t ignore_index, int32_t* __restrict__ n_out) {
  __shared__ float red[16];
  const float c = sum_rows(T, red, [&](int64_t i) { return labels[i] != ignore_index ? 1.f : 0.f; });
  if (threadIdx.x == 0) *n_out = (int32_t)(c + 0.5f);
}

template <typename T> struct Io;
template <> struct Io<bf16> {
  static constexpr int VEC = 8;
  static __device__ __forceinline__ void load(const bf16* p, float* f) {
    Pack8 t;
    t.u = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
    for (int e = 0; e < 8; e++) f[e] = bf2f(t.e[e]);
  }
  static __device__ __forceinline__ void store(bf16* p, const float* f) {
    Pack8 t;
#pragma unroll
    for (int e = 0; e < 8; e++) t.e[e] = f2bf(f[e]);
    *reinterpret_cast<u32x4*>(p) = t.u;
  }
  static __device__ __forceinline__ float ld1(const bf16* p) { return bf2f(*p); }
  static __device__ __forceinline__ void st1(bf16* p, float f) { *p = f2bf(f); }
};
template <> struct Io<float> {
  static constexpr int VEC = 4;
  static __device__ __forceinline__ void load(const float* p, float* f) {
    f32x4 t = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
    for (int e = 0; e < 4; e++) f[e] = t[e];
  }
  static __device__ __forceinline__ void store(float* p, const float* f) {
    f32x4 t;
#pragma unroll
    for (int e = 0; e < 4; e++) t[e] = f[e];
    *reinterpret_cast<f32x4*>(p) = t;
  }
  static __device__ __forceinline__ float ld1(const float* p) { return *p; }
  static __device__ __forceinline__ void st1(float* p, float f) { *p = f; }
};

template <typename T, bool CAP, int THREADS>
__global__ __launch_bounds__(THREADS) void ce_row_kernel(
    const T* __restrict__ logits, T* __restrict__ dlogits, const int32_t* __restrict__ labels,
    float* __restrict__ row_loss, float* __restrict__ lse_out, const int32_t* __restrict__ n_counted,
    int64_t rows, int V, int64_t ld, int64_t ldd, int32_t ignore_index, float cap, float dloss,
    int vec_ok, const float* __restrict__ drow, int mean, int pad) {
  constexpr int VEC = Io<T>::VEC;
  constexpr int NW = THREADS / 64;
  __shared__ float red[NW];
  __shared__ float label_logit;
  const int64_t row = blockIdx.x;
  const T* zr = logits + row * ld;
  const int label = labels[row];
  const float inv_cap = CAP ? 1.f / cap : 0.f;
  const bool counted = label != ignore_index;
  const bool inrange = label >= 0 && label < V;
  // The label's logit is fetched and parked in LDS BEFORE the first block barrier: with dlogits
  // aliasing logits, other waves overwrite the row as soon as they are past the last reduction,
  // and no load of the row may be left to race with those stores.
  if (threadIdx.x == 0) {
    float zl = 0.f;
    if (counted && inrange) {
      zl = Io<T>::ld1(zr + label);
      if (CAP) zl = cap * fast_tanh(zl * inv_cap);
    }
    label_logit = zl;
  }
  // ---- pass 1: online max / sum-exp ----
  float mx = -INFINITY, sm = 0.f;
  const int nvec = vec_ok ? V / VEC : 0;
  for (int i = threadIdx.x; i < nvec; i += THREADS) {
    float f[VEC];
    Io<T>::load(zr + i * VEC, f);
    float cm = -INFINITY;
#pragma unroll
    for (int e = 0; e < VEC; e++) {
      if (CAP) f[e] = cap * fast_tanh(f[e] * inv_cap);
      cm = fmaxf(cm, f[e]);
    }
    if (cm > mx) {
      sm *= __expf(mx - cm);
      mx = cm;
    }
#pragma unroll
    for (int e = 0; e < VEC; e++) sm += __expf(f[e] - mx);
  }
  for (int i = nvec * VEC + threadIdx.x; i < V; i += THREADS) {
    float f = Io<T>::ld1(zr + i);
    if (CAP) f = cap * fast_tanh(f * inv_cap);
    if (f > mx) {
      sm *= __expf(mx - f);
      mx = f;
    }
    sm += __expf(f - mx);
  }
  const float gmx = block_max<NW>(mx, red);
  sm = (mx == -INFINITY) ? 0.f : sm * __expf(mx - gmx);
  const float gsm = block_sum<NW>(sm, red);
  const float lse = gmx + __logf(gsm);
  if (threadIdx.x == 0) {
    row_loss[row] = (counted && inrange) ? (lse - label_logit) : 0.f;
    if (lse_out) lse_out[row] = counted ? lse : 0.f;
  }
  if (!dlogits) return;
  // ---- pass 2: gradient, in place allowed ----
  T* dr = dlogits + row * ldd;
  // d(reduced loss) / d(row loss): 1/n for "mean", 1 for "sum", the row's own cotangent for "none"
  const float scale = (counted && inrange) ? dloss * (drow ? drow[row] : 1.f) / (mean ? (float)(*n_counted) : 1.f) : 0.f;
  for (int i = threadIdx.x; i < nvec; i += THREADS) {
    float f[VEC];
    Io<T>::load(zr + i * VEC, f);
#pragma unroll
    for (int e = 0; e < VEC; e++) {
      float z = f[e], chain = 1.f;
      if (CAP) {
        const float t = fast_tanh(z * inv_cap);
        z = cap * t;
        chain = 1.f - t * t;
      }
      float p = __expf(z - lse);
      if (i * VEC + e == label) p -= 1.f;
      f[e] = p * scale * chain;
    }
    Io<T>::store(dr + i * VEC, f);
  }
  for (int i = nvec * VEC + threadIdx.x; i < V; i += THREADS) {
    float z = Io<T>::ld1(zr + i), chain = 1.f;
    if (CAP) {
      const float t = fast_tanh(z * inv_cap);
      z = cap * t;
      chain = 1.f - t * t;
    }
    float p = __expf(z - lse);
    if (i == label) p -= 1.f;
    Io<T>::st1(dr + i, p * scale * chain);
  }
  for (int i = V + threadIdx.x; i < V + pad; i += THREADS) Io<T>::st1(dr + i, 0.f);
}

// The same row computation for bf16 rows kept in registers between the two passes (THREADS x MAXV
// vectors of 8): the logits are read from memory once and the gradient
// written once, 4 B per logit instead of 6.  Max and sum-exp are two plain block reductions (no
// online rescaling needed when the whole row is at hand).  PAD: V is not a multiple of 8 and the rows
// have room up to the next one; those logits are left out and their gradient is written as zero.
// TAIL: a longer row; what the registers do not hold is reduced online and read a second time, right after
// (4096 x 262144: 1.26 ms all read twice by 4 waves, 1.10 by 16, 1.04 with half of the row held).
//
// Bound by memory (8192 x 50304: 1.65 GB in 316 us = 5.2 TB/s) as long as the vector instructions stay below it,
// about 12 a logit: the maximum is taken of raw values, missing logits are minus infinity instead of a test in each pass,
// only the one vector that holds the label looks for it, and the gradient's exponential is one fma and exp2.  The fma's
// constant lse * log2(e) is rounded: half an ulp of it is a factor of exp(1.1e-5) at 256 (0.04 in the exponent at 1e6, and infinite at the type's
// lowest value); the row's scale has the factor that takes it back.  rms error of p with an exact exp2: 2.0e-7 at
// lse 10 to 250 (without the factor 3.9e-7 at 10, 6.1e-6 at 250), as with lse subtracted first, which rows from 256 on and the label's vector do.
template <bool CAP, int THREADS, int MAXV, bool PAD, bool TAIL>
__global__ __launch_bounds__(THREADS, 4) void ce_row_regs_kernel(
    const bf16* __restrict__ logits, bf16* __restrict__ dlogits, const int32_t* __restrict__ labels,
    float* __restrict__ row_loss, float* __restrict__ lse_out, const int32_t* __restrict__ n_counted,
    int V, int64_t ld, int64_t ldd, int32_t ignore_index, float cap, float dloss,
    const float* __restrict__ drow, int mean) {
  static_assert(!(CAP && TAIL), "soft-capped rows beyond the registers take the streaming form");
  constexpr int NW = THREADS / 64;
  constexpr int HELD = MAXV * THREADS;  // vectors in registers
  constexpr uint32_t NEG_INF2 = 0xff80ff80u;
  constexpr float LOG2E = 1.4426950408889634f;
  __shared__ float red[NW];
  __shared__ float label_logit;
  const int64_t row = blockIdx.x;
  const bf16* zr = logits + row * ld;
  const int label = labels[row];
  const float inv_cap = CAP ? 1.f / cap : 0.f;
  const int nvec = PAD ? (V + 7) / 8 : V / 8;
  const bool counted = label != ignore_index;
  const bool inrange = label >= 0 && label < V;
  // label logit into LDS before the first barrier (see ce_row_kernel): nothing reads the row
  // from memory once any wave may be storing the gradient over it
  if (threadIdx.x == 0) {
    float zl = 0.f;
    if (counted && inrange) {
      zl = bf2f(zr[label]);
      if (CAP) zl = cap * fast_tanh(zl * inv_cap);
    }
    label_logit = zl;
  }
  // a vector of the row; logits that do not exist are minus infinity: nothing to the maximum, nothing to the sum
  auto fetch = [&](int idx) {
    Pack8 v;
    v.u = u32x4{NEG_INF2, NEG_INF2, NEG_INF2, NEG_INF2};
    if (idx < nvec) {
      v.u = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(zr) + idx);
      if (PAD && idx == nvec - 1) {
#pragma unroll
        for (int e = 1; e < 8; e++)
          if (idx * 8 + e >= V) v.u[e >> 1] = e & 1 ? (v.u[e >> 1] & 0xffffu) | (NEG_INF2 & 0xffff0000u) : NEG_INF2;
      }
    }
    return v;
  };
  // the soft-cap t = tanh(z / cap) with its factors in one multiply; it takes minus infinity to -cap, so under
  // it the logits that do not exist are left out by their index (exists)
  const float cap_k = CAP ? 2.f * LOG2E * inv_cap : 0.f;
  auto soft = [&](float f) { return 1.f - 2.f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(f * cap_k) + 1.f); };
  auto value = [&](bf16 x) {
    const float f = bf2f(x);
    return CAP ? cap * soft(f) : f;
  };
  auto exists = [&](int idx, int e) { return !CAP || !PAD || idx * 8 + e < V; };
  // exponentials of a vector against ref, added in pairs
  auto exps = [&](const Pack8& v, int idx, float ref) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = exists(idx, e) ? __expf(value(v.e[e]) - ref) : 0.f;
    return ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
  };
  Pack8 c[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; i++) c[i] = fetch(i * THREADS + threadIdx.x);
  float mx = -INFINITY, tsm = 0.f;
  if (TAIL) {
    constexpr int U = 4;
    for (int i0 = HELD + threadIdx.x; i0 < nvec; i0 += U * THREADS) {
      Pack8 t[U];
#pragma unroll
      for (int u = 0; u < U; u++) t[u] = fetch(i0 + u * THREADS);
      float cm = -INFINITY;
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int e = 0; e < 8; e++) cm = fmaxf(cm, bf2f(t[u].e[e]));
      if (cm > mx) {
        tsm *= __expf(mx - cm);
        mx = cm;
      }
      const float ref = mx == -INFINITY ? 0.f : mx;  // nothing but minus infinity so far: the sum stays 0
#pragma unroll
      for (int u = 0; u < U; u++)
        tsm += exps(t[u], i0 + u * THREADS, ref);
    }
  }
  const float tmx = mx;
  float rmx = -INFINITY;  // of the raw logits: the soft-cap rises with them
  // each pass unpacks a vector when its turn comes: hidden from the compiler, which otherwise keeps all
  // unpacked logits of a pass for the next and spills; so it did with the offsets of 25 vectors, loaded with and kept for the
  // stores (13 to 18 registers, up to 76 bytes a lane: 8192 x 100352 715 us, 621 with the offsets computed again)
  auto keep = [](Pack8& v) {
    asm volatile("" : "+v"(v.u));
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < MAXV; i++) {
    keep(c[i]);
#pragma unroll
    for (int e = 0; e < 8; e++) rmx = fmaxf(rmx, bf2f(c[i].e[e]));
  }
  mx = fmaxf(mx, CAP ? cap * soft(rmx) : rmx);
  const float gmx = block_max<NW>(mx, red);
  float sm = TAIL ? (tmx == -INFINITY ? tsm : tsm * __expf(tmx - gmx)) : 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; i++) {
    keep(c[i]);
    if (!CAP || i * THREADS + threadIdx.x < nvec) sm += exps(c[i], i * THREADS + threadIdx.x, gmx);
  }
  const float gsm = block_sum<NW>(sm, red);
  const float lse = gmx + __logf(gsm);
  if (threadIdx.x == 0) {
    row_loss[row] = (counted && inrange) ? (lse - label_logit) : 0.f;
    if (lse_out) lse_out[row] = counted ? lse : 0.f;
  }
  if (!dlogits) return;
  bf16* dr = dlogits + row * ldd;
  // d(reduced loss) / d(row loss): 1/n for "mean", 1 for "sum", the row's own cotangent for "none"
  const float scale = (counted && inrange) ? dloss * (drow ? drow[row] : 1.f) / (mean ? (float)(*n_counted) : 1.f) : 0.f;
  const float lse2 = lse * LOG2E;
  const float scale2 = scale * __builtin_amdgcn_exp2f(-__builtin_fmaf(lse, LOG2E, -lse2));
  const bool far = !(fabsf(lse) < 256.f);
  auto store = [&](int idx, const Pack8& v) {
    Pack8 o;
    auto grads = [&](auto general) {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        float z = bf2f(v.e[e]), chain = 1.f;
        if (CAP) {
          const float t = soft(z);
          z = cap * t;
          chain = 1.f - t * t;
        }
        float p = general ? __expf(z - lse) : __builtin_amdgcn_exp2f(__builtin_fmaf(z, LOG2E, -lse2));
        if (general && idx * 8 + e == label) p -= 1.f;
        o.e[e] = f2bf(p * (general ? scale : scale2) * chain);
      }
    };
    if (far || idx == label >> 3) grads(std::true_type());
    else grads(std::false_type());
    if (PAD && idx == nvec - 1) {
#pragma unroll
      for (int e = 1; e < 8; e++)
        if (idx * 8 + e >= V) o.e[e] = f2bf(0.f);
    }
    *(reinterpret_cast<u32x4*>(dr) + idx) = o.u;
  };
  if (TAIL) {  // what was read last first
    constexpr int U = 4;
    for (int i0 = HELD + (nvec - HELD - 1 - (int)threadIdx.x) / (U * THREADS) * (U * THREADS) + (int)threadIdx.x; i0 >= HELD; i0 -= U * THREADS) {
      Pack8 t[U];
#pragma unroll
      for (int u = 0; u < U; u++)
        if (i0 + u * THREADS < nvec) t[u].u = *(reinterpret_cast<const u32x4*>(zr) + i0 + u * THREADS);
#pragma unroll
      for (int u = 0; u < U; u++)
        if (i0 + u * THREADS < nvec) store(i0 + u * THREADS, t[u]);
    }
  }
#pragma unroll
  for (int i = 0; i < MAXV; i++) {
    int tid = threadIdx.x;
    if (MAXV >= 25 || TAIL) asm volatile("" : "+v"(tid));
    const int idx = i * THREADS + tid;
    keep(c[i]);
    if (idx < nvec) store(idx, c[i]);
  }
}

// loss = sum(row_loss) / n_counted, or the plain sum (single block; deterministic order)
__global__ __launch_bounds__(1024) void ce_finalize_kernel(const float* __restrict__ row_loss, int64_t T,
                                                           const int32_t* __restrict__ n_counted,
                                                           float* __restrict__ loss, int mean) {
  __shared__ float red[16];
  const float s = sum_rows(T, red, [&](int64_t i) { return row_loss[i]; });
  if (threadIdx.x == 0) *loss = mean ? s / (float)(*n_counted) : s;
}

}  // namespace

// Workspace: T floats (row losses) + 16 bytes (counted-row count), 16-byte aligned.
extern "C" int64_t olmax_cross_entropy_workspace_bytes(int64_t T) { return ((T * 4 + 15) / 16) * 16 + 16; }

// logits [T, V] (bf16 when logits_f32 == 0, else fp32) -> loss (device fp32: a scalar, or [T] row
// losses for reduction "none"); dlogits (same dtype, may alias logits, may be NULL) <-
// d loss / d logits times the incoming cotangent (the scalar dloss; for "none" also the per-row
// device array dloss_rows when given); lse_out (optional, [T]) <- log-normaliser *
// (label != ignore_index)  (the reference's fused_cross_entropy_loss second output,
// src/olmax/nn/functional.py:94-121).  reduction: 0 "mean", 1 "sum", 2 "none" (functional.py:84-91).
// padded (in place, bf16): the rows have room up to the next multiple of 8 logits, which may be read
// and is written with zeros.
static int cross_entropy(hipStream_t stream, const void* logits, void* dlogits, const int32_t* labels, float* loss, float* lse_out,
                         const float* dloss_rows, void* workspace, int64_t workspace_bytes, int64_t T, int32_t V, int64_t ld,
                         int64_t ldd, int32_t logits_f32, int32_t ignore_index, float softcap, float dloss, int32_t reduction,
                         bool padded) {
  OLMAX_CHECK(logits && labels && loss && workspace, OLMAX_ERR_ARG, "olmax_cross_entropy: null pointer");
  OLMAX_CHECK(T > 0 && V > 0 && ld >= V && (!dlogits || ldd >= V), OLMAX_ERR_SHAPE, "olmax_cross_entropy: bad shape T=%ld V=%d", (long)T, V);
  OLMAX_CHECK(reduction >= 0 && reduction <= 2, OLMAX_ERR_ARG, "olmax_cross_entropy: reduction must be 0 (mean), 1 (sum) or 2 (none)");
  OLMAX_CHECK(!dloss_rows || reduction == 2, OLMAX_ERR_ARG, "olmax_cross_entropy: a per-row cotangent only goes with reduction none");
  OLMAX_CHECK(workspace_bytes >= olmax_cross_entropy_workspace_bytes(T) && aligned16(workspace), OLMAX_ERR_WORKSPACE, "olmax_cross_entropy: workspace too small or misaligned");
  // "none": the row kernels write the row losses straight into the caller's array
  float* row_loss = reduction == 2 ? loss : (float*)workspace;
  int32_t* n_counted = (int32_t*)((char*)workspace + ((T * 4 + 15) / 16) * 16);
  const int mean = reduction == 0;
  hipLaunchKernelGGL(ce_count_kernel, dim3(1), dim3(1024), 0, stream, labels, T, ignore_index, n_counted);
  const int vecw = logits_f32 ? 4 : 8;
  const int vec_ok = aligned16(logits) && (!dlogits || aligned16(dlogits)) && ld % vecw == 0 && (!dlogits || ldd % vecw == 0);
  const bool cap = softcap > 0.f;
  dim3 grid((unsigned)T);
#define CE_GO(TY, CAPV, TH)                                                                      \
  hipLaunchKernelGGL((ce_row_kernel<TY, CAPV, TH>), grid, dim3(TH), 0, stream, (const TY*)logits, \
                     (TY*)dlogits, labels, row_loss, lse_out, n_counted, T, V, ld, ldd,          \
                     ignore_index, softcap, dloss, vec_ok, dloss_rows, mean, padded ? (8 - V % 8) % 8 : 0)
#define CE_REGS_P(CAPV, TH, MV, PADV, TAILV)                                                                          \
  hipLaunchKernelGGL((ce_row_regs_kernel<CAPV, TH, MV, PADV, TAILV>), grid, dim3(TH), 0, stream, (const bf16*)logits, \
                     (bf16*)dlogits, labels, row_loss, lse_out, n_counted, V, ld, ldd, ignore_index, softcap, dloss, dloss_rows, mean)
#define CE_REGS_T(CAPV, TH, MV, TAILV)                                                                         \
  do { if (V % 8) CE_REGS_P(CAPV, TH, MV, true, TAILV); else CE_REGS_P(CAPV, TH, MV, false, TAILV); } while (0)
#define CE_REGS(TH, MV) do { if (cap) CE_REGS_T(true, TH, MV, false); else CE_REGS_T(false, TH, MV, false); } while (0)
  const bool regs_ok = !logits_f32 && vec_ok && (V % 8 == 0 || padded);
  if (logits_f32) {
    if (cap) CE_GO(float, true, 256); else CE_GO(float, false, 256);
  } else if (regs_ok && V <= 1024 * 8 * 20) {
    // The fewest threads that hold the row, so that as many rows as possible are on a CU in different phases: us with the
    // workgroup below | the one of 512 threads x 26 vectors (1024 x 20) that held all rows: 2048 x 4096 20 | 46, 1500 x 16384 27 | 51, 8192 x 50304 316 | 425,
    // 8192 x 100352 609 | 740, 4096 x 128256 424 | 493 (the last two only from the arithmetic).  Rows that all find room
    // at once, two workgroups of 512 threads (84 registers) or one of 1024 on a CU, take twice the threads: us with them | with half as many, 16 x 50304 12.6 | 16.9,
    // 257 x 50304 20.3 | 21.7, 512 x 50304 25.3 | 26.9 (513: 31.5 | 29.0), 512 x 20000 16.8 | 18.3, 256 x 100352 29.7 | 34.7.
    if (V <= 256 * 8 * 2) CE_REGS(256, 2);
    else if (V <= 256 * 8 * 8) CE_REGS(256, 8);
    else if (V <= 256 * 8 * 25 && T > 512) CE_REGS(256, 25);
    else if (V <= 256 * 8 * 25) CE_REGS(512, 13);
    else if (V <= 512 * 8 * 25 && T > 256) CE_REGS(512, 25);
    else CE_REGS(1024, 20);
  } else if (regs_ok && !cap) {
    CE_REGS_T(false, 1024, 16, true);
  } else if (V > 1024 * 8 * 20) {
    // rows of half a megabyte: a whole GPU of 16-wave workgroups has 134 to 268 MB of them in flight, which the memory-side
    // cache still holds for the second pass (8192 x 256000, soft-cap: 2.55 ms with 4 waves, 2.34 with 16)
    if (cap) CE_GO(bf16, true, 1024); else CE_GO(bf16, false, 1024);
  } else {
    if (cap) CE_GO(bf16, true, 256); else CE_GO(bf16, false, 256);
  }
#undef CE_GO
#undef CE_REGS
#undef CE_REGS_T
#undef CE_REGS_P
  if (reduction != 2) hipLaunchKernelGGL(ce_finalize_kernel, dim3(1), dim3(1024), 0, stream, row_loss, T, n_counted, loss, mean);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

extern "C" int32_t olmax_cross_entropy_reduce(hipStream_t stream, const void* logits, void* dlogits,
                                              const int32_t* labels, float* loss, float* lse_out,
                                              const float* dloss_rows, void* workspace, int64_t workspace_bytes,
                                              int64_t T, int32_t V, int64_t ld, int64_t ldd, int32_t logits_f32,
                                              int32_t ignore_index, float softcap, float dloss, int32_t reduction) {
  return cross_entropy(stream, logits, dlogits, labels, loss, lse_out, dloss_rows, workspace, workspace_bytes, T, V, ld, ldd,
                       logits_f32, ignore_index, softcap, dloss, reduction, false);
}

// reduction "mean": what the benchmark's loss_fun and the fused LM head use
extern "C" int32_t olmax_cross_entropy(hipStream_t stream, const void* logits, void* dlogits,
                                       const int32_t* labels, float* loss, float* lse_out,
                                       void* workspace, int64_t workspace_bytes, int64_t T, int32_t V,
                                       int64_t ld, int64_t ldd, int32_t logits_f32,
                                       int32_t ignore_index, float softcap, float dloss) {
  return olmax_cross_entropy_reduce(stream, logits, dlogits, labels, loss, lse_out, nullptr, workspace, workspace_bytes, T, V, ld,
                                    ldd, logits_f32, ignore_index, softcap, dloss, 0);
}

// Row stride of the LM head's own logits: whole 128-byte lines, so that the three GEMMs around the
// cross entropy fetch 16-byte chunks whatever the vocabulary (100278 logits are rows of 2-byte
// alignment when packed).
static int64_t logits_stride(int32_t V) { return ((int64_t)V + 63) / 64 * 64; }

// Workspace for the fused LM head: bf16 logits [T, logits_stride(V)] + the CE workspace.
extern "C" int64_t olmax_lmhead_ce_workspace_bytes(int64_t T, int32_t V) {
  return ((T * logits_stride(V) * 2 + 255) / 256) * 256 + olmax_cross_entropy_workspace_bytes(T);
}

// Fused LM head + cross entropy, forward and backward in one call:
//   logits = h W^T (bf16) ; loss = CE(softcap(logits), labels) ;
//   dlogits overwrites logits in the workspace ; dh = dlogits W ; dW = dlogits^T h.
// h [T, d] bf16, W [V, d] bf16, labels [T] int32.  dh [T, d] bf16 and dW [V, d] (bf16, or
// fp32 when dw_f32 != 0) may be NULL to skip that product (forward-only when both are NULL).
int olmax_lmhead_ce_scratch(hipStream_t stream, const void* h, const void* W, const int32_t* labels, float* loss, void* dh, void* dW,
                            void* workspace, int64_t workspace_bytes, int64_t T, int32_t d, int32_t V, int32_t ignore_index,
                            float softcap, int32_t dw_f32, GemmScratch scratch) {
  OLMAX_CHECK(h && W && labels && loss && workspace, OLMAX_ERR_ARG, "olmax_lmhead_ce: null pointer");
  OLMAX_CHECK(T > 0 && d > 0 && V > 0 && T < (1LL << 31), OLMAX_ERR_SHAPE, "olmax_lmhead_ce: bad shape");
  OLMAX_CHECK(workspace_bytes >= olmax_lmhead_ce_workspace_bytes(T, V) && (((uintptr_t)workspace) & 255) == 0, OLMAX_ERR_WORKSPACE,
              "olmax_lmhead_ce: workspace needs %ld bytes, 256-byte aligned", (long)olmax_lmhead_ce_workspace_bytes(T, V));
  const int64_t ldl = logits_stride(V);
  bf16* logits = (bf16*)workspace;
  void* ce_ws = (char*)workspace + ((T * ldl * 2 + 255) / 256) * 256;
  const bf16 *hp = (const bf16*)h, *wp = (const bf16*)W;
  int rc = olmax_gemm_padded(stream, hp, wp, logits, nullptr, (int)T, V, d, d, d, ldl, 0, true, true, false, false);
  if (rc) return rc;
  const bool need_grad = dh || dW;
  rc = cross_entropy(stream, logits, need_grad ? logits : nullptr, labels, loss, nullptr, nullptr, ce_ws,
                     olmax_cross_entropy_workspace_bytes(T), T, V, ldl, ldl, 0, ignore_index, softcap, 1.f, 0, true);
  if (rc) return rc;
  if (dh && dW)
    return olmax_gemm_grads(stream, logits, wp, hp, (bf16*)dh, nullptr, dW, (int)T, d, V, ldl, d, d, d, 0, d, dw_f32 != 0, true, scratch);
  if (dh) {
    rc = olmax_gemm_padded(stream, logits, wp, dh, nullptr, (int)T, d, V, ldl, d, d, 0, true, false, false, true, scratch);
    if (rc) return rc;
  }
  if (dW) {
    rc = olmax_gemm_padded(stream, logits, hp, dW, nullptr, V, d, (int)T, ldl, d, d, 0, false, false, dw_f32 != 0, true, scratch);
    if (rc) return rc;
  }
  return OLMAX_OK;
}

extern "C" int32_t olmax_lmhead_ce(hipStream_t stream, const void* h, const void* W,
                                   const int32_t* labels, float* loss, void* dh, void* dW,
                                   void* workspace, int64_t workspace_bytes, int64_t T, int32_t d,
                                   int32_t V, int32_t ignore_index, float softcap, int32_t dw_f32) {
  return olmax_lmhead_ce_scratch(stream, h, W, labels, loss, dh, dW, workspace, workspace_bytes, T, d, V, ignore_index, softcap, dw_f32,
                                 GemmScratch());
}
