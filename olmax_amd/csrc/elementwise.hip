// HBM-bound elementwise / gather kernels: gated-MLP activation, embedding gather and
// scatter-add, fused fp32 AdamW (with the bf16 working-copy write), utility fills/casts.
// 128-bit accesses, grid-stride loops.
//
// Reference semantics:
//   GatedMLP      src/olmax/nn/mlp.py:69-73 (act = jax.nn.silu; jax.nn.gelu(tanh) for Gemma,
//                 src/olmax/nn/transformer/layer.py:133)
//   Embedding     src/olmax/nn/embedding.py:30-32
//   AdamW         optax.adamw configured at src/olmax/optim/config.py:136-156, applied at
//                 src/olmax/train/trainer.py:745-752; the bf16 copy replaces the per-step
//                 cast_tree(params, bf16) of src/olmax/train/trainer.py:728
#include "common.h"
#include <atomic>

namespace {

// gate/up are column blocks of one [T, ld] buffer (or separate buffers); out [T, F].
template <bool GELU>
__global__ __launch_bounds__(256) void glu_fwd_kernel(const bf16* __restrict__ gate,
                                                      const bf16* __restrict__ up,
                                                      bf16* __restrict__ out, int64_t T, int F,
                                                      int64_t ldg, int64_t ldu, int64_t ldo) {
  const int cpr = F / 8;
  const int64_t total = T * cpr;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t t = i / cpr;
    const int c = (int)(i % cpr) * 8;
    Pack8 g, u, o;
    g.u = *reinterpret_cast<const u32x4*>(gate + t * ldg + c);
    u.u = *reinterpret_cast<const u32x4*>(up + t * ldu + c);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float gf = bf2f(g.e[e]);
      const float a = bf2f(f2bf(GELU ? act_gelu(gf) : act_silu(gf)));  // act output is a bf16 array
      o.e[e] = f2bf(a * bf2f(u.e[e]));
    }
    *reinterpret_cast<u32x4*>(out + t * ldo + c) = o.u;
  }
}

template <bool GELU>
__global__ __launch_bounds__(256) void glu_bwd_kernel(const bf16* __restrict__ gate,
                                                      const bf16* __restrict__ up,
                                                      const bf16* __restrict__ dh,
                                                      bf16* __restrict__ dgate,
                                                      bf16* __restrict__ dup, int64_t T, int F,
                                                      int64_t ldg, int64_t ldu, int64_t lddh,
                                                      int64_t lddg, int64_t lddu) {
  const int cpr = F / 8;
  const int64_t total = T * cpr;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t t = i / cpr;
    const int c = (int)(i % cpr) * 8;
    Pack8 g, u, d, og, ou;
    g.u = *reinterpret_cast<const u32x4*>(gate + t * ldg + c);
    u.u = *reinterpret_cast<const u32x4*>(up + t * ldu + c);
    d.u = *reinterpret_cast<const u32x4*>(dh + t * lddh + c);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float gf = bf2f(g.e[e]), uf = bf2f(u.e[e]), df = bf2f(d.e[e]);
      og.e[e] = f2bf(df * uf * (GELU ? act_gelu_grad(gf) : act_silu_grad(gf)));
      ou.e[e] = f2bf(df * (GELU ? act_gelu(gf) : act_silu(gf)));
    }
    *reinterpret_cast<u32x4*>(dgate + t * lddg + c) = og.u;
    *reinterpret_cast<u32x4*>(dup + t * lddu + c) = ou.u;
  }
}

template <bool GELU>
__global__ void glu_fwd_scalar(const bf16* gate, const bf16* up, bf16* out, int64_t T, int F,
                               int64_t ldg, int64_t ldu, int64_t ldo) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= T * F) return;
  const int64_t t = i / F;
  const int c = (int)(i % F);
  const float gf = bf2f(gate[t * ldg + c]);
  const float a = bf2f(f2bf(GELU ? act_gelu(gf) : act_silu(gf)));
  out[t * ldo + c] = f2bf(a * bf2f(up[t * ldu + c]));
}
template <bool GELU>
__global__ void glu_bwd_scalar(const bf16* gate, const bf16* up, const bf16* dh, bf16* dgate,
                               bf16* dup, int64_t T, int F, int64_t ldg, int64_t ldu, int64_t lddh,
                               int64_t lddg, int64_t lddu) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= T * F) return;
  const int64_t t = i / F;
  const int c = (int)(i % F);
  const float gf = bf2f(gate[t * ldg + c]), uf = bf2f(up[t * ldu + c]), df = bf2f(dh[t * lddh + c]);
  dgate[t * lddg + c] = f2bf(df * uf * (GELU ? act_gelu_grad(gf) : act_silu_grad(gf)));
  dup[t * lddu + c] = f2bf(df * (GELU ? act_gelu(gf) : act_silu(gf)));
}

// ------------------------------------------------------------------ gradient accumulation
// Running mean over micro-batches, acc += (g - acc) / (k + 1) for the k-th (0-based) micro-batch
// (optax.MultiSteps with use_grad_mean, which the reference wraps its optimizer in,
// src/olmax/optim/config.py:153-154); k = 0 overwrites acc.
// [i, end) in vectors of 4 elements, `step` apart, and the ntail (< 4) elements behind vector n4
template <bool G_BF16, typename Int>
__device__ __forceinline__ void grad_accum_span(float* __restrict__ acc, const void* __restrict__ gv, Int i, Int end, Int step, Int n4,
                                                int ntail, float inv, int first) {
  for (; i < end; i += step) {
    float g[4];
    if (G_BF16) {
      Pack4 gp;
      gp.u = reinterpret_cast<const u32x2*>(gv)[i];
#pragma unroll
      for (int e = 0; e < 4; e++) g[e] = bf2f(gp.e[e]);
    } else {
      const f32x4 gf = reinterpret_cast<const f32x4*>(gv)[i];
#pragma unroll
      for (int e = 0; e < 4; e++) g[e] = gf[e];
    }
    f32x4 a;
    if (first) {
#pragma unroll
      for (int e = 0; e < 4; e++) a[e] = g[e];
    } else {
      a = reinterpret_cast<const f32x4*>(acc)[i];
#pragma unroll
      for (int e = 0; e < 4; e++) a[e] = a[e] + (g[e] - a[e]) * inv;
    }
    reinterpret_cast<f32x4*>(acc)[i] = a;
  }
  if ((int)threadIdx.x < ntail) {
    const Int j = n4 * 4 + (Int)threadIdx.x;
    const float g = G_BF16 ? bf2f(reinterpret_cast<const bf16*>(gv)[j]) : reinterpret_cast<const float*>(gv)[j];
    acc[j] = first ? g : acc[j] + (g - acc[j]) * inv;
  }
}
template <bool G_BF16>
__global__ __launch_bounds__(256) void grad_accum_kernel(float* __restrict__ acc, const void* __restrict__ gv, int64_t n,
                                                         float inv, int first) {
  grad_accum_span<G_BF16>(acc, gv, (int64_t)blockIdx.x * 256 + threadIdx.x, n / 4, (int64_t)gridDim.x * 256, n / 4,
                          blockIdx.x == 0 ? (int)(n & 3) : 0, inv, first);
}

// ------------------------------------------------------------------ ranges of the flat buffers
// A model has two to six vectors of a few KB per layer (norm weights, gradients in fp32) between its matrices, and
// a small one matrices of a few hundred KB: a launch for each is 3 to 5 us of latency and 2 us of gap.  One launch takes up to
// 32 of them: CHUNK elements to a workgroup, one vector of 4 to a lane; a workgroup finds its range with one load per lane and a ballot.
__device__ __forceinline__ int find_range(const FlatRanges& t) {
  const int lane = threadIdx.x & 63;
  const int first = lane < t.count ? t.r[lane & (FlatRanges::MAX - 1)].first : 0x7fffffff;
  return __builtin_amdgcn_readfirstlane((int)__builtin_popcountll(__builtin_amdgcn_ballot_w64(first <= (int)blockIdx.x)) - 1);
}
// a workgroup's part of a range: its first element, vectors of 4, and the elements (< 4) behind them
struct RangeSpan {
  int64_t at;
  int n4, ntail;
  __device__ __forceinline__ explicit RangeSpan(const FlatRange& r) {
    const int skip = ((int)blockIdx.x - r.first) * FlatRanges::CHUNK, n = min(r.n - skip, FlatRanges::CHUNK);
    at = skip;
    n4 = n >> 2;
    ntail = n & 3;
  }
};
__global__ __launch_bounds__(256) void grad_accum_ranges_kernel(FlatRanges t, float* __restrict__ acc, const bf16* __restrict__ g,
                                                                const float* __restrict__ gf, float inv, int first) {
  const FlatRange r = t.r[find_range(t)];
  const RangeSpan sp(r);
  acc += r.off + sp.at;
  if (r.g_f32) grad_accum_span<false>(acc, gf + r.goff + sp.at, (int)threadIdx.x, sp.n4, 256, sp.n4, sp.ntail, inv, first);
  else grad_accum_span<true>(acc, g + r.goff + sp.at, (int)threadIdx.x, sp.n4, 256, sp.n4, sp.ntail, inv, first);
}

// ------------------------------------------------------------------ synthetic token batches
// inputs[b, s] = (s + offset[b]) mod V, targets = inputs + 1 (a target equals V, one past the
// vocabulary, whenever the input is V - 1: the loss treats such a label as an all-zero one-hot).
__global__ __launch_bounds__(256) void sequential_tokens_kernel(const int32_t* __restrict__ offsets,
                                                                int32_t* __restrict__ inputs,
                                                                int32_t* __restrict__ targets, int B, int S, int V) {
  const int64_t total = (int64_t)B * S;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int b = (int)(i / S), sidx = (int)(i % S);
    const int32_t tok = (int32_t)(((int64_t)sidx + offsets[b]) % V);
    inputs[i] = tok;
    targets[i] = tok + 1;
  }
}

// ------------------------------------------------------------------ embedding
// ids follow NumPy/JAX indexing of `weight[ids]` (src/olmax/nn/embedding.py:32): a negative id
// counts from the end, and what is still outside [0, V) is clamped (JAX's gather mode for
// out-of-bounds reads; upstream semantics, the data path never produces such ids).  The
// scatter-add is the transpose of exactly that gather.
__device__ __forceinline__ int wrap_clamp_id(int id, int V) {
  if (id < 0) id += V;
  return id < 0 ? 0 : (id >= V ? V - 1 : id);
}
__global__ __launch_bounds__(256) void embed_fwd_kernel(const int32_t* __restrict__ ids,
                                                        const bf16* __restrict__ W,
                                                        bf16* __restrict__ out, int64_t T, int d,
                                                        int V) {
  const int cpr = d / 8;
  const int64_t total = T * cpr;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t t = i / cpr;
    const int c = (int)(i % cpr) * 8;
    const int id = wrap_clamp_id(ids[t], V);
    *reinterpret_cast<u32x4*>(out + t * d + c) = *reinterpret_cast<const u32x4*>(W + (int64_t)id * d + c);
  }
}
__global__ void embed_fwd_scalar(const int32_t* ids, const bf16* W, bf16* out, int64_t T, int d, int V) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= T * d) return;
  const int id = wrap_clamp_id(ids[i / d], V);
  out[i] = W[(int64_t)id * d + i % d];
}
// dW[ids[t], :] += dh[t, :]   (fp32 accumulate; duplicates sum through atomics)
__global__ __launch_bounds__(256) void embed_bwd_kernel(const int32_t* __restrict__ ids,
                                                        const bf16* __restrict__ dh,
                                                        float* __restrict__ dW, int64_t T, int d,
                                                        int V) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < T * d; i += (int64_t)gridDim.x * 256) {
    const int64_t t = i / d;
    const int c = (int)(i % d);
    const int id = wrap_clamp_id(ids[t], V);
    atomicAdd(&dW[(int64_t)id * d + c], bf2f(dh[i]));
  }
}

// ------------------------------------------------------------------ AdamW
// p, m, v fp32 in place; g bf16 or fp32; optional bf16 working copy of the new p.
// bc1 = 1 - b1^t, bc2 = 1 - b2^t (computed on the host in double), or, with hyper_dev, lr and the
// two bias corrections read from device memory (a host whose schedule and step count live on
// the device, like optax's injected hyper-parameters inside a jitted step).
// p - lr (m_hat / (sqrt(v_hat) + eps) + wd p) with the hardware square root and reciprocal (1 ulp
// each) instead of the correctly rounded library forms: those expand to ~22 vector instructions
// per element, and when this kernel shares a CU with a GEMM every vector instruction it issues
// takes an issue slot from the GEMM's MFMAs.  The update moves by a few 1e-7 of its own size
// (lr-sized), far below one ulp of p.
__device__ __forceinline__ float adamw_new_p(float p, float mh, float vh, float lr, float eps, float wd) {
  const float r = __builtin_amdgcn_rcpf(__builtin_amdgcn_sqrtf(vh) + eps);
  return __builtin_fmaf(-lr, __builtin_fmaf(mh, r, wd * p), p);
}

struct AdamwScalars {
  float lr, b1, b2, eps, wd, ibc1, ibc2, gscale;
};
__device__ __forceinline__ AdamwScalars adamw_scalars(float lr, float b1, float b2, float eps, float wd, float bc1, float bc2, float gscale,
                                                      const float* __restrict__ gscale_dev, const float* __restrict__ hyper_dev) {
  if (gscale_dev) gscale *= *gscale_dev;
  if (hyper_dev) {  // step-dependent scalars from device memory (wave-uniform scalar loads)
    lr = hyper_dev[0];
    bc1 = hyper_dev[1];
    bc2 = hyper_dev[2];
  }
  // (results of vector instructions that are the same in every lane: back to scalar registers)
  auto uniform = [](float x) { return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x))); };
  return {lr, b1, b2, eps, wd, uniform(1.f / bc1), uniform(1.f / bc2), uniform(gscale)};
}

// The vector of 4 elements `lane` vectors behind the (wave-uniform) pointers.  Every element is touched exactly once: streaming
// (non-temporal) accesses keep the 28 B/param out of the way of the L2.  One 32-bit offset register addresses all five arrays and
// the four loads are requested together: with a 64-bit pointer register pair per array they did not fit the 32 registers of
// the kernels below and waited for each other.
// HAS_G false: the gradient is zero and not read.
template <bool G_BF16, bool HAS_G = true>
__device__ __forceinline__ void adamw_vec(float* __restrict__ p, const void* __restrict__ gv, float* __restrict__ m, float* __restrict__ v,
                                          bf16* __restrict__ shadow, uint32_t lane, const AdamwScalars& c) {
  const float lr = c.lr, b1 = c.b1, b2 = c.b2, eps = c.eps, wd = c.wd, ibc1 = c.ibc1, ibc2 = c.ibc2, gscale = c.gscale;
  const float omb1 = 1.f - b1, omb2 = 1.f - b2;
  // opaque scalar bases and lane: a loop's pointer arithmetic stays in scalar registers
  uint64_t pa = (uint64_t)p, ga = (uint64_t)gv, ma = (uint64_t)m, va = (uint64_t)v, sa = (uint64_t)shadow;
  asm volatile("" : "+v"(lane), "+s"(pa), "+s"(ga), "+s"(ma), "+s"(va), "+s"(sa));
  const uint32_t o16 = lane * 16, o8 = lane * 8;
#define GLOBAL(T, base, bytes) ((__attribute__((address_space(1))) T*)((__attribute__((address_space(1))) char*)(base) + (bytes)))
  f32x4 gf;
  Pack4 gp;
  if (!HAS_G) gf = f32x4{0.f, 0.f, 0.f, 0.f};
  else if (G_BF16) gp.u = __builtin_nontemporal_load(GLOBAL(u32x2, ga, o8));
  else gf = __builtin_nontemporal_load(GLOBAL(f32x4, ga, o16));
  f32x4 mv = __builtin_nontemporal_load(GLOBAL(f32x4, ma, o16));
  f32x4 vv = __builtin_nontemporal_load(GLOBAL(f32x4, va, o16));
  f32x4 pv = __builtin_nontemporal_load(GLOBAL(f32x4, pa, o16));
  __builtin_amdgcn_sched_barrier(0);
  Pack4 sh;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const float ge = (G_BF16 ? bf2f(gp.e[e]) : gf[e]) * gscale;
    mv[e] = b1 * mv[e] + omb1 * ge;
    vv[e] = b2 * vv[e] + omb2 * ge * ge;
    pv[e] = adamw_new_p(pv[e], mv[e] * ibc1, vv[e] * ibc2, lr, eps, wd);
    sh.e[e] = f2bf(pv[e]);
  }
  __builtin_nontemporal_store(pv, GLOBAL(f32x4, pa, o16));
  __builtin_nontemporal_store(mv, GLOBAL(f32x4, ma, o16));
  __builtin_nontemporal_store(vv, GLOBAL(f32x4, va, o16));
  if (sa) __builtin_nontemporal_store(sh.u, GLOBAL(u32x2, sa, o8));
#undef GLOBAL
}
// element j (of the last n % 4)
template <bool G_BF16, typename Int>
__device__ __forceinline__ void adamw_one(float* __restrict__ p, const void* __restrict__ gv, float* __restrict__ m, float* __restrict__ v,
                                          bf16* __restrict__ shadow, Int j, const AdamwScalars& c) {
  const float lr = c.lr, b1 = c.b1, b2 = c.b2, eps = c.eps, wd = c.wd, ibc1 = c.ibc1, ibc2 = c.ibc2, gscale = c.gscale;
  const float omb1 = 1.f - b1, omb2 = 1.f - b2;
  const float ge = (G_BF16 ? bf2f(reinterpret_cast<const bf16*>(gv)[j]) : reinterpret_cast<const float*>(gv)[j]) * gscale;
  // the same operations in the same order as the vector body: where a range is cut does not
  // change any element's result
  const float mm = b1 * m[j] + omb1 * ge;
  const float vv = b2 * v[j] + omb2 * ge * ge;
  const float pp = adamw_new_p(p[j], mm * ibc1, vv * ibc2, lr, eps, wd);
  m[j] = mm;
  v[j] = vv;
  p[j] = pp;
  if (shadow) shadow[j] = f2bf(pp);
}

// The kernel is held to 32 registers (amdgpu_num_vgpr counts pairs
// of the unified file on this target) so that one of its waves fits on a SIMD beside two
// 240-register GEMM waves when it runs on a second stream, and it is launched as a small
// grid-stride grid (two workgroups per CU): the whole grid then sweeps five arrays as
// contiguous 2 MB fronts, which measured 5.6 TB/s against 4.7 TB/s for one workgroup per 8 KB.  The scalar bases of adamw_vec
// bring the width-1024 step from 7490 to 7226 us; two layers of the 7B step move by less than boxes differ (everything since the ragged GEMM forms
// came, together: 44.6 -> 43.3 and 44.7 -> 43.6 ms).
template <bool G_BF16>
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_vgpr(16))) void adamw_kernel(
    float* __restrict__ p, const void* __restrict__ gv, float* __restrict__ m, float* __restrict__ v,
    bf16* __restrict__ shadow, int64_t n, float lr, float b1, float b2, float eps, float wd, float bc1,
    float bc2, float gscale, const float* __restrict__ gscale_dev, const float* __restrict__ hyper_dev) {
  const AdamwScalars c = adamw_scalars(lr, b1, b2, eps, wd, bc1, bc2, gscale, gscale_dev, hyper_dev);
  const int64_t n4 = n / 4, stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256; i < n4; i += stride)
    if (threadIdx.x < (uint32_t)min(n4 - i, (int64_t)256))
      adamw_vec<G_BF16>(p + i * 4, reinterpret_cast<const char*>(gv) + i * (G_BF16 ? 8 : 16), m + i * 4, v + i * 4,
                        shadow ? shadow + i * 4 : nullptr, threadIdx.x, c);
  // tail (n % 4) handled by the first threads of block 0
  if (blockIdx.x == 0 && threadIdx.x < (n & 3)) adamw_one<G_BF16>(p, gv, m, v, shadow, n4 * 4 + threadIdx.x, c);
}
// (also beside GEMM waves, hence the same 32 registers)
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_vgpr(16))) void adamw_ranges_kernel(
    FlatRanges t, float* __restrict__ p, const bf16* __restrict__ g, const float* __restrict__ gf, float* __restrict__ m, float* __restrict__ v,
    bf16* __restrict__ shadow, float lr, float b1, float b2, float eps, float wd, float bc1, float bc2,
    const float* __restrict__ gscale_dev, const float* __restrict__ hyper_dev) {
  const FlatRange r = t.r[find_range(t)];
  const RangeSpan sp(r);
  const AdamwScalars c = adamw_scalars(lr, b1, b2, eps, r.decay ? wd : 0.f, bc1, bc2, 1.f, gscale_dev, hyper_dev);
  const int64_t o = r.off + sp.at, go = r.goff + sp.at;
  const int i = threadIdx.x, j = sp.n4 * 4 + i;
  const void* gr = r.g_f32 ? (const void*)(gf + go) : g + go;
  p += o, m += o, v += o, shadow += o;
  if (r.g_f32) {
    if (i < sp.n4) adamw_vec<false>(p, gr, m, v, shadow, (uint32_t)i, c);
    if (i < sp.ntail) adamw_one<false>(p, gr, m, v, shadow, j, c);
  } else {
    if (i < sp.n4) adamw_vec<true>(p, gr, m, v, shadow, (uint32_t)i, c);
    if (i < sp.ntail) adamw_one<true>(p, gr, m, v, shadow, j, c);
  }
}

// An embedding's update in two parts, so that the larger one need not wait for the scatter-add at the end of the backward pass: rows that no
// token of the batch names (their gradient is zero, or under a tied head final with the head's weight gradient), and the
// others.  first_use[row]: the first token that names it, INT32_MAX if none does.  (gscale, 1 here, is an argument as in adamw_kernel: as a
// constant the multiplication goes, other products become fused ones, and an element depends on the kernel by an ulp.)
__global__ __launch_bounds__(256) void first_use_kernel(const int32_t* __restrict__ ids, int32_t* __restrict__ first_use, int64_t T, int V) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t < T) atomicMin(&first_use[wrap_clamp_id(ids[t], V)], (int32_t)t);
}
// n elements from element `off` of row `row` on (both multiples of 4, rows of d >= 1024: a workgroup's 1024 elements lie in two
// rows at most, whose flags are scalar loads).  Registers and grid as adamw_kernel.
template <bool HAS_G>
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_vgpr(16))) void adamw_unused_rows_kernel(
    float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v, bf16* __restrict__ shadow, int64_t n,
    const int32_t* __restrict__ first_use, int row, int off, int d, float lr, float b1, float b2, float eps, float wd, float bc1, float bc2,
    float gscale, const float* __restrict__ hyper_dev) {
  const AdamwScalars c = adamw_scalars(lr, b1, b2, eps, wd, bc1, bc2, gscale, nullptr, hyper_dev);
  const int64_t n4 = n / 4, stride = (int64_t)gridDim.x * 256;
  const int step_rows = (int)(stride * 4 / d), step_off = (int)(stride * 4 % d);
  const int64_t at = (int64_t)off + (int64_t)blockIdx.x * 1024;
  row += (int)(at / d);
  off = (int)(at % d);
  for (int64_t i = (int64_t)blockIdx.x * 256; i < n4; i += stride) {
    const bool here = first_use[row] == INT32_MAX, next = off + 1024 > d && i + (d - off) / 4 < n4 && first_use[row + 1] == INT32_MAX;
    if ((off + (int)threadIdx.x * 4 < d ? here : next) && threadIdx.x < (uint32_t)min(n4 - i, (int64_t)256))
      adamw_vec<false, HAS_G>(p + i * 4, g + i * 4, m + i * 4, v + i * 4, shadow + i * 4, threadIdx.x, c);
    row += step_rows;
    off += step_off;
    if (off >= d) off -= d, row++;
  }
}
__global__ __launch_bounds__(256) void adamw_used_rows_kernel(
    float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v, bf16* __restrict__ shadow,
    const int32_t* __restrict__ ids, const int32_t* __restrict__ first_use, int64_t T, int V, int d, float lr, float b1, float b2, float eps,
    float wd, float bc1, float bc2, float gscale, const float* __restrict__ hyper_dev) {
  const AdamwScalars c = adamw_scalars(lr, b1, b2, eps, wd, bc1, bc2, gscale, nullptr, hyper_dev);
  for (int64_t t = blockIdx.x; t < T; t += gridDim.x) {
    const int row = wrap_clamp_id(ids[t], V);
    if (first_use[row] != t) continue;
    const int64_t o = (int64_t)row * d;
    for (int j = 0; j < d; j += 1024)
      if (j + (int)threadIdx.x * 4 < d) adamw_vec<false>(p + o + j, g + o + j, m + o + j, v + o + j, shadow + o + j, threadIdx.x, c);
  }
}

// sum of squares of a gradient leaf, accumulated (fp32 atomics) into *out
// Bound by HBM at large sizes (4 TB/s), by what meets at one address at small ones: all workgroups end together and their atomics take 13 ns each.  So few and
// large ones, 512 of sixteen waves at most, eight loads of a lane in flight over a contiguous span.  us, up to 2048 workgroups of four waves with two
// loads -> so: fp32 in the cache 1 M 17.0 -> 7.0, 6.3 M 30.6 -> 9.7, 60 M 54 -> 37, from HBM 6.3 M 35 -> 15, 60 M 92 -> 89, 155 M 164 -> 162; bf16 6.3 M 30.2 -> 7.2.  A step
// with clipping: 6.3 M parameters 690 -> 622, 155 M 6917 -> 6807.  (Non-temporal loads read 155 M in 97 us, but then the update that follows
// writes back what they leave in the cache, 503 -> 546: nothing gained.)
// Up to 16384 vectors workgroups of four waves, with one load a lane up to 1024 and four beyond: sixteen waves and code for eight loads take 0.5 to 0.8 us more (a call on cold fp32, with
// the events around it, 4096 9.4 -> 8.8, 65536 9.4 -> 9.2).  A vector is two chains of additions: as one, 4096 numbers were 1.28 times as far from the exact sum.
template <bool G_BF16, int NT, int U>
__global__ __launch_bounds__(NT) void sumsq_kernel(const void* __restrict__ gv, int64_t n, int64_t head, int width, float* __restrict__ out) {
  constexpr int VEC = G_BF16 ? 8 : 4;
  __shared__ float red[NT / 64];
  float s[8] = {};
  auto element = [&](int64_t j) {
    const float x = G_BF16 ? bf2f(reinterpret_cast<const bf16*>(gv)[j]) : reinterpret_cast<const float*>(gv)[j];
    s[0] += x * x;
  };
  const u32x4* g = reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(gv) + head * (16 / VEC));
  const int64_t nv = (n - head) / VEC;
  for (int64_t b = blockIdx.x; b * NT * width < nv; b += gridDim.x) {
    const int64_t i = b * NT * width + threadIdx.x;
    u32x4 q[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      q[u] = u32x4{0, 0, 0, 0};
      if (u < width && i + u * NT < nv) q[u] = g[i + u * NT];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      Pack8 b8;
      b8.u = q[u];
      const f32x4 f = (const f32x4&)q[u];
#pragma unroll
      for (int e = 0; e < VEC; e++) {
        const float x = G_BF16 ? bf2f(b8.e[e]) : f[e & 3];
        s[(u + (e & 1) * 4) % 8] += x * x;  // (two chains to a vector)
      }
    }
  }
  for (int64_t j = (int64_t)blockIdx.x * NT + threadIdx.x; j < head; j += (int64_t)gridDim.x * NT) element(j);
  if (const int64_t at = head + nv * VEC + threadIdx.x; blockIdx.x == 0 && at < n) element(at);
  const float t = block_sum<NT / 64>(((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])), red);
  if (threadIdx.x == 0) atomicAdd(out, t);
}

__global__ void cast_f32_bf16_kernel(const float* __restrict__ in, bf16* __restrict__ out, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = f2bf(in[i]);
}
__global__ void cast_bf16_f32_kernel(const bf16* __restrict__ in, float* __restrict__ out, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = bf2f(in[i]);
}
__global__ void fill_u32_kernel(uint32_t* __restrict__ p, uint32_t val, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = val;
}
// out = a + b (bf16), 8 per lane
__global__ __launch_bounds__(256) void add_bf16_kernel(const bf16* __restrict__ a, const bf16* __restrict__ b,
                                                       bf16* __restrict__ out, int64_t n8) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    Pack8 x, y, o;
    x.u = reinterpret_cast<const u32x4*>(a)[i];
    y.u = reinterpret_cast<const u32x4*>(b)[i];
#pragma unroll
    for (int e = 0; e < 8; e++) o.e[e] = f2bf(bf2f(x.e[e]) + bf2f(y.e[e]));
    reinterpret_cast<u32x4*>(out)[i] = o.u;
  }
}

int grid_1d(int64_t items, int cap = 8192) {
  int64_t g = (items + 255) / 256;
  return (int)(g < 1 ? 1 : (g > cap ? cap : g));
}

}  // namespace

extern "C" int32_t olmax_glu_fwd(hipStream_t stream, const void* gate, const void* up, void* out,
                                 int64_t T, int32_t F, int64_t ldg, int64_t ldu, int64_t ldo,
                                 int32_t act) {
  if (T == 0) return OLMAX_OK;
  OLMAX_CHECK(gate && up && out, OLMAX_ERR_ARG, "olmax_glu_fwd: null pointer");
  OLMAX_CHECK(T >= 0 && F > 0 && ldg >= F && ldu >= F && ldo >= F, OLMAX_ERR_SHAPE, "olmax_glu_fwd: bad shape");
  OLMAX_CHECK(act == 0 || act == 1, OLMAX_ERR_ARG, "olmax_glu_fwd: act must be 0 (silu) or 1 (gelu-tanh)");
  const bf16 *g = (const bf16*)gate, *u = (const bf16*)up;
  bf16* o = (bf16*)out;
  const bool vec = F % 8 == 0 && ldg % 8 == 0 && ldu % 8 == 0 && ldo % 8 == 0 && aligned16(gate) && aligned16(up) && aligned16(out);
  if (vec) {
    const int grid = grid_1d(T * (F / 8));
    if (act) hipLaunchKernelGGL(glu_fwd_kernel<true>, dim3(grid), dim3(256), 0, stream, g, u, o, T, F, ldg, ldu, ldo);
    else hipLaunchKernelGGL(glu_fwd_kernel<false>, dim3(grid), dim3(256), 0, stream, g, u, o, T, F, ldg, ldu, ldo);
  } else {
    const unsigned grid = (unsigned)((T * F + 255) / 256);
    if (act) hipLaunchKernelGGL(glu_fwd_scalar<true>, dim3(grid), dim3(256), 0, stream, g, u, o, T, F, ldg, ldu, ldo);
    else hipLaunchKernelGGL(glu_fwd_scalar<false>, dim3(grid), dim3(256), 0, stream, g, u, o, T, F, ldg, ldu, ldo);
  }
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

extern "C" int32_t olmax_glu_bwd(hipStream_t stream, const void* gate, const void* up,
                                 const void* dh, void* dgate, void* dup, int64_t T, int32_t F,
                                 int64_t ldg, int64_t ldu, int64_t lddh, int64_t lddg, int64_t lddu,
                                 int32_t act) {
  if (T == 0) return OLMAX_OK;
  OLMAX_CHECK(gate && up && dh && dgate && dup, OLMAX_ERR_ARG, "olmax_glu_bwd: null pointer");
  OLMAX_CHECK(T >= 0 && F > 0 && ldg >= F && ldu >= F && lddh >= F && lddg >= F && lddu >= F, OLMAX_ERR_SHAPE, "olmax_glu_bwd: bad shape");
  OLMAX_CHECK(act == 0 || act == 1, OLMAX_ERR_ARG, "olmax_glu_bwd: act must be 0 (silu) or 1 (gelu-tanh)");
  const bf16 *g = (const bf16*)gate, *u = (const bf16*)up, *d = (const bf16*)dh;
  bf16 *og = (bf16*)dgate, *ou = (bf16*)dup;
  const bool vec = F % 8 == 0 && ldg % 8 == 0 && ldu % 8 == 0 && lddh % 8 == 0 && lddg % 8 == 0 && lddu % 8 == 0 &&
                   aligned16(gate) && aligned16(up) && aligned16(dh) && aligned16(dgate) && aligned16(dup);
  if (vec) {
    const int grid = grid_1d(T * (F / 8));
    if (act) hipLaunchKernelGGL(glu_bwd_kernel<true>, dim3(grid), dim3(256), 0, stream, g, u, d, og, ou, T, F, ldg, ldu, lddh, lddg, lddu);
    else hipLaunchKernelGGL(glu_bwd_kernel<false>, dim3(grid), dim3(256), 0, stream, g, u, d, og, ou, T, F, ldg, ldu, lddh, lddg, lddu);
  } else {
    const unsigned grid = (unsigned)((T * F + 255) / 256);
    if (act) hipLaunchKernelGGL(glu_bwd_scalar<true>, dim3(grid), dim3(256), 0, stream, g, u, d, og, ou, T, F, ldg, ldu, lddh, lddg, lddu);
    else hipLaunchKernelGGL(glu_bwd_scalar<false>, dim3(grid), dim3(256), 0, stream, g, u, d, og, ou, T, F, ldg, ldu, lddh, lddg, lddu);
  }
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

extern "C" int32_t olmax_embed_fwd(hipStream_t stream, const int32_t* ids, const void* W, void* out,
                                   int64_t T, int32_t d, int32_t V) {
  if (T == 0) return OLMAX_OK;
  OLMAX_CHECK(ids && W && out, OLMAX_ERR_ARG, "olmax_embed_fwd: null pointer");
  OLMAX_CHECK(T >= 0 && d > 0 && V > 0, OLMAX_ERR_SHAPE, "olmax_embed_fwd: bad shape");
  if (d % 8 == 0 && aligned16(W) && aligned16(out))
    hipLaunchKernelGGL(embed_fwd_kernel, dim3(grid_1d(T * (d / 8))), dim3(256), 0, stream, ids, (const bf16*)W, (bf16*)out, T, d, V);
  else
    hipLaunchKernelGGL(embed_fwd_scalar, dim3((unsigned)((T * d + 255) / 256)), dim3(256), 0, stream, ids, (const bf16*)W, (bf16*)out, T, d, V);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

extern "C" int32_t olmax_grad_accumulate(hipStream_t stream, float* acc, const void* g, int64_t n, int32_t grad_is_bf16,
                                         int32_t mini_step) {
  if (n == 0) return OLMAX_OK;
  OLMAX_CHECK(acc && g && n >= 0 && mini_step >= 0, OLMAX_ERR_ARG, "olmax_grad_accumulate: bad argument");
  OLMAX_CHECK(aligned16(acc) && (((uintptr_t)g) & (grad_is_bf16 ? 7 : 15)) == 0, OLMAX_ERR_ALIGN,
              "olmax_grad_accumulate: acc / fp32 g must be 16-byte aligned, bf16 g 8-byte aligned");
  const int grid = grid_1d((n + 3) / 4, 2048);
  const float inv = 1.f / (float)(mini_step + 1);
  if (grad_is_bf16) hipLaunchKernelGGL(grad_accum_kernel<true>, dim3(grid), dim3(256), 0, stream, acc, g, n, inv, mini_step == 0);
  else hipLaunchKernelGGL(grad_accum_kernel<false>, dim3(grid), dim3(256), 0, stream, acc, g, n, inv, mini_step == 0);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

static bool ranges_aligned(const FlatRanges& t) {
  for (int i = 0; i < t.count; i++)
    if (t.r[i].off % 4 || t.r[i].goff % 4) return false;
  return true;
}

int olmax_grad_accumulate_ranges(hipStream_t stream, const FlatRanges& t, float* acc, const bf16* g, const float* gf, int mini_step) {
  if (t.blocks == 0) return OLMAX_OK;
  OLMAX_CHECK(aligned16(acc) && aligned16(gf) && (((uintptr_t)g) & 7) == 0 && ranges_aligned(t), OLMAX_ERR_ALIGN,
              "olmax_grad_accumulate: acc / fp32 g must be 16-byte aligned, bf16 g 8-byte aligned");
  hipLaunchKernelGGL(grad_accum_ranges_kernel, dim3((unsigned)t.blocks), dim3(256), 0, stream, t, acc, g, gf,
                     1.f / (float)(mini_step + 1), (int)(mini_step == 0));
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

extern "C" int32_t olmax_sequential_tokens(hipStream_t stream, const int32_t* start_offsets, int32_t* inputs,
                                           int32_t* targets, int32_t B, int32_t S, int32_t V) {
  if (B == 0 || S == 0) return OLMAX_OK;
  OLMAX_CHECK(start_offsets && inputs && targets, OLMAX_ERR_ARG, "olmax_sequential_tokens: null pointer");
  OLMAX_CHECK(B > 0 && S > 0 && V > 0, OLMAX_ERR_SHAPE, "olmax_sequential_tokens: bad shape");
  hipLaunchKernelGGL(sequential_tokens_kernel, dim3(grid_1d((int64_t)B * S)), dim3(256), 0, stream, start_offsets, inputs,
                     targets, B, S, V);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

// dW (fp32 [V, d]) is ACCUMULATED into: the caller zeroes it (or seeds it, for tied heads).
extern "C" int32_t olmax_embed_bwd(hipStream_t stream, const int32_t* ids, const void* dh, float* dW,
                                   int64_t T, int32_t d, int32_t V) {
  if (T == 0) return OLMAX_OK;
  OLMAX_CHECK(ids && dh && dW, OLMAX_ERR_ARG, "olmax_embed_bwd: null pointer");
  OLMAX_CHECK(T >= 0 && d > 0 && V > 0, OLMAX_ERR_SHAPE, "olmax_embed_bwd: bad shape");
  hipLaunchKernelGGL(embed_bwd_kernel, dim3(grid_1d(T * d)), dim3(256), 0, stream, ids, (const bf16*)dh, dW, T, d, V);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

// As olmax_adamw, with an additional device-resident gradient scale (NULL = none) so that
// global-norm clipping needs no host round trip.
extern "C" int32_t olmax_adamw_dscale(hipStream_t stream, float* p, const void* g, float* m, float* v,
                                      void* shadow_bf16, int64_t n, int32_t grad_is_bf16, float lr, float b1,
                                      float b2, float eps, float wd, int64_t step, float grad_scale,
                                      const float* grad_scale_dev) {
  // two workgroups per CU: the fastest grid when the kernel has the GPU to itself
  return olmax_adamw_grid(stream, p, g, m, v, shadow_bf16, n, grad_is_bf16, lr, b1, b2, eps, wd, step, grad_scale,
                          grad_scale_dev, 512, nullptr);
}

// As olmax_adamw_dscale with lr and the bias corrections in device memory:
// hyper_dev = {lr, 1 - b1^step, 1 - b2^step} (fp32), written by earlier work on the same stream.
extern "C" int32_t olmax_adamw_dev(hipStream_t stream, float* p, const void* g, float* m, float* v, void* shadow_bf16,
                                   int64_t n, int32_t grad_is_bf16, float b1, float b2, float eps, float wd,
                                   const float* hyper_dev, const float* grad_scale_dev) {
  OLMAX_CHECK(hyper_dev, OLMAX_ERR_ARG, "olmax_adamw_dev: hyper_dev is null");
  return olmax_adamw_grid(stream, p, g, m, v, shadow_bf16, n, grad_is_bf16, 0.f, b1, b2, eps, wd, 1, 1.f, grad_scale_dev, 512,
                          hyper_dev);
}

// Library-internal form with the grid size exposed: the overlapped train step runs it with one
// workgroup per CU on its second stream, which disturbs the GEMMs it shares the GPU with least.
int olmax_first_use(hipStream_t stream, const int32_t* ids, int32_t* first_use, int64_t T, int V) {
  hipLaunchKernelGGL(fill_u32_kernel, dim3(grid_1d(V)), dim3(256), 0, stream, (uint32_t*)first_use, 0x7fffffffu, (int64_t)V);
  hipLaunchKernelGGL(first_use_kernel, dim3((unsigned)((T + 255) / 256)), dim3(256), 0, stream, ids, first_use, T, V);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

int olmax_adamw_unused_rows(hipStream_t stream, float* p, const float* g, float* m, float* v, bf16* shadow, const int32_t* first_use, int64_t at,
                            int64_t n, int d, float lr, float b1, float b2, float eps, float wd, int64_t step, int grid_cap,
                            const float* hyper_dev) {
  if (n == 0) return OLMAX_OK;
  const float bc1 = (float)(1.0 - pow((double)b1, (double)step)), bc2 = (float)(1.0 - pow((double)b2, (double)step));
  auto kern = g ? adamw_unused_rows_kernel<true> : adamw_unused_rows_kernel<false>;
  hipLaunchKernelGGL(kern, dim3(grid_1d(n / 4, grid_cap)), dim3(256), 0, stream, p + at, g ? g + at : nullptr, m + at, v + at, shadow + at, n,
                     first_use, (int)(at / d), (int)(at % d), d, lr, b1, b2, eps, wd, bc1, bc2, 1.f, hyper_dev);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

int olmax_adamw_used_rows(hipStream_t stream, float* p, const float* g, float* m, float* v, bf16* shadow, const int32_t* ids,
                          const int32_t* first_use, int64_t T, int V, int d, float lr, float b1, float b2, float eps, float wd, int64_t step,
                          const float* hyper_dev) {
  const float bc1 = (float)(1.0 - pow((double)b1, (double)step)), bc2 = (float)(1.0 - pow((double)b2, (double)step));
  hipLaunchKernelGGL(adamw_used_rows_kernel, dim3((unsigned)(T < 2048 ? T : 2048)), dim3(256), 0, stream, p, g, m, v, shadow, ids, first_use, T, V, d,
                     lr, b1, b2, eps, wd, bc1, bc2, 1.f, hyper_dev);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

int olmax_adamw_grid(hipStream_t stream, float* p, const void* g, float* m, float* v, void* shadow_bf16, int64_t n,
                     int32_t grad_is_bf16, float lr, float b1, float b2, float eps, float wd, int64_t step,
                     float grad_scale, const float* grad_scale_dev, int grid_cap, const float* hyper_dev) {
  if (n == 0) return OLMAX_OK;
  OLMAX_CHECK(p && g && m && v, OLMAX_ERR_ARG, "olmax_adamw: null pointer");
  OLMAX_CHECK(n >= 0 && step >= 1, OLMAX_ERR_ARG, "olmax_adamw: n must be >= 0 and step >= 1 (1-based)");
  OLMAX_CHECK(aligned16(p) && aligned16(m) && aligned16(v) && (((uintptr_t)g) & (grad_is_bf16 ? 7 : 15)) == 0 &&
                  (!shadow_bf16 || (((uintptr_t)shadow_bf16) & 7) == 0),
              OLMAX_ERR_ALIGN, "olmax_adamw: buffers must be 16-byte aligned (bf16 buffers 8-byte)");
  const float bc1 = (float)(1.0 - pow((double)b1, (double)step));
  const float bc2 = (float)(1.0 - pow((double)b2, (double)step));
  const int grid = grid_1d((n + 3) / 4, grid_cap);
  if (grad_is_bf16)
    hipLaunchKernelGGL(adamw_kernel<true>, dim3(grid), dim3(256), 0, stream, p, g, m, v, (bf16*)shadow_bf16, n, lr, b1, b2, eps, wd, bc1, bc2, grad_scale, grad_scale_dev, hyper_dev);
  else
    hipLaunchKernelGGL(adamw_kernel<false>, dim3(grid), dim3(256), 0, stream, p, g, m, v, (bf16*)shadow_bf16, n, lr, b1, b2, eps, wd, bc1, bc2, grad_scale, grad_scale_dev, hyper_dev);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

int olmax_adamw_ranges(hipStream_t stream, const FlatRanges& t, float* p, const bf16* g, const float* gf, float* m, float* v, bf16* shadow,
                       float lr, float b1, float b2, float eps, float wd, int64_t step, const float* grad_scale_dev,
                       const float* hyper_dev) {
  if (t.blocks == 0) return OLMAX_OK;
  OLMAX_CHECK(step >= 1, OLMAX_ERR_ARG, "olmax_adamw: step must be >= 1 (1-based)");
  OLMAX_CHECK(aligned16(p) && aligned16(m) && aligned16(v) && aligned16(gf) && (((uintptr_t)g) & 7) == 0 && (((uintptr_t)shadow) & 7) == 0 &&
                  ranges_aligned(t),
              OLMAX_ERR_ALIGN, "olmax_adamw: buffers must be 16-byte aligned (bf16 buffers 8-byte)");
  const float bc1 = (float)(1.0 - pow((double)b1, (double)step));
  const float bc2 = (float)(1.0 - pow((double)b2, (double)step));
  hipLaunchKernelGGL(adamw_ranges_kernel, dim3((unsigned)t.blocks), dim3(256), 0, stream, t, p, g, gf, m, v, shadow, lr, b1, b2, eps, wd,
                     bc1, bc2, grad_scale_dev, hyper_dev);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

extern "C" int32_t olmax_adamw(hipStream_t stream, float* p, const void* g, float* m, float* v,
                               void* shadow_bf16, int64_t n, int32_t grad_is_bf16, float lr, float b1,
                               float b2, float eps, float wd, int64_t step, float grad_scale) {
  return olmax_adamw_dscale(stream, p, g, m, v, shadow_bf16, n, grad_is_bf16, lr, b1, b2, eps, wd, step, grad_scale, nullptr);
}

// *out (fp32 scalar) += sum(g^2); the caller zeroes it.
extern "C" int32_t olmax_sumsq(hipStream_t stream, const void* g, int64_t n, int32_t is_bf16, float* out) {
  if (n == 0) return OLMAX_OK;
  OLMAX_CHECK(g && out && n >= 0, OLMAX_ERR_ARG, "olmax_sumsq: bad argument");
  const int size = is_bf16 ? 2 : 4;
  // elements before the first aligned vector (all of them where they are not aligned to their size)
  const int64_t head = (uintptr_t)g % size ? n : std::min<int64_t>(n, (-(uintptr_t)g & 15) / size), nv = n * size / 16;
  const int nt = nv <= 16384 ? 256 : 1024, most = nv <= 1024 ? 1 : nv <= 16384 ? 4 : 8;
  const int width = (int)std::min<int64_t>(std::max<int64_t>(nv / (nt == 256 ? 1024 : 65536), 1), most);  // loads of a lane: 4 or 64 workgroups before they grow
  const dim3 grid((unsigned)std::min<int64_t>(std::max<int64_t>((nv + nt * width - 1) / (nt * width), 1), 512));
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(nt), 0, stream, g, n, head, width, out); };
  if (most == 1) go(is_bf16 ? sumsq_kernel<true, 256, 1> : sumsq_kernel<false, 256, 1>);
  else if (most == 4) go(is_bf16 ? sumsq_kernel<true, 256, 4> : sumsq_kernel<false, 256, 4>);
  else go(is_bf16 ? sumsq_kernel<true, 1024, 8> : sumsq_kernel<false, 1024, 8>);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}

extern "C" int32_t olmax_cast_f32_to_bf16(hipStream_t stream, const float* in, void* out, int64_t n) {
  if (n == 0) return OLMAX_OK;
  OLMAX_CHECK(in && out && n >= 0, OLMAX_ERR_ARG, "olmax_cast_f32_to_bf16: bad argument");
  hipLaunchKernelGGL(cast_f32_bf16_kernel, dim3(grid_1d(n)), dim3(256), 0, stream, in, (bf16*)out, n);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}
extern "C" int32_t olmax_cast_bf16_to_f32(hipStream_t stream, const void* in, float* out, int64_t n) {
  if (n == 0) return OLMAX_OK;
  OLMAX_CHECK(in && out && n >= 0, OLMAX_ERR_ARG, "olmax_cast_bf16_to_f32: bad argument");
  hipLaunchKernelGGL(cast_bf16_f32_kernel, dim3(grid_1d(n)), dim3(256), 0, stream, (const bf16*)in, out, n);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}
// Fill kernel (graph-capture safe replacement for memset); nbytes must be a multiple of 4.
extern "C" int32_t olmax_fill_zero(hipStream_t stream, void* p, int64_t nbytes) {
  OLMAX_CHECK(p && nbytes >= 0 && nbytes % 4 == 0 && (((uintptr_t)p) & 3) == 0, OLMAX_ERR_ARG, "olmax_fill_zero: need 4-byte aligned pointer and size");
  if (nbytes == 0) return OLMAX_OK;
  hipLaunchKernelGGL(fill_u32_kernel, dim3(grid_1d(nbytes / 4)), dim3(256), 0, stream, (uint32_t*)p, 0u, nbytes / 4);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}
extern "C" int32_t olmax_add_bf16(hipStream_t stream, const void* a, const void* b, void* out, int64_t n) {
  if (n == 0) return OLMAX_OK;
  OLMAX_CHECK(a && b && out && n >= 0 && n % 8 == 0 && aligned16(a) && aligned16(b) && aligned16(out), OLMAX_ERR_ARG, "olmax_add_bf16: need n % 8 == 0 and 16-byte alignment");
  hipLaunchKernelGGL(add_bf16_kernel, dim3(grid_1d(n / 8)), dim3(256), 0, stream, (const bf16*)a, (const bf16*)b, (bf16*)out, n / 8);
  OLMAX_LAUNCH_CHECK();
  return OLMAX_OK;
}
