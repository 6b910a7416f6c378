"""GPU tests of the launches that take many short pieces of the flat parameter buffers at once: AdamW, gradient
accumulation and the gradient norm over a model's leaves against the same thing leaf by leaf."""
import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu

# d_model and hidden decide where a leaf ends inside a workgroup's 1024 elements (or is shorter than that); 24 layers are 49 vectors
# and 24 runs of matrices, more than one table; width 1032 has runs that are too long for a table
CASES = [(24, 64, 136), (3, 256, 1024), (2, 1032, 1048), (1, 8, 8)]


def _model(layers, d, hidden):
    from olmax_amd import TransformerRecipe
    cfg = dataclasses.replace(TransformerRecipe.tiny_llama(), vocab_size=72, d_model=d, hidden_size=hidden, num_layers=layers,
                              n_heads=2, n_kv_heads=2, head_dim=8)
    m = cfg.build(batch_size=1, sequence_length=16, seed=1)
    g = torch.Generator(device="cuda").manual_seed(2)
    m.grad_bf16.normal_(0.0, 1e-2, generator=g)
    m.grad_f32.normal_(0.0, 1e-2, generator=g)
    m.init_optimizer_state()
    m.m.normal_(0.0, 1e-3, generator=g)
    m.v.uniform_(1e-6, 1e-4, generator=g)
    return m


def _leaf_grad(m, l):
    return m.grad_f32[l.grad_f32_offset:l.grad_f32_offset + l.numel] if l.grad_f32 else m.grad_bf16[l.offset:l.offset + l.numel]


@pytest.mark.parametrize("layers,d,hidden", CASES)
@pytest.mark.parametrize("clip", [None, 1e-3])
def test_adamw_over_all_leaves_equals_adamw_per_leaf(layers, d, hidden, clip):
    """Bit for bit without clipping (the same operations per element); with it the gradient norm against float64: fp32 sums
    of positive terms, at most 2^12 in a chain, 2^-24 each."""
    from olmax_amd import ops
    print(f"[case] adamw ranges L{layers} d{d} F{hidden} clip {clip}", flush=True)
    m = _model(layers, d, hidden)
    p, mm, vv = m.master.clone(), m.m.clone(), m.v.clone()
    shadow = m.params_bf16.clone()
    kw = dict(step=3, lr=1e-3, b1=0.9, b2=0.95, eps=1e-8)
    m.adamw_step(**kw, weight_decay=0.1, no_decay_modules=["*norm*"], max_grad_norm=clip)
    scale = 1.0
    if clip:
        norm = sum(_leaf_grad(m, l).double().square().sum() for l in m.leaves).sqrt().item()
        assert abs(m.norm_scratch[1].item() - norm) < 2 ** -12 * norm
        scale = m.norm_scratch[0].item()
        assert abs(scale - clip / norm) < 2 ** -11 * scale
    mask = m.weight_decay_mask(["*norm*"])
    for i, l in enumerate(m.leaves):
        s = slice(l.offset, l.offset + l.numel)
        ops.adamw_(p[s], _leaf_grad(m, l), mm[s], vv[s], wd=0.1 if mask[i] else 0.0, shadow=shadow[s], grad_scale=scale, **kw)
    assert torch.equal(m.master, p) and torch.equal(m.m, mm) and torch.equal(m.v, vv) and torch.equal(m.params_bf16, shadow)


@pytest.mark.parametrize("layers,d,hidden", CASES)
def test_accumulation_over_all_leaves(layers, d, hidden):
    """The running mean over three micro-batches; acc + (g - acc) / (k + 1) in fp32, three roundings of 2^-24 per step."""
    print(f"[case] accumulate ranges L{layers} d{d} F{hidden}", flush=True)
    m = _model(layers, d, hidden)
    want = torch.zeros(m.num_params, device="cuda", dtype=torch.float64)
    g = torch.Generator(device="cuda").manual_seed(5)
    for k in range(3):
        m.grad_bf16.normal_(0.0, 1.0, generator=g)
        m.grad_f32.normal_(0.0, 1.0, generator=g)
        m.accumulate_grads(k)
        for l in m.leaves:
            s = slice(l.offset, l.offset + l.numel)
            want[s] += (_leaf_grad(m, l).double() - want[s]) / (k + 1)
    assert (m.grad_acc.double() - want).abs().max().item() < 12 * 2 ** -24 * 6


@pytest.mark.parametrize("n,shift", [(1, 0), (7, 0), (4099, 0), (4099, 1), (3 << 20, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sum_of_squares(n, shift, dtype):
    """Vector and element loads; bound as for the norm above."""
    from olmax_amd import ops
    print(f"[case] sumsq n{n} shift{shift} {dtype}", flush=True)
    x = torch.randn(n + shift, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).to(dtype)[shift:]
    want = x.double().square().sum().item()
    assert abs(ops.sumsq(x).item() - want) < 2 ** -12 * want


@pytest.mark.parametrize("n", [8, 1023, 8192, 65536 * 4 + 4, 65536 * 8 * 8 + 9, 512 * 65536 + 3, (128 << 20) + 40])
@pytest.mark.parametrize("shift", [0, 1, 3])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sum_of_squares_by_spans(n, shift, dtype):
    """Ends of spans, of the elements before the first aligned vector and of the last one, one load of a lane to eight, several spans a workgroup, leaves beyond the
    cache.  Whole numbers: exact below 2^24, whatever the order; above it no chain has more than 573 additions (4 elements of each of
    9 spans, 3 + 6 + 16 in the workgroup, 512 workgroups), 2^-24 each; the test below is the exact one there."""
    from olmax_amd import ops
    print(f"[case] sumsq spans n{n} shift{shift} {dtype}", flush=True)
    x = torch.randint(-3, 4, (n + shift,), device="cuda", generator=torch.Generator(device="cuda").manual_seed(2), dtype=torch.int8).to(dtype)[shift:]
    x[0] = x[-1] = 64.0
    want = sum(c.double().square().sum().item() for c in x.split(1 << 20))
    got = ops.sumsq(x).item()
    assert got == want if want < 2 ** 24 else abs(got - want) < 712 * 2 ** -24 * want


@pytest.mark.parametrize("n", [8, 1000, 4096, 8192 + 5, 65536, 65536 * 4 + 4, 65536 * 8 * 8 + 9, 512 * 65536 + 3, (128 << 20) + 40])
@pytest.mark.parametrize("shift", [0, 1, 3])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sum_of_squares_counts_every_element_once(n, shift, dtype):
    """Zeros but for whole numbers around every power of two, the ends of all spans of 1024 to 65536 elements that the sizes above meet first and last, and both ends of the
    leaf: a sum below 2^24, exact in any order, to which each adds a share of its own."""
    from olmax_amd import ops
    print(f"[case] sumsq sparse n{n} shift{shift} {dtype}", flush=True)
    at = {0, 1, 2, 7, 8, n - 1, n - 2, n - 7, n - 8, n - 9}
    for span in [1 << i for i in range(2, 28)] + [n // 2, n // 3]:
        at |= {span + d for d in (-9, -8, -1, 0, 1, 7, 8)} | {n // span * span + d for d in (-1, 0, 1)}
    at = sorted(i for i in at if 0 <= i < n)
    x = torch.zeros(n + shift, device="cuda", dtype=dtype)[shift:]
    value = torch.arange(1, len(at) + 1, device="cuda") % 240 + 1  # whole numbers that bf16 holds
    x[torch.tensor(at, device="cuda")] = value.to(dtype)
    want = value.square().sum().item()
    assert want < 2 ** 24
    assert ops.sumsq(x).item() == want


@pytest.mark.parametrize("n", [8, 1000, 4096, 10000, 65536, 1 << 20])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sum_of_squares_adds_a_vector_as_two_chains(n, dtype):
    """2^24 and a 1 in every other place of the same 16 bytes: behind it in one chain the ones would be lost, 2^24 + 1 = 2^24 in fp32."""
    from olmax_amd import ops
    vec = 16 // dtype.itemsize
    for first in (0, (n // vec // 2) * vec, n // vec * vec - vec):
        print(f"[case] sumsq chains n{n} at {first} {dtype}", flush=True)
        x = torch.zeros(n, device="cuda", dtype=dtype)
        x[first] = 4096.0
        x[first + 1:first + vec:2] = 1.0
        assert ops.sumsq(x).item() == 2 ** 24 + vec // 2
