"""GPU parity test of forward products whose reductions several workgroups share (few tokens, a long reduction)."""
import dataclasses

import pytest
import torch

from test_gemm_choice_gpu import recorded, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("recipe,seq", [("llama3_8B", 512), ("llama3_8B", 600), ("olmo2_7B", 2048), ("olmo2_7B", 333)])
def test_down_projection(recipe, seq):
    """Pre-norm (a residual joins behind the sum) and post-norm blocks, whole and ragged rows, against the same block with its buffer cut to
    what it keeps, which leaves no room for parts: y differs by the order of fp32 additions in front of one or two roundings to bf16, 2^-9 each."""
    import ctypes
    from olmax_amd import TransformerRecipe
    from olmax_amd._lib import check, i32, i64, ptr, stream_ptr
    from olmax_amd.layer import TransformerBlock
    print(f"[case] forward split {recipe} S{seq}", flush=True)
    cfg = dataclasses.replace(getattr(TransformerRecipe, recipe)(), num_layers=1)
    block = TransformerBlock(cfg, batch_size=1, sequence_length=seq)
    g = torch.Generator(device="cuda").manual_seed(1)
    for w in (block.wqkv, block.wo, block.wgu, block.wdown):
        w.normal_(0.0, 0.02, generator=g)
    x, out = rnd(seq, cfg.d_model, seed=2), []
    got = recorded(lambda: out.append(block.forward(x)))
    assert any(key >> 18 & 1 and key >> 12 & 3 == 3 for key, *_ in got), got
    room = 256 << 18
    y = torch.empty_like(x)
    w = block._weights()
    got = recorded(lambda: check(block._L.olmax_block_fwd(stream_ptr(), ctypes.byref(block.c), ctypes.byref(w), i32(block.window), ptr(block.cos),
                                                          ptr(block.sin), ptr(x), ptr(y), ptr(block.acts), i64(block.acts.numel() - room))))
    assert not any(key >> 18 & 1 for key, *_ in got), got
    assert ((out[0].double() - y.double()).norm() / y.double().norm()).item() < 2 ** -8


@pytest.mark.parametrize("recipe,seq,split", [("llama3_8B", 1500, True), ("gemma2_like_27B", 2048, False)])
def test_a_larger_buffer(recipe, seq, split):
    """Behind the olmax_block_acts_bytes of a larger buffer nothing is written, though more parts would fit there (the second case: three for each
    of 144 tiles, 108 MB); the result is that of the exact buffer, bit for bit."""
    import ctypes
    from olmax_amd import TransformerRecipe
    from olmax_amd._lib import check, i32, i64, ptr, stream_ptr
    from olmax_amd.layer import TransformerBlock
    print(f"[case] larger buffer {recipe} S{seq}", flush=True)
    cfg = dataclasses.replace(getattr(TransformerRecipe, recipe)(), num_layers=1)
    block = TransformerBlock(cfg, batch_size=1, sequence_length=seq)
    g = torch.Generator(device="cuda").manual_seed(1)
    for w in (block.wqkv, block.wo, block.wgu, block.wdown):
        w.normal_(0.0, 0.02, generator=g)
    x = rnd(seq, cfg.d_model, seed=2)
    want, w, need = block.forward(x), block._weights(), block.acts.numel()
    acts = torch.full((need + (256 << 20),), 77, device="cuda", dtype=torch.uint8)
    y = torch.empty_like(x)
    got = recorded(lambda: check(block._L.olmax_block_fwd(stream_ptr(), ctypes.byref(block.c), ctypes.byref(w), i32(block.window), ptr(block.cos),
                                                          ptr(block.sin), ptr(x), ptr(y), ptr(acts), i64(acts.numel()))))
    assert any(key >> 18 & 1 for key, *_ in got) == split, got
    assert (acts[need:] == 77).all()
    assert torch.equal(y, want)
