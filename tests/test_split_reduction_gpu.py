"""GPU parity tests of reductions that several workgroups share: the LM head's and the blocks' gradient products
at shapes with few tiles and a long reduction (whole tiles, ragged rows, a partial k-tile, a residual)."""
import pytest
import torch

from oracle import ref
from test_gemm_choice_gpu import recorded

pytestmark = pytest.mark.gpu


def shared(call):
    """(M, N, K, fp32 result) of the products of `call` whose reductions several workgroups share."""
    return {(m, n, k, key >> 15 & 1) for key, m, n, k, _ in recorded(call) if key >> 18 & 1}


def worst(got, want, dim):
    """Largest relative error of a row (dim 1) or column (dim 0): a misplaced edge shows in one of them."""
    got, want = got.double(), want.double()
    return ((got - want).norm(dim=dim) / (want.norm(dim=dim) + 1e-3 * want.norm() / want.shape[1 - dim] ** 0.5)).max().item()


@pytest.mark.parametrize("T,d,V,tied", [
    (2048, 1024, 20480, False),  # dh: 32 whole tiles over 320 k-tiles
    (520, 264, 20007, False),    # dh: 3 x 2 ragged tiles, a partial k-tile at the end of the last part
    (2500, 1032, 16384, False),  # dh: ragged rows and columns, whole k-tiles
    (8200, 1024, 2061, False),   # dW: a padded M that is no multiple of 8, partial k-tile
    (8200, 1024, 2061, True),    # the same in fp32
    (8192, 1000, 2064, True),    # ragged columns in fp32, whole k-tiles
    (8192, 1024, 4096, True),    # whole tiles in fp32
])
def test_lm_head_gradients(T, d, V, tied):
    """Against float64 on the rounded operands.  dlogits and the outputs are rounded to bf16 (2^-9 each, and a
    handful of dlogits round the other way): a row's error stays under 4 of those, 8e-3."""
    from olmax_amd import TransformerConfig
    print(f"[case] split lm head T{T} d{d} V{V} tied{tied}", flush=True)
    cfg = TransformerConfig(vocab_size=V, d_model=d, hidden_size=8192, num_layers=0, n_heads=2, head_dim=128, tie_embeddings=tied)
    model = cfg.build(batch_size=1, sequence_length=T, seed=1)
    gen = torch.Generator(device="cuda").manual_seed(2)
    ids = torch.randperm(V, device="cuda", generator=gen).repeat(5)[:T].to(torch.int32)
    labels = torch.randint(0, V, (T,), device="cuda", generator=gen, dtype=torch.int32)
    runs = shared(lambda: model.loss_and_grads(ids, labels))
    assert ((V, d, T, int(tied)) if V < T else (T, d, V, 0)) in runs, runs
    G = model.named_gradients()
    E, W = (model.named_parameters()[k].to(torch.bfloat16).double() for k in ("embedding.weight", "embedding.weight" if tied else "lm_head.proj.weight"))
    x = E[ids.long()]
    r = (x.square().mean(-1, keepdim=True) + cfg.norm_eps).rsqrt()
    hn = ref.bf16_round((x * r).float()).double()
    with torch.device("cuda"):
        _, dh, dW = ref.lm_head_ce(hn, W, labels.long(), softcap=0.0, rt=ref.bf16_round)
    dh = ref.bf16_round(dh.float()).double()
    dx = r * dh - x * r ** 3 * (x * dh).mean(-1, keepdim=True)
    want = torch.zeros_like(E).index_add_(0, ids.long(), dx)
    if tied:
        want += dW
    for dim in (0, 1):
        assert tied or worst(G["lm_head.proj.weight"], dW, dim) < 8e-3
        assert worst(G["embedding.weight"], want, dim) < 8e-3


def test_block_gradients_with_a_residual():
    """A post-norm block adds the residual's gradient in the product's epilogue: shared reductions against whole
    ones (a forced tile size has no shared form); they differ by fp32 orders, hence bf16 roundings, only."""
    from olmax_amd import TransformerConfig, _lib
    from olmax_amd.layer import TransformerBlock
    cfg = TransformerConfig(vocab_size=64, d_model=1024, hidden_size=8192, num_layers=1, n_heads=16, head_dim=128, layer_type="reordered_norm",
                            qk_norm_headwise=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    block = TransformerBlock(cfg, batch_size=2, sequence_length=1300)
    for w in (block.wqkv, block.wo, block.wgu, block.wdown):
        w.normal_(0.0, 0.02, generator=gen)
    x, dy = (torch.randn(2600, 1024, device="cuda", generator=gen).to(torch.bfloat16) for _ in range(2))

    def grads():
        block.forward(x)
        dx = block.backward(dy)
        return {"dx": dx.clone(), **{k: v.clone() for k, v in block.grads.items()}}

    print("[case] split block", flush=True)
    got = {}
    runs = shared(lambda: got.update(grads()))
    assert (2600, 1024, 16384, 0) in runs, runs  # dx of the gated projection, the residual's gradient added
    L = _lib.load()
    try:
        L.olmax_gemm_set_tile(256)
        want = {}
        assert not shared(lambda: want.update(grads()))
    finally:
        L.olmax_gemm_set_tile(0)
    for k in want:
        if want[k].dim() == 2:
            assert max(worst(got[k], want[k], d) for d in (0, 1)) < 1.5e-2, k
