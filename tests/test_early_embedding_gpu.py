"""GPU test of the overlapped train step's update of a large embedding in two parts: rows that no token names, and the others."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers,d,vocab,tied,decay", [(2, 1032, 65040, True, False), (3, 1032, 65040, False, True), (1, 1024, 65544, False, False),
                                                       (1, 2048, 32776, True, True),
                                                       (2, 1032, 65016, True, False), (2, 1024, 65528, False, True)])  # too small for two parts
def test_rows_of_the_batch_and_the_others(layers, d, vocab, tied, decay):
    """Against the sequential step from the same state, three steps.  Rows that no token names have deterministic gradients: bit-equal
    (a row updated twice, left out or taken at the wrong offset shows); the others are summed by atomics in fp32, 1e-5 as for every such leaf.
    Negative and too large ids wrap and clamp."""
    from olmax_amd import TransformerConfig, _lib
    print(f"[case] early embedding L{layers} d{d} V{vocab} tied{tied} decay{decay}", flush=True)
    cfg = TransformerConfig(vocab_size=vocab, d_model=d, hidden_size=512, num_layers=layers, n_heads=2, head_dim=128, tie_embeddings=tied,
                            layer_ac_policy="nothing_saveable")
    B, S = 2, 192
    seq, ovl = (cfg.build(batch_size=B, sequence_length=S, seed=3) for _ in range(2))
    for m in (seq, ovl):
        m.init_optimizer_state()
    kw = dict(lr=1e-3, b1=0.9, b2=0.95, weight_decay=0.1, no_decay_modules=[] if decay else ["embedding.weight"])
    gen = torch.Generator(device="cuda").manual_seed(5)
    for step in range(1, 4):
        ids = torch.randint(0, vocab, (B * S,), device="cuda", generator=gen, dtype=torch.int32)
        ids[:8] = torch.tensor([0, vocab - 1, -1, -vocab, vocab + 5, 7, 7, -7 * vocab], dtype=torch.int32)
        labels = torch.randint(0, vocab, (B * S,), device="cuda", generator=gen, dtype=torch.int32)
        for name in ("master", "m", "v", "params_bf16"):
            getattr(ovl, name).copy_(getattr(seq, name))
        l0 = seq.train_step(ids, labels, step=step, overlap_optimizer=False, **kw).item()
        l1 = ovl.train_step(ids, labels, step=step, overlap_optimizer=True, **kw).item()
        assert l0 == l1
        # layers, final norm and embedding; the head in a share per window (a layer's worth first, the rest with layer 0's update if there is one window
        # only); the embedding in a share per window
        got = _lib.load().olmax_model_last_step_overlapped_launches()
        assert got == layers + 2 + (0 if tied else max(layers, 2)) + (layers if vocab * d >= 1 << 26 else 0), got
        rows = torch.where(ids < 0, ids + vocab, ids).clamp(0, vocab - 1).long().unique()
        other = torch.ones(vocab, dtype=torch.bool, device="cuda")
        other[rows] = False
        for buf in ("master", "m", "v", "params_bf16"):
            a, b = (getattr(m, buf)[: vocab * d].view(vocab, d) for m in (seq, ovl))
            assert torch.equal(a[other], b[other]), (step, buf)
            # (a weight rounds to the neighbouring bf16 where its fp32 value moved by an ulp)
            tol = 2 ** -7 if buf == "params_bf16" else 1e-5
            assert ((a[rows].float() - b[rows].float()).abs() <= tol * a.float().abs().max()).all(), (step, buf)
            c, e = (getattr(m, buf)[vocab * d:].float() for m in (seq, ovl))
            # norm weights have gradients summed by atomics too, and an update lr m / (sqrt(v) + eps) passes a change of g on as lr / (sqrt(v) + eps) of it at
            # most in each of m (0.1 of g, corrected by 0.1 or more) and sqrt(v), where g is hardly more than eps itself as well
            dg = (seq.m[vocab * d:] - ovl.m[vocab * d:]).abs() / 0.1
            moved = 4 * kw["lr"] * dg / ((seq.v[vocab * d:] / (1 - kw["b2"] ** step)).sqrt() + 1e-8) if buf in ("master", "params_bf16") else 0
            assert ((c - e).abs() <= tol * c.abs().max() + moved).all(), (step, buf)
