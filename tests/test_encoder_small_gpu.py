"""Small batches of the BERT family (eos_enc_lin8 / eos_enc_lin16 launches):
bit-identical to the unfused launches at the edges of their tiles (32 and 64
rows, 256 and 128 columns) for every width, both GELUs, both poolings and
token types, and within the contract of the CPU oracle; and bit-identical to
the same sequence in batches that take the other paths (LayerNorm launches
with the wide GEMM, 64-row tiles, the fused tail); and batches above the
tail's line by the tail kernels."""
import numpy as np
import pytest

import oracle
from eos_amd import datagen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,heads,inter,lens,gelu,pooling", [
    (128, 4, 128, [1], 1, "masked_mean"),
    (256, 8, 640, [31, 8], 2, "masked_mean"),
    (384, 12, 1536, [32], 1, "cls"),
    (384, 12, 384, [33, 1, 30], 2, "masked_mean"),
    (512, 8, 2048, [64, 65], 1, "masked_mean"),
    (768, 12, 3072, [57, 9], 1, "cls"),
])
def test_small_batch_matches_oracle(rt, hidden, heads, inter, lens, gelu, pooling):
    from eos_amd.encoder import Encoder
    print(f"[case] small batch H={hidden} F={inter} lens={lens} gelu={gelu} {pooling}", flush=True)
    w = datagen.bert_q8_weights(3, hidden, heads, inter, 500, 80, seed=hidden + inter, gelu=gelu,
                                random_affine=True)
    T = max(lens)
    ids = datagen.uniform_int(5, len(lens) * T, 0, 500).astype(np.int32).reshape(len(lens), T)
    types = datagen.uniform_int(6, ids.size, 0, 2).astype(np.int32).reshape(ids.shape)
    mask = (np.arange(T)[None, :] < np.array(lens)[:, None]).astype(np.int32)
    enc = Encoder(rt, w)
    if pooling != "masked_mean":
        enc.set_pooling(pooling)
    got = enc.embed(ids, mask, types)
    # every value is rounded where the unfused GEMM and LayerNorm launches round it
    enc.set_fused_tail(False)
    np.testing.assert_array_equal(got, enc.embed(ids, mask, types))
    if gelu == 1:  # the oracle's GELU
        want = oracle.bert_embed(w.tok, w.pos, w.typ, w.emb_gamma, w.emb_beta,
                                 [L.dequantized() for L in w.layers], ids, mask, types, heads,
                                 w.ln_eps, pooling=pooling)
        # the package's contract for every embedding
        cos = (got * want).sum(1) / np.linalg.norm(got, axis=1) / np.linalg.norm(want, axis=1)
        assert cos.min() >= 0.9999 and np.abs(got - want).max() <= 2e-2
    enc.release()


@pytest.mark.parametrize("hidden,heads,batch", [(384, 12, 12), (384, 12, 32), (512, 8, 8),
                                                (512, 8, 32), (768, 12, 6), (768, 12, 24),
                                                (256, 8, 36)])
def test_small_and_large_batches_agree_bit_for_bit(rt, hidden, heads, batch):
    from eos_amd.encoder import Encoder
    print(f"[case] small against large batch H={hidden}", flush=True)
    w = datagen.bert_q8_weights(2, hidden, heads, 2 * hidden, 500, 250, seed=hidden,
                                random_affine=True)
    ids, mask, _ = datagen.encoder_batch(batch, 250, 500, 3, 250, 7, 8)
    enc = Encoder(rt, w)
    large = enc.embed(ids, mask)
    for b in (0, 3, batch - 1):
        n = int(mask[b].sum())
        np.testing.assert_array_equal(enc.embed(ids[b:b + 1, :n], mask[b:b + 1, :n])[0], large[b])
    enc.release()


@pytest.mark.parametrize("hidden,heads,inter,gelu,batch,least", [
    (384, 12, 1536, 1, 40, 1),
    (384, 6, 384, 2, 30, 1),      # the tail from fewer rows on at F <= 2 H
    (384, 12, 1536, 2, 64, 150),
    (512, 8, 1024, 1, 30, 1),
    (512, 8, 2048, 2, 110, 150),  # rows past one 64-row block per CU: the 32-row launch
])
def test_large_batches_take_the_fused_tail(rt, hidden, heads, inter, gelu, batch, least):
    """Batches of more than 7,680 packed rows (5,632 at F <= 2 H) run the fused
    layer tail at hidden 384 and 512 (a single sequence does not): bit-identical
    to the unfused launches, and within the contract of the CPU oracle."""
    from eos_amd.encoder import Encoder
    print(f"[case] fused tail H={hidden} F={inter} gelu={gelu} batch={batch}", flush=True)
    w = datagen.bert_q8_weights(2, hidden, heads, inter, 500, 250, seed=hidden + batch, gelu=gelu,
                                random_affine=True)
    ids, mask, _ = datagen.encoder_batch(batch, 200, 500, least, 200, 17, 18)
    enc = Encoder(rt, w)
    enc.embed(ids[:1], mask[:1])
    rt.profile(True)
    rt.profile_reset()
    got = enc.embed(ids, mask)
    assert rt.profile_read("enc_tail")[0] >= 2
    rt.profile_reset()
    enc.embed(ids[:1], mask[:1])
    assert rt.profile_read("enc_tail")[0] == 0
    rt.profile(False)
    enc.set_fused_tail(False)
    np.testing.assert_array_equal(got, enc.embed(ids, mask))
    if gelu == 1:  # the oracle's GELU
        for b in (0, batch // 2, batch - 1):
            n = int(mask[b].sum())
            want = oracle.bert_embed(w.tok, w.pos, w.typ, w.emb_gamma, w.emb_beta,
                                     [L.dequantized() for L in w.layers], ids[b:b + 1, :n],
                                     mask[b:b + 1, :n], None, heads, w.ln_eps)
            cos = (got[b] @ want[0]) / np.linalg.norm(got[b]) / np.linalg.norm(want[0])
            assert cos >= 0.9999 and np.abs(got[b] - want[0]).max() <= 2e-2
    enc.release()
