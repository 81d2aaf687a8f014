"""The encoder's F16 path where it can go wrong: attention at the edges of its
16-query blocks and 32-key steps, every head width, a wave or a workgroup to
a query block, alone and in a batch bit for bit (other tiles of the products), and activations split by their producer (bounds of the weights)
or from each token's own maximum (F32 producers, bounds that are none)."""
import gc
import zlib

import numpy as np
import pytest

from ligguf_amd import encode
from ligguf_amd.bert import BERT_TINY, Bert, BertConfig, HostBert
from ligguf_amd.lib import F16, F32, Q8_0

pytestmark = pytest.mark.gpu

LENGTHS = [1, 13, 14, 15, 30, 31, 62, 63, 125, 126, 127, 158, 159, 257]      # with CLS and SEP: at the blocks' and steps' ends
REL = 2e-5   # fp32 sums in another order, activations to 2^-21: the bar of the encoder tests


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(np.asarray(b, np.float64)))


def texts(cfg, lengths):
    return [np.random.default_rng(n).integers(5, cfg.vocab, n).astype(np.int32) for n in lengths]


@pytest.mark.parametrize("hd", [16, 32, 48, 64, 80, 96, 112, 128])
def test_attention_edges(gpu, oracle, hd):
    hb = HostBert.synthetic(BERT_TINY.with_(n_heads=2, n_embed=2 * hd, n_ff=416, n_layers=2, n_context=288,
                                            layer_type=F16, embd_type=F16))
    dev = Bert(0)
    dev.load(hb, 4096)
    seqs = texts(hb.cfg, LENGTHS)
    one = np.stack([dev.embed(s) for s in seqs])
    many = dev.embed_batch(seqs * 3)
    dev.close()
    for i, s in enumerate(seqs):
        ref = oracle.bert_embed(hb, s)
        assert rel(one[i], ref) < REL, (hd, len(s), rel(one[i], ref))
    assert np.array_equal(many.view(np.uint32), np.tile(one, (3, 1)).view(np.uint32))


def scale(hb, norm, m, channel=slice(None)):
    for part in ("weight", "bias"):
        v = hb.vectors[f"{norm}.{part}"].copy()
        v[channel] *= np.float32(m)
        hb.vectors[f"{norm}.{part}"] = v


def test_wide_encoder_alone_and_in_a_batch(gpu, oracle):
    """4096 tokens of 768 and 3072 values: Q|K|V and up on 128 x 128 tiles, where
    a text alone takes 32 x 32 and 64 x 64."""
    cfg = BERT_TINY.with_(name="bert-wide", n_layers=1, n_embed=768, n_heads=12, n_ff=3072, n_context=256, layer_type=F16,
                          embd_type=F16)
    hb = HostBert.synthetic(cfg)
    dev = Bert(0)
    dev.load(hb, 4224)
    seqs = texts(hb.cfg, [126, 3, 200, 61] + [126] * 28 + [120])      # 4104 tokens: an uneven end
    many = dev.embed_batch(seqs)
    for i in (0, 1, 2, 3, 32):
        one = dev.embed(seqs[i])
        assert np.array_equal(one.view(np.uint32), many[i].view(np.uint32)), i
        if i < 3:
            ref = oracle.bert_embed(hb, seqs[i])
            assert rel(one, ref) < REL, (i, rel(one, ref))
    dev.close()


@pytest.mark.parametrize("f32", [("attn_q", "attn_k", "attn_v", "ffn_up"), ("attn_v",), ("attn_output", "ffn_down"), ("ffn_up",)])
def test_split_follows_the_producer(gpu, oracle, f32):
    cfg = BERT_TINY.with_(layer_type=F16, embd_type=F16)
    hb = HostBert.synthetic(cfg)
    for name, (t, rows, cols, _) in list(hb.weights.items()):
        if name.split(".")[-2] in f32:
            hb.weights[name] = (F32, rows, cols, encode.random_tensor(F32, 3, zlib.crc32(name.encode()), rows, cols, cfg.sigma))
    # LayerNorm outputs, and so the bounds, of very different sizes
    assert cfg.n_layers == 2
    for n, m in (("token_embd_norm", 1e-3), ("blk.0.attn_output_norm", 1e-6), ("blk.0.layer_output_norm", 1e3),
                 ("blk.1.attn_output_norm", 1e4)):
        scale(hb, n, m)
    dev = Bert(0)
    dev.load(hb)
    for s in texts(hb.cfg, [2, 40]):
        assert rel(dev.embed(s), oracle.bert_embed(hb, s)) < REL
    dev.close()


def large_norm_weight(norm):
    """one channel of a LayerNorm far above the rest: x's or x1's split takes each token's own maximum"""
    return lambda hb: scale(hb, norm, 2.0 ** 11, 5)


def silent_neuron(hb):
    """up's bias keeps one neuron at gelu = 0 and puts its bound at 1e9: the other neurons' values stay exact"""
    for l in range(hb.cfg.n_layers):
        hb.vectors[f"blk.{l}.ffn_up.bias"][7] = -1e9


def no_bound(hb):
    """the bound of h is no use at all (1e30 and more)"""
    for l in range(hb.cfg.n_layers):
        hb.vectors[f"blk.{l}.ffn_up.bias"][7] = -1e30


def squares_underflow(hb):
    """x1 near 1e-22: the squares in the bound of h would be zero, and h far above such a bound"""
    scale(hb, "blk.0.attn_output_norm", 1e-22)
    hb.vectors["blk.0.attn_output_norm.bias"][:] = 0
    hb.vectors["blk.0.ffn_up.bias"][:] = 0


@pytest.mark.parametrize("change", [large_norm_weight("token_embd_norm"), large_norm_weight("blk.0.attn_output_norm"),
                                    large_norm_weight("blk.0.layer_output_norm"), silent_neuron, no_bound, squares_underflow],
                         ids=["x-of-0", "x1", "x-of-1", "silent-neuron", "no-bound", "squares-underflow"])
def test_bounds_that_say_too_little(gpu, oracle, change):
    hb = HostBert.synthetic(BERT_TINY.with_(layer_type=F16, embd_type=F16))
    hb.vectors = {n: v.copy() for n, v in hb.vectors.items()}
    change(hb)
    dev = Bert(0)
    dev.load(hb)
    for s in texts(hb.cfg, [2, 40, 200]):
        assert rel(dev.embed(s), oracle.bert_embed(hb, s)) < REL
    dev.close()


def test_split_buffers_for_f16_only(gpu):
    """Encoders without an F16 layer matrix have no split activations to hold:
    4096 tokens of 384 and of 1536 values take 31 MB of them."""
    import torch
    cfg = BertConfig("bert-mem", 1, 384, 12, 1536, 512, 128)
    used, devs = {}, []
    for t in (F16, Q8_0, F16, Q8_0):      # (the first two also load the kernels)
        hb = HostBert.synthetic(cfg.with_(layer_type=t))
        dev = Bert(0)
        gc.collect()      # what earlier tests left goes back now, not in between
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        dev.load(hb, 4096)
        used[t] = free - torch.cuda.mem_get_info()[0]
        devs.append(dev)
    for dev in devs:
        dev.close()
    assert used[Q8_0] + 24 * 2 ** 20 <= used[F16], used
