"""The prefill attention (lg_pfattn.hip) at the edges of its 32-token blocks and
64- or 32-key tiles, with keys in one and in several chunks, for every number
of query heads per KV head and head width: a prompt in one pass against the
token-sequential path, over an unquantized model of two layers."""
import gc

import numpy as np
import pytest

from ligguf_amd.lib import F32, PREFILL_BATCHED, PREFILL_STEPS
from ligguf_amd.model import Engine, HostModel, ModelConfig

pytestmark = pytest.mark.gpu

# heads, KV heads, head width (1 to 8 query heads per KV head)
SHAPES = [(6, 6, 48), (3, 3, 128), (4, 2, 64), (12, 4, 64), (8, 2, 128), (10, 2, 64), (12, 2, 128), (14, 2, 48), (8, 1, 128)]
# tokens, positions before: one block and its ends, an own key in the next tile, keys in chunks of a few tiles; with
# (300, 250) chunks of 384 keys of which blocks of queries see the first alone, both, and some of their tokens the second
PROMPTS = [(1, 0), (31, 0), (33, 5), (64, 64), (65, 100), (160, 450), (5, 1300), (40, 1011), (300, 250)]
# the same in more than 20 chunks
LONG = [(1, 5999), (3, 6000), (40, 6037)]


@pytest.mark.parametrize("nh,nkv,hd", SHAPES, ids=[f"{a}on{b}x{c}" for a, b, c in SHAPES])
def test_prompt_against_steps(gpu, nh, nkv, hd):
    against_steps(nh, nkv, hd, 1408, PROMPTS)


@pytest.mark.parametrize("nh,nkv,hd", [(6, 6, 48), (8, 1, 128)], ids=["6on6x48", "8on1x128"])
def test_many_chunks_against_steps(gpu, nh, nkv, hd):
    against_steps(nh, nkv, hd, 6144, LONG)


def test_first_prompt_allocates_no_partials(gpu):
    """The partials of split keys go where up|gate's output comes later: the
    first prompt of an engine takes the buffers of the layer pass and nothing
    the size of the partials (17 MB here) beside them."""
    import torch
    ne, kvd, nff = 1024, 128, 4352
    used = []
    for _ in range(2):      # the first engine also loads the kernels
        eng = Engine(0)
        eng.load(HostModel.synthetic(ModelConfig("pfmem", 0, 1, ne, 16, 2, 64, nff, 64, 1024, 1e4, 1e-5, F32, F32, F32)))
        gc.collect()      # what earlier tests left goes back now, not in between
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        eng.set_prefill_path(PREFILL_BATCHED)
        eng.prefill(np.arange(20, dtype=np.int32), 0)
        used.append(free - torch.cuda.mem_get_info()[0])
        eng.close()
    # x, qkv, attention output, up|gate and the widest activation of 512 tokens, 2 MiB steps
    assert used[1] <= 512 * 4 * (ne + (ne + 2 * kvd) + ne + 2 * nff + nff) + 5 * 2 ** 21, used


def against_steps(nh, nkv, hd, ctx, prompts):
    ne, kvd = nh * hd, nkv * hd
    eng = Engine(0)
    eng.load(HostModel.synthetic(ModelConfig("pfattn", 0, 2, ne, nh, nkv, hd, 256, 64, ctx, 1e4, 1e-5, F32, F32, F32)))
    rng = np.random.default_rng(nh + hd)
    past = rng.standard_normal((2, 2, ctx, kvd)).astype(np.float16).view(np.uint16)
    for T, pos in prompts:
        toks = rng.integers(0, 64, T).astype(np.int32)
        out = []
        for path in (PREFILL_BATCHED, PREFILL_STEPS):
            eng.kv_write(0, 2, 0, ctx, past[0].reshape(-1), past[1].reshape(-1))
            eng.set_prefill_path(path)
            logits = np.asarray(eng.prefill(toks, pos), np.float64)
            kv = [np.asarray(a).reshape(-1).view(np.float16).astype(np.float64).reshape(2, T, kvd)[1]
                  for a in eng.kv_read(0, 2, pos, T)]
            out.append((logits, *kv))
        (la, *ka), (lb, *kb) = out
        # fp32 sums in another order (1.2e-6 a matrix product, two before layer 1's cache) move a share e / 2^-11 of its
        # values across an fp16 rounding boundary, by a step of up to 2^-10: sqrt(e 2^11) 2^-10 = 6.8e-5 (e = 2.4e-6) of
        # the rows that the last token's attention sums, in the mean; twice that for one prompt
        assert np.linalg.norm(la - lb) <= 1.4e-4 * np.linalg.norm(lb), (T, pos)
        # layer 1's K and V rows see layer 0's attention of every token: an fp16 step, and the same difference of the
        # cache rows before (6.8e-5 of the rms; 6 of those over some thousand values, the largest value ~3 rms)
        for a, b in zip(ka, kb):
            assert np.all(np.abs(a - b) <= 2.0 ** -10 * np.abs(b) + 1.4e-4 * np.abs(b).max()), (T, pos)
