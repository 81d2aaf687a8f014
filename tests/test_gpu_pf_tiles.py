"""The quantized token GEMMs (lg_matmul_tokens) at the edges of every tile the
batched prefill picks -- 128 x 64, 64 x 32 and 32 x 32 with K in one, two or
four parts, fewer blocks of K than parts, ends of rows and tokens -- against
float64 over the same quantized operands."""
import ctypes as C

import numpy as np
import pytest
import torch

from ligguf_amd import encode, ops
from ligguf_amd.lib import Q1_0, Q1_G, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q8_0, TYPE_NAMES, load, row_size

pytestmark = pytest.mark.gpu

# rows, width, tokens, the tile taken (rows x tokens, parts of K) and Q1_G's where it is another one: ends of rows and
# tokens, one step of K in two parts, as many steps as parts and fewer, an uneven last part
SHAPES = [(33, 256, 1, (64, 32, 2), None), (600, 2304, 95, (32, 32, 4), None), (4090, 1280, 33, (32, 32, 4), None),
          (65, 768, 40, (32, 32, 4), None), (4097, 512, 65, (64, 32, 2), None), (4065, 1280, 100, (64, 32, 2), None),
          (4033, 1792, 97, (64, 32, 2), (64, 32, 4)), (4097, 4864, 65, (64, 32, 4), None), (3970, 2304, 449, (128, 64, 2), None),
          (6145, 768, 100, (128, 64, 1), (64, 32, 2)), (3970, 1280, 449, (128, 64, 1), (128, 64, 2)),
          (12289, 512, 165, (128, 64, 1), None)]
TYPES = [Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q8_0, Q1_0, Q1_G]


def activations(x, kq):
    """float64 values of the rows of x as quantize_q8_K / quantize_q8_0 leave them"""
    T, n = x.shape
    raw = (ops.quantize_q8_K if kq else ops.quantize_q8_0)(x.reshape(-1)).cpu().numpy().reshape(T, -1)
    size, d_bytes, count = (292, 4, 256) if kq else (34, 2, 32)
    b = raw.reshape(T, n // count, size)
    d = np.ascontiguousarray(b[:, :, :d_bytes]).view(np.float32 if kq else np.float16).astype(np.float64)
    q = np.ascontiguousarray(b[:, :, d_bytes:d_bytes + count]).view(np.int8).astype(np.float64)
    return torch.from_numpy((d * q).reshape(T, n)).to(x.device)


@pytest.mark.parametrize("wt", TYPES, ids=[TYPE_NAMES[t] for t in TYPES])
@pytest.mark.parametrize("R,n,T,tile,q1g", SHAPES)
def test_tiles(gpu, wt, R, n, T, tile, q1g):
    got = [C.c_int() for _ in range(3)]
    assert load().lg_prefill_tile(wt, R, n, T, *(C.byref(o) for o in got)) == 0
    assert tuple(o.value for o in got) == (q1g if q1g and wt == Q1_G else tile)
    rsz = row_size(wt, n)
    distinct = min(R, 512)   # encoding is host work: the rows repeat, with a stride that no tile edge divides
    rows = encode.random_tensor(wt, R + n, wt, distinct, n).reshape(distinct, rsz)
    rows = np.ascontiguousarray(rows[np.arange(R) * 37 % distinct])
    w = torch.from_numpy(rows.reshape(-1)).to(gpu)
    x = torch.from_numpy(np.random.default_rng(T).standard_normal((T, n)).astype(np.float32)).to(gpu)
    wd = ops.dequantize_row(wt, w, R * n).reshape(R, n).double()
    a = activations(x, wt not in (Q8_0, Q1_0, Q1_G))
    got = ops.matmul_tokens(wt, w, rsz, n, R, x).double()
    # the matvec bar: integer block sums are exact, their fp32 combination within 2e-6 of the sum of |terms|
    assert bool(((got - a @ wd.T).abs() <= 2e-6 * (a.abs() @ wd.abs().T)).all())
