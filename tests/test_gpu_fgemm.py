"""F16 weights x fp32 activations on fp16 MFMA (lg_fgemm.hip), through
lg_matmul_tokens, at the edges of every tile it picks, against float64."""
import numpy as np
import pytest
import torch

from ligguf_amd import ops
from ligguf_amd.lib import F16

pytestmark = pytest.mark.gpu


def product(w, x):
    rows, cols = w.shape
    return ops.matmul_tokens(F16, w.contiguous().view(torch.uint8).reshape(-1), 2 * cols, cols, rows, x)


def bound(w, x, K):
    """Per output: the split keeps each activation to 2^-21 of itself (hi
    toward zero, lo to nearest) and to 2^-38 of the token's largest; the K / 16
    accumulation steps round to 2^-24 each, adding like a random walk (6
    sigma); all times the sum of |terms|."""
    wa = w.double().abs()
    terms = x.double().abs() @ wa.T
    peak = x.double().abs().amax(1, keepdim=True) * wa.sum(1)
    return (2.0 ** -21 + 6 * (K / 16 + 4) ** 0.5 * 2.0 ** -24) * terms + 2.0 ** -38 * peak


# 32 x 32 tile and its ends, a part of K of one to five steps, fewer steps than parts, the last part short, few rows
# and many; 64 x 64 with K split and unsplit; 128 x 64 split and unsplit; 128 x 128; either side of where
# the tokens are taken in halves, uneven ones
@pytest.mark.parametrize("R,K,T", [(100001, 96, 31), (40003, 224, 32), (26001, 352, 31), (18001, 512, 32), (15001, 608, 32),
                                   (40, 224, 20), (70, 352, 9), (33, 512, 31), (50, 608, 17),
                                   (1, 32, 1), (33, 96, 31), (32, 2016, 32), (24576, 32, 13), (100, 64, 33), (65, 12288, 64),
                                   (4095, 1056, 129), (8200, 96, 130), (6145, 416, 257), (4100, 4096, 449), (12289, 160, 193),
                                   (8193, 1024, 512), (1024, 1024, 511), (1024, 1024, 512), (520, 4096, 127), (520, 4096, 150)])
def test_f16_product_tiles(gpu, R, K, T):
    g = torch.Generator(device="cuda").manual_seed(R + K + T)
    w = (torch.randn(R, K, generator=g, device=gpu) * 0.02).half()
    # token magnitudes from 1e-9 to 1e9: each has its own scale
    x = torch.randn(T, K, generator=g, device=gpu) * torch.exp(torch.randn(T, 1, generator=g, device=gpu) * 7)
    err = (product(w, x).double() - x.double() @ w.double().T).abs()
    assert bool((err <= bound(w, x, K)).all()), float((err / bound(w, x, K)).max())


@pytest.mark.parametrize("T", [16, 70])
def test_f16_product_keeps_infinities_and_nan(gpu, T):
    """An infinite or NaN weight or activation gives the class that the fp32
    products give: also under an activation that is exactly fp16 (its low
    part is zero) or far below its token's largest (its high part is)."""
    g = torch.Generator(device="cuda").manual_seed(T)
    w, x = torch.randn(64, 128, generator=g, device=gpu).half(), torch.randn(T, 128, generator=g, device=gpu)
    w[3, 5], w[4, 7], w[5, 1], w[6, 9], w[6, 10] = np.inf, -np.inf, np.nan, np.inf, -np.inf
    w[7, :] = 0
    x[1, 5], x[2, 5], x[3, 5], x[8, 5] = 1.0, 0.0, -2.0, 1e-30
    x[4, 20], x[5, 20], x[9, 20], x[9, 21] = np.inf, np.nan, -np.inf, 3e5
    x[6], x[7], x[10] = 0, x[7] * 1e-38, x[10] * 1e30
    got, ref = product(w, x), (x.double() @ w.double().T).float()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], ref[inf])
    fin = torch.isfinite(ref)
    fw, fx = (torch.where(torch.isfinite(a), a, torch.zeros_like(a)) for a in (w, x))
    assert bool(((got.double() - ref.double()).abs() <= bound(fw, fx, 128) + 2.0 ** -149)[fin].all())
