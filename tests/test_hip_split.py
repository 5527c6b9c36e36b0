"""Parity of the key-split forward (at most 64 queries over more than 512
keys, 16-bit I/O, no bias) against the float64 oracle: one and two query
strips, key lengths around a tile, at the first and beyond the last split
count, head dims at and between the three widths, masks with whole tiles and
whole splits removed, and the backward that follows (which must not expect
the forward's tile map)."""

from __future__ import annotations

import numpy as np
import pytest
import torch
from test_hip_parity import _check, _dev, _draw, _to

pytestmark = pytest.mark.gpu

BF, HF = torch.bfloat16, torch.float16


@pytest.mark.parametrize('dtype', [BF, HF], ids=['bf16', 'f16'])
@pytest.mark.parametrize('B, H, s, t, d, dv', [
    (1, 1, 1, 513, 64, 64), (2, 3, 28, 544, 32, 32), (1, 2, 32, 1000, 128, 128),
    (2, 2, 33, 2049, 40, 64), (1, 2, 64, 5000, 64, 24), (1, 1, 7, 40001, 128, 72),
    (40, 16, 5, 600, 8, 8),
])
def test_few_queries(dtype, B, H, s, t, d, dv):
    _check(dtype, B, H, s, t, d, dv=dv, seed=t, grads=t < 6000)
    _check(dtype, B, H, s, t, d, dv=dv, mask_kind='keypad', scale=-0.2, seed=t + 1, grads=t < 6000)
    if t < 6000:
        _check(dtype, B, H, s, t, d, dv=dv, mask_kind='rowbcast', seed=t + 2)


def test_masks_that_empty_splits_and_batches():
    """Keys kept in one short run, in none (rows NaN, as the reference) and at
    the very end."""
    rng = np.random.default_rng(3)
    B, H, s, t, d = 4, 2, 20, 9000, 64
    q, k, v = (_draw(rng, (B, H, n, d), BF) for n in (s, t, t))
    mask = np.zeros((B, 1, 1, t), bool)
    mask[0, ..., 4000:4010] = True
    mask[2, ..., -1] = True
    mask[3] = True
    from nitrix_amd import scaled_dot_product_attention
    from oracle import attention as O

    out = scaled_dot_product_attention(_to(q, BF), _to(k, BF), _to(v, BF),
                                       mask=torch.from_numpy(mask).to(_dev()), backend='hip')
    got = out.float().cpu().numpy()
    assert np.isnan(got[1]).all()
    keep = [0, 2, 3]
    ref = O.sdpa_forward(q[keep], k[keep], v[keep], mask=mask[keep], scale=d ** -0.5,
                         acc_dtype=np.float64)
    assert np.isfinite(got[keep]).all()
    assert np.abs(got[keep] - ref).max() / np.abs(ref).max() <= 2e-2


@pytest.mark.parametrize('dtype', [BF, HF], ids=['bf16', 'f16'])
@pytest.mark.parametrize('t', [545, 9000])
def test_scores_of_minus_infinity(dtype, t):
    """A wave whose only kept key scores -inf for half of the rows (an
    overflowing bf16 product, an infinite fp16 key) and more for the others:
    the key weighs nothing in those rows."""
    rng = np.random.default_rng(7)
    B, H, s, d = 2, 2, 20, 64
    q, k, v = (_draw(rng, (B, H, n, d), dtype) for n in (s, t, t))
    lone = t - 1 if t == 545 else 40
    mask = np.zeros((1, 1, 1, t), bool)
    mask[..., :20] = mask[..., lone] = True
    k[..., lone, :] = 0
    k[..., lone, 5] = 3e38 if dtype == BF else np.inf
    q[..., ::2, 5] = -2
    q[..., 1::2, 5] = 0 if dtype == BF else 1
    k[..., :20, 5] = 0
    rows = slice(None) if dtype == BF else slice(0, None, 2)
    from nitrix_amd import scaled_dot_product_attention
    from oracle import attention as O

    out = scaled_dot_product_attention(_to(q, dtype), _to(k, dtype), _to(v, dtype),
                                       mask=torch.from_numpy(mask).to(_dev()), backend='hip')
    got = out.float().cpu().numpy()[:, :, rows]
    ref = O.sdpa_forward(q[:, :, rows], k, v, mask=mask, scale=d ** -0.5, acc_dtype=np.float64)
    assert np.isfinite(got).all()
    assert np.abs(got - ref).max() / np.abs(ref).max() <= (2e-2 if dtype == BF else 2e-3)


def test_a_call_repeats_itself():
    from nitrix_amd import scaled_dot_product_attention

    g = torch.Generator(device=_dev()).manual_seed(2)
    q, k, v = (torch.randn(4, 8, n, 64, generator=g, device=_dev()).to(HF) for n in (28, 8192, 8192))
    mask = (torch.arange(8192, device=_dev()) < 7001)[None, None, None]
    outs = [scaled_dot_product_attention(q, k, v, mask=mask, backend='hip') for _ in range(3)]
    assert all(torch.equal(outs[0], o) for o in outs[1:])
