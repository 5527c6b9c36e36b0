"""Parity of the fp32 backward whose waves split the streamed tiles (head dims
up to 64, at most 128 blocks of 128 rows, more than 64 streamed rows) against
the float64 oracle: lengths around its 32-row tiles and around the two limits,
with causality, masks that leave waves without a tile, and biases whose
gradient is full, a column sum, or summed over pairs."""

from __future__ import annotations

import pytest
import torch
from test_hip_parity import _check

pytestmark = pytest.mark.gpu

F32 = torch.float32


@pytest.mark.parametrize('B, H, s, t, d, dv', [
    (1, 1, 1, 65, 64, 64), (1, 2, 65, 17, 64, 64), (2, 3, 31, 97, 40, 64), (2, 2, 129, 128, 64, 24),
    (1, 2, 344, 344, 64, 64), (1, 1, 160, 1000, 8, 8), (128, 1, 64, 65, 64, 64),
    (129, 1, 65, 66, 64, 64),
])
def test_lengths(B, H, s, t, d, dv):
    _check(F32, B, H, s, t, d, dv=dv, seed=s + t)
    _check(F32, B, H, s, t, d, dv=dv, mask_kind='keypad', scale=0.3, seed=s)
    if s > 1:  # one query keeps one key: its dq is exactly 0, and no relative error is defined
        _check(F32, B, H, s, t, d, dv=dv, causal=True, seed=t)


@pytest.mark.parametrize('shape', [(1, 2, 200, 333), (1, 2, 1, 333), (2, 1, 200, 333), (2, 2, 200, 333)],
                         ids=['heads', 'row', 'batch', 'full'])
@pytest.mark.parametrize('mask', [None, 'block'])
def test_bias_gradients(shape, mask):
    _check(F32, 2, 2, 200, 333, 64, bias_shape=shape, bias_dtype=F32, mask_kind=mask, seed=7)
