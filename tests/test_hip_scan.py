"""Parity of the fused scan kernels (up to 16 states, x, delta, B and C in
fp32, bf16 or fp16) against the float64 oracle at the edges of their chunks,
channel groups and dispatch: lengths around 8 and the steps of one
iteration, channel counts around a group, state counts around the padding,
batches that select each states-per-lane variant, and the first shapes that
stay with the chunk-parallel kernels."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import ssm as S

pytestmark = pytest.mark.gpu

DTYPES = {'f32': torch.float32, 'bf16': torch.bfloat16, 'f16': torch.float16}
# Relative 2-norm of the gradients written in the scan's dtype: its rounding.
TOL = {'f32': 2e-6, 'bf16': 4e-3, 'f16': 5e-4}


def _check(name, nb, length, d, n, with_d=True, seed=0):
    dtype, dev = DTYPES[name], torch.device('cuda:0')
    g = torch.Generator().manual_seed(seed)

    def rnd(*shape):
        return torch.randn(*shape, generator=g)

    x, B, C = rnd(nb, length, d), rnd(nb, length, n), rnd(nb, length, n)
    delta = 0.01 + 0.3 * torch.sigmoid(rnd(nb, length, d))
    io = [t.to(dtype) for t in (x, delta, B, C)]
    A = -(0.2 + rnd(d, n).abs())
    D = rnd(d) if with_d else None
    dy = rnd(nb, length, d)
    from nitrix_amd import selective_scan

    leaves = [t.to(dev).requires_grad_(True) for t in (io[0], io[1], A, io[2], io[3])]
    if with_d:
        leaves.append(D.to(dev).requires_grad_(True))
    print(f'[case] scan {name} b{nb} L{length} d{d} n{n} D={with_d}', flush=True)
    y = selective_scan(*leaves, backend='hip')
    with torch.no_grad():
        y0 = selective_scan(*[t.detach() for t in leaves], backend='hip')
    grads = torch.autograd.grad(y, leaves, dy.to(dev))
    a64 = [t.double().numpy() for t in (io[0], io[1], A, io[2], io[3])]
    a64.append(D.double().numpy() if with_d else None)
    want = [S.selective_scan(*a64)] + [w for w in S.selective_scan_vjp(*a64, dy.double().numpy())
                                       if w is not None]
    assert y.dtype == y0.dtype == torch.float32
    for i, (got, ref) in enumerate(zip([y, *grads], want)):
        got = got.detach().double().cpu().numpy()
        tol = TOL['f32'] if i == 0 or i == 3 or i == 6 else TOL[name]
        # (dA is exactly zero for a single step: both sides then are)
        assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref), i
    err = np.linalg.norm(y0.double().cpu().numpy() - want[0]) / np.linalg.norm(want[0])
    assert err <= TOL['f32'], err


@pytest.mark.parametrize('name', ['f32', 'bf16', 'f16'])
@pytest.mark.parametrize('nb, length, d, n', [
    (1, 1, 1, 1), (2, 7, 5, 3), (1, 8, 16, 8), (3, 9, 17, 9), (1, 129, 33, 16), (2, 257, 31, 5),
    (1, 1025, 8, 16), (700, 20, 9, 16), (300, 33, 40, 8),
])
def test_chunks_groups_and_states(name, nb, length, d, n):
    _check(name, nb, length, d, n, with_d=n % 2 == 0, seed=length)


@pytest.mark.parametrize('name', ['f32', 'bf16', 'f16'])
@pytest.mark.parametrize('nb, length, d, n, eight', [
    (30, 20, 145, 8, True), (30, 300, 137, 5, True), (40, 33, 60, 16, True), (40, 129, 58, 9, True),
    (25, 20, 145, 8, False), (32, 20, 60, 16, False),
])
def test_both_sides_of_the_eight_wave_rule(name, nb, length, d, n, eight):
    """Blocks of 8 waves (one state a lane forward, two backward) where more
    than 512 forward and 256 backward blocks fill the chip without 16; below,
    blocks of 16."""
    np_ = 8 if n <= 8 else 16

    def groups(states):  # blocks with so many states a lane
        return nb * -(-d // (64 * states // np_))

    assert groups(4) < 512
    assert (groups(1) > 512) == (groups(2) > 256) == eight
    _check(name, nb, length, d, n, seed=length + d)


@pytest.mark.parametrize('name', ['f32', 'bf16', 'f16'])
@pytest.mark.parametrize('nb, length, d, n', [
    (1, 1, 1, 1), (2, 7, 5, 3), (1, 33, 17, 2), (3, 100, 300, 4), (1, 129, 33, 5), (2, 33, 257, 16),
    (2, 96, 128, 8), (1, 257, 64, 12), (700, 20, 9, 16), (1, 700, 40, 8),
])
@pytest.mark.parametrize('fused', [False, True], ids=['chunked', 'fused'])
def test_either_engine(monkeypatch, name, nb, length, d, n, fused):
    """Both engines at up to 16 states, whichever the host rule would take."""
    from nitrix_amd import ssm

    monkeypatch.setattr(ssm, '_takes_fused', lambda *a: fused)
    _check(name, nb, length, d, n, with_d=n % 2 == 0, seed=length)


@pytest.mark.parametrize('n', [8, 16])
@pytest.mark.parametrize('length, fused', [(2400, True), (2500, False)])
def test_the_engine_of_a_long_training_step(length, fused, n):
    from nitrix_amd import ssm

    assert ssm._takes_fused(1, length, 12, n, True) == fused
    _check('f32', 1, length, 12, n, seed=n)


@pytest.mark.parametrize('name, length', [('f32', 2400), ('bf16', 2403), ('f32', 2600)])
def test_both_sides_of_the_long_sequence_rule(name, length):
    _check(name, 1, length, 12, 4, seed=length)


def test_seventeen_states_and_mixed_dtypes():
    _check('bf16', 2, 100, 20, 17)
    dev = torch.device('cuda:0')
    g = torch.Generator().manual_seed(1)
    x, B, C = (torch.randn(2, 50, k, generator=g) for k in (24, 8, 8))
    delta = 0.1 * torch.rand(2, 50, 24, generator=g)
    A = -torch.rand(24, 8, generator=g)
    from nitrix_amd import selective_scan

    xb = x.to(torch.bfloat16)
    y = selective_scan(*[t.to(dev) for t in (xb, delta, A, B, C)], backend='hip')
    ref = S.selective_scan(*[t.double().numpy() for t in (xb, delta, A, B, C)], None)
    assert np.linalg.norm(y.double().cpu().numpy() - ref) / np.linalg.norm(ref) <= 2e-6


@pytest.mark.parametrize('length', [13, 16, 130])
def test_an_infinite_decay_rate(length):
    """States that forget at once (A = -inf, an overflowed exponential): the
    other states' gradients do not see the padded steps of a ragged end."""
    from nitrix_amd import selective_scan

    dev, nb, d, n = torch.device('cuda:0'), 2, 20, 8
    g = torch.Generator().manual_seed(length)
    x, dy = torch.randn(nb, length, d, generator=g), torch.randn(nb, length, d, generator=g)
    B, C = torch.randn(nb, length, n, generator=g), torch.randn(nb, length, n, generator=g)
    delta = 0.01 + torch.rand(nb, length, d, generator=g)
    A = -(0.2 + torch.rand(d, n, generator=g))
    A[:, ::3] = -float('inf')
    ins = [t.to(dev) for t in (x, delta, A, B, C)]
    for i in (0, 3, 4):
        ins[i].requires_grad_(True)
    y = selective_scan(*ins, backend='hip')
    got = [y, *torch.autograd.grad(y, [ins[i] for i in (0, 3, 4)], dy.to(dev))]
    a64 = [t.double().numpy() for t in (x, delta, A.clamp(min=-1e30), B, C)]
    vjp = S.selective_scan_vjp(*a64, None, dy.double().numpy())
    for a, w in zip(got, [S.selective_scan(*a64, None), vjp[0], vjp[3], vjp[4]]):
        a = a.detach().double().cpu().numpy()
        assert np.linalg.norm(a - w) <= TOL['f32'] * np.linalg.norm(w)
