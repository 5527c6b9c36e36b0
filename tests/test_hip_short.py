"""Parity of the short-sequence kernels (at most 512 queries and keys, head
dims up to 64, 16-bit I/O) against the float64 oracle, at the edges of their
strips, tiles and limits: lengths around 32 and 64 rows and at 512, head dims
around the 32-wide variant, a bias shared by many pairs in every broadcast
pattern and dtype (odd row lengths, so that nothing is aligned), key padding
over an odd length, causal with s != t, and the first lengths and shapes the
general kernels take again."""

from __future__ import annotations

import numpy as np
import pytest
import torch
from _golden import relerr
from test_hip_parity import REL, _check, _dev, _draw, _to

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize('dtype', [BF, HF], ids=['bf16', 'f16'])
@pytest.mark.parametrize('s, t, d, dv', [
    (5, 7, 8, 8), (31, 33, 32, 32), (64, 65, 40, 40), (95, 129, 32, 64), (343, 343, 32, 32),
    (512, 512, 64, 64), (512, 513, 64, 64), (513, 300, 24, 24), (300, 17, 64, 16),
])
def test_lengths_and_head_dims(dtype, s, t, d, dv):
    _check(dtype, 3, 4, s, t, d, dv=dv, seed=s + t + d)
    _check(dtype, 3, 4, s, t, d, dv=dv, mask_kind='keypad', seed=s + t)
    _check(dtype, 2, 4, s, t, d, dv=dv, causal=True, seed=s)


@pytest.mark.parametrize('bias_dtype', [BF, F32], ids=['bf16', 'f32'])
@pytest.mark.parametrize('B, H, bias', [
    (8, 3, (3, 0, 0)), (4, 5, (1, 1, 0, 0)), (3, 8, (3, 1, 0, 0)), (5, 2, (1, 2, 1, 0)),
    (64, 4, (4, 0, 0)), (3, 3, (3, 0, 0)),
], ids=['heads', 'one', 'batch', 'row', 'many', 'share3'])
@pytest.mark.parametrize('s, t, d', [(49, 49, 32), (343, 343, 32), (100, 130, 64), (33, 511, 48)])
def test_shared_bias(bias_dtype, B, H, bias, s, t, d):
    shape = tuple(n or m for n, m in zip(bias, (*(1,) * (len(bias) - 2), s, t)))
    _check(BF, B, H, s, t, d, bias_shape=shape, bias_dtype=bias_dtype, seed=s + B)
    if B < 64:
        _check(BF, B, H, s, t, d, bias_shape=shape, bias_dtype=bias_dtype, mask_kind='keypad',
               causal=s == t, scale=0.3, seed=t + B)


@pytest.mark.parametrize('dtype', [BF, HF], ids=['bf16', 'f16'])
def test_large_and_negative_infinite_bias(dtype):
    """A shared bias used as a mask (-inf on some keys of every row) and one
    whose logits rise far above the first tiles' (the row reference moves)."""
    rng = np.random.default_rng(3)
    B, H, s, t, d = 4, 2, 100, 201, 32
    q, k, v = (_draw(rng, (B, H, n, d), dtype) for n in (s, t, t))
    bias = np.linspace(0, 300, t, dtype=np.float32)[None, None] + np.zeros((H, s, 1), np.float32)
    bias = bias.astype(np.float16).astype(np.float32) if dtype == HF else np.floor(bias)
    bias[:, :, 1::3] = -np.inf
    from nitrix_amd import scaled_dot_product_attention
    from oracle import attention as O

    if dtype == BF:
        bias = O.round_bf16(np.where(np.isinf(bias), 0, bias)).astype(np.float32)
        bias[:, :, 1::3] = -np.inf
    out = scaled_dot_product_attention(_to(q, dtype), _to(k, dtype), _to(v, dtype),
                                       bias=_to(bias, dtype), backend='hip')
    ref = O.sdpa_forward(q, k, v, bias=bias, scale=d ** -0.5, acc_dtype=np.float64)
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all()
    assert np.abs(got - ref).max() / np.abs(ref).max() <= (2e-2 if dtype == BF else 2e-3)


LOWEST = float(np.finfo(np.float32).min)


@pytest.mark.parametrize('dtype, bias_dtype', [(HF, F32), (BF, F32), (BF, BF)],
                         ids=['f16', 'bf16', 'bf16b'])
@pytest.mark.parametrize('d', [16, 24, 32, 40, 64])
@pytest.mark.parametrize('const', [-1e4, -1e9, -1e10, -1e30, LOWEST])
def test_large_finite_bias_as_a_mask(dtype, bias_dtype, d, const):
    """A shared bias that masks with a large finite constant: on the first
    keys (the first tiles hold nothing else), on the last, and on whole rows.
    The whole rows' output is the softmax of what float32 keeps of their
    scores (from 1e8 on nothing: the mean of v), and with a zero cotangent
    they leave every gradient alone."""
    from nitrix_amd import scaled_dot_product_attention
    from oracle import attention as O

    rng = np.random.default_rng(d)
    B, H, s, t = 72, 4, 40, 131
    q, k, v, g = (_draw(rng, (B, H, n, d), dtype) for n in (s, t, t, s))
    bias = _draw(rng, (1, H, s, t), bias_dtype)
    if bias_dtype == BF:
        const = max(const, float(torch.finfo(BF).min))
        const = float(torch.tensor(const).to(BF))
    bias[:, :, :20, :64] = const
    bias[:, :, 20:30] = const
    bias[:, :, 30:, 70:] = const
    if const < -1e38:
        bias[:, :, 29, 100:] = const / 2  # larger: these keys take the row
    g[:, :, 20:30] = 0
    tq, tk, tv, tb = _to(q, dtype, True), _to(k, dtype, True), _to(v, dtype, True), _to(bias, bias_dtype, True)
    print(f'[case] {dtype} {bias_dtype} d{d} const {const}', flush=True)
    out = scaled_dot_product_attention(tq, tk, tv, bias=tb, backend='hip')
    grads = torch.autograd.grad(out, (tq, tk, tv, tb), _to(g, dtype))
    b64 = np.broadcast_to(bias, (B, H, s, t)).astype(np.float64)
    ref = O.sdpa_forward(q, k, v, bias=b64, scale=d ** -0.5, acc_dtype=np.float64)
    if const < -1e8:
        ref[:, :, 20:30] = v.astype(np.float64).mean(2, keepdims=True)
    if const < -1e38:
        ref[:, :, 29] = v[:, :, 100:].astype(np.float64).mean(2)
    want = O.sdpa_backward(q, k, v, g, bias=bias, scale=d ** -0.5, acc_dtype=np.float64)
    for name, got, w in zip(('out', 'dq', 'dk', 'dv', 'dbias'), (out, *grads), (ref, *want)):
        got = got.detach().float().cpu().numpy()
        assert np.isfinite(got).all(), name
        err = relerr(got, w.reshape(got.shape))
        tol = max(REL[dtype], REL[bias_dtype]) if name == 'dbias' else REL[dtype]
        assert err <= tol, (name, err)


@pytest.mark.parametrize('dtype, d, dv', [(BF, 64, 64), (HF, 40, 56)], ids=['bf16', 'f16'])
@pytest.mark.parametrize('s, t', [(343, 343), (511, 449)])
@pytest.mark.parametrize('kind', ['plain', 'causal', 'keypad', 'bias'])
def test_eight_wave_blocks(dtype, d, dv, s, t, kind):
    """Blocks of 8 waves in the forward, dQ and dK / dV: more than 53 KB
    resident and more than 256 blocks of 128 rows (the launcher's rule; a
    bias of odd rows is packed in the forward too)."""
    B, H = 24, 4
    for resident, strips in ((t, s), (s, t)):
        assert 2 * -(-resident // 64) * 64 * 64 * 2 > 53 * 1024
        assert B * H * -(-strips // 128) > 256
    kw = {'plain': {}, 'causal': dict(causal=True), 'keypad': dict(mask_kind='keypad'),
          'bias': dict(bias_shape=(1, H, s, t), bias_dtype=F32)}[kind]
    _check(dtype, B, H, s, t, d, dv=dv, seed=s + d, **kw)


@pytest.mark.parametrize('L, d', [(296, 32), (304, 64)])
def test_packed_forward_of_aligned_bias_rows(L, d):
    """A bias the general forward could read as it is, packed where enough
    pairs share it."""
    B, H = 33, 8
    from nitrix_amd import _lib
    from nitrix_amd.attention import _Prepared

    q = torch.zeros(B, H, L, d, device=_dev(), dtype=BF)
    bias = torch.zeros(1, H, L, L, device=_dev(), dtype=BF)
    prep = _Prepared(q, q, q, bias, None, d ** -0.5, False)
    assert prep.workspace_bytes(_lib.NXA_WS_PACK) > prep.workspace_bytes(_lib.NXA_WS_FWD)
    _check(BF, B, H, L, L, d, bias_shape=(1, H, L, L), seed=L, grads=False)
    _check(BF, B, H, L, L, d, bias_shape=(1, H, L, L), causal=True, mask_kind='keypad', seed=L,
           grads=False)


@pytest.mark.parametrize('dtype', [BF, HF], ids=['bf16', 'f16'])
def test_a_large_positive_bias_takes_its_rows(dtype):
    """One key at +1e9: every row's output is that key's value, its value's
    gradient the sum of the cotangents, and no other gradient is larger than
    the rounding of P (dP - delta)."""
    from nitrix_amd import scaled_dot_product_attention

    rng = np.random.default_rng(11)
    B, H, s, t, d = 72, 4, 40, 131, 32
    q, k, v, g = (_draw(rng, (B, H, n, d), dtype) for n in (s, t, t, s))
    bias = _draw(rng, (1, H, s, t), F32)
    bias[..., 77] = 1e9
    tq, tk, tv = _to(q, dtype, True), _to(k, dtype, True), _to(v, dtype, True)
    out = scaled_dot_product_attention(tq, tk, tv, bias=_to(bias, F32), backend='hip')
    dq, dk, dv = (x.float().cpu().numpy() for x in
                  torch.autograd.grad(out, (tq, tk, tv), _to(g, dtype)))
    assert relerr(out.detach().float().cpu().numpy(), np.broadcast_to(v[:, :, 77:78], out.shape)) == 0
    want = np.zeros_like(v, dtype=np.float64)
    want[:, :, 77] = g.astype(np.float64).sum(2)
    assert relerr(dv, want) <= REL[dtype]
    # dP - delta: two sums of d products of unit size, in fp32
    assert np.abs(dq).max() <= 1e-3 and np.abs(dk).max() <= s * 1e-3


def _forms(x, dtype):
    """The same values under other strides: [B, L, H, D] memory, rows apart,
    a slice of a longer sequence."""
    B, H, L, D = x.shape
    t = _to(x, dtype)
    wide = torch.zeros(B, H, L, D + 16, device=_dev(), dtype=dtype)
    wide[..., 8:8 + D] = t
    long = torch.zeros(B, H, L + 5, D, device=_dev(), dtype=dtype)
    long[:, :, 3:3 + L] = t
    return {'plain': t, 'blhd': t.transpose(1, 2).contiguous().transpose(1, 2),
            'rows': wide[..., 8:8 + D], 'slice': long[:, :, 3:3 + L]}


@pytest.mark.parametrize('form', ['blhd', 'rows', 'slice'])
@pytest.mark.parametrize('s, t, d, bias', [
    (70, 131, 32, None), (70, 131, 64, 'heads'), (200, 131, 32, 'batch'), (28, 700, 64, None),
])
def test_strided_inputs(form, s, t, d, bias):
    """Any strides give the bytes of contiguous inputs: outputs and gradients
    of the short-sequence and key-split paths, a bias of spaced rows among them."""
    from nitrix_amd import scaled_dot_product_attention

    rng = np.random.default_rng(s + d)
    B, H = 72, 4
    fq, fk, fv, fg = (_forms(_draw(rng, (B, H, n, d), BF), BF) for n in (s, t, t, s))
    b = None if bias is None else _draw(rng, {'heads': (1, H, s, t), 'batch': (B, 1, s, t)}[bias], BF)
    runs = []
    for f in ('plain', form):
        ins = [x[f].detach().requires_grad_(True) for x in (fq, fk, fv)]
        tb = None
        if b is not None:
            tb = _to(b, BF)
            if f != 'plain':
                tb = torch.nn.functional.pad(tb, (3, 2))[..., 3:3 + t].detach()
            ins.append(tb.requires_grad_(True))
        out = scaled_dot_product_attention(*ins[:3], bias=tb, backend='hip')
        runs.append((out, *torch.autograd.grad(out, ins, fg[f])))
    for a, c in zip(*runs):
        assert torch.equal(a, c)


@pytest.mark.parametrize('s, t', [(70, 131), (28, 700)])
def test_inputs_broadcast_over_heads_and_batch(s, t):
    """Keys shared by all heads, values by all batches, as views."""
    from nitrix_amd import scaled_dot_product_attention

    rng = np.random.default_rng(t)
    B, H, d = 3, 4, 64
    q, k, v, g = (_to(_draw(rng, sh, BF), BF, True) for sh in
                  ((B, H, s, d), (B, 1, t, d), (1, H, t, d), (B, H, s, d)))
    runs = []
    for expand in (False, True):
        ke, ve = k.expand(B, H, t, d), v.expand(B, H, t, d)
        if not expand:
            ke, ve = ke.contiguous(), ve.contiguous()
        with torch.no_grad():
            o = scaled_dot_product_attention(q, ke, ve, backend='hip')
        out = scaled_dot_product_attention(q, ke, ve, backend='hip')
        runs.append((o, out, *torch.autograd.grad(out, (q, k, v), g.detach())))
    for a, c in zip(*runs):
        assert torch.equal(a, c)


def test_a_call_repeats_itself():
    from nitrix_amd import scaled_dot_product_attention

    g = torch.Generator(device=_dev()).manual_seed(2)
    q, k, v, do = (torch.randn(16, 4, 343, 32, generator=g, device=_dev()).to(BF) for _ in range(4))
    bias = torch.randn(1, 4, 343, 343, generator=g, device=_dev()).to(BF)
    ins = [t.requires_grad_(True) for t in (q, k, v, bias)]
    runs = []
    for _ in range(3):
        out = scaled_dot_product_attention(q, k, v, bias=bias, backend='hip')
        runs.append((out, *torch.autograd.grad(out, ins, do)))
    for run in runs[1:]:
        for a, b in zip(runs[0], run):
            assert torch.equal(a, b)


def test_the_packed_bias_is_not_kept_for_the_backward():
    """Between forward and backward a call holds its output, the row values
    and no packed bias (which is larger than the bias itself)."""
    from nitrix_amd import scaled_dot_product_attention

    B, H, n, d = 96, 4, 343, 32
    q, k, v = (torch.randn(B, H, n, d, device=_dev(), dtype=BF) for _ in range(3))
    bias = torch.randn(B, 1, n, n, device=_dev(), dtype=BF)
    for want in (False, True):
        q.requires_grad_(True)
        bias.requires_grad_(want)
        before = torch.cuda.memory_allocated()
        out = scaled_dot_product_attention(q, k, v, bias=bias, backend='hip')
        held = torch.cuda.memory_allocated() - before
        packed = B * 12 * 12 * 4096
        assert held <= out.numel() * 2 + B * H * n * 4 + 4096 < packed
        torch.autograd.grad(out, (q, bias) if want else q, torch.ones_like(out))


def test_workspace_without_room_for_the_packed_bias():
    """A caller that passes no workspace to a mask-free forward with a shared
    bias is served by the general kernels, to rounding."""
    import ctypes

    from nitrix_amd import _lib
    from nitrix_amd.attention import _Prepared

    g = torch.Generator(device=_dev()).manual_seed(5)
    q, k, v = (torch.randn(8, 2, 70, 32, generator=g, device=_dev()).to(BF) for _ in range(3))
    bias = torch.randn(2, 70, 70, generator=g, device=_dev()).to(BF)
    prep = _Prepared(q, k, v, bias, None, 32 ** -0.5, False)
    outs = []
    for ws in (prep.workspace(_lib.NXA_WS_PACK), None):
        o = torch.empty_like(q)
        lse = torch.empty(8, 2, 70, device=_dev())
        _lib.check(_lib.lib().nxa_fwd(
            ctypes.byref(prep.desc), prep.q.data_ptr(), prep.k.data_ptr(), prep.v.data_ptr(),
            prep.bias.data_ptr(), None, o.data_ptr(), lse.data_ptr(),
            None if ws is None else ws.data_ptr(), 0 if ws is None else ws.numel(),
            prep.stream()))
        outs.append((o.float(), lse))
    assert prep.workspace_bytes(_lib.NXA_WS_PACK) > prep.workspace_bytes(_lib.NXA_WS_FWD) == 0
    torch.testing.assert_close(outs[0][0], outs[1][0], rtol=0, atol=2e-2)
    torch.testing.assert_close(outs[0][1], outs[1][1], rtol=0, atol=2e-3)
