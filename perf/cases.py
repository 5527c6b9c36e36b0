"""Performance cases: the calls a program makes of this package's two operators.

Attention (``scaled_dot_product_attention``) and the selective scan
(``selective_scan``), each through its public entry point with the default
backend, over the range of sizes, data types, masks and biases that the
package's benchmark, tests and documents use.  :func:`listed` names twelve of
them, :func:`draw` gives more of the same ranges.

A case is a dict of plain values.  Attention: ``op='attention'``, ``dtype``
(``bf16`` / ``f16`` / ``f32``), ``B``, ``H``, ``Lq``, ``Lk``, ``D``, ``bias``
(``none``; ``full`` ``[B, H, Lq, Lk]``; ``head`` ``[1, H, Lq, Lk]``; ``row``
``[1, H, 1, Lk]``), ``mask`` (``none``; ``keypad`` ``[B, 1, 1, Lk]``;
``blocks`` ``[1, 1, Lq, Lk]`` of 128 x 128 blocks), ``causal``, ``qk_norm``
and ``train`` (with the gradients of q, k, v and the bias).  Scan:
``op='scan'``, ``dtype`` (of x, delta, B and C; A and D are float32, as
programs keep them), ``B``, ``L``, ``Dm``, ``N``, ``train``.
"""

from __future__ import annotations

import math

import torch

from nitrix_amd import scaled_dot_product_attention, selective_scan

_DTYPES = {'bf16': torch.bfloat16, 'f16': torch.float16, 'f32': torch.float32}


def _attention(name, dtype, B, H, Lq, Lk, D, *, bias='none', mask='none', causal=False,
               qk_norm=False, train=False):
    case = dict(op='attention', dtype=dtype, B=B, H=H, Lq=Lq, Lk=Lk, D=D, bias=bias, mask=mask,
                causal=causal, qk_norm=qk_norm, train=train)
    if name:
        case['name'] = name
    return case


def _scan(name, dtype, B, L, Dm, N, *, train):
    case = dict(op='scan', dtype=dtype, B=B, L=L, Dm=Dm, N=N, train=train)
    if name:
        case['name'] = name
    return case


def listed():
    return [
        # One small float32 layer call with a position bias: latency and
        # launches (the benchmark's c1).
        _attention('small_bias_f32', 'f32', 1, 4, 256, 256, 64, bias='head'),
        # A float32 transformer layer over 344 tokens of a volume, forward and
        # backward: an ordinary, odd-sized training call.
        _attention('volume_f32_train', 'f32', 4, 6, 344, 344, 64, train=True),
        # Window attention over 7 x 7 x 7 voxels with a learned relative
        # position bias shared by all windows, forward and backward: many
        # short, odd-sized problems at a small head dim.
        _attention('window_bf16_train', 'bf16', 512, 4, 343, 343, 32, bias='head', train=True),
        # A few prompt tokens attending a long padded sequence at inference:
        # few queries, many keys.
        _attention('prompt_f16', 'f16', 4, 8, 28, 8192, 64, mask='keypad'),
        # A layer with normalised q and k at an odd length, causal, forward
        # and backward in float16.
        _attention('qknorm_f16_train', 'f16', 2, 16, 1500, 1500, 128, causal=True, qk_norm=True,
                   train=True),
        # Training on padded batches of long sequences (the benchmark's c2,
        # its default).
        _attention('padded_bf16_train', 'bf16', 8, 16, 4096, 4096, 128, mask='keypad', train=True),
        # Causal training at twice the length and heads (c3): the largest.
        _attention('causal_bf16_train', 'bf16', 4, 32, 8192, 8192, 128, causal=True, train=True),
        # Inference with a full per-head bias, bound by the bias stream (c4).
        _attention('full_bias_bf16', 'bf16', 2, 16, 8192, 8192, 64, bias='full'),
        # Training on one very long sequence with a block-sparse mask and a
        # bias per key (c5).
        _attention('sparse_bf16_train', 'bf16', 1, 8, 32768, 32768, 64, bias='row', mask='blocks',
                   train=True),
        # A float32 scan layer, forward and backward (the benchmark's ssm).
        _scan('scan_f32_train', 'f32', 8, 2048, 1536, 16, train=True),
        # One long sequence of odd sizes through a scan layer at inference.
        _scan('scan_bf16', 'bf16', 1, 5000, 1000, 16, train=False),
        # A scan layer in mixed precision with odd sizes, forward and backward.
        _scan('scan_bf16_train', 'bf16', 4, 1023, 1200, 8, train=True),
    ]


def _spread(rng, lo, hi):
    """A whole number in [lo, hi], spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _cost(case):
    # float32 products run at a sixteenth of the 16-bit rate.
    w = work(case)
    rate = 16 if case['op'] == 'attention' and case['dtype'] == 'f32' else 1
    return max(w['bytes'] * 250, w['flops'] * (rate if case['op'] == 'attention' else 32))


def draw(rng):
    """One more case of the ranges behind the listed ones."""
    top = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(['layer', 'layer', 'layer', 'window', 'prompt', 'bias', 'sparse',
                           'scan', 'scan'])
        wide = rng.choice(['bf16', 'bf16', 'f16'])
        if kind == 'layer':
            L = _spread(rng, 64, 8192)
            mask = rng.choice(['none', 'keypad'])
            case = _attention(None, rng.choice([wide, wide, 'f32']), _spread(rng, 1, 8),
                              _spread(rng, 4, 32), L, L, rng.choice([64, 64, 96, 128, 128, 256]),
                              mask=mask, causal=mask == 'none' and rng.random() < 0.5,
                              qk_norm=rng.random() < 0.25, train=rng.random() < 0.7)
        elif kind == 'window':
            L = rng.choice([rng.randint(4, 8) ** 3, rng.randint(6, 16) ** 2])
            case = _attention(None, rng.choice([wide, wide, 'f32']), _spread(rng, 16, 1024),
                              _spread(rng, 3, 12), L, L, rng.choice([32, 32, 64]), bias='head',
                              train=rng.random() < 0.7)
        elif kind == 'prompt':
            case = _attention(None, wide, _spread(rng, 1, 16), _spread(rng, 4, 32),
                              _spread(rng, 1, 64), _spread(rng, 1024, 32768),
                              rng.choice([32, 64, 128]), mask=rng.choice(['none', 'keypad']))
        elif kind == 'bias':
            L = 8 * _spread(rng, 32, 1024) if rng.random() < 0.5 else _spread(rng, 256, 4096)
            case = _attention(None, wide, _spread(rng, 1, 4), _spread(rng, 4, 16), L, L,
                              rng.choice([64, 128]), bias='full')
        elif kind == 'sparse':
            L = 128 * _spread(rng, 32, 256)
            case = _attention(None, wide, 1, _spread(rng, 4, 8), L, L, rng.choice([64, 128]),
                              bias='row', mask='blocks', train=rng.random() < 0.7)
        else:
            case = _scan(None, rng.choice(['f32', 'bf16']), _spread(rng, 1, 8),
                         _spread(rng, 64, 8192), _spread(rng, 64, 2048), rng.choice([4, 8, 16, 32]),
                         train=rng.random() < 0.6)
        if _cost(case) <= top:
            return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _randn(gen, dtype, *shape):
    x = torch.empty(*shape, device=gen.device, dtype=dtype)
    flat = x.view(-1)
    step = 1 << 28  # float32 draws of large tensors go in pieces
    for i in range(0, flat.numel(), step):
        n = min(step, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, generator=gen, device=gen.device)
    return x


def _mask(gen, case):
    B, Lq, Lk = case['B'], case['Lq'], case['Lk']
    if case['mask'] == 'keypad':
        # Valid lengths uniform in [Lk / 4, Lk].
        lo = max(1, Lk // 4)
        valid = torch.randint(lo, Lk + 1, (B, 1), generator=gen, device=gen.device)
        return (torch.arange(Lk, device=gen.device)[None, :] < valid)[:, None, None, :]
    if case['mask'] == 'blocks':
        # 128 x 128 blocks kept with probability 1/4, the diagonal always.
        nq, nk = -(-Lq // 128), -(-Lk // 128)
        keep = torch.rand(nq, nk, generator=gen, device=gen.device) < 0.25
        keep |= torch.eye(nq, nk, device=gen.device, dtype=torch.bool)
        keep = keep.repeat_interleave(128, 0).repeat_interleave(128, 1)[:Lq, :Lk]
        return keep.contiguous()[None, None]
    return None


def _bias(gen, dtype, case):
    shape = {
        'none': None,
        'full': (case['B'], case['H'], case['Lq'], case['Lk']),
        'head': (1, case['H'], case['Lq'], case['Lk']),
        'row': (1, case['H'], 1, case['Lk']),
    }[case['bias']]
    return None if shape is None else _randn(gen, dtype, *shape)


def prepare(case, seed):
    dev = torch.device('cuda', torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    dtype = _DTYPES[case['dtype']]
    train = case['train']
    if case['op'] == 'attention':
        B, H, D = case['B'], case['H'], case['D']
        inputs = dict(
            q=_randn(gen, dtype, B, H, case['Lq'], D),
            k=_randn(gen, dtype, B, H, case['Lk'], D),
            v=_randn(gen, dtype, B, H, case['Lk'], D),
            bias=_bias(gen, dtype, case),
        )
        state = dict(mask=_mask(gen, case))
        out_shape, out_dtype = (B, H, case['Lq'], D), dtype
    else:
        B, L, Dm, N = case['B'], case['L'], case['Dm'], case['N']
        inputs = dict(
            x=_randn(gen, dtype, B, L, Dm),
            # Step sizes in [0.01, 0.1], decay rates 1 .. N per channel.
            delta=(0.01 + 0.09 * torch.sigmoid(_randn(gen, torch.float32, B, L, Dm))).to(dtype),
            A=-(torch.arange(N, device=dev, dtype=torch.float32) + 1.0).repeat(Dm, 1),
            B=_randn(gen, dtype, B, L, N),
            C=_randn(gen, dtype, B, L, N),
            D=_randn(gen, torch.float32, Dm),
        )
        state = {}
        out_shape, out_dtype = (B, L, Dm), torch.float32
    if train:
        for t in inputs.values():
            if t is not None:
                t.requires_grad_(True)
        state['dout'] = _randn(gen, out_dtype, *out_shape)
    return dict(state, case=case, inputs=inputs)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(state):
    case, t = state['case'], state['inputs']
    if case['op'] == 'attention':
        out = scaled_dot_product_attention(
            t['q'], t['k'], t['v'], bias=t['bias'], mask=state['mask'], causal=case['causal'],
            qk_norm=case['qk_norm'],
        )
    else:
        out = selective_scan(t['x'], t['delta'], t['A'], t['B'], t['C'], t['D'])
    if not case['train']:
        return {'out': out}
    names = [n for n, x in t.items() if x is not None]
    grads = torch.autograd.grad(out, [t[n] for n in names], state['dout'])
    return {'out': out, **{'d' + n: g for n, g in zip(names, grads)}}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------


def work(case):
    e = 4 if case['dtype'] == 'f32' else 2
    if case['op'] == 'scan':
        rows = case['B'] * case['L']
        x, bc, a = rows * case['Dm'], rows * case['N'], case['Dm'] * (case['N'] + 1)
        steps = float(x * case['N'])
        if not case['train']:
            return {'bytes': (2 * x + 2 * bc) * e + 4 * a + 4 * x, 'flops': 7 * steps}
        return {'bytes': (4 * x + 4 * bc) * e + 8 * a + 2 * 4 * x, 'flops': 27 * steps}
    B, H, Lq, Lk, D = (case[n] for n in ('B', 'H', 'Lq', 'Lk', 'D'))
    pairs = float(Lq) * Lk
    kept = 1.0
    if case['causal']:
        pairs = float(sum(min(i + 1, Lk) for i in range(Lq)))
    elif case['mask'] == 'keypad':
        kept = 0.625  # the mean valid length over Lk
    elif case['mask'] == 'blocks':
        n = -(-Lk // 128)
        kept = (1 + 0.25 * (n - 1)) / n
    bias = {'none': 0, 'full': B * H * Lq * Lk, 'head': H * Lq * Lk, 'row': H * Lk}[case['bias']]
    mask = {'none': 0, 'keypad': B * Lk, 'blocks': Lq * Lk}[case['mask']]
    keys = kept if case['mask'] == 'keypad' else 1.0
    qo, kv = B * H * Lq * D * 2, B * H * Lk * D * 2
    flops = 4.0 * D * B * H * pairs * kept
    if not case['train']:
        return {'bytes': int((qo + kv * keys + bias) * e + mask), 'flops': flops}
    # Forward and backward: q, k, v, bias and dout read, out and the gradients written.
    return {'bytes': int((2 * qo + kv * (keys + 1) + 2 * bias) * e + mask), 'flops': 3.5 * flops}


def tolerance(case):
    # Relative error (2-norm) that another correct implementation at the same
    # precision shows: about four times the measured distance from float64
    # (scan 2e-7 to 5e-7 in float32, 1.7e-3 for gradients rounded to bf16;
    # attention 2.5e-3 in bf16, 5e-4 in f16, 4e-7 to 7e-7 in float32).
    if case['op'] == 'scan':
        return {'rel': 7e-3} if case['dtype'] == 'bf16' and case['train'] else {'rel': 2e-6}
    return {'rel': {'bf16': 1e-2, 'f16': 2e-3, 'f32': 3e-6}[case['dtype']]}


# ---------------------------------------------------------------------------
# The same in float64
# ---------------------------------------------------------------------------


def _norm64(z):
    """RMS-normalised rows of z and the reciprocal root they were scaled by."""
    r = torch.rsqrt(z.square().mean(-1, keepdim=True) + 1e-6)
    return z * r, r


def _norm64_vjp(z, r, g):
    y = z * r
    return r * (g - y * (g * y).mean(-1, keepdim=True))


def _exact_attention(case, state):
    t, mask, train = state['inputs'], state['mask'], case['train']
    B, H, Lq, Lk, D = (case[n] for n in ('B', 'H', 'Lq', 'Lk', 'D'))
    dev = t['q'].device
    q, k, v = (t[n].detach().view(B * H, -1, D) for n in ('q', 'k', 'v'))
    bias = None if t['bias'] is None else t['bias'].detach()
    dout = state['dout'].view(B * H, Lq, D) if train else None
    out = torch.empty(B * H, Lq, D, dtype=torch.float64, device=dev)
    grads = None
    if train:
        grads = [torch.zeros(B * H, n, D, dtype=torch.float64, device=dev) for n in (Lq, Lk, Lk)]
    dbias = torch.zeros(bias.shape, dtype=torch.float64, device=dev) if train and bias is not None else None
    scale = 1.0 / math.sqrt(D)
    rows = max(1, min(Lq, (1 << 27) // Lk))          # query rows at a time
    heads = max(1, (1 << 27) // (rows * Lk))          # (batch, head) pairs at a time
    keys = torch.arange(Lk, device=dev)
    for i0 in range(0, B * H, heads):
        # Pairs of one batch entry, so that a batch's mask broadcasts.
        i = i0
        while i < min(i0 + heads, B * H):
            b = i // H
            j = min(i0 + heads, B * H, (b + 1) * H)
            h0, h1 = i - b * H, j - b * H
            kk, vv = k[i:j].double(), v[i:j].double()
            kr = None
            if case['qk_norm']:
                kk, kr = _norm64(kk)
            for r0 in range(0, Lq, rows):
                r1 = min(Lq, r0 + rows)
                qq = q[i:j, r0:r1].double()
                qr = None
                if case['qk_norm']:
                    qq, qr = _norm64(qq)
                s = torch.matmul(qq, kk.transpose(1, 2).contiguous()).mul_(scale)
                if bias is not None:
                    bb = bias[b if bias.shape[0] > 1 else 0, h0:h1]
                    s += bb[:, r0:r1] if bias.shape[2] > 1 else bb
                if mask is not None:
                    m = mask[b if mask.shape[0] > 1 else 0, 0]
                    s.masked_fill_(~(m[r0:r1] if m.shape[0] > 1 else m), -math.inf)
                if case['causal']:
                    s.masked_fill_(keys[None, :] > torch.arange(r0, r1, device=dev)[:, None], -math.inf)
                p = torch.softmax(s, -1)
                del s
                out[i:j, r0:r1] = torch.matmul(p, vv)
                if not train:
                    continue
                do = dout[i:j, r0:r1].double()
                grads[2][i:j] += torch.matmul(p.transpose(1, 2).contiguous(), do)
                ds = torch.matmul(do, vv.transpose(1, 2).contiguous())
                ds -= (do * out[i:j, r0:r1]).sum(-1, keepdim=True)
                ds *= p
                del p
                if dbias is not None:
                    db = dbias[b if bias.shape[0] > 1 else 0, h0:h1]
                    if bias.shape[2] > 1:
                        db[:, r0:r1] += ds
                    else:
                        db += ds.sum(1, keepdim=True)
                ds *= scale
                dq = torch.matmul(ds, kk)
                grads[0][i:j, r0:r1] = _norm64_vjp(q[i:j, r0:r1].double(), qr, dq) if case['qk_norm'] else dq
                grads[1][i:j] += torch.matmul(ds.transpose(1, 2).contiguous(), qq)
                del ds
            if train and case['qk_norm']:
                grads[1][i:j] = _norm64_vjp(k[i:j].double(), kr, grads[1][i:j].clone())
            i = j
    got = {'out': out.view(B, H, Lq, D)}
    if train:
        for n, g in zip('qkv', grads):
            got['d' + n] = g.view(B, H, -1, D)
        if dbias is not None:
            got['dbias'] = dbias
    return got


def _exact_scan(case, state):
    t = {n: x.detach().double() for n, x in state['inputs'].items()}
    x, delta, A, Bm, Cm, Dv = (t[n] for n in ('x', 'delta', 'A', 'B', 'C', 'D'))
    nb, L, Dm = x.shape
    N = A.shape[1]
    train = case['train']
    h = torch.zeros(nb, Dm, N, dtype=torch.float64, device=x.device)
    # States entering every step, for the backward (float64: a few GB at most).
    hist = torch.empty(L + 1, nb, Dm, N, dtype=torch.float64, device=x.device) if train else None
    y = torch.empty_like(x)
    dx_in = delta * x
    for s in range(L):
        if train:
            hist[s] = h
        h = torch.exp(delta[:, s, :, None] * A) * h + dx_in[:, s, :, None] * Bm[:, s, None, :]
        y[:, s] = torch.einsum('bdn,bn->bd', h, Cm[:, s]) + Dv * x[:, s]
    if not train:
        return {'out': y}
    hist[L] = h
    dy = state['dout'].double()
    g = torch.zeros_like(h)  # adjoint of the state after the step, from the right
    dx, ddelta = torch.empty_like(x), torch.empty_like(x)
    dA, dB, dC = torch.zeros_like(A), torch.empty_like(Bm), torch.empty_like(Cm)
    for s in range(L - 1, -1, -1):
        a = torch.exp(delta[:, s, :, None] * A)
        g = g + Cm[:, s, None, :] * dy[:, s, :, None]
        dC[:, s] = torch.einsum('bdn,bd->bn', hist[s + 1], dy[:, s])
        gb = torch.einsum('bdn,bn->bd', g, Bm[:, s])
        gah = g * a * hist[s]
        dx[:, s] = Dv * dy[:, s] + delta[:, s] * gb
        ddelta[:, s] = x[:, s] * gb + (gah * A).sum(-1)
        dA += (gah * delta[:, s, :, None]).sum(0)
        dB[:, s] = torch.einsum('bdn,bd->bn', g, dx_in[:, s])
        g = a * g
    dD = (dy * x).sum((0, 1))
    return {'out': y, 'dx': dx, 'ddelta': ddelta, 'dA': dA, 'dB': dB, 'dC': dC, 'dD': dD}


def exact(case, seed):
    state = prepare(case, seed)
    if case['op'] == 'scan':
        # The float64 states of a training pass are kept: skip what would not fit.
        if case['train'] and case['B'] * case['L'] * case['Dm'] * case['N'] > 3e9:
            return None
        return _exact_scan(case, state)
    with torch.no_grad():
        return _exact_attention(case, state)
