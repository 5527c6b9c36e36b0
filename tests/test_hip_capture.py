"""The short-sequence, key-split and one-kernel scan paths in a captured HIP
graph and on a stream of their own: every replay gives the bytes of an eager
call on the inputs it finds (the paths launch kernels only, and their
workspaces live in the graph's pool)."""

from __future__ import annotations

import pytest
import torch

from nitrix_amd import scaled_dot_product_attention, selective_scan

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def _randn(gen, *shape, dtype=BF):
    return torch.randn(*shape, generator=gen, device='cuda:0').to(dtype)


def _window(gen):
    ins = [_randn(gen, 72, 4, 131, 32) for _ in range(3)] + [_randn(gen, 1, 4, 131, 131)]
    do = _randn(gen, 72, 4, 131, 32)

    def run():
        out = scaled_dot_product_attention(*ins[:3], bias=ins[3], backend='hip')
        return (out, *torch.autograd.grad(out, ins, do))

    return ins, run, True


def _prompt(gen):
    ins = [_randn(gen, 4, 8, n, 64) for n in (28, 8192, 8192)]
    mask = (torch.arange(8192, device='cuda:0') < 7000)[None, None, None]

    def run():
        return (scaled_dot_product_attention(*ins, mask=mask, backend='hip'),)

    return ins, run, False


def _scan(gen):
    f32 = torch.float32
    ins = [_randn(gen, 2, 300, 40, dtype=f32), torch.rand(2, 300, 40, generator=gen, device='cuda:0'),
           -torch.rand(40, 16, generator=gen, device='cuda:0'), _randn(gen, 2, 300, 16, dtype=f32),
           _randn(gen, 2, 300, 16, dtype=f32)]
    dy = _randn(gen, 2, 300, 40, dtype=f32)

    def run():
        y = selective_scan(*ins, backend='hip')
        return (y, *torch.autograd.grad(y, ins, dy))

    return ins, run, True


@pytest.mark.parametrize('make', [_window, _prompt, _scan])
def test_replays_and_streams_give_the_eager_bytes(make):
    gen = torch.Generator(device='cuda:0').manual_seed(3)
    ins, run, train = make(gen)
    for t in ins:
        t.requires_grad_(train)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            run()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = run()
    for step in range(4):
        with torch.no_grad():
            ins[0].copy_(torch.randn(ins[0].shape, generator=gen, device='cuda:0'))
        graph.replay()
        torch.cuda.synchronize()
        got = [t.detach().clone() for t in captured]
        eager = run()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            other = run()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        for a, b, c in zip(got, eager, other):
            assert torch.equal(a, b) and torch.equal(b, c), step
