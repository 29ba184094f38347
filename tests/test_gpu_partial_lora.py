"""Adapters on some segments of a fused projection (the reference adapts q, v
and o by default): one GEMM over all segments gives what the segments give one
by one, forward, input gradient and adapter gradients, immediate and deferred."""
import pytest
import torch

from spilltune_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


class _L:
    def __init__(self, g, rank, fin, fout, dev):
        self.rank, self.scale = rank, 2.0
        self.A = (torch.randn(rank, fin, generator=g, device=dev) * 0.05).requires_grad_(True)
        self.B = (torch.randn(fout, rank, generator=g, device=dev) * 0.05).requires_grad_(True)
        self.grad_A, self.grad_B = torch.zeros_like(self.A.detach()), torch.zeros_like(self.B.detach())


@pytest.mark.parametrize("deferred", [False, True])
@pytest.mark.parametrize("has", [(1, 0, 1), (0, 1, 0), (0, 0, 1)])
@pytest.mark.parametrize("M,rank", [(5, 3), (130, 8)])
def test_partial_adapters_equal_separate_projections(M, rank, has, deferred):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + rank)
    K, widths = 256, (160, 32, 64)
    N = sum(widths)
    payload = torch.randint(0, 256, (N * K // 2,), dtype=torch.uint8, device=dev, generator=g)
    scales = torch.rand(N * K // 128, device=dev, generator=g) * 0.03 + 0.01
    full = ops.Q4Weight(payload, scales, (N, K), "nf4-g128", widths)
    x0 = torch.randn(M, K, device=dev, generator=g).to(BF)
    dy = torch.randn(M, N, device=dev, generator=g).to(BF)
    loras = [_L(g, rank, K, n, dev) if h else None for n, h in zip(widths, has)]
    leaves = [t for l in loras if l is not None for t in (l.A, l.B)]

    def grads(out, x):
        if not deferred:
            return torch.autograd.grad(out, [x, *leaves], dy)
        with ops.lora_grad_sink(dev) as sink:
            (dx, *_) = torch.autograd.grad(out, [x, *leaves], dy, allow_unused=True)
            sink.flush()
        return [dx] + [t.clone() for l in loras if l is not None for t in (l.grad_A, l.grad_B)]

    x = x0.clone().requires_grad_(True)
    with pytest.raises(ValueError):
        ops.q4_lora_linear(x, full, loras)  # only on request
    y = ops.q4_lora_linear(x, full, loras, partial=True)
    got = grads(y, x)
    xs = x0.clone().requires_grad_(True)
    parts, at = [], 0
    for n, l in zip(widths, loras):
        w = ops.Q4Weight(payload[at * K // 2:(at + n) * K // 2], scales[at * K // 128:(at + n) * K // 128],
                         (n, K), "nf4-g128")
        parts.append(ops.q4_lora_linear(xs, w, [l]))
        at += n
    ys = torch.cat(parts, 1)
    want = grads(ys, xs)
    assert torch.equal(y, ys)  # the same sums, and + 0 where there is no adapter
    # dx: one bf16 sum over all segments against three bf16 sums added in bf16
    assert torch.allclose(got[0].float(), want[0].float(), rtol=2 ** -6, atol=2 ** -6 * want[0].float().abs().mean().item() * 4)
    for a, b in zip(got[1:], want[1:]):  # fp32 sums of the same products
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-4 * b.abs().max().item())


@pytest.mark.parametrize("has", [(1, 0, 1), (0, 1, 0)])
def test_infinite_rows_stay_infinite_without_an_adapter(has):
    """An infinity in a row of x (or dY) makes that row's outputs (or input
    gradient) infinite, not NaN, in the segments without an adapter: they have
    no adapter term.  The weights hold no zeros (0 * inf is NaN by itself)."""
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(11)
    M, K, rank, widths = 40, 256, 4, (64, 32, 64)
    N = sum(widths)
    nibble = torch.randint(8, 16, (2, N * K // 2), dtype=torch.uint8, device=dev, generator=g)
    w = ops.Q4Weight(nibble[0] | nibble[1] << 4,  # codes 8..15: positive weights
                     torch.full((N * K // 128,), 0.02, device=dev), (N, K), "nf4-g128", widths)
    x = torch.randn(M, K, device=dev, generator=g).to(BF)
    dy = torch.randn(M, N, device=dev, generator=g).to(BF)
    x[7, 3] = float("inf")
    loras = [_L(g, rank, K, n, dev) if h else None for n, h in zip(widths, has)]
    col = 0
    for n, h in zip(widths, has):
        if not h:
            dy[9, col] = float("-inf")
        col += n
    xg = x.clone().requires_grad_(True)
    y = ops.q4_lora_linear(xg, w, loras, partial=True)
    (dx,) = torch.autograd.grad(y, [xg], dy)
    base = ops.q4_lora_linear(x, w, None)
    col = 0
    for n, h in zip(widths, has):
        if not h:
            assert torch.equal(y[:, col:col + n], base[:, col:col + n])
            assert (y[7, col:col + n] == float("inf")).all()
        col += n
    rest = torch.arange(M, device=dev) != 9
    assert (dx[9] == float("-inf")).all() and torch.isfinite(dx[rest]).all()
