"""Grouped (per-expert) 4-bit GEMMs over uneven groups: group counts around the
8 XCDs that row tiles are dealt to, empty groups, groups of one row, and groups
at and past the row counts where a tile takes fewer matrix blocks (32, 64, 96,
128).  Reference: fp32 matmul per group with the device decode (itself checked
bit for bit elsewhere); bf16 results of fp32 sums agree to 2^-8."""
import pytest
import torch

from spilltune_amd import _lib, moe

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

GROUPS = [[5], [0, 130, 1], [33, 64, 65, 96, 97, 128, 129, 32], [64] * 9, [0] * 19 + [200]]


@pytest.mark.parametrize("hi_first", [False, True])
@pytest.mark.parametrize("N,K", [(256, 256), (200, 384), (520, 128)])
@pytest.mark.parametrize("rows", GROUPS, ids=[str(len(r)) for r in GROUPS])
def test_grouped_gemms_over_uneven_groups(rows, N, K, hi_first):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(sum(rows) + N + K)
    E, R, T = len(rows), sum(rows), 50
    flags = _lib.ST_FLAG_HI_NIBBLE_FIRST if hi_first else 0
    q = moe.Q4Experts(
        torch.randint(0, 256, (E * N * K // 2,), dtype=torch.uint8, device=dev, generator=g),
        torch.rand(E * N * K // 128, device=dev, generator=g) * 0.03 + 0.01, E, N, K, "nf4-g128",
        flags)
    W = q.dequantize().float()
    off = torch.tensor([0] + rows, device=dev).cumsum(0).int()
    tok = torch.randint(0, T, (R,), device=dev, generator=g).int()
    x = torch.randn(T, K, device=dev, generator=g).to(BF)
    dy = torch.randn(R, N, device=dev, generator=g).to(BF)
    gu = torch.randn(R, 2 * K, device=dev, generator=g).to(BF)
    y = torch.full((R, N), 7.0, dtype=BF, device=dev)
    dx, dgu, P = torch.full((R, K), 7.0, dtype=BF, device=dev), torch.empty_like(gu), _lib.ptr
    st = _lib.stream_handle(dev)
    _lib.call("st_q4_grouped_fwd", P(x), T, K, P(tok), R, K, P(off), E, P(q.payload), P(q.scales),
              N, q.lut(), flags, None, 0, None, 0, 1.0, 0, None, P(y), N, st)
    _lib.call("st_q4_grouped_dgrad", P(dy), N, R, N, P(off), E, P(q.payload), P(q.scales), K,
              q.lut(), flags, None, 0, None, 0, P(dx), K, st)
    _lib.call("st_q4_grouped_dgrad_swiglu", P(dy), N, R, N, P(off), E, P(q.payload), P(q.scales),
              K, q.lut(), flags, None, 0, None, 0, P(gu), 2 * K, P(dgu), 2 * K, st)
    ref_gu = torch.empty_like(dgu)
    _lib.call("st_swiglu_bwd", P(dx), K, P(gu), 2 * K, P(gu[:, K:]), 2 * K, R, K, P(ref_gu), 2 * K,
              P(ref_gu[:, K:]), 2 * K, st)
    assert torch.equal(dgu, ref_gu)  # the fused SwiGLU VJP of the same sums
    at = 0
    for e, n in enumerate(rows):
        sl = slice(at, at + n)
        at += n
        for got, a, b in ((y[sl], x[tok[sl].long()].float(), W[e].t()),
                          (dx[sl], dy[sl].float(), W[e])):
            slack = (a.abs() @ b.abs()) / a.shape[1] ** 0.5
            ref = a @ b
            assert ((got.float() - ref).abs() <= 2 ** -8 * (ref.abs() + slack)).all(), (e, n)


def test_half_row_tiles_equal_the_256_row_tile(monkeypatch):
    """Expert tails of at most 64 rows take half a 128-row tile: the same sums,
    adapters included, as the 256-row tile (bit for bit), on odd columns."""
    dev, rows, N, K, r = torch.device("cuda:0"), [1, 63, 64, 65, 128, 129, 192, 193, 300], 328, 512, 8
    g = torch.Generator(device=dev).manual_seed(5)
    E, R = len(rows), sum(rows)
    q = moe.Q4Experts(
        torch.randint(0, 256, (E * N * K // 2,), dtype=torch.uint8, device=dev, generator=g),
        torch.rand(E * N * K // 128, device=dev, generator=g) * 0.03 + 0.01, E, N, K, "nf4-g128")
    off = torch.tensor([0] + rows, device=dev).cumsum(0).int()
    x = torch.randn(R, K, device=dev, generator=g).to(BF)
    T = torch.randn(R, r, device=dev, generator=g)
    B = torch.randn(E, N, r, device=dev, generator=g) * 0.1
    P, got = _lib.ptr, []
    for tile in ("2568", "2566"):
        monkeypatch.setenv("ST_GROUPED_TILE", tile)
        for lora in (False, True):
            y = torch.full((R, N), 7.0, dtype=BF, device=dev)
            args = (P(T), r, P(B), r, 0.5, 1, _lib.i64_array([N])) if lora else \
                (None, 0, None, 0, 1.0, 0, None)
            _lib.call("st_q4_grouped_fwd", P(x), R, K, None, R, K, P(off), E, P(q.payload),
                      P(q.scales), N, q.lut(), 0, *args, P(y), N, _lib.stream_handle(dev))
            got.append(y)
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3])
    assert not torch.equal(got[0], got[1])
