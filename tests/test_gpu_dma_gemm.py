"""bf16 GEMM tiles whose operands move by DMA, and the 4-bit linears that
decode W into a workspace and run on them.

Oracle: fp32 matmul of the same bf16 operands.  A bf16 result of an fp32 sum
is within half a bf16 ulp (2^-9) of it plus the sum's own error; the tolerance
takes 2^-8 of the value and 2^-8 of the sum of the terms' sizes over sqrt(K).
The decode-first linears must also give the bits of the fused kernels (the
same sums in the same order)."""
import pytest
import torch

from spilltune_amd import _lib, ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
TILES = ("256", "2561", "128", "1284")


@pytest.fixture()
def dev():
    return torch.device("cuda:0")


def _close(got, a, b):
    """``got`` against fp32 a @ b."""
    a, b = a.float(), b.float()
    ref = a @ b
    slack = (a.abs() @ b.abs()) / a.shape[1] ** 0.5
    assert torch.isfinite(got).all()
    assert ((got.float() - ref).abs() <= 2 ** -8 * (ref.abs() + slack)).all()


def _rand(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g, device="cuda:0") * scale).to(BF)


# contraction tails of every chunk count, one k-step, fewer k-steps than the
# operand rings hold; rows and columns short of, at and past a tile's edge
SHAPES = [(1, 8, 8), (3, 40, 56), (255, 256, 64), (257, 264, 72), (128, 136, 200), (300, 512, 1000)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_bf16_linear_tiles(dev, monkeypatch, tile, M, N, K):
    monkeypatch.setenv("ST_GEMM_DMA", tile)
    g = torch.Generator(device=dev).manual_seed(M * N + K)
    x, w, dy = _rand(g, M, K), _rand(g, N, K), _rand(g, M, N)
    _close(ops.linear_bf16(x, w), x, w.t())
    _close(ops.linear_bf16_dgrad(dy, w), dy, w)


def test_long_contraction_on_few_tiles(dev, monkeypatch):
    """The input gradient of a few rows over many (the terminal's short chunks)
    takes the deeper ring by itself; every tile sums in the same order."""
    g = torch.Generator(device=dev).manual_seed(8)
    M, N, K = 130, 256 * 64 + 8, 264
    w, dy = _rand(g, N, K, scale=0.02), _rand(g, M, N)
    got = ops.linear_bf16_dgrad(dy, w)
    _close(got, dy, w)
    for tile in TILES:
        monkeypatch.setenv("ST_GEMM_DMA", tile)
        assert torch.equal(ops.linear_bf16_dgrad(dy, w), got), tile


@pytest.mark.parametrize("tile", TILES)
def test_bf16_linear_odd_width_and_neighbours(dev, monkeypatch, tile):
    """N not a multiple of 8 (2-byte stores), and nothing written beside y."""
    monkeypatch.setenv("ST_GEMM_DMA", tile)
    g = torch.Generator(device=dev).manual_seed(3)
    M, N, K = 130, 261, 264
    x, w = _rand(g, M, K), _rand(g, N, K)
    y = torch.full((M + 2, N + 3), 7.0, dtype=BF, device=dev)
    _lib.call("st_linear_bf16_fwd", _lib.ptr(x), M, K, K, _lib.ptr(w), N, K, _lib.ptr(y[1:]), N + 3,
              _lib.stream_handle(dev))
    _close(y[1:M + 1, :N], x, w.t())
    assert (y[0] == 7).all() and (y[M + 1] == 7).all() and (y[:, N:] == 7).all()


def test_bf16_linear_keeps_nan_and_inf(dev):
    """A NaN or infinity reaches its own row only; rows past M and the
    contraction tail are zeros, not products with it."""
    g = torch.Generator(device=dev).manual_seed(5)
    x, w = _rand(g, 65, 72), _rand(g, 48, 72)
    x[7, 3], x[64, 71] = float("nan"), float("inf")
    y = ops.linear_bf16(x, w)
    assert torch.isnan(y[7]).all() and not torch.isfinite(y[64]).any()
    rest = torch.ones(65, dtype=torch.bool, device=dev)
    rest[7] = rest[64] = False
    _close(y[rest], x[rest], w.t())


def _q4(g, N, K, flags=0):
    group = 64 if flags & _lib.ST_FLAG_GROUP64 else 128
    groups = -(-N * K // group)
    payload = torch.randint(0, 256, (groups * group // 2,), dtype=torch.uint8, device="cuda:0",
                            generator=g)
    scales = torch.rand(groups, device="cuda:0", generator=g) * 0.03 + 0.01
    return ops.Q4Weight(payload, scales, (N, K), "nf4-g128", flags=flags)


HI64 = _lib.ST_FLAG_HI_NIBBLE_FIRST | _lib.ST_FLAG_GROUP64
# (M, N, K, rank, segments, flags): 1792 x 7168 gives 196 register-operand
# 256x256 tiles, whose contraction order differs from the other kernels'
LINEARS = [(70, 136, 200, 0, 1, 0), (130, 256, 256, 5, 1, 0), (257, 96, 128, 16, 3, 0),
           (300, 512, 320, 64, 1, HI64), (1000, 264, 688, 8, 1, 0), (1792, 7168, 512, 16, 2, 0)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,rank,nseg,flags", LINEARS)
def test_decode_first_linear_gives_the_fused_bits(dev, monkeypatch, tile, M, N, K, rank, nseg,
                                                  flags):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    w = _q4(g, N, K, flags)
    x, dy, res = _rand(g, M, K), _rand(g, M, N), _rand(g, M, N)
    gu, st, P = _rand(g, M, 2 * K), _lib.stream_handle(dev), _lib.ptr
    T = torch.randn(M, nseg * rank, device=dev, generator=g) if rank else None
    B = torch.randn(N, rank, device=dev, generator=g) if rank else None
    A = torch.randn(nseg * rank, K, device=dev, generator=g) if rank else None
    ends = _lib.i64_array([N * (i + 1) // nseg for i in range(nseg)])

    W, ws = w.dequantize(), torch.empty(2 * N * K + 256, dtype=torch.uint8, device=dev)
    start = -ws.data_ptr() % 256

    def call(decode, name, form, *args):
        wa = (P(ws), ws.numel()) if decode else (None, 0)
        ws.fill_(0xA5)
        _lib.call(name, *args, *wa, st)
        # the workspace then holds W's decode, on every tile that the query says
        # it runs on: all but the 64 KiB one with 64 LoRA columns
        need = _lib.query("st_q4_linear_workspace_bytes", form, M, N, K, flags, rank,
                          rank * nseg, -1)
        decodes = decode and not (tile == "128" and rank * nseg == 64)
        assert torch.equal(ws[start:start + 2 * N * K].view(BF).view(N, K), W) == decodes, name
        assert not decode or need == (ws.numel() if decodes else 0), name

    def run(decode):
        monkeypatch.setenv("ST_GEMM_DECODE", str(int(decode)))
        y, dx, dgu = torch.empty_like(dy), torch.empty_like(x), torch.empty_like(gu)
        lf = (P(T), nseg * rank, P(B), rank, 0.5, nseg, ends) if rank else (None, 0, None, 0, 1.0,
                                                                            0, None)
        lb = (P(T), nseg * rank, P(A), nseg * rank) if rank else (None, 0, None, 0)
        call(decode, "st_q4_linear_fwd", _lib.ST_Q4_FWD, P(x), M, K, K, P(w.payload),
             P(w.scales), N, w.lut(), flags, *lf, P(res), N, P(y), N)
        call(decode, "st_q4_linear_dgrad", _lib.ST_Q4_DGRAD, P(dy), M, N, N, P(w.payload),
             P(w.scales), K, w.lut(), flags, *lb, P(dx), K)
        call(decode, "st_q4_linear_dgrad_swiglu", _lib.ST_Q4_DGRAD_SWIGLU, P(dy), M, N, N,
             P(w.payload), P(w.scales), K, w.lut(), flags, *lb, P(gu), 2 * K, P(dgu), 2 * K)
        return y, dx, dgu

    fused = run(False)
    monkeypatch.setenv("ST_GEMM_DMA", tile)
    for name, a, b in zip(("y", "dx", "dgate|up"), fused, run(True)):
        # every sum is the same one; only the fp32 LoRA product, added to the
        # bf16 base, may differ in its last bit (at most one bf16 ulp, rarely)
        off = a != b
        if not rank:
            assert not off.any(), name
        assert off.float().mean() <= 1e-3, name
        assert torch.allclose(a.float(), b.float(), rtol=2 ** -6, atol=1e-2), name


def test_decode_first_rule_and_small_workspace(dev):
    """Many rows decode W once, few rows of a wide matrix do not; a workspace
    below what the query asks for leaves the call on the packed weight."""
    q = _lib.query
    N, K = 4096, 14336
    assert q("st_q4_linear_fwd_workspace_bytes", 2048, N, K) >= 2 * N * K
    assert q("st_q4_linear_dgrad_workspace_bytes", 2048, N, K) >= 2 * N * K
    assert q("st_q4_linear_fwd_workspace_bytes", 256, 28672, 4096) == 0
    g = torch.Generator(device=dev).manual_seed(9)
    M, N, K = 2048, 2048, 1024
    w, x = _q4(g, N, K), _rand(g, M, K)
    ys = []
    for nbytes in (0, 4096, 2 * N * K + 256):
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        y = torch.empty(M, N, dtype=BF, device=dev)
        _lib.call("st_q4_linear_fwd", _lib.ptr(x), M, K, K, _lib.ptr(w.payload),
                  _lib.ptr(w.scales), N, w.lut(), 0, None, 0, None, 0, 1.0, 0, None, None, 0,
                  _lib.ptr(y), N, _lib.ptr(ws), nbytes, _lib.stream_handle(dev))
        ys.append(y)
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])


def test_slot_budget_bounds_the_decoded_weights(dev):
    """A session whose slots take its whole device budget decodes inside the
    GEMMs: the same bits, no scratch of a decoded matrix on the device."""
    from spilltune_amd import codecs, slots
    N, K, M = 4096, 2048, 2103
    host_w = torch.randn(N, K, generator=torch.Generator().manual_seed(1)) * 0.02
    rec = codecs.encode(host_w.to(BF), "nf4-g128")
    name = "self_attn.o_proj.weight"
    host = {f"@{name}/{part}": t for part, t in rec.parts.items()}
    specs = {name: {"spec": rec.spec, "parts": {part: f"@{name}/{part}" for part in rec.parts}}}
    block = slots.BlockPlan(0, "full_attention", None, {}, host, {}, specs)
    g = torch.Generator(device=dev).manual_seed(2)
    x = _rand(g, M, K)
    probe = slots.Q4SlotSession([block], dev, host_budget_bytes=1 << 30,
                                device_budget_bytes=1 << 30)
    got = []
    for budget in (2 * probe.capacity, 1 << 30):
        session = slots.Q4SlotSession([block], dev, host_budget_bytes=1 << 30,
                                      device_budget_bytes=budget)
        with session.run():
            with session.reloader(block).borrow("forward") as views:
                w = views[name]
                assert w.decode_limit == budget - 2 * probe.capacity
                torch.cuda.synchronize()
                torch.cuda.reset_peak_memory_stats(dev)
                before = torch.cuda.memory_allocated(dev)
                y = ops.q4_lora_linear(x, w, None)
                torch.cuda.synchronize()
                got.append((y, torch.cuda.max_memory_allocated(dev) - before))
    (y0, peak0), (y1, peak1) = got
    assert torch.equal(y0, y1)
    assert peak0 < 2 * M * N + (1 << 20) and peak1 - peak0 >= 2 * N * K  # y, and the decoded W
