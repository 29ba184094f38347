"""Host-side logic of the differentiable ops that runs before any kernel
(CPU only): when fused projections may share one weight view, and the
terminal's label rules (native_terminal.py:39-47: device labels are never
scanned on the host)."""
import threading

import pytest
import torch

from spilltune_amd import _lib, ops


def _q4(payload, scales, rows, K=128):
    return ops.Q4Weight(payload, scales, (rows, K), "nf4-g128")


def test_concat_rows_views_one_storage():
    rows = (64, 32)
    K = 128
    pay = torch.zeros(sum(rows) * K // 2, dtype=torch.uint8)
    sc = torch.ones(sum(rows) * K // 128, dtype=torch.float32)
    a = _q4(pay[:rows[0] * K // 2], sc[:rows[0]], rows[0])
    b = _q4(pay[rows[0] * K // 2:], sc[rows[0]:], rows[1])
    fused = ops.concat_rows([a, b])
    assert fused is not None and fused.shape == (96, K) and fused.segments == rows
    assert fused.payload.data_ptr() == pay.data_ptr() and fused.payload.numel() == pay.numel()
    assert fused.scales.numel() == sc.numel()


def test_concat_rows_rejects_adjacent_separate_allocations():
    """Two allocations that lie back to back in memory are not one buffer:
    the fused view would run off the first storage."""
    K = 128
    raw_p = bytearray(96 * K // 2)
    raw_s = bytearray(96 * K // 128 * 4)
    pa = torch.frombuffer(raw_p, dtype=torch.uint8, count=64 * K // 2, offset=0)
    pb = torch.frombuffer(raw_p, dtype=torch.uint8, count=32 * K // 2, offset=64 * K // 2)
    sa = torch.frombuffer(raw_s, dtype=torch.float32, count=64, offset=0)
    sb = torch.frombuffer(raw_s, dtype=torch.float32, count=32, offset=64 * 4)
    assert pa.data_ptr() + pa.numel() == pb.data_ptr()          # adjacent pointers ...
    assert pa.untyped_storage().data_ptr() != pb.untyped_storage().data_ptr()  # ... two storages
    assert ops.concat_rows([_q4(pa, sa, 64), _q4(pb, sb, 32)]) is None
    # one storage but a gap between the parts is not adjacent either
    pay = torch.zeros(100 * K // 2, dtype=torch.uint8)
    sc = torch.ones(100, dtype=torch.float32)
    a = _q4(pay[:64 * K // 2], sc[:64], 64)
    b = _q4(pay[68 * K // 2:], sc[68:], 32)
    assert ops.concat_rows([a, b]) is None


def test_terminal_device_labels_need_prepared_chunks():
    normalized = torch.zeros(1, 8, 16, dtype=torch.bfloat16, device="meta")
    head = torch.zeros(32, 16, dtype=torch.bfloat16, device="meta")
    labels = torch.zeros(1, 8, dtype=torch.int64, device="meta")
    with pytest.raises(RuntimeError, match="prepared supervised chunks"):
        ops.chunked_causal_loss(normalized, head, labels, normalization=7.0, token_chunk=4)
    with pytest.raises(RuntimeError, match="host labels"):
        ops.supervised_chunk_intervals(labels, 4)


def test_supervised_chunk_intervals_host_rule():
    labels = torch.full((2, 10), -100)
    labels[1, 6] = 3                       # only the target of position 5 is supervised
    assert ops.supervised_chunk_intervals(labels, 4) == ((4, 8),)
    with pytest.raises(ValueError, match="token chunk"):
        ops.supervised_chunk_intervals(labels, 0)


def test_router_parts_sum_exactly_and_follow_the_version():
    """The fp32 router's bf16 parts [hi; mid; lo] (the operand of its input
    gradient on the rank-r kernel) sum back to every fp32 value exactly,
    including values far from 1 and with low-order bits set; they are kept
    on the tensor and remade only after an in-place change (version)."""
    from spilltune_amd import moe
    g = torch.Generator().manual_seed(5)
    E, H = 8, 96
    w = torch.randn(E, H, generator=g) * torch.exp2(torch.randint(-30, 30, (E, H), generator=g).float())
    w[0, :4] = torch.tensor([1.0 + 2 ** -23, -(2 - 2 ** -22), 2 ** -100, 3.0e20])
    parts = moe._router_parts(w)
    assert parts.shape == (3 * E, H) and parts.dtype == torch.bfloat16
    back = parts[:E].double() + parts[E:2 * E].double() + parts[2 * E:].double()
    assert torch.equal(back, w.double())
    assert moe._router_parts(w) is parts  # unchanged tensor: the kept split
    w.mul_(0.5)
    again = moe._router_parts(w)
    assert again is not parts
    back = again[:E].double() + again[E:2 * E].double() + again[2 * E:].double()
    assert torch.equal(back, w.double())


def test_stream_handle_takes_what_current_stream_takes(monkeypatch):
    """A torch.device, its name, an index or nothing; only CUDA devices."""
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 1000 + i, raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 7)
    h = _lib.stream_handle
    assert h() == h(None) == h("cuda") == h(torch.device("cuda")) == 1007
    assert h(2) == h("cuda:2") == h(torch.device("cuda", 2)) == 1002
    for bad in ("cpu", torch.device("cpu")):
        with pytest.raises(ValueError, match="cuda device"):
            h(bad)


def test_gemm_scratch_is_bounded(monkeypatch):
    """Decoded weights stay within the weight's limit (the tighter one of a
    concatenation), and give way when the device has no room; split-K partials
    do not (without them the sums run in another order)."""
    empty = torch.empty(0, dtype=torch.uint8)
    N, K = 4096, 14336
    decode = 2 * N * K + 256

    def scratch(form, M, limit=None):
        ws = ops._gemm_scratch(ops.Q4Weight(empty, empty, (N, K), "nf4-g128", decode_limit=limit),
                               form, M, 0, 0)
        return 0 if ws is None else ws.numel()
    split = scratch(_lib.ST_Q4_DGRAD, 256)
    assert scratch(_lib.ST_Q4_FWD, 2048) == decode != split > 0
    assert scratch(_lib.ST_Q4_FWD, 2048, decode) == decode
    assert scratch(_lib.ST_Q4_FWD, 2048, decode - 1) == scratch(_lib.ST_Q4_FWD, 2048, 0) == 0
    assert scratch(_lib.ST_Q4_FWD, 2048, -5) == 0
    assert scratch(_lib.ST_Q4_DGRAD, 256, 0) == split

    payload, scales = torch.zeros(128 * 64, dtype=torch.uint8), torch.zeros(128)
    a, b = (_q4(payload[i * 4096:], scales[i * 64:], 64) for i in (0, 1))
    a.payload, a.scales = payload[:4096], scales[:64]
    assert ops.concat_rows([a, b]).decode_limit is None
    a.decode_limit, b.decode_limit = None, 7
    assert ops.concat_rows([a, b]).decode_limit == 7
    a.decode_limit = 3
    assert ops.concat_rows([a, b]).decode_limit == 3

    def full(*args, **kwargs):
        raise torch.OutOfMemoryError("full")
    monkeypatch.setattr(torch, "empty", full)
    assert scratch(_lib.ST_Q4_FWD, 2048) == 0
    with pytest.raises(torch.OutOfMemoryError):
        scratch(_lib.ST_Q4_DGRAD, 256)


def test_calls_in_flight_do_not_share_scratch(monkeypatch):
    """Two calls that overlap (two threads or two streams) get workspaces of
    their own: the second must not write its partials over the first's."""
    barrier, seen = threading.Barrier(2, timeout=30), []

    def call(name, *args):
        seen.append((args[-3], args[-2]))  # workspace and its size; the stream is last
        barrier.wait()  # both calls have their workspace in hand
    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(_lib, "stream_handle", lambda device=None: 0)
    x, A, T = torch.zeros(64, 2048), torch.zeros(8, 2048), torch.zeros(64, 8)
    assert _lib.query("st_lora_gemm_workspace_bytes", 64, 8, 2048) > 0
    for _ in range(2):  # also with a buffer that an earlier call left behind
        threads = [threading.Thread(target=ops.lora_gemm,
                                    args=(64, 8, 2048, x, 2048, 1, A, 1, 2048, 1.0, T))
                   for _ in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    for (a, size), (b, _) in (seen[:2], seen[2:]):
        assert abs(a - b) >= size > 0
