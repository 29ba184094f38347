"""The C ABI library loads, exports exactly what include/spilltune_hip.h
declares, and rejects bad arguments before touching the device (CPU only)."""
import ctypes
import re
from pathlib import Path

import pytest

from spilltune_amd import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "spilltune_hip.h"


def declared_symbols():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(st_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    names = declared_symbols()
    assert len(names) >= 20
    for name in names:
        assert hasattr(lib, name), name
    assert sorted(_lib.EXPORTED) == names


def test_abi_version_and_error_mapping():
    lib = _lib.load()
    assert lib.st_abi_version() == 1
    lut = _lib.lut_array(range(16))
    with pytest.raises(ValueError, match="group must be 64 or 128"):
        _lib.call("st_dequant4", None, None, 10, 96, lut, 0, None, None)
    with pytest.raises(ValueError, match="NULL"):
        _lib.call("st_dequant4", None, None, 10, 128, lut, 0, None, None)
    # zero-size work is a no-op that succeeds without a device
    _lib.call("st_dequant4", None, None, 0, 128, lut, 0, None, None)
    with pytest.raises(ValueError, match="multiple of 8"):
        _lib.call("st_q4_linear_dgrad", ctypes.c_void_p(16), 4, 100, 100, ctypes.c_void_p(16),
                  ctypes.c_void_p(16), 128, lut, 0, None, 0, None, 0, ctypes.c_void_p(16), 128,
                  None, 0, None)
    with pytest.raises(ValueError, match="dtype codes"):
        _lib.call("st_lora_gemm", 4, 4, 4, ctypes.c_void_p(16), 7, 1, 1, ctypes.c_void_p(16), 0,
                  1, 1, 1.0, ctypes.c_void_p(16), 4, 0, None, 0, None)


def test_lut_array_keeps_the_sign_of_zero():
    """Codebooks that are equal as numbers but not in their bits each get
    their own table, in either order; equal bits share one."""
    pos = [0.0] + [0.5] * 15
    neg = [-0.0] + [0.5] * 15
    for values, sign in ((pos, "0000"), (neg, "8000"), (pos, "0000")):
        assert bytes(_lib.lut_array(values))[:4][::-1].hex() == sign + "0000"
    assert bytes(_lib.lut_array(range(16))) == bytes((ctypes.c_float * 16)(*range(16)))


def test_linear_workspace_query_knows_the_call():
    """The workspace that is asked for is one the call would use."""
    def q(form, M, N, K, flags=0, rank=0, cols=0, limit=-1):
        return _lib.query("st_q4_linear_workspace_bytes", form, M, N, K, flags, rank, cols, limit)
    fwd, dgrad, swiglu = _lib.ST_Q4_FWD, _lib.ST_Q4_DGRAD, _lib.ST_Q4_DGRAD_SWIGLU
    g64 = _lib.ST_FLAG_GROUP64
    down = (4096, 14336)  # [N, K]
    assert q(fwd, 2048, *down) == q(fwd, 2048, *down, rank=16, cols=16) == 2 * 4096 * 14336 + 256
    # the SwiGLU form never splits the contraction: no partials, decode or nothing
    assert 0 < q(dgrad, 256, *down) != 2 * 4096 * 14336 + 256
    assert q(swiglu, 256, *down) in (0, 2 * 4096 * 14336 + 256)
    # 64-element groups do not straddle rows of 1088, 128-element groups do
    assert q(fwd, 300, 8000, 1088, flags=g64) == 0 < q(fwd, 1000, 8000, 1088)
    # more LoRA columns than any tile holds beside the DMA rings
    assert q(fwd, 2048, *down, rank=128, cols=128) == 0
    assert q(dgrad, 2048, *down, rank=192, cols=192) == 0
    assert q(fwd, 2048, *down, limit=2 * 4096 * 14336 + 255) == 0
    assert q(fwd, 2048, *down, limit=2 * 4096 * 14336 + 256) > 0
    assert q(3, 2048, *down) == q(-1, 2048, *down) == q(fwd, 0, *down) == 0


def test_lora_rank_limits_rejected_before_any_launch():
    """Rank bounds of the LoRA entry points: checked on the host, before any
    device work (fake pointers never reach a kernel)."""
    lut = _lib.lut_array(range(16))
    p = ctypes.c_void_p(16)
    ends = _lib.i64_array([256])

    def fwd(rank):
        _lib.call("st_q4_linear_fwd", p, 4, 256, 256, p, p, 256, lut, 0, p, 256, p, rank, 1.0, 1,
                  ends, None, 0, p, 256, None, 0, None)
    for rank in (0, -3, 70000):
        with pytest.raises(ValueError, match="out of range"):
            fwd(rank)
    # the batched dY-side products take r <= 64: the query says so with 0
    assert _lib.query("st_lora_bwd_dy_workspace_bytes", 2048, 4096, 16, 1, _lib.i64_array([4096])) > 0
    assert _lib.query("st_lora_bwd_dy_workspace_bytes", 2048, 4096, 65, 1, _lib.i64_array([4096])) == 0
    with pytest.raises(ValueError, match="rank must be 1..64"):
        _lib.call("st_lora_bwd_dy", p, 4, 256, 256, p, p, 65, 65, 1, ends, 1.0, p, 65, None, p,
                  1 << 20, None)
    with pytest.raises(ValueError, match="0 < R"):
        _lib.call("st_moe_lora_rows", 4, 0, 256, 1, p, 256, 4, None, p, 1, 256, 0, p, 1, 1.0, p,
                  1, None)


def test_workspace_queries():
    assert _lib.query("st_q4_linear_fwd_workspace_bytes", 16, 256, 4096) == 0
    # K % 128 != 0 runs on the flat-group kernels from the packed weight
    assert _lib.query("st_q4_linear_fwd_workspace_bytes", 16, 256, 688) == 0
    assert _lib.query("st_q4_linear_dgrad_workspace_bytes", 16, 256, 688) == 0
    ws = _lib.query("st_lora_gemm_workspace_bytes", 2048, 16, 4096)
    assert ws > 0 and ws % (2048 * 16 * 4) == 0


def test_product_does_not_import_the_oracle():
    root = Path(__file__).resolve().parents[1] / "spilltune_amd"
    for path in root.rglob("*.py"):
        src = path.read_text()
        assert "import oracle" not in src and "from oracle" not in src, path
