"""The C ABI: the built library loads and exports every declared symbol (CPU).

No compute call is made here (no GPU); the GPU tests call through the same
entry points.
"""

from __future__ import annotations

import ctypes
import importlib

import torch
import re
from pathlib import Path

import pytest

from maple_amd import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "maple_amd.h"


def declared_in_header() -> list[str]:
    text = HEADER.read_text()
    return sorted(set(re.findall(r"\b(ma_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_path():
    names = declared_in_header()
    for must in ("ma_ternary_gemv", "ma_router_topk", "ma_moe_dispatch", "ma_ternary_expert_swiglu",
                 "ma_ternary_expert_gemv", "ma_ternary_expert_down_sum", "ma_moe_reduce_add",
                 "ma_rtn4_gemv", "ma_rtn4_embedding", "ma_rms_norm", "ma_add_rms_norm"):
        assert must in names


def test_library_exports_every_declared_symbol():
    if not _lib.LIB_PATH.exists():
        pytest.fail(f"{_lib.LIB_PATH} not built; run __graft_entry__.build()")
    lib = ctypes.CDLL(str(_lib.LIB_PATH))
    missing = [n for n in declared_in_header() if not hasattr(lib, n)]
    assert not missing, f"declared but not exported: {missing}"


def test_binding_covers_header():
    assert set(declared_in_header()) <= set(_lib.declared_symbols())


def test_version_and_error_string():
    lib = _lib.load()
    assert lib.ma_version() >= 100
    assert isinstance(lib.ma_last_error(), bytes)


def test_size_errors_map_without_a_gpu():
    """Bad sizes are rejected on the host before any launch: status -> ValueError."""
    with pytest.raises(ValueError, match="bad sizes"):
        _lib.call("ma_ternary_gemv", None, 1, -1, 16, None, 4, 1, 0, None, 0, None, 0, 1e-6,
                  None, 4, None)
    with pytest.raises(ValueError, match="top_k"):
        _lib.call("ma_router_topk", None, 1, 1, 16, None, 1, 4, 16, None, 5, None, None, None, 0, None)
    with pytest.raises(ValueError, match="n_experts"):
        _lib.call("ma_moe_dispatch", None, 0, 8, 0, None, None, None, None, None)
    with pytest.raises(ValueError, match="groups"):
        _lib.call("ma_rtn4_gemv", None, 1, 1, 96, None, 4, 12, 0, None, 1, None, 1, 64, None, 4, None)
    # 2^22 tokens x hidden 2048: x' holds 2^32 uint32 words, past the batched
    # kernels' 32-bit copy offsets (rejected before any launch; the pointers
    # are never dereferenced)
    fake = 0x10000
    with pytest.raises(ValueError, match="split the batch"):
        _lib.call("ma_moe_grouped", fake, 2048, None, None, 1 << 22, 8, fake, fake, fake, fake,
                  _lib.dtype_code(torch.empty(0, dtype=torch.bfloat16), "a"), 64, 2048, 768, fake, fake,
                  fake, fake, None, 0, None, 0, fake, fake, 1 << 62, None)


@pytest.mark.parametrize("rms", [0, 1])
def test_ternary_gemv_call_workspace_is_what_the_call_uses(rms):
    """The scaled 8-bit form's bytes only for calls it takes (from 64 tokens, past
    4 x 2^16 outputs); below, the two-launch RMS form's, or none; never above the
    query that does not know the rows."""
    lib = _lib.load()
    call, most = lib.ma_ternary_gemv_call_workspace_bytes, lib.ma_ternary_gemv_workspace_bytes
    for batch in (1, 16, 17, 63, 64, 65, 127, 128, 2048):
        for n_out in (8, 2048, 2049, 4096, 4097, 5120):
            used = call(batch, n_out, 128, rms)
            assert used <= most(batch, 128, rms)
            if batch >= 64 and batch * n_out > 4 * 65536:
                assert used == most(batch, 128, rms) > 0
            else:
                assert (used > 0) == (rms == 1 and batch >= 17)
    assert call(2048, 5120, 120, rms) == 0


def test_ternary_gemv_takes_no_workspace_it_does_not_use(monkeypatch):
    """The wrapper allocates by that query (the launch is a stand-in): 64 tokens x
    2048 rows without the RMSNorm go to ma_ternary_gemv, 64 x 5120 to the
    workspace entry; float16 x, which no workspace form takes, to the first."""
    mod = importlib.import_module("maple_amd.kernels.ternary_gemv")  # (the package has a function of that name)
    called = []
    monkeypatch.setattr(mod._lib, "call", lambda name, *args: called.append(name))
    monkeypatch.setattr(mod._lib, "stream_of", lambda t: None)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda self: True))
    for rows, dtype in ((2048, torch.bfloat16), (5120, torch.bfloat16), (5120, torch.float16)):
        mod.ternary_gemv(torch.zeros(64, 2048, dtype=dtype), torch.zeros(rows, 128, dtype=torch.uint32),
                         torch.ones(rows, dtype=torch.bfloat16))
    assert called == ["ma_ternary_gemv", "ma_ternary_gemv_ws", "ma_ternary_gemv"]


def test_rtn4_gemv_mx_rejects_null_pointers_without_a_gpu():
    """A null x, codes, scales, biases or y is refused on the host: null passes the
    alignment checks, and the launch would have read it."""
    fake, bf16 = 0x10000, _lib.BF16
    nbytes = _lib.load().ma_rtn4_gemv_mx_workspace_bytes(8, 256, 128)
    for null in range(5):
        x, w, sc, bs, y = (None if i == null else fake for i in range(5))
        with pytest.raises(ValueError, match="null pointer"):
            _lib.call("ma_rtn4_gemv_mx", x, bf16, 8, 2048, w, 128, 256, 0, sc, bf16, bs, bf16, 128, y, 128, fake,
                      nbytes, None)


@pytest.mark.parametrize("batch", [5, 16, 17, 256])
def test_rtn4_gemv_mx_workspace_covers_the_calls_it_passes_on(batch):
    """The query's bytes hold the scaled form's rows and, for every K in groups of
    128, those of ma_rtn4_gemv_ws too, which takes K a multiple of 128 but not of
    256; no other shape uses a workspace."""
    lib = _lib.load()
    for nwords in range(16, 1025, 16):
        ws, mx = (int(f(batch, nwords, 128)) for f in (lib.ma_rtn4_gemv_workspace_bytes,
                                                       lib.ma_rtn4_gemv_mx_workspace_bytes))
        assert mx >= ws > 0 and (nwords % 32 == 0 or mx == ws)
    assert lib.ma_rtn4_gemv_mx_workspace_bytes(batch, 80, 64) == 0
    assert lib.ma_rtn4_gemv_mx_workspace_bytes(4, 256, 128) == 0


def test_stamped_variant_exports_the_same_symbols_and_its_stamps_fit():
    """libmaple_amd_stamps.so (the one-launch layer with phase stamps) exports
    everything the header declares; only it reports a stamp layout, and the
    stamp rows lie inside the workspace ma_moe_fused_workspace_bytes sizes."""
    if not _lib.STAMPED_LIB_PATH.exists():
        pytest.fail(f"{_lib.STAMPED_LIB_PATH} not built; run __graft_entry__.build()")
    st = ctypes.CDLL(str(_lib.STAMPED_LIB_PATH))
    missing = [n for n in declared_in_header() if not hasattr(st, n)]
    assert not missing, f"declared but not exported: {missing}"
    off, words, wgs = ctypes.c_size_t(), ctypes.c_int(), ctypes.c_int()
    fn = st.ma_moe_phase_stamps
    fn.argtypes = [ctypes.c_void_p] * 3
    assert fn(ctypes.byref(off), ctypes.byref(words), ctypes.byref(wgs)) == 0
    assert words.value == 16 and wgs.value == 256 and off.value % 256 == 0
    size = st.ma_moe_fused_workspace_bytes
    size.argtypes = [ctypes.c_int64] * 4
    size.restype = ctypes.c_size_t
    for inter in (768, 512):
        assert off.value + 4 * words.value * wgs.value <= size(64, 2048, inter, 8)
    plain = _lib.load()
    assert plain.ma_moe_phase_stamps(ctypes.byref(off), ctypes.byref(words), ctypes.byref(wgs)) != 0
