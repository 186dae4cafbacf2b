"""CPU tests of the C ABI: the library loads, exports every declared symbol, and rejects
invalid arguments with a status (no GPU is touched on these paths)."""

import ctypes as C
import re
from pathlib import Path

import numpy as np
import pytest

from qcom_htp_amd import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "qhtp.h"


def declared_functions():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(qh_[a-z0-9_]+)\s*\(", text)))


def test_header_declarations_match_binding():
    assert declared_functions() == sorted(_lib.EXPORTED)


def test_library_exports_every_declared_symbol(qhtp_lib):
    for name in declared_functions():
        assert hasattr(qhtp_lib, name), name


def test_status_strings(qhtp_lib):
    names = [qhtp_lib.qh_status_string(i).decode() for i in range(5)]
    assert names == ["ok", "invalid_argument", "unsupported", "runtime_error", "shape_unsupported"]
    assert qhtp_lib.qh_status_string(99).decode() == "unknown"
    assert qhtp_lib.qh_version() >= 0x000100


def _desc(**kw):
    w = kw.pop("w", np.zeros((32, 64), np.int8))
    s = kw.pop("s", np.full(32, 0.01, np.float32))
    d = _lib.QmmDesc(k=w.shape[1], n=w.shape[0], act_bits=8, out_bits=8, weight_format=0, lpbq_block=0,
                     act_zp=128, out_zp=0, act_scale=0.02, out_scale=0.05,
                     weight_nk=w.ctypes.data, lpbq_block_scale=None, weight_scale=s.ctypes.data, bias_q=None)
    for k, v in kw.items():
        setattr(d, k, v)
    return d, (w, s)


@pytest.mark.parametrize(
    "field,value,status",
    [
        ("act_bits", 12, _lib.QH_STATUS_UNSUPPORTED),
        ("out_bits", 4, _lib.QH_STATUS_UNSUPPORTED),
        ("weight_format", 7, _lib.QH_STATUS_UNSUPPORTED),
        ("k", 48, _lib.QH_STATUS_SHAPE_UNSUPPORTED),
        ("n", 0, _lib.QH_STATUS_SHAPE_UNSUPPORTED),
        ("act_zp", 300, _lib.QH_STATUS_INVALID_ARGUMENT),
        ("out_scale", 0.0, _lib.QH_STATUS_INVALID_ARGUMENT),
        ("act_scale", float("nan"), _lib.QH_STATUS_INVALID_ARGUMENT),
        ("weight_nk", None, _lib.QH_STATUS_INVALID_ARGUMENT),
    ],
)
def test_prepare_rejects_invalid_descriptors(qhtp_lib, field, value, status):
    d, keep = _desc(**{field: value})
    h = C.c_void_p()
    assert qhtp_lib.qh_qmm_prepare(C.byref(d), C.byref(h)) == status
    assert h.value is None
    assert qhtp_lib.qh_last_error().decode() != ""


def test_prepare_rejects_out_of_range_codes(qhtp_lib):
    w = np.zeros((32, 64), np.int8)
    w[3, 5] = -128
    d, keep = _desc(w=w)
    h = C.c_void_p()
    assert qhtp_lib.qh_qmm_prepare(C.byref(d), C.byref(h)) == _lib.QH_STATUS_INVALID_ARGUMENT
    assert "outside" in qhtp_lib.qh_last_error().decode()
    w = np.full((32, 64), 8, np.int8)  # int4 codes must be within [-7, 7]
    d, keep = _desc(w=w, weight_format=_lib.QH_WEIGHT_I4)
    assert qhtp_lib.qh_qmm_prepare(C.byref(d), C.byref(h)) == _lib.QH_STATUS_INVALID_ARGUMENT


def test_prepare_rejects_bad_lpbq(qhtp_lib):
    w = np.zeros((32, 128), np.int8)
    blk = np.zeros((32, 4), np.uint8)  # factor 0 is outside [1, 16]
    d, keep = _desc(w=w, weight_format=_lib.QH_WEIGHT_I4_LPBQ, lpbq_block=32, lpbq_block_scale=blk.ctypes.data)
    h = C.c_void_p()
    assert qhtp_lib.qh_qmm_prepare(C.byref(d), C.byref(h)) == _lib.QH_STATUS_INVALID_ARGUMENT
    d, keep = _desc(w=w, weight_format=_lib.QH_WEIGHT_I4_LPBQ, lpbq_block=48, lpbq_block_scale=blk.ctypes.data)
    assert qhtp_lib.qh_qmm_prepare(C.byref(d), C.byref(h)) == _lib.QH_STATUS_UNSUPPORTED


def test_run_rejects_null_and_bad_shapes(qhtp_lib):
    L = qhtp_lib
    assert L.qh_qmm_run(None, 4, 16, 16, None) == _lib.QH_STATUS_INVALID_ARGUMENT
    assert L.qh_qmm_accumulate(None, 4, 16, 16, None) == _lib.QH_STATUS_INVALID_ARGUMENT
    assert L.qh_qmm_query(None, None) == _lib.QH_STATUS_INVALID_ARGUMENT
    assert L.qh_qmm_release(None) == _lib.QH_STATUS_OK
    # GDN: C not a multiple of 16 / too large / zero heads / NULL
    assert L.qh_gdn_solve_f32(16, 16, 1, 40, 0, None) == _lib.QH_STATUS_SHAPE_UNSUPPORTED
    assert L.qh_gdn_solve_f32(16, 16, 1, 512, 0, None) == _lib.QH_STATUS_SHAPE_UNSUPPORTED
    assert L.qh_gdn_solve_f32(16, 16, 0, 64, 0, None) == _lib.QH_STATUS_SHAPE_UNSUPPORTED
    assert L.qh_gdn_solve_f32(None, 16, 1, 64, 0, None) == _lib.QH_STATUS_INVALID_ARGUMENT
    assert L.qh_gdn_solve_f32(16, 16, 1, 64, 5, None) == _lib.QH_STATUS_UNSUPPORTED
    assert L.qh_gdn_solve_u16(16, 16, 1, 64, 70000, 0, 1.0, 1.0, 0, None) == _lib.QH_STATUS_INVALID_ARGUMENT
    assert L.qh_gdn_solve_u16(16, 16, 1, 64, 0, 0, 0.0, 1.0, 0, None) == _lib.QH_STATUS_INVALID_ARGUMENT
    assert L.qh_gdn_solve_u16(8, 16, 1, 64, 0, 0, 1.0, 1.0, 0, None) == _lib.QH_STATUS_INVALID_ARGUMENT


def test_gdn_prefill_rejects_bad_arguments(qhtp_lib):
    """Every refusal comes before a launch (the buffers are made-up addresses)."""
    L, INV, UNS, SHP = qhtp_lib, _lib.QH_STATUS_INVALID_ARGUMENT, _lib.QH_STATUS_UNSUPPORTED, _lib.QH_STATUS_SHAPE_UNSUPPORTED
    B, T, H = 4, 100, 32  # more sequences than any device runs on the route of few
    need = L.qh_gdn_prefill_workspace(B, T, H, _lib.QH_GDN_FP32)
    assert need == B * H * 2 * 2 * 64 * 64 * 2  # two chunks' T, hi and lo parts
    assert L.qh_gdn_prefill_workspace(B, T, H, _lib.QH_GDN_BF16) == need // 2
    names = ("q", "k", "v", "g", "beta", "s_in", "s_out", "o", "batch", "tokens", "heads", "head_dim", "flags", "precision", "ws",
             "ws_bytes", "stream")
    good = dict(zip(names, (4096, 4096, 4096, 4096, 4096, 0, 8192, 4096, B, T, H, 128, 0, 0, 16384, need, None)))
    bad = [(dict([(p, None)]), INV) for p in ("q", "k", "v", "g", "beta", "s_out", "o", "ws")]
    bad += [(dict([(p, 4104)]), INV) for p in ("q", "k", "v", "s_in", "s_out", "o", "ws")]
    bad += [({"s_in": 8192}, INV), ({"ws_bytes": need - 1}, INV), ({"ws_bytes": 0}, INV), ({"head_dim": 64}, SHP),
            ({"flags": _lib.QH_GDN_RAGGED}, UNS), ({"flags": _lib.QH_GDN_WU_F32}, UNS), ({"flags": 1 << 31}, UNS),
            ({"precision": _lib.QH_GDN_OP_MODEL}, UNS), ({"batch": 0}, SHP), ({"tokens": 0}, SHP), ({"heads": 0}, SHP),
            ({"tokens": 1 << 24}, SHP), ({"batch": 1 << 31, "heads": 1 << 31}, SHP)]
    for change, status in bad:
        args = {**good, **change}
        assert L.qh_gdn_prefill(*(args[n] for n in names)) == status, change
        assert L.qh_last_error().decode().startswith("qh_gdn_prefill")


def test_gdn_chunk_rejects_bad_ragged_and_workspace_arguments(qhtp_lib):
    L, INV, UNS, SHP = qhtp_lib, _lib.QH_STATUS_INVALID_ARGUMENT, _lib.QH_STATUS_UNSUPPORTED, _lib.QH_STATUS_SHAPE_UNSUPPORTED
    uw = lambda T, chunk, flags: L.qh_gdn_chunk_uw(4096, 4096, 4096, 4096, 4096, 4096, 1, T, 1, 128, chunk, flags, None)  # noqa: E731
    assert uw(100, 64, 0) == SHP
    assert uw(0, 64, _lib.QH_GDN_RAGGED) == SHP
    assert uw(100, 128, _lib.QH_GDN_RAGGED) == UNS and uw(256, 256, _lib.QH_GDN_RAGGED) == UNS

    def state(T=64, flags=0, s_in=0, ws=0, ws_bytes=0, chunk=64):
        return L.qh_gdn_chunk_state_ws(4096, 4096, 4096, 4096, 4096, s_in, 8192, 4096, 1, T, 1, 128, chunk, flags, 0, ws, ws_bytes, None)

    assert state(T=100) == SHP and state(T=0, flags=_lib.QH_GDN_RAGGED) == SHP
    assert state(T=100, flags=_lib.QH_GDN_RAGGED, chunk=128) == SHP
    assert state(s_in=8192) == INV and state(ws=4104, ws_bytes=1 << 20) == INV
    assert state(flags=_lib.QH_GDN_W_DECAY) == UNS
    for query in (L.qh_gdn_chunk_state_workspace, L.qh_gdn_prefill_workspace):
        assert query(0, 64, 1, 0) == 0 and query(1, 0, 1, 0) == 0 and query(1, 64, 0, 0) == 0
        assert query(1 << 12, 1 << 12, 2, 0) == 0  # batch * tokens * heads over 2^24


def test_gdn_sizes_whose_product_wraps_are_refused(qhtp_lib):
    """batch * tokens * heads of these is 2^64 + 10 and 2^64."""
    L, SHP = qhtp_lib, _lib.QH_STATUS_SHAPE_UNSUPPORTED
    for B, T, H in ((21398, 289529, 2977518503), (289529, 2977518503, 21398), (1 << 24, 1 << 16, 1 << 24)):
        for precision in (0, 1):
            assert L.qh_gdn_prefill_workspace(B, T, H, precision) == 0
            assert L.qh_gdn_chunk_state_workspace(B, T, H, precision) == 0
        p = 4096
        assert L.qh_gdn_prefill(p, p, p, p, p, 0, 8192, p, B, T, H, 128, 0, 0, p, 1 << 62, None) == SHP
        assert L.qh_gdn_chunk_uw(p, p, p, p, p, p, B, T, H, 128, 64, _lib.QH_GDN_RAGGED, None) == SHP
        assert L.qh_gdn_chunk_state(p, p, p, p, p, 0, 8192, p, B, T, H, 128, 64, _lib.QH_GDN_RAGGED, 0, None) == SHP


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "libqhtp.so")
    monkeypatch.setattr(_lib, "_lib", None)
    with pytest.raises(RuntimeError, match="no fallback"):
        _lib.lib()
