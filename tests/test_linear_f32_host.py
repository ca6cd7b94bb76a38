"""Argument checks of the split fp32 product's entry point (no GPU): every call here is
one the library answers before any HIP call."""

import ctypes

from kla.ops.hip import _lib


def test_linear_f32_validation():
    """kla_linear_f32_fwd checks sizes, strides, options, alignment and workspace before any launch."""
    lib = _lib.lib()
    P, WS = 0x7F0000000000, 0x7F0000100000
    fine = dict(epilogue=_lib.KLA_ROWS_PLAIN, x=P, ldx=64, w=P, ldw=64, y=P, ldy=80, rows=300, n=80, k=64)

    def call(ws=WS, nbytes=1 << 40, **over):
        args = _lib.LinearF32(**{**fine, **over})
        return lib.kla_linear_f32_fwd(ctypes.byref(args), ws, nbytes, None)

    assert lib.kla_linear_f32_fwd(None, WS, 1 << 40, None) == _lib.KLA_ERR_INVALID_ARG
    assert call(rows=0) == _lib.KLA_OK and call(n=0) == _lib.KLA_OK
    residual, swiglu = {"epilogue": _lib.KLA_ROWS_RESIDUAL}, {"epilogue": _lib.KLA_ROWS_SWIGLU}
    for bad in ({"rows": -1}, {"n": -1}, {"k": 0}, {"x": None}, {"w": None}, {"y": None}, {"ldx": 63}, {"ldw": 63},
                {"ldy": 79}, {"epilogue": 7}, residual, {**residual, "res": P, "ldres": 79}, {**swiglu, "glu_off": 79}):
        assert call(**bad) == _lib.KLA_ERR_INVALID_ARG, bad
    assert call(x=P + 2) == _lib.KLA_ERR_ALIGN and call(norm_w=P + 1) == _lib.KLA_ERR_ALIGN
    need = lib.kla_linear_f32_workspace_bytes(300, 80, 64, _lib.KLA_ROWS_PLAIN)
    assert need == (10 + 3) * (2 * 4096 + 128)      # 32-row blocks x (two 32-wide chunks and the row exponents)
    assert lib.kla_linear_f32_workspace_bytes(300, 80, 64, _lib.KLA_ROWS_SWIGLU) == (10 + 6) * (2 * 4096 + 128)
    for bad in ({"ws": None}, {"ws": WS + 8}, {"nbytes": need - 1}):
        assert call(**bad) == _lib.KLA_ERR_WORKSPACE, bad
    huge = 2**62
    assert lib.kla_linear_f32_workspace_bytes(huge, huge, huge, 0) == 0
    refused = (_lib.KLA_ERR_WORKSPACE, _lib.KLA_ERR_INVALID_ARG)
    assert call(rows=huge) in refused and call(rows=2**40, n=2**40, ldy=2**40, nbytes=2**61) in refused
