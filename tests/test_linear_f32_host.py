"""Argument checks of the split fp32 product's entry point (no GPU): every call here is
one the library answers before any HIP call."""

import ctypes

from kla.ops.hip import _lib
from kla.ops.hip import linear as lin


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


# (rows, n, k), split product and library in us on MI355X (one graph of six calls each),
# where the GPU's time counts (rows * k of 2^22 and more).
TIMED = [((2048, 96, 2048), 38.1, 12.8), ((2048, 160, 2048), 37.8, 20.4), ((4096, 64, 1024), 22.7, 9.5),
         ((4096, 96, 1024), 23.0, 15.7), ((4096, 64, 2048), 38.1, 14.1), ((8192, 64, 512), 17.8, 8.3),
         ((8192, 96, 2048), 59.0, 29.1), ((8192, 160, 1024), 36.7, 25.7), ((8192, 160, 2048), 66.6, 45.8),
         ((4096, 512, 1365), 41.5, 51.7), ((4096, 2048, 1024), 70.3, 142.1), ((8188, 1024, 2048), 136.9, 256.1),
         ((8188, 4096, 1024), 214.8, 514.6)]


def test_the_rule_takes_what_was_measured_the_faster():
    for (rows, n, k), split, library in TIMED:
        assert lin.f32_pays(rows, n, k, False) == (split < library), (rows, n, k)
        if split < library:
            assert lin.f32_pays(rows, n, k, True)
    # Narrow products of long rows (low-rank sensors): never where the GPU's time counts.
    for rows in (2048, 4096, 5000, 8192):
        for n in (48, 64, 96, 128, 160):
            for k in (1536, 2048):
                assert lin.f32_pays(rows, n, k, False) == (rows * k < 1 << 22), (rows, n, k)
    # Where the host's does, the call that takes less of it.
    assert lin.f32_pays(256, 64, 1024, False) and lin.f32_pays(2048, 512, 1024, False)
