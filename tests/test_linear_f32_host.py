"""Argument checks of the split fp32 product's entry point (no GPU): every call here is
one the library answers before any HIP call."""

from kla.ops.hip import _lib


def test_linear_f32_validation():
    """kla_linear_f32_fwd checks sizes, strides, alignment and workspace before any launch."""
    lib = _lib.lib()
    P, WS = 0x7F0000000000, 0x7F0000100000

    def call(x=P, ldx=64, w=P, ldw=64, y=P, ldy=80, rows=300, n=80, k=64, ws=WS, nbytes=1 << 40):
        return lib.kla_linear_f32_fwd(x, ldx, w, ldw, None, y, ldy, rows, n, k, ws, nbytes, None)

    assert call(rows=0) == _lib.KLA_OK and call(n=0) == _lib.KLA_OK
    for bad in ({"rows": -1}, {"n": -1}, {"k": 0}, {"x": None}, {"w": None}, {"y": None}, {"ldx": 63}, {"ldw": 63},
                {"ldy": 79}):
        assert call(**bad) == _lib.KLA_ERR_INVALID_ARG, bad
    assert call(x=P + 2) == _lib.KLA_ERR_ALIGN
    need = lib.kla_linear_f32_workspace_bytes(300, 80, 64)
    assert need == (10 + 3) * (2 * 4096 + 128)      # 32-row blocks x (two 32-wide chunks and the row exponents)
    for bad in ({"ws": None}, {"ws": WS + 8}, {"nbytes": need - 1}):
        assert call(**bad) == _lib.KLA_ERR_WORKSPACE, bad
    huge = 2**62
    assert lib.kla_linear_f32_workspace_bytes(huge, huge, huge) == 0
    assert call(rows=huge, n=80, k=64) in (_lib.KLA_ERR_WORKSPACE, _lib.KLA_ERR_INVALID_ARG)
    assert call(rows=2**40, n=2**40, ldy=2**40, nbytes=2**61) in (_lib.KLA_ERR_WORKSPACE, _lib.KLA_ERR_INVALID_ARG)
