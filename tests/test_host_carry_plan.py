"""la_carry_bytes over a grid of shapes (host logic only; 256 CUs assumed without a device): the plain matrices'
bytes where la_saved_state_bytes has any, else nothing or exactly the workspace of the forward pass (its state slots, a
whole number per sequence); nothing for float32 and when the launch options pin another form."""
import ctypes

from lightning_attn.ops.hip import _lib


def test_carry_bytes():
    L = _lib.lib()
    used = 0
    for b, h in ((1, 1), (1, 8), (2, 12), (1, 40), (1, 64), (3, 24), (4, 32), (8, 32)):
        for n in (1, 64, 1000, 4096, 8192, 65536):
            for d, e in ((16, 64), (64, 64), (64, 128), (72, 128), (128, 128), (128, 64), (192, 192), (256, 256)):
                for dtype in (0, 1, 2):
                    got = L.la_carry_bytes(b, h, n, d, e, dtype, None)
                    saved = L.la_saved_state_bytes(b, h, n, d, e, dtype, None)
                    if saved:
                        assert got == saved
                    elif got:
                        wide = d > 64
                        assert dtype != 2 and (e > 64) == wide and d <= 128 and e <= 128
                        assert got == L.la_workspace_bytes(0, b, h, n, d, e, dtype)
                        assert got % (b * h * (128 * 128 if wide else 64 * 64) * 4) == 0
                        used += 1
                        for args in ((2, 0, 0, 0, 0), (0, _lib.LA_OPT_OFF, 0, 0, 0), (0, 0, _lib.LA_OPT_ON, 0, 0), (0, 0, 0, _lib.LA_OPT_OFF, 0)):
                            assert L.la_carry_bytes(b, h, n, d, e, dtype, ctypes.byref(_lib.LaunchOpts(*args))) == 0
    assert used
    assert L.la_carry_bytes(0, 8, 8192, 128, 128, 0, None) == 0
