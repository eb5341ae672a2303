"""The product with both operands in LDS forms 32-bit offsets into X: the library itself refuses an X, or a row list over
one, that they do not reach.  (No rows are asked for: nothing is launched.)"""
import ctypes

import torch


def test_rows_of_x_beyond_the_offsets_are_refused():
    from spite_amd.csrc import hipops
    buf = torch.zeros(64, dtype=torch.float32)
    p = ctypes.c_void_p((buf.data_ptr() + 63) // 64 * 64)
    call = lambda M, ldx, rows, x_rows: hipops.lib().spite_gemm_lds(p, ldx, p, 0, p, hipops.F32, 16, M, 16, 64, None, 1, p if rows else None, None,
                                                                 None, 0, 0.0, 0, x_rows, None)
    assert call(0, 64, False, 0) == 0 and call(0, 8192, True, 131071) == 0
    assert call(0, 8192, True, 131072) != 0              # 2 GiB of X behind a list of no rows
    assert call(0, 64, True, 0) != 0                     # a list over an X of unknown height
    assert b"rows of X" in hipops.lib().spite_hip_last_error()
