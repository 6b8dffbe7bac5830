"""CPU: which kernel a call takes (no GPU is touched; without one the router
counts 256 CUs).  The sizes are measured ones at which an earlier rule picked
the slower kernel; us of both in the comments, taken kernel first."""
import ctypes

import pytest

from dsl_tool_amd import _native as N

MODES = {"tensor": 0, "block": 1, "mxfp4": 2, "nvfp4": 3, "bf16": 4, "group": 5}
BF16, F32 = N.OUT_BF16, N.OUT_F32


def route(mode, m, n, k, out=BF16):
    f = N.lib().dsl_test_gemm_route
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_int] + [ctypes.c_int64] * 3 + [
        ctypes.c_int, ctypes.c_char_p, ctypes.c_size_t]
    buf = ctypes.create_string_buffer(96)
    assert f(MODES[mode], m, n, k, out, buf, len(buf)) == 0
    return buf.value.decode()


def test_routes_of_the_common_calls():
    assert route("block", 16, 7168, 4096) == "decode"
    assert route("block", 4096, 7168, 4096) == "persist 256x256"
    assert route("tensor", 128, 4096, 4096).startswith("stream ")
    assert route("group", 777, 5000, 2880, F32) == "pipe 128x128"
    assert route("mxfp4", 8192, 8192, 8192) == "persist 256x256"
    assert route("nvfp4", 2048, 14336, 4096) == "persist 256x256"
    assert route("bf16", 3001, 5120, 5120, F32) == "persist 256x256"
    assert route("block", 1500, 22016, 4096) == "persist 256x256 + pipe 64x128 deep"
    assert route("block", 1500, 4096, 11008) == "persist 256x128"
    assert route("bf16", 512, 4096, 4096, F32) == "pipe 64x128 deep"
