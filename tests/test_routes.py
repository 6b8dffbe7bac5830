"""CPU: which kernel a call takes (no GPU is touched; without one the router
counts 256 CUs).  The sizes are measured ones at which an earlier rule picked
the slower kernel; us of both in the comments, taken kernel first."""
import ctypes
import os
import subprocess
import sys

import pytest

from dsl_tool_amd import _native as N

MODES = {"tensor": 0, "block": 1, "mxfp4": 2, "nvfp4": 3, "bf16": 4, "group": 5}
BF16, F32 = N.OUT_BF16, N.OUT_F32


def route(mode, m, n, k, out=BF16, accumulate=False):
    f = N.lib().dsl_test_gemm_route
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_int] + [ctypes.c_int64] * 3 + [
        ctypes.c_int, ctypes.c_char_p, ctypes.c_size_t, ctypes.c_int]
    buf = ctypes.create_string_buffer(96)
    assert f(MODES[mode], m, n, k, out, buf, len(buf), int(accumulate)) == 0
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


@pytest.mark.parametrize("mode,m,n,k", [
    ("bf16", 180, 1248, 1664),      # 5.3 / 7.8
    ("tensor", 150, 1368, 1280),    # 3.8 / 5.5
    ("nvfp4", 235, 1040, 7680),     # 16.5 / 25.1
    ("nvfp4", 376, 3156, 12800),    # 89 / 113
    ("mxfp4", 133, 2392, 2560)])    # 5.1 / 7.1
def test_odd_chunk_rows_keep_the_plain_streaming_form(mode, m, n, k):
    assert route(mode, m, n, k).startswith("stream 32x")


@pytest.mark.parametrize("mode,m,n,k,bm", [
    ("bf16", 812, 136, 11008, 64),     # 30.1 / 38.8
    ("tensor", 384, 296, 24576, 64),   # 27.1 / 36.0
    ("block", 357, 280, 18432, 64),    # 24.3 / 33.4
    ("nvfp4", 544, 144, 1024, 32),     # 4.1 / 7.9: short chains overlap on a CU
    ("mxfp4", 41, 2592, 8192, 64),     # 6.9 / 9.1: three times the workgroups of one round
    ("bf16", 64, 512, 4096, 16)])      # 6.7 / 8.4
def test_streaming_row_blocks_of_one_round(mode, m, n, k, bm):
    assert route(mode, m, n, k).startswith(f"stream {bm}x")


@pytest.mark.parametrize("mode,m,n,k,want", [
    ("tensor", 724, 3200, 640, "pipe 128x128"),         # 6.3 / 8.2
    ("tensor", 410, 7680, 1664, "pipe 128x128"),        # 10.3 / 12.1
    ("bf16", 424, 5368, 320, "pipe 128x128"),           # 6.3 / 8.2
    ("tensor", 350, 6232, 512, "pipe 128x128"),         # 5.9 / 6.4
    ("tensor", 395, 3400, 896, "pipe 128x128"),         # 6.6 / 7.1
    ("tensor", 724, 3200, 4096, "pipe 128x128 deep"),   # 19.9 / 22.9
    ("tensor", 395, 3400, 1664, "pipe 64x128 deep"),
    ("block", 724, 3200, 640, "pipe 128x128 deep")])    # group-scaled forms gain at any K
def test_deep_rings_need_a_long_k(mode, m, n, k, want):
    assert route(mode, m, n, k) == want


@pytest.mark.parametrize("mode,m,n,k,want", [
    # a partial last column of tiles stores element by element
    ("tensor", 583, 9952, 512, "pipe 128x128"),        # 11.0 / 18.5
    ("block", 6720, 752, 1024, "pipe 128x128"),        # 13.5 / 25.3
    ("block", 528, 7016, 512, "pipe 128x128"),         # 9.1 / 17.0
    ("nvfp4", 716, 4432, 512, "pipe 128x128"),         # 12.8 / 19.6
    ("tensor", 691, 5632, 768, "persist 256x128"),     # 9.3 / 11.8: whole columns
    ("tensor", 2048, 4000, 11008, "persist 256x128"),  # ragged, long K
    ("nvfp4", 1024, 5000, 4096, "persist 256x128"),
    # scale rows that are no whole quads, rows of whole 128 bytes
    ("block", 6569, 1520, 768, "pipe 128x128"),        # 16.9 / 43.5
    ("block", 7493, 2784, 640, "pipe 256x256"),        # 28.1 / 50.5
    ("mxfp4", 1319, 8624, 768, "pipe 128x128"),        # 15.4 / 33.4
    ("mxfp4", 1124, 13624, 256, "pipe 256x256"),       # 15.4 / 22.1
    ("block", 4128, 7680, 768, "pipe 256x256"),        # 38.1 / 36.1: the line is at 1024
    ("block", 6027, 3072, 1792, "persist 256x256 + pipe 128x128 deep"),    # 46.4 / 58.0
    ("mxfp4", 6956, 1792, 2304, "persist 256x256")])   # 27.1 / 39.7
def test_persistent_tiles_need_whole_columns_or_a_long_k(mode, m, n, k, want):
    assert route(mode, m, n, k) == want
    if want.startswith("pipe"):      # fp32 results: those tiles store element by element too
        assert route(mode, m, n, k, F32).startswith("persist")


@pytest.mark.parametrize("mode,m,n,k,want", [
    ("bf16", 129, 3840, 10528, "split"),       # 41 / 80
    ("bf16", 681, 512, 14872, "split"),        # 48 / 105
    ("block", 49, 4480, 14960, "split"),       # 26.8 / 53.8
    ("group", 48, 4736, 12416, "split"),       # 24.2 / 36.1
    ("tensor", 2253, 128, 29776, "split"),     # 36 / 102
    ("nvfp4", 218, 13312, 256, "pipe"),        # 8.3 / 44.9
    ("mxfp4", 87, 4840, 4608, "stream"),       # 7.1 / 10.7
    ("tensor", 16, 4096, 4224, "stream tail"), # 6.1 / 11.4
    ("mxfp4", 256, 4096, 4224, "stream tail"), # 12.4 / 76
    ("block", 16, 4096, 4224, "stream tail")]) # 6.6 / 12.2
def test_ragged_forms_are_compared_with_the_kernel_they_replaced(mode, m, n, k, want):
    assert route(mode, m, n, k).startswith(want)


def test_a_call_without_the_splits_room_keeps_the_ragged_form():
    """The split's partial sums are in the workspace contract of its shapes."""
    for mode, op in (("bf16", N.OP_BF16), ("block", N.OP_FP8), ("mxfp4", N.OP_FP4)):
        for m, n, k in ((129, 3840, 10528), (36, 4480, 7456), (681, 512, 14880)):
            r = route(mode, m, n, k)
            if r.startswith("split"):
                parts = int(r.split("/")[1])
                assert N.lib().dsl_gemm_workspace_bytes(op, m, n, k) >= 4 * parts * m * n


@pytest.mark.parametrize("mode,m,n,k", [
    ("group", 5, 45352, 1184),      # 14.0 / 16.0
    ("block", 5, 44096, 1200),      # 14.5 / 16.6
    ("mxfp4", 3, 36464, 256)])      # 10.1 / 10.1
def test_up_to_16_rows_of_ragged_k_stream(mode, m, n, k):
    assert route(mode, m, n, k).startswith("stream tail")


@pytest.mark.parametrize("m,n,k,want", [     # the whole layer at rank 8 to 32
    (541, 1024, 64, "stream tail 64x32"),    # 18.1 / 24.2
    (300, 2992, 64, "stream tail 64x64"),    # 37.4 / 40.3
    (276, 3216, 64, "pipe 128x128"),         # 25.8 / 28.0
    (773, 3496, 64, "pipe 128x128"),         # 30.6 / 41.4
    (773, 3496, 128, "stream 32x64")])       # whole chunks stream
def test_adapter_adds_of_no_whole_chunk_stream_few_columns(m, n, k, want):
    assert route("bf16", m, n, k, F32, accumulate=True) == want


def grouped_route(g, rows, n, k, gather=False):
    f = N.lib().dsl_test_grouped_route
    f.restype, f.argtypes = ctypes.c_char_p, [ctypes.c_int64] * 4 + [ctypes.c_int]
    return f(g, rows, n, k, int(gather)).decode()


@pytest.mark.parametrize("g,rows,n,k,want", [
    (64, 1147, 2824, 128, "persist"),        # 19.4 / 32.4: K of less than a chunk
    (64, 99, 2456, 64, "pipe 128x256"),      # 11.5 / 20.1
    (64, 2202, 1912, 3776, "persist"),       # 128.7 / 193.8: two row blocks read W twice
    (64, 2367, 352, 2896, "tiled"),          # 34.7 / 42.0
    (32, 1036, 1112, 2944, "stream"),        # 34.8 / 40.6
    (64, 256, 1536, 2048, "stream"),
    (8, 73, 3736, 128, "stream"),            # 6.5 / 9.5
    (2, 1982, 704, 144, "tiled"),            # 18.5 / 31.6: a round of small tiles, partial columns
    (2, 1351, 2656, 3376, "tiled"),          # 48.2 / 56.9
    (8, 891, 648, 3264, "pipe 128x256"),     # 38.7 / 50.7
    (16, 1165, 1280, 448, "persist"),        # 14.7 / 24.1: whole columns
    (16, 8192, 2048, 1168, "persist")])      # many tiles
def test_grouped_routes(g, rows, n, k, want):
    assert grouped_route(g, rows, n, k) == want


def test_gathered_groups_have_the_persistent_or_the_streaming_kernel():
    assert grouped_route(64, 1147, 2824, 128, True) == "persist"
    assert grouped_route(64, 256, 1536, 1152, True) == "stream"
    assert grouped_route(64, 8192, 1536, 2048, True) == "persist"
    assert grouped_route(64, 8192, 1536, 1168, True) == "none"   # refused by dsl_moe_grouped_fp8_gemm


def transposed(rows, cols, gr, gc, f32=False, ptr=1 << 20):
    f = N.lib().dsl_test_quant_transposed
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_int] + [ctypes.c_int64] * 6
    return bool(f(ptr, N.IN_F32 if f32 else N.IN_BF16, rows, cols, 1, rows, gr, gc))


@pytest.mark.parametrize("rows,cols,gr,gc,f32,want", [
    # one scale per row: us of the strided / the transposed kernel
    (64, 8192, 1, 8192, False, False),      # 22.9 / 68.0
    (512, 2048, 1, 2048, True, False),      # 13.3 / 27.9
    (1280, 2048, 1, 2048, False, True),     # 28.6 / 20.0
    (1024, 512, 1, 512, True, False),       # 7.1 / 9.3
    (1536, 2048, 1, 2048, True, True),      # 45.0 / 28.3
    (1500, 2048, 1, 2048, False, False),    # 31.5 / 60.7: rows of no whole runs of 8
    (4100, 512, 1, 512, False, True),       # 20.7 / 16.2
    (64, 2048, 1, 512, False, False),       # 4.8 / 7.1
    (64, 28672, 1, 512, False, True),       # 17.1 / 7.4
    (2, 1 << 20, 1, 512, False, False),     # 13.8 / 41.4
    (4, 512, 128, 128, True, False),        # 3.7 / 4.6
    (8, 512, 128, 128, True, True),         # 5.1 / 4.4
    (4, 512, 1, 128, False, True),          # 46 / 3.7
    (4, 512, 1, 256, False, True),
    ((1 << 29) + 8, 2, 1, 2, False, False)])   # past the grid's threads
def test_transposed_quantizer_needs_enough_scales(rows, cols, gr, gc, f32, want):
    assert transposed(rows, cols, gr, gc, f32) == want


@pytest.mark.parametrize("g,rows,cols,esize,want", [
    (1, 64, 8192, 2, False),      # copy and row quantizer 7.9 us, in place 68.3
    (2, 512, 2048, 2, False),     # 16.6 / 19.9
    (4, 512, 2048, 2, True),      # 26.0 / 20.3
    (16, 64, 512, 2, True),       # 8.3 / 7.1
    (16, 64, 8192, 2, False),     # 45.1 / 69.3
    (8, 300, 2048, 2, False),     # 30.1 / 60.2: rows of no whole runs of 8
    (8, 1001, 2048, 2, True),     # 81.8 / 62.2
    (16, 333, 2048, 4, True),     # 86.6 / 73.8
    (16, 333, 2048, 2, False)])   # 56.4 / 62.8
def test_grouped_weights_are_read_in_place_where_that_fills_the_chip(g, rows, cols, esize, want):
    from dsl_tool_amd import quant as Q
    assert Q._rows_in_place(g, rows, cols, esize, rows * cols, rows, 1 << 20) == want
    if rows % 8 == 0:             # a pointer or pitch off the 16-byte grid is read element by element
        assert not Q._rows_in_place(4, 512, cols, esize, rows * cols, rows, (1 << 20) + 2)
        assert not Q._rows_in_place(4, 512, cols, esize, 512 * cols, 513, 1 << 20)


@pytest.mark.parametrize("value", ["off", "1"])
def test_pipe_switch_also_holds_for_column_strips(value):
    """DSL_GEMM_PIPE=off never uses the pipelined kernels; a number names one."""
    call = "from tests.test_routes import route; print(route('bf16', 4300, 4300, 4096))"
    env = dict(os.environ, DSL_GEMM_PIPE=value)
    got = subprocess.run([sys.executable, "-c", call], env=env, capture_output=True, text=True, check=True,
                         cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__)))).stdout.strip()
    assert route("bf16", 4300, 4300, 4096).startswith("persist 256x256 + pipe")
    assert got == "persist 256x256"


def test_column_strips_of_few_rows_stream_their_rest():
    assert route("tensor", 1000, 16640, 1024).startswith("persist 256x256 + stream")
    assert route("bf16", 1000, 16640, 1024).startswith("persist 256x256 + stream")
