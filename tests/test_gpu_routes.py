"""Both sides of the routing lines, each on the kernel its route names (asserted),
against the oracle: ragged K split over workgroups or streamed, the deep rings
at whole, odd and partial pair counts, persistent tiles with whole, partial
and element-stored last columns, grouped K of no whole 128 bytes on each
kernel, and column strips whose rest streams."""
import numpy as np
import pytest
import torch

from dsl_tool_amd import _native as N
from dsl_tool_amd import gemm as G
from dsl_tool_amd import quant as Q
from dsl_tool_amd import workloads as W
from tests.test_gpu_lora import test_lora_fused_gemm as check_lora
from tests.test_gpu_random_shapes import test_random_shape as check
from tests.test_routes import BF16, F32, grouped_route, route
from tests.util import assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("mode,m,n,k,want", [
    ("bf16", 700, 512, 14880, "split"), ("bf16", 40, 1800, 16008, "split"), ("tensor", 70, 1544, 20016, "split"),
    ("block", 60, 1552, 20016, "split"), ("group", 41, 2104, 20016, "split"), ("mxfp4", 40, 2304, 28032, "split"),
    ("tensor", 1500, 128, 8208, "split"),
    ("nvfp4", 218, 3400, 256, "pipe 128x128"),
    ("bf16", 180, 1248, 640, "stream 32x"), ("nvfp4", 235, 1040, 2560, "stream 32x"),
    ("tensor", 560, 136, 8704, "stream 64x"), ("mxfp4", 700, 168, 2048, "stream"),
    # the deep rings: whole pairs, an odd last stage, a partial one
    ("tensor", 900, 4000, 1536, "pipe 128x128 deep"), ("tensor", 900, 4000, 2688, "pipe 128x128 deep"),
    ("tensor", 900, 4000, 2576, "pipe 128x128 deep"), ("bf16", 900, 4000, 768, "pipe 128x128 deep"),
    ("bf16", 900, 4000, 1288, "pipe 128x128 deep"), ("tensor", 300, 2050, 1664, "pipe 64x128 deep"),
    ("tensor", 900, 4000, 640, "pipe 128x128"), ("bf16", 424, 2632, 448, "pipe 128x128"),
    # persistent tiles
    ("tensor", 1300, 3200, 1536, "persist 256x128"), ("block", 1300, 3216, 1280, "persist 256x128"),
    ("mxfp4", 1300, 3216, 1024, "persist 256x128"), ("tensor", 1300, 3301, 512, "persist 256x128"),
    ("tensor", 1300, 3300, 512, "pipe 128x128"), ("block", 1300, 3300, 512, "pipe 128x128"),
    ("block", 4352, 4352, 1152, "persist 256x256"), ("mxfp4", 4352, 4352, 1280, "persist 256x256"),
    ("block", 4352, 4304, 640, "pipe 256x256"), ("mxfp4", 4352, 4304, 768, "pipe 256x256"),
    ("block", 1300, 7000, 640, "pipe 128x128"),
    # the last columns of a barely started round
    ("tensor", 1000, 16640, 256, "persist 256x256 + stream"), ("block", 1000, 16640, 512, "persist 256x256 + "),
    ("mxfp4", 1000, 16640, 512, "persist 256x256 + stream"), ("nvfp4", 1000, 16640, 256, "persist 256x256 + stream"),
    ("bf16", 1000, 16640, 256, "persist 256x256 + stream")], ids=lambda v: str(v))
def test_routed_kernel(mode, m, n, k, want):
    got = route(mode, m, n, k, F32 if (m + n + k) % 2 else BF16)     # the check's output type
    if "+" not in want:
        got = got.split(" + ")[0]
    assert got.startswith(want) and ("deep" in want or "deep" not in got), got
    check(mode, m, n, k)


@pytest.mark.parametrize("counts,n,k,want", [
    ((20,) * 64, 1100, 128, "persist"), ((1, 2) * 32, 4200, 64, "pipe 128x256"), ((3,) * 64, 2400, 192, "pipe 128x256"),
    ((34,) * 64, 712, 2064, "persist"), ((37,) * 64, 136, 3600, "stream"), ((37,) * 64, 360, 2896, "tiled"),
    ((60, 100), 200, 144, "tiled"), ((0, 300, 99, 513), 264, 144, "persist"), ((700, 400), 712, 192, "persist"),
    ((90, 0, 111), 520, 1088, "persist"), ((90, 0, 111), 600, 1472, "pipe 128x256"),
    ((80,) * 16, 2100, 400, "persist")])
def test_routed_grouped_kernel(counts, n, k, want):
    g, t = len(counts), sum(counts)
    assert grouped_route(g, t, n, k) == want
    x, w = W.randn_bf16((t, k), 11).to(DEV), W.randn_bf16((g * n, k), 12, 0.02).to(DEV)
    off = torch.tensor([0] + list(np.cumsum(counts)), dtype=torch.int32, device=DEV)
    qx, sx = Q.quant_fp8_blocks(x, 1, k)
    qw, sw = Q.quant_fp8_blocks(w, 1, k)
    y = G.grouped_fp8_gemm_packed(qx, sx, qw.view(g, n, k), sw.view(g, n), off)
    xd = (qx.view(torch.float8_e4m3fn).double() * sx.double()).float()
    wd = (qw.view(torch.float8_e4m3fn).double() * sw.double()).float().view(g, n, k)
    ref = torch.cat([xd[off[e]:off[e + 1]] @ wd[e].t() for e in range(g)])
    assert_close(y, ref.cpu().numpy(), what=f"grouped {want} {g}x{t} {n}x{k}")


@pytest.mark.parametrize("m,n,k,r,l,want", [   # want: the adapter add
    (541, 1024, 1032, 8, 4, "stream tail"), (300, 1000, 832, 8, 2, "stream tail"),
    (773, 3496, 832, 8, 2, "pipe 128x128"), (773, 3496, 1096, 16, 2, "pipe 128x128"),
    (773, 3496, 576, 16, 4, "stream 32x"), (700, 1200, 1096, 16, 4, "stream 32x")])
def test_lora_adapter_adds(m, n, k, r, l, want):
    """K of whole 64s that are no whole 128s (T from the plain GEMM) and ragged K."""
    got = route("bf16", m, n, (2 * r * l + 63) // 64 * 64, F32, accumulate=True)
    assert got.startswith(want) and "deep" not in got, got
    check_lora(m, n, k, r, l)


def test_unaligned_scales_do_not_take_a_split_they_have_no_room_for():
    """Scale arrays off the 4-byte grid: without the whole-row kernels the shape
    would split K, but its workspace contract (aligned scales) has no room."""
    m, n, k = 40, 2304, 28672
    assert route("mxfp4", m, n, k).startswith("stream ")
    assert N.lib().dsl_gemm_workspace_bytes(N.OP_FP4, m, n, k) == 0
    a, w = W.randn_bf16((m, k), 13).to(DEV), W.randn_bf16((n, k), 14, 0.02).to(DEV)
    (qa, sa), (qw, sw) = Q.quant_mxfp4(a), Q.quant_mxfp4(w)

    def shifted(s):
        buf = torch.zeros(s.numel() + 1, dtype=torch.uint8, device=DEV)
        v = buf[1:].view(s.shape)
        v.copy_(s)
        return v

    ref = G.fp4_gemm_packed(qa, sa, qw, sw, out_dtype=torch.float32)
    assert_close(G.fp4_gemm_packed(qa, shifted(sa), qw, shifted(sw), out_dtype=torch.float32), ref.cpu().numpy())
