"""K that is no multiple of the kernels' 128- / 256-byte steps, on every mode:
the last, partly filled step of a row must add nothing, and scale rows that
start at any byte must reach their own blocks only."""
import numpy as np
import pytest
import torch

from dsl_tool_amd import gemm as G
from dsl_tool_amd import quant as Q
from dsl_tool_amd import workloads as W
from tests.test_gpu_random_shapes import test_random_shape as check
from tests.util import assert_close, np_f32

pytestmark = pytest.mark.gpu
DEV = "cuda"

# K of 1..3 steps plus a remainder: one 16-byte chunk, half a step, one chunk short
KS = {"tensor": (16, 272, 1152, 1280 + 112), "block": (16, 272, 1152, 1280 + 112),
      "group": (16, 272, 1152, 1280 + 112), "mxfp4": (32, 544, 640, 1024 + 480),
      "nvfp4": (32, 544, 640, 1024 + 480), "bf16": (8, 136, 1152, 1280 + 56)}


@pytest.mark.parametrize("m", [1, 16, 17, 50, 100, 130])
@pytest.mark.parametrize("mode", sorted(KS))
def test_ragged_k_streamed(mode, m):
    for k in KS[mode]:
        check(mode, m, 200, k)
        check(mode, m, 77, k)


@pytest.mark.parametrize("m", [3, 40, 300])
@pytest.mark.parametrize("mode", ["mxfp4", "nvfp4", "block", "group"])
def test_nan_scales_stay_in_their_row(mode, m):
    """A NaN scale of one row (its neighbours share the words that the copies
    move) makes that row NaN and no other."""
    n, k = 96, 544
    a, w = W.randn_bf16((m, k), 1, 1.0).to(DEV), W.randn_bf16((n, k), 2, 0.02).to(DEV)
    bad = m // 2
    if mode in ("block", "group"):
        qa, sa = Q.quant_fp8_blocks(a, 1, 128)
        qw, sw = Q.quant_fp8_blocks(w, 128 if mode == "block" else 1, 128)
        sw = sw if mode == "block" else sw.t().contiguous()
        good = G.fp8_gemm_packed(qa, qw, sa, sw, block=mode == "block", group=mode == "group")
        sa[bad] = float("nan")
        c = G.fp8_gemm_packed(qa, qw, sa, sw, block=mode == "block", group=mode == "group")
    elif mode == "mxfp4":
        qa, sa = Q.quant_mxfp4(a)
        qw, sw = Q.quant_mxfp4(w)
        good = G.fp4_gemm_packed(qa, sa, qw, sw)
        sa[bad] = 0xFF
        c = G.fp4_gemm_packed(qa, sa, qw, sw)
    else:
        qa, sa, ga = Q.quant_nvfp4(a)
        qw, sw, gw = Q.quant_nvfp4(w)
        good = G.fp4_gemm_packed(qa, sa, qw, sw, fmt="nvfp4", global_a=ga, global_w=gw)
        sa[bad] = 0x7F
        c = G.fp4_gemm_packed(qa, sa, qw, sw, fmt="nvfp4", global_a=ga, global_w=gw)
    rows = [i for i in range(m) if i != bad]
    assert np.isnan(np_f32(c)[bad]).all()
    assert torch.equal(c[rows], good[rows])


@pytest.mark.parametrize("mode", ["mxfp4", "nvfp4"])
def test_misaligned_scale_rows(mode):
    """Scale arrays that start at an odd byte, over an aligned K."""
    m, n, k = 20, 96, 1024
    a, w = W.randn_bf16((m, k), 3, 1.0).to(DEV), W.randn_bf16((n, k), 4, 0.02).to(DEV)

    def shifted(s):
        buf = torch.zeros(s.numel() + 3, dtype=torch.uint8, device=DEV)
        v = buf[3:].view(s.shape)
        v.copy_(s)
        return v

    if mode == "mxfp4":
        (qa, sa), (qw, sw) = Q.quant_mxfp4(a), Q.quant_mxfp4(w)
        assert torch.equal(G.fp4_gemm_packed(qa, shifted(sa), qw, shifted(sw)),
                           G.fp4_gemm_packed(qa, sa, qw, sw))
    else:
        (qa, sa, ga), (qw, sw, gw) = Q.quant_nvfp4(a), Q.quant_nvfp4(w)
        kw = dict(fmt="nvfp4", global_a=ga, global_w=gw)
        assert torch.equal(G.fp4_gemm_packed(qa, shifted(sa), qw, shifted(sw), **kw),
                           G.fp4_gemm_packed(qa, sa, qw, sw, **kw))


@pytest.mark.parametrize("k", [16, 144, 272, 1408])
@pytest.mark.parametrize("counts", [(1, 0, 3, 2), (17, 5, 40, 1, 0)])
def test_ragged_k_grouped_stream(counts, k):
    """Groups of a few rows on the streaming tiles (and, where K is whole 128s, the row map)."""
    g, n, t = len(counts), 136, sum(counts)
    x, w = W.randn_bf16((t, k), 5).to(DEV), W.randn_bf16((g * n, k), 6, 0.02).to(DEV)
    off = torch.tensor([0] + list(np.cumsum(counts)), dtype=torch.int32, device=DEV)
    qx, sx = Q.quant_fp8_blocks(x, 1, k)
    qw, sw = Q.quant_fp8_blocks(w, 1, k)
    y = G.grouped_fp8_gemm_packed(qx, sx, qw.view(g, n, k), sw.view(g, n), off)
    xd = qx.view(torch.float8_e4m3fn).double().cpu() * sx.double().cpu()
    wd = (qw.view(torch.float8_e4m3fn).double().cpu() * sw.double().cpu()).view(g, n, k)
    ref = torch.cat([xd[off[e]:off[e + 1]] @ wd[e].t() for e in range(g)])
    assert_close(y, ref.float().numpy(), what=f"grouped stream {counts} K={k}")


# the persistent tiles: more than one tile per workgroup at short K (partial
# pairs as a tile's only, second and later one), ragged rows and columns
@pytest.mark.parametrize("mode,k", [("tensor", 16 * 9), ("tensor", 400), ("tensor", 1168), ("block", 640),
                                    ("block", 400), ("block", 1168), ("mxfp4", 288), ("mxfp4", 1056),
                                    ("mxfp4", 1408), ("nvfp4", 288), ("nvfp4", 1056), ("nvfp4", 1344),
                                    ("bf16", 72), ("bf16", 200), ("bf16", 584)])
def test_ragged_k_persistent(mode, k):
    check(mode, 4352, 4300, k)
    check(mode, 1025, 1000, k)


@pytest.mark.parametrize("k", [144, 400, 1168])
def test_ragged_k_grouped_persistent(k):
    counts, n = (300, 0, 97, 513), 264
    g, t = len(counts), sum(counts)
    x, w = W.randn_bf16((t, k), 7).to(DEV), W.randn_bf16((g * n, k), 8, 0.02).to(DEV)
    off = torch.tensor([0] + list(np.cumsum(counts)), dtype=torch.int32, device=DEV)
    qx, sx = Q.quant_fp8_blocks(x, 1, k)
    qw, sw = Q.quant_fp8_blocks(w, 1, k)
    y = G.grouped_fp8_gemm_packed(qx, sx, qw.view(g, n, k), sw.view(g, n), off)
    xd = qx.view(torch.float8_e4m3fn).double().cpu() * sx.double().cpu()
    wd = (qw.view(torch.float8_e4m3fn).double().cpu() * sw.double().cpu()).view(g, n, k)
    ref = torch.cat([xd[off[e]:off[e + 1]] @ wd[e].t() for e in range(g)])
    assert_close(y, ref.float().numpy(), what=f"grouped persistent {counts} K={k}")


# one round of the 128x128 tiles: partial first, odd and even last stages
@pytest.mark.parametrize("mode,k", [("tensor", 48), ("tensor", 336), ("tensor", 1072), ("block", 144),
                                    ("block", 1072), ("group", 144), ("group", 1072), ("mxfp4", 96),
                                    ("mxfp4", 672), ("mxfp4", 2144), ("nvfp4", 96), ("nvfp4", 672),
                                    ("nvfp4", 2144), ("bf16", 24), ("bf16", 168), ("bf16", 536)])
def test_ragged_k_pipelined(mode, k):
    check(mode, 1100, 1000, k)
    check(mode, 1200, 1029, k)


def test_padded_scale_rows_need_their_workspace():
    """The query covers the padded scale rows; a caller who brings less (here
    none: no kernel for whole rows would need any) is served all the same."""
    from dsl_tool_amd import _native as N
    m, n, k = 4100, 4200, 1056
    a, w = W.randn_bf16((m, k), 9).to(DEV), W.randn_bf16((n, k), 10, 0.02).to(DEV)
    (qa, sa), (qw, sw) = Q.quant_mxfp4(a), Q.quant_mxfp4(w)
    nb = N.lib().dsl_gemm_workspace_bytes(N.OP_FP4, m, n, k)
    assert nb >= (m + n) * 48
    want = G.fp4_gemm_packed(qa, sa, qw, sw)
    ws = torch.empty(nb, dtype=torch.uint8, device=DEV)
    for p, b in ((ws.data_ptr(), nb), (ws.data_ptr(), nb - 16), (None, 0)):
        c = torch.empty_like(want)
        N.call("dsl_fp4_gemm", qa.data_ptr(), qw.data_ptr(), c.data_ptr(), m, n, k, n, N.OUT_BF16,
               N.FMT_MXFP4, sa.data_ptr(), sw.data_ptr(), None, None, p, b, N.stream_of(a.device))
        assert_close(c, np_f32(want), what=f"mxfp4 workspace {b}")


# 256x128 persistent tiles (one round of them, more than one of 128x128), whole
# and ragged K, and a problem of one round and a few tiles more, whose last
# columns run as a second launch
@pytest.mark.parametrize("mode", ["tensor", "block", "mxfp4", "nvfp4", "bf16"])
@pytest.mark.parametrize("m,n,k", [(1300, 2500, 512), (1281, 4000, 608), (4100, 4200, 512), (2100, 7500, 256)])
def test_narrow_tiles_and_column_strips(mode, m, n, k):
    check(mode, m, n, k)


# 64x128 and deep-ring 128x128 tiles: one round, ragged rows and columns, whole,
# odd and partial stages, fewer stages than the ring holds
@pytest.mark.parametrize("mode", ["tensor", "block", "group", "mxfp4", "bf16"])
@pytest.mark.parametrize("m,n", [(300, 2050), (1025, 1000), (900, 4000)])
def test_small_tiles(mode, m, n):
    unit = {"mxfp4": 32, "bf16": 8}.get(mode, 16)
    for k in (unit, 128, 256, 640, 1024, 1152 + unit):
        check(mode, m, n, k)



@pytest.mark.parametrize("mode", sorted(KS))
@pytest.mark.parametrize("m,n", [(33, 500), (64, 1030), (100, 260), (200, 130)])
def test_few_weight_slices(mode, m, n):
    """Small row blocks where N gives few workgroups."""
    for k in (512, 4096, KS[mode][2]):
        check(mode, m, n, k)


@pytest.mark.parametrize("k", [65536, 65536 + 144])
def test_more_scale_groups_than_the_ring_holds(k):
    """Block-scaled tiles keep 512 weight scales of a row in LDS; longer K
    takes the tiles that read them from memory."""
    m, n = 320, 2048
    gen = torch.Generator(device=DEV).manual_seed(k)
    a = torch.randn((m, k), generator=gen, device=DEV).bfloat16()
    w = torch.randn((n, k), generator=gen, device=DEV).bfloat16()
    qa, sa = Q.quant_fp8_blocks(a, 1, 128)
    qw, sw = Q.quant_fp8_blocks(w, 128, 128)
    c = G.fp8_gemm_packed(qa, qw, sa, sw, block=True, out_dtype=torch.float32)
    ref = torch.zeros((m, n), dtype=torch.float64, device=DEV)
    for g in range(0, k, 8192):
        e = min(g + 8192, k)
        f = lambda q, s: q[:, g:e].view(torch.float8_e4m3fn).double() * s.double()[:, g // 128:].repeat_interleave(
            128, 1)[:, :e - g]
        ref += f(qa, sa) @ f(qw, sw.repeat_interleave(128, 0)[:n]).t()
    # fp32 sums of k products: sqrt(k) * 2^-24 relative to the largest output, 8x margin
    assert (c.double() - ref).abs().max() <= 8 * k ** 0.5 * 2.0 ** -24 * ref.abs().max()
