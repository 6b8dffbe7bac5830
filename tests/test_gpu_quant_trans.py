"""Quantizers on [K, N] sources (the reference's B, read as its [N, K] view):
the transposed-tile kernels, bit for bit against the oracle, at the edges of
their 64- and 128-row x 128- and 256-column tiles."""
import numpy as np
import pytest
import torch

from oracle import quant as OQ
from dsl_tool_amd import quant as Q
from tests.util import np_f32, np_u8

pytestmark = pytest.mark.gpu
DEV = "cuda"

# rows (N), columns (K)
SHAPES = [(2, 32), (8, 128), (63, 96), (64, 128), (65, 160), (72, 256), (127, 288), (128, 512),
          (136, 544), (200, 1056), (513, 128)]


def _source(r, c, dt, pad, off):
    """([r, c] view with unit row stride on the GPU, its values in fp32)."""
    g = torch.Generator().manual_seed(1000 * r + c + pad)
    x = torch.randn((c, r), generator=g) * torch.exp(torch.empty((1, r)).uniform_(-3, 3, generator=g))
    x = torch.where(torch.rand((c, r), generator=g) < 2e-3, x * 50, x)
    x[:, r // 2] = 0.0                         # an all-zero row: the scale floors
    x = x.to(dt)
    buf = torch.zeros(c * (r + pad) + off, dtype=dt, device=DEV)
    view = buf[off:].view(c, r + pad)[:, :r]
    view.copy_(x)
    return view.t(), x.t().float().contiguous().numpy()


@pytest.mark.parametrize("r,c", SHAPES)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("pad,off", [(0, 0), (8, 0), (3, 1)])
def test_transposed_sources_match_oracle(r, c, dt, pad, off):
    x, ref = _source(r, c, dt, pad, off)
    q, s = Q.quant_fp8_tensor(x)
    q_ref, s_ref = OQ.quant_fp8_per_tensor(ref)
    assert np_f32(s)[0] == s_ref and np.array_equal(np_u8(q), q_ref)
    for gr, gc in ((1, 128), (1, 256), (1, c), (128, 128)):
        q, s = Q.quant_fp8_blocks(x, gr, gc)
        q_ref, s_ref = OQ.quant_fp8_blockwise(ref, gr, gc)
        assert np.array_equal(np_f32(s), s_ref), (gr, gc)
        assert np.array_equal(np_u8(q), q_ref), (gr, gc)
    q, s = Q.quant_mxfp4(x)
    q_ref, s_ref = OQ.quant_mxfp4(ref)
    assert np.array_equal(np_u8(s), s_ref) and np.array_equal(np_u8(q), q_ref)
    q, s, sg = Q.quant_nvfp4(x)
    q_ref, s_ref, sg_ref = OQ.quant_nvfp4(ref)
    assert np_f32(sg)[0] == sg_ref
    assert np.array_equal(np_u8(s), s_ref) and np.array_equal(np_u8(q), q_ref)


@pytest.mark.parametrize("c", [40, 130, 272])
def test_transposed_sources_odd_columns(c):
    """Code rows of no whole 16 bytes (FP8 any K; NVFP4 an odd number of blocks)."""
    x, ref = _source(72, c, torch.bfloat16, 0, 0)
    for gr, gc in ((1, 128), (128, 128)):
        q, s = Q.quant_fp8_blocks(x, gr, gc)
        q_ref, s_ref = OQ.quant_fp8_blockwise(ref, gr, gc)
        assert np.array_equal(np_f32(s), s_ref) and np.array_equal(np_u8(q), q_ref)
    if c % 16 == 0:
        q, s, sg = Q.quant_nvfp4(x)
        q_ref, s_ref, sg_ref = OQ.quant_nvfp4(ref)
        assert np_f32(sg)[0] == sg_ref
        assert np.array_equal(np_u8(s), s_ref) and np.array_equal(np_u8(q), q_ref)


@pytest.mark.parametrize("g,n,k", [(1, 64, 128), (3, 72, 400), (5, 130, 1040), (2, 513, 2064)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("pad", [0, 3, 8])
def test_batched_rows_match_oracle(g, n, k, dt, pad):
    """[G, K, N] weights, one scale per output row, read in place."""
    gen = torch.Generator().manual_seed(g * n + k)
    w = (torch.randn((g, k, n), generator=gen) * 0.02).to(dt)
    buf = torch.zeros((g, k, n + pad), dtype=dt, device=DEV)
    buf[:, :, :n] = w.to(DEV)
    q, s = Q.quant_fp8_rows_batched(buf[:, :, :n].transpose(1, 2))
    q_ref, s_ref = OQ.quant_fp8_blockwise(w.transpose(1, 2).reshape(g * n, k).float().numpy(), 1, k)
    assert np.array_equal(np_f32(s), s_ref)
    assert np.array_equal(np_u8(q), q_ref)


@pytest.mark.parametrize("r,c,gr,gc", [
    (1024, 384, 1, 384), (1536, 384, 1, 384), (1016, 384, 1, 384), (3072, 272, 1, 272), (3071, 272, 1, 272),
    (64, 8192, 1, 512), (64, 8704, 1, 512), (15, 8192, 1, 512), (7, 384, 128, 128), (8, 384, 128, 128)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_both_sides_of_the_occupancy_rule(r, c, gr, gc, dt):
    """Few long scale groups take the strided kernel, many the transposed one."""
    x, ref = _source(r, c, dt, 0, 0)
    q, s = Q.quant_fp8_blocks(x, gr, gc)
    q_ref, s_ref = OQ.quant_fp8_blockwise(ref, gr, gc)
    assert np.array_equal(np_f32(s), s_ref) and np.array_equal(np_u8(q), q_ref)


@pytest.mark.parametrize("r,c", [(333, 2048), (1500, 1024), (513, 1024), (4100, 512), (4616, 512)])
def test_nvfp4_of_odd_fp32_sources(r, c):
    x, ref = _source(r, c, torch.float32, 1, 1)
    q, s, sg = Q.quant_nvfp4(x)
    q_ref, s_ref, sg_ref = OQ.quant_nvfp4(ref)
    assert np_f32(sg)[0] == sg_ref
    assert np.array_equal(np_u8(s), s_ref) and np.array_equal(np_u8(q), q_ref)


@pytest.mark.parametrize("g,n,k", [(1, 64, 1040), (2, 512, 400), (4, 512, 144), (16, 64, 400), (32, 40, 144),
                                   (9, 1001, 80), (3, 72, 400)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_grouped_weights_in_place_or_copied(g, n, k, dt):
    test_batched_rows_match_oracle(g, n, k, dt, 0)
