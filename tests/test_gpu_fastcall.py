"""The native call path against the Python path it stands in for: the same
bytes for well-formed calls, and None (so the Python path decides) for
anything else."""
import pytest
import torch

from dsl_tool_amd import _native as N
from dsl_tool_amd import fused as F
from dsl_tool_amd import gemm as G
from dsl_tool_amd import moe as M
from dsl_tool_amd import quant as Q

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bf16(shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(torch.bfloat16).to(DEV)


def _calls(m, n, k):
    x, w = _bf16((m, k), 1), _bf16((n, k), 2, 0.05)
    out = {}
    for nm, src in (("bf16", x), ("fp32", x.float()), ("kn", w.t())):
        out[f"tensor {nm}"] = lambda s=src: Q.quant_fp8_tensor(s)
        out[f"blocks {nm}"] = lambda s=src: Q.quant_fp8_blocks(s, 1, 128)
        if src.shape[1] % 32 == 0:
            out[f"mx {nm}"] = lambda s=src: Q.quant_mxfp4(s)
            out[f"nv {nm}"] = lambda s=src: Q.quant_nvfp4(s)
    qa, sa = Q.quant_fp8_tensor(x)
    qw, sw = Q.quant_fp8_tensor(w)
    ba, bsa = Q.quant_fp8_blocks(x, 1, 128)
    bw, bsw = Q.quant_fp8_blocks(w, 128, 128)
    gw, gsw = Q.quant_fp8_blocks(w, 1, 128)
    gsw = gsw.t().contiguous()
    for dt in (torch.bfloat16, torch.float32):
        out[f"fp8 {dt}"] = lambda d=dt: G.fp8_gemm_packed(qa, qw, sa, sw, out_dtype=d)
        out[f"fp8 block {dt}"] = lambda d=dt: G.fp8_gemm_packed(ba, bw, bsa, bsw, block=True, out_dtype=d)
        out[f"fp8 group {dt}"] = lambda d=dt: G.fp8_gemm_packed(ba, gw, bsa, gsw, group=True, out_dtype=d)
        out[f"bf16 {dt}"] = lambda d=dt: G.bf16_gemm(x, w.t(), out_dtype=d)
    ma, msa = Q.quant_mxfp4(x)
    mw, msw = Q.quant_mxfp4(w)
    va, vsa, vga = Q.quant_nvfp4(x)
    vw, vsw, vgw = Q.quant_nvfp4(w)
    out["mxfp4"] = lambda: G.fp4_gemm_packed(ma, msa, mw, msw)
    out["nvfp4"] = lambda: G.fp4_gemm_packed(va, vsa, vw, vsw, fmt="nvfp4", global_a=vga, global_w=vgw)
    gam = _bf16((k,), 3)
    for f in ("fp8", "mxfp4"):
        out[f"rmsnorm {f}"] = lambda f=f: F.rmsnorm_quant(x, gam, fmt=f)
        out[f"swiglu {f}"] = lambda f=f: F.swiglu_quant(x, fmt=f)
    e, topk = 8, 2
    ids = torch.randint(0, e, (m, topk), generator=torch.Generator().manual_seed(4), dtype=torch.int32).to(DEV)
    tw = torch.rand((m, topk), generator=torch.Generator().manual_seed(5)).to(DEV)
    we = _bf16((e * n, k), 6, 0.05)
    qe, se = Q.quant_fp8_blocks(we, 1, k)
    qe, se = qe.view(e, n, k), se.view(e, n)
    off = torch.arange(0, e * m + 1, m, dtype=torch.int32, device=DEV)
    xg = _bf16((e * m, k), 7)
    qx, sx = Q.quant_fp8_blocks(xg, 1, k)
    out["grouped"] = lambda: G.grouped_fp8_gemm_packed(qx, sx, qe, se, off)
    out["moe"] = lambda: M.routed_grouped_gemm(x, ids, tw, (qe, se))
    la, lb = _bf16((2, k, 8), 8, 0.05), _bf16((2, 8, n), 9, 0.05)
    ls = torch.tensor([0.5, 2.0], device=DEV)
    out["lora"] = lambda: G.lora_fused_gemm(x, w.t(), la, lb, ls)
    return out


def _flat(r):
    return list(r) if isinstance(r, tuple) else [r]


@pytest.mark.parametrize("m,n,k", [(1, 256, 512), (33, 200, 640), (700, 264, 2304)])
def test_native_calls_give_the_python_paths_bytes(m, n, k, monkeypatch):
    calls = _calls(m, n, k)
    fast = {nm: _flat(f()) for nm, f in calls.items()}
    taken = []
    real = N.fast()

    class Spy:
        def __getattr__(self, nm):
            def f(*a):
                r = getattr(real, nm)(*a)
                taken.append((nm, r is not None))
                return r
            return f

    monkeypatch.setattr(N, "fast", Spy)
    for f in calls.values():
        f()
    assert all(ok for nm, ok in taken), [t for t in taken if not t[1]]
    monkeypatch.setattr(N, "fast", N._NoFast)
    for nm, f in calls.items():
        for a, b in zip(fast[nm], _flat(f())):
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride(), nm
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), nm


def test_odd_calls_are_left_to_python():
    fast = N.fast()
    x, w = _bf16((32, 512), 1), _bf16((64, 512), 2)
    (qa, sa), (qw, sw) = Q.quant_fp8_tensor(x), Q.quant_fp8_tensor(w)
    bf = torch.bfloat16

    class Sub(torch.Tensor):
        pass

    assert fast.quant_fp8_tensor(x.half()) is None
    assert fast.quant_fp8_tensor(x.cpu()) is None
    assert fast.quant_fp8_tensor(x[:0]) is None
    assert fast.quant_fp8_tensor(x.as_subclass(Sub)) is None
    assert fast.quant_fp8_tensor(3) is None
    assert fast.quant_fp8_blocks(x, 0, 128) is None
    assert fast.quant_fp8_blocks(x, 1 << 80, 128) is None
    assert fast.quant_fp8_blocks(x, 1.0, 128) is None
    assert fast.quant_mxfp4(x[:, :500]) is None
    assert fast.fp8_gemm(qa, qw, sa, sw, N.SCALE_TENSOR, "bfloat16") is None
    assert fast.fp8_gemm(qa[:, :496], qw, sa, sw, N.SCALE_TENSOR, bf) is None
    assert fast.fp8_gemm(qa, qw[:, 16:], sa, sw, N.SCALE_TENSOR, bf) is None
    assert fast.fp8_gemm(qa, qw, 1.0, sw, N.SCALE_TENSOR, bf) is None
    assert fast.fp8_gemm(qa, qw, sa, sw, N.SCALE_BLOCK128, bf) is None
    assert fast.fp8_gemm(qa, qw, sa, sw, 7, bf) is None
    assert fast.fp4_gemm(qa, sa, qw, sw, N.FMT_MXFP4, None, None, bf) is None
    assert fast.bf16_gemm(x, w, bf) is None
    assert fast.bf16_gemm(x, w.t().contiguous(), bf) is None
    assert fast.bf16_gemm(x, w.t(), torch.float16) is None
    assert fast.rmsnorm_quant(x, w[0], 1, N.QFMT_MXFP4) is None
    with pytest.raises(ValueError, match="K mismatch"):
        G.fp8_gemm_packed(qa[:, :256].contiguous(), qw, sa, sw)


@pytest.mark.parametrize("m,n,k,rank,loras", [
    (1, 200, 136, 8, 1), (2, 72, 64, 16, 3), (40, 200, 136, 8, 3), (300, 264, 1096, 16, 5),
    (512, 1024, 512, 16, 4), (700, 2056, 320, 72, 1), (1500, 2048, 1024, 32, 4)])
def test_lora_adapters_packed_by_the_call(m, n, k, rank, loras):
    """Contiguous adapters are turned to K-major rows by the call's own kernel;
    a strided view of the same values takes the copies, with the same bytes."""
    g = torch.Generator(device="cuda").manual_seed(m + n)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").bfloat16()
    x, w, a, b = r(m, k), r(n, k).t(), r(loras, k, rank), r(loras, rank, n)
    s = torch.rand(loras, generator=g, device="cuda")
    a2 = torch.zeros((loras, k, rank + 1), dtype=a.dtype, device="cuda")
    a2[:, :, :rank] = a
    got = G.lora_fused_gemm(x, w, a, b, s)
    assert torch.equal(got, G.lora_fused_gemm(x, w, a2[:, :, :rank], b, s))
    ref = x.double() @ w.double()
    for l in range(loras):
        ref += s[l].double() * (x.double() @ a[l].double()) @ b[l].double()
    assert (got.double() - ref).abs().max() <= 2e-5 * ref.abs().max()


def test_native_calls_run_on_the_current_stream_and_in_threads():
    """The extension looks up the stream itself and runs without the GIL: calls on
    side streams and from threads of their own give the bytes of calls in order."""
    import threading
    shapes = [(33, 200, 640), (16, 512, 1024)]
    want = {}
    for s in shapes:
        want[s] = {nm: [t.clone() for t in _flat(f())] for nm, f in _calls(*s).items()}
    torch.cuda.synchronize()
    bad = []

    def work(s):
        try:
            st = torch.cuda.Stream()
            with torch.cuda.stream(st):
                calls = _calls(*s)
                got = [{nm: _flat(f()) for nm, f in calls.items()} for _ in range(4)]
                busy = torch.empty(1 << 22, device=DEV).normal_()      # later work on the stream's freed scratch
                busy.mul_(2)
            st.synchronize()
            for r in got:
                for nm, ts in r.items():
                    bad.extend(nm for a, b in zip(ts, want[s][nm])
                               if not torch.equal(a.view(torch.uint8), b.view(torch.uint8)))
        except Exception as exc:          # a thread's error is the test's
            bad.append(repr(exc))

    threads = [threading.Thread(target=work, args=(s,)) for s in shapes * 2]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad


def test_a_call_waits_for_its_stream_only():
    """Work queued on a side stream first: the call's result needs it, so a launch
    on another stream would read the inputs before they are written."""
    x = torch.zeros((512, 4096), dtype=torch.bfloat16, device=DEV)
    src = _bf16((512, 4096), 21)
    big = torch.empty(1 << 28, device=DEV)
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        for _ in range(4):
            big.fill_(1.0)                # a few hundred microseconds
        x.copy_(src)
        q, s = Q.quant_fp8_blocks(x, 1, 128)
    st.synchronize()
    q_ref, s_ref = Q.quant_fp8_blocks(src, 1, 128)
    assert torch.equal(q, q_ref) and torch.equal(s, s_ref)
