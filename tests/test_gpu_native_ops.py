"""The native entry of the torch-facing ops (csrc/torch_ops.cpp) against their
Python form: the same calls, once as they are and once under an empty torch
function mode, which sends every op down its Python form.  Results have to be
the same bits, whether a call's operands are plain (the native entry takes
it) or not (views, ranks, strides and workspaces it leaves alone)."""
import numpy as np
import pytest
import torch
from torch.overrides import TorchFunctionMode

from gpu_util import normal

pytestmark = pytest.mark.gpu


class PythonForm(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def n(dev, *shape, seed=1, std=1.0, dtype=torch.float16):
    return normal(shape, seed, std, dtype=dtype).to(dev)


def calls(pkg, dev):
    """(name, whether the native entry takes it, call)"""
    x, w, b = n(dev, 40, 64), n(dev, 96, 64, seed=2), n(dev, 96, seed=3)
    wide = n(dev, 40, 80)
    qkv = n(dev, 2, 50, 3, 4, 64, seed=4)
    q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))  # [2, 4, 50, 64], heads 64 apart
    one = [t[:1] for t in (q, k, v)]
    kx = n(dev, 2, 1, 50, 64, seed=5).expand(2, 4, 50, 64)
    q3 = n(dev, 2, 3, 4, 50, 64, seed=12)
    masks = [(n(dev, *sh, seed=13), True) for sh in
             ((1, 1, 1, 50, 50), (2, 1, 1, 50, 50), (2, 3, 1, 50, 50), (2, 3, 4, 50, 50))]
    masks += [(n(dev, *sh, seed=13), False) for sh in ((1, 3, 1, 50, 50), (1, 1, 4, 50, 50), (2, 1, 4, 50, 50))]
    masks += [(n(dev, *sh, seed=13), True) for sh in ((1, 50, 50), (1, 1, 50, 50))]
    masks += [(n(dev, *sh, seed=13), False) for sh in ((4, 50, 50), (3, 1, 50, 50))]
    masks += [(n(dev, 2, 3, 1, 50, 64, seed=13)[..., 7:57], True), (n(dev, 2, 3, 1, 50, 50) > 0, False)]
    s, g = n(dev, 64, 96, 40, seed=6), n(dev, 40, seed=7)
    wq = torch.randint(-127, 128, (96, 64), dtype=torch.int8, generator=torch.Generator().manual_seed(8)).to(dev)
    sc = (torch.rand(96, generator=torch.Generator().manual_seed(9)) * 9e-3 + 1e-3).half().to(dev)
    bx, bw = x.bfloat16(), w.bfloat16()
    long_x, long_w = n(dev, 33, 4096), n(dev, 128, 4096, seed=10)  # splits K into a workspace
    out = lambda *sh, dt=torch.float16: torch.empty(sh, dtype=dt, device=dev)  # noqa: E731
    rs = torch.rand(40, generator=torch.Generator().manual_seed(11)).to(dev)
    return [
        ("gemm nt", True, lambda: pkg.gemm(x, w, b_layout="nt")),
        ("gemm nn bias alpha out", True,
         lambda: pkg.gemm(x, w.t().contiguous(), epilogue="bias", bias=b, alpha=0.5, out=out(40, 96))),
        ("gemm silu", True, lambda: pkg.gemm(x, w, b_layout="nt", epilogue="silu_mul")),
        ("gemm padded rows", True, lambda: pkg.gemm(wide[:, 8:72], w, b_layout="nt", out=out(40, 104)[:, :96])),
        ("gemm strided bias", False, lambda: pkg.gemm(x, w, b_layout="nt", epilogue="bias", bias=n(dev, 192)[::2])),
        ("gemm workspace", True, lambda: pkg.gemm(long_x, long_w, b_layout="nt")),
        ("gemm no rows", True, lambda: pkg.gemm(x[:0], w, b_layout="nt")),
        ("gemm bf16", True, lambda: pkg.gemm(bx, bw, b_layout="nt")),
        ("linear 3-D gelu", True, lambda: pkg.linear(x.view(5, 8, 64), w, b, epilogue="gelu_tanh")),
        ("linear 3-D view", False, lambda: pkg.linear(wide.view(5, 8, 80)[..., :64], w, b)),
        ("linear vector", True, lambda: pkg.linear(x[3], w)),
        ("bgemm", True, lambda: pkg.bgemm(x.view(4, 10, 64), w.view(4, 24, 64), b_layout="nt")),
        ("bgemm slices", True, lambda: pkg.bgemm(s[:, :, :24], s.transpose(1, 2)[:, :24].contiguous(),
                                                 out=out(64, 96, 104)[..., :96])),
        ("rms_norm_linear", True, lambda: pkg.rms_norm_linear(x, w, 1e-5, bias=b)),
        ("rms_norm_linear scales", True, lambda: pkg.rms_norm_linear(x, w, epilogue="silu_mul", rscale_in=rs)),
        ("rms_norm_linear out", False, lambda: pkg.rms_norm_linear(x, w, 1e-5, out=out(40, 96))),
        ("gemv", True, lambda: pkg.gemv(x[:3], w, b)),
        ("gemv wide M", True, lambda: pkg.gemv(x, w)),
        ("w8a16", True, lambda: pkg.w8a16_linear(x[:5], wq, sc, b)),
        ("rms_norm", True, lambda: pkg.rms_norm(s, g, 1e-5)),
        ("rms_norm rows", False, lambda: pkg.rms_norm(wide[:, :64], w[0], 1e-5)),
        ("softmax", True, lambda: pkg.softmax(s, 0.3)),
        ("softmax out", True, lambda: pkg.softmax(x, 0.3, out=out(40, 64))),
        ("softmax column", False, lambda: pkg.softmax(wide[:, 1:2], 0.3)),
        ("attention", True, lambda: pkg.attention(q.contiguous(), k.contiguous(), v.contiguous(), causal=1)),
        ("attention heads of one row", True, lambda: pkg.attention(*one, 0.2)),
        ("attention heads of two rows", False, lambda: pkg.attention(q, k, v, causal=2)),
        ("attention expanded keys", False, lambda: pkg.attention(q.contiguous(), kx, kx)),
        ("attention grouped bf16", True, lambda: pkg.attention(q.bfloat16().contiguous(), kx[:, :1].bfloat16(),
                                                               kx[:, 1:2].bfloat16())),
        ("attention negative scale", False, lambda: pkg.attention(*one, -0.2)),
        ("attention masked", True, lambda: pkg.attention(*one, mask=n(dev, 50, 50))),
        ("attention out", True, lambda: pkg.attention(*one, out=out(1, 4, 50, 64))),
        ("attention padded out", True, lambda: pkg.attention(*one, out=out(1, 4, 50, 72)[..., 8:])),
        ("attention out off the grid", False, lambda: pkg.attention(*one, out=out(1, 4, 50, 72)[..., 4:68])),
        *((f"attention mask of {tuple(m.shape)} {m.stride()}", plain, lambda m=m: pkg.attention(q3, q3, q3, mask=m))
          for m, plain in masks),
    ]


def test_native_form_equals_python_form(pkg, dev, monkeypatch):
    ops, taken = pkg.hxmi._ops, []
    getattr(ops, "gemm")  # loads the module
    real = pkg.hxmi._ops

    class Spy:
        def __getattr__(self, name):
            def f(*args):
                y = getattr(real, name)(*args)
                taken.append(y is not None)
                return y
            return f

    monkeypatch.setattr(pkg.hxmi, "_ops", Spy())
    for name, native, call in calls(pkg, dev):
        taken.clear()
        got = call()
        assert (True in taken[:1]) == native, name
        with PythonForm():
            taken.clear()
            want = call()
            assert True not in taken, name
        assert got.shape == want.shape and got.dtype == want.dtype, name
        assert torch.equal(got, want), name


def test_native_form_runs_on_the_current_stream(pkg, dev):
    x, w = n(dev, 64, 512), n(dev, 512)
    want = pkg.rms_norm(x, w, 1e-5)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):  # a launch on any other stream would not be captured
        y = pkg.rms_norm(x, w, 1e-5)
    y.zero_()
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        y.zero_()


def test_native_form_leaves_errors_to_python(pkg, dev):
    x, w = n(dev, 4, 64), n(dev, 8, 64)
    for bad in (lambda: pkg.gemm(x, w, b_layout="nn"), lambda: pkg.gemv(x, w.float()), lambda: pkg.softmax(x.cpu()),
                lambda: pkg.rms_norm(x, w[:, :8]), lambda: pkg.attention(x, x, x)):
        with pytest.raises((pkg.HxmiError, IndexError)):
            bad()


def shared_rows(pkg, dev):
    """(name, call, operands whose rows share elements): each operand in turn,
    expanded from one row or a window that moves less than a row."""
    x, w, b = n(dev, 40, 64), n(dev, 96, 64, seed=2), n(dev, 96, seed=3)
    one, window = x[:1].expand(40, 64), n(dev, 1000, seed=21).as_strided((40, 64), (8, 1))
    w1, ww = w[:1].expand(96, 64), n(dev, 1000, seed=22).as_strided((96, 64), (8, 1))
    x3, w3 = window.view(40, 64).as_strided((4, 10, 64), (80, 8, 1)), ww.as_strided((4, 24, 64), (200, 8, 1))
    wq = torch.randint(-127, 128, (96, 64), dtype=torch.int8, generator=torch.Generator().manual_seed(8)).to(dev)
    q1 = wq[:1].expand(96, 64)
    sc = (torch.rand(96, generator=torch.Generator().manual_seed(9)) * 9e-3 + 1e-3).half().to(dev)
    q, k = n(dev, 4, 50, 64, seed=4), n(dev, 4, 1, 64, seed=5).expand(4, 50, 64)
    for xx in (one, window):
        yield "gemm a", lambda a: pkg.gemm(a, w, b_layout="nt"), xx
        yield "linear x", lambda a: pkg.linear(a, w, b), xx
        yield "rms_norm_linear x", lambda a: pkg.rms_norm_linear(a, w, 1e-5), xx
        yield "gemv x", lambda a: pkg.gemv(a, w), xx[:3]
        yield "w8a16 x", lambda a: pkg.w8a16_linear(a, wq, sc), xx[:3]
        yield "w8a16 x, many rows", lambda a: pkg.w8a16_linear(a, wq, sc), xx
        yield "rms_norm x", lambda a: pkg.rms_norm(a, w[0], 1e-5), xx
        yield "softmax x", lambda a: pkg.softmax(a, 0.3), xx
    for yy in (w1, ww):
        yield "gemm b", lambda a: pkg.gemm(x, a, b_layout="nt"), yy
        yield "linear w", lambda a: pkg.linear(x, a, b), yy
        yield "rms_norm_linear w", lambda a: pkg.rms_norm_linear(x, a, 1e-5), yy
        yield "gemv w", lambda a: pkg.gemv(x[:3], a), yy
        yield "fold_rms_weight w", lambda a: pkg.fold_rms_weight(a, x[0]), yy
        yield "quantize_int8 w", lambda a: pkg.hxmi.quantize_int8(a)[0], yy
        yield "gemm nn b", lambda a: pkg.gemm(n(dev, 40, 96), a), yy
    yield "w8a16 wq", lambda a: pkg.w8a16_linear(x[:3], a, sc), q1
    yield "bgemm a", lambda a: pkg.bgemm(a, w.view(4, 24, 64), b_layout="nt"), x3
    yield "bgemm b", lambda a: pkg.bgemm(x.view(4, 10, 64), a, b_layout="nt"), w3
    for dt in (torch.float16, torch.bfloat16):
        yield "attention k", lambda a: pkg.attention(q.to(a.dtype), a, q.to(a.dtype)), k.to(dt)[:, :1].expand(4, 50, 64)
        yield "attention q", lambda a: pkg.attention(a, q.to(a.dtype), q.to(a.dtype)), k.to(dt)[:, :1].expand(4, 50, 64)


def test_rows_that_share_elements(pkg, dev):
    """The results are those of a copy with rows of its own, on the native
    entry's way and on the Python form's."""
    for name, call, t in shared_rows(pkg, dev):
        print(name, tuple(t.shape), t.stride(), flush=True)
        assert t.stride(-2) < t.size(-1)
        want = call(t.clone(memory_format=torch.contiguous_format))
        assert torch.equal(call(t), want), name
        with PythonForm():
            assert torch.equal(call(t), want), name


def test_out_rows_that_share_elements_are_refused(pkg, dev):
    x, w, b = n(dev, 8, 64), n(dev, 96, 64, seed=2), n(dev, 1, 96)
    wq = torch.ones(96, 64, dtype=torch.int8, device=dev)
    out = b.expand(8, 96)
    for bad in (lambda: pkg.gemm(x, w, b_layout="nt", out=out), lambda: pkg.linear(x, w, out=out),
                lambda: pkg.gemv(x, w, out=out), lambda: pkg.w8a16_linear(x, wq, b[0], out=out),
                lambda: pkg.rms_norm_linear(x, w, 1e-5, out=out), lambda: pkg.softmax(x, out=x[:1].expand(8, 64)),
                lambda: pkg.rms_norm(x, w[0], out=x[:1].expand(8, 64)),
                lambda: pkg.bgemm(x.view(1, 8, 64), w.view(1, 96, 64), b_layout="nt", out=out.unsqueeze(0)),
                lambda: pkg.attention(x.view(1, 8, 64), x.view(1, 8, 64), x.view(1, 8, 64),
                                      out=x[:1].expand(1, 8, 64))):
        with pytest.raises(pkg.HxmiError):
            bad()


class Half:
    def __float__(self):
        return 0.5


def test_numbers_that_only_the_python_form_takes(pkg, dev):
    """causal and scale in other forms than int and float: what the Python
    form converts gives its results, what it refuses is refused by its name."""
    q = n(dev, 2, 50, 64)
    for dt in (torch.float16, torch.bfloat16):
        t = q.to(dt)
        want = pkg.attention(t, t, t, causal=1)
        for causal in (1.0, True, np.bool_(True), np.int64(1), np.float32(1)):
            assert torch.equal(pkg.attention(t, t, t, causal=causal), want)
        assert torch.equal(pkg.attention(t, t, t, np.float32(0.5)), pkg.attention(t, t, t, 0.5))
        for causal in (None, 1.5, "1", 3, -1, 1 << 70):
            with pytest.raises(pkg.HxmiError):
                pkg.attention(t, t, t, causal=causal)
    x, w = n(dev, 8, 64), n(dev, 96, 64, seed=2)
    assert torch.equal(pkg.gemm(x, w, b_layout="nt", alpha=Half()), pkg.gemm(x, w, b_layout="nt", alpha=0.5))
    assert torch.equal(pkg.gemm(x, w, b_layout="nt", alpha=2), pkg.gemm(x, w, b_layout="nt", alpha=2.0))
    assert torch.equal(pkg.softmax(x, Half()), pkg.softmax(x, 0.5))
    for bad in (lambda: pkg.gemm(x, w, b_layout="nt", alpha="one"), lambda: pkg.softmax(x, None),
                lambda: pkg.rms_norm(x, w[0], None), lambda: pkg.rms_norm_linear(x, w, "eps")):
        with pytest.raises((TypeError, ValueError)):
            bad()
