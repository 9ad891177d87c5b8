"""The native entry of the torch-facing ops (csrc/torch_ops.cpp) against their
Python form: the same calls, once as they are and once under an empty torch
function mode, which sends every op down its Python form.  Results have to be
the same bits, whether a call's operands are plain (the native entry takes
it) or not (views, ranks, strides and workspaces it leaves alone)."""
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
