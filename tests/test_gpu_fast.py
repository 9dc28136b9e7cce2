"""The C++ call path of fastmlx_amd/ops.py against its Python path: the same bits for the
calls both take, the Python path's errors for the calls only it answers."""
import numpy as np
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu


def _weights(lead, K, bits, group, gpu, seed):
    g = torch.Generator().manual_seed(seed)
    w = torch.randint(-2**31, 2**31 - 1, (*lead, K * bits // 32), generator=g, dtype=torch.int32)
    s = (torch.rand(*lead, K // group, generator=g) * 0.01 + 0.002).bfloat16()
    return w.to(gpu), s.to(gpu), (-8 * s).to(gpu)


def _calls(gpu, bits, group):
    from fastmlx_amd import ops

    w = _weights((96,), 512, bits, group, gpu, 1)
    x = torch.randn(2, 3, 512, generator=torch.Generator().manual_seed(2)).bfloat16().to(gpu)
    bias = torch.randn(96, generator=torch.Generator().manual_seed(3)).bfloat16().to(gpu)
    E, T, D, I = 6, 5, 512, 256
    up = [_weights((E, I), D, bits, group, gpu, 4 + i) for i in range(2)]
    down = _weights((E, D), I, bits, group, gpu, 6)
    shared = [_weights((1, I), D, bits, group, gpu, 7), _weights((1, I), D, bits, group, gpu, 8),
              _weights((1, D), I, bits, group, gpu, 9)]
    xt = x.view(-1, D)[:T].contiguous()
    logits = torch.randn(T, E, generator=torch.Generator().manual_seed(5)).bfloat16().to(gpu)

    def run():
        out = torch.empty(2, 3, 96, dtype=torch.bfloat16, device=gpu)
        y = ops.quantized_matmul(x, *w, True, group, bits, None, out)
        assert y is out
        d = ops.dequantize(*w, group, bits)
        inds, wts = ops.route_softmax_topk(logits, 2)
        gi, gw = ops.route_group_topk(logits.float(), None, 2, 3, 2, 1.5)
        return [y, ops.quantized_matmul(x, *w, True, group, bits, bias), d,
                *ops.quantize(d, group, bits), inds, wts, gi, gw,
                ops.moe_layer(xt, inds, *up, down, wts, shared, None, group, bits),
                ops.switch_glu_combine(xt, inds, *up, down, wts, xt, logits[:, 0].contiguous(), group,
                                       bits)]

    return run


@pytest.mark.parametrize("bits,group", [(4, 64), (8, 32)])
@pytest.mark.parametrize("mode", ["plain", "inference", "graph"])
def test_fast_path_matches_python_path(gpu, monkeypatch, bits, group, mode):
    from fastmlx_amd import ops

    assert ops._fast is not None, "fastmlx_amd/_fast.so is not built"
    announce(f"fast path {bits}-bit group {group} {mode}")
    run = _calls(gpu, bits, group)
    got = run()
    if mode == "inference":
        with torch.inference_mode():
            got = run()
        assert all(t.is_inference() for t in got)
    elif mode == "graph":
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            run()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            got = run()
        for t in got:
            t.zero_()
        for _ in range(2):
            graph.replay()
            torch.cuda.synchronize()
    monkeypatch.setattr(ops, "_fast", None)
    want = run()
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)


def test_fast_path_refusals(gpu):
    """What the Python path refuses stays refused with its message, and what only it takes
    is answered."""
    from fastmlx_amd import FmxqError, ops

    announce("fast path refusals")
    w, s, b = _weights((64,), 256, 4, 64, gpu, 1)
    x = torch.randn(4, 512, device=gpu).bfloat16()
    with pytest.raises(ValueError, match="contiguous"):
        ops.quantized_matmul(x[:, ::2], w, s, b)
    with pytest.raises(ValueError, match="K=512"):
        ops.quantized_matmul(x, w, s, b)
    with pytest.raises(TypeError, match="dtype"):
        ops.quantized_matmul(x[:, :256].float(), w, s, b)
    with pytest.raises(ValueError, match="GPU"):
        ops.quantized_matmul(x[:, :256].contiguous(), w.cpu(), s, b)
    with pytest.raises(FmxqError):
        ops.quantized_matmul(x[:, :256].contiguous(), w, s, b, False)
    with pytest.raises(FmxqError):
        ops.dequantize(w, s, b, 16)
    with pytest.raises(FmxqError):
        ops.route_softmax_topk(x, 65)
    misaligned = torch.zeros(256 + 8, dtype=torch.bfloat16, device=gpu)[1:257].view(1, 256)
    with pytest.raises(FmxqError):
        ops.quantized_matmul(misaligned, w, s, b)
    assert ops.quantized_matmul(x[:0, :256], w, s, b).shape == (0, 64)
    param = torch.nn.Parameter(x[:, :256].contiguous())
    y = ops.quantized_matmul(param, w, s, b)
    assert not y.requires_grad and torch.equal(y, ops.quantized_matmul(param.data, w, s, b))


class _Recorder:
    """fastmlx_amd._fast with a note of what each call returned."""

    def __init__(self, mod):
        self.mod, self.calls = mod, []

    def __getattr__(self, name):
        def call(*args):
            r = getattr(self.mod, name)(*args)
            self.calls.append((name, r is not None))
            return r
        return call


NAMES = {"quantized_matmul", "dequantize", "quantize", "moe_layer", "route_softmax_topk",
         "route_group_topk"}


@pytest.mark.parametrize("mode", ["plain", "inference", "graph"])
def test_fast_path_answers_plain_calls(gpu, monkeypatch, mode):
    """Every function of the module answers the plain calls itself."""
    from fastmlx_amd import ops

    announce(f"fast path answers {mode}")
    run = _calls(gpu, 4, 64)
    run()
    rec = _Recorder(ops._fast)
    monkeypatch.setattr(ops, "_fast", rec)
    if mode == "plain":
        run()
    elif mode == "inference":
        with torch.inference_mode():
            run()
    else:
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            run()
        stream.synchronize()
        rec.calls.clear()
        with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=stream):
            run()
    torch.cuda.synchronize()
    assert {n for n, _ in rec.calls} == NAMES and all(ok for _, ok in rec.calls), rec.calls


class _Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("what", ["dispatch mode", "function mode", "subclass"])
def test_fast_path_declines(gpu, monkeypatch, what):
    """Modes that watch calls and tensor subclasses take the Python path, with its values."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from fastmlx_amd import ops

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    announce(f"fast path declines: {what}")
    w, s, b = _weights((64,), 256, 4, 64, gpu, 1)
    x = torch.randn(4, 256, generator=torch.Generator().manual_seed(2)).bfloat16().to(gpu)
    want = ops.quantized_matmul(x, w, s, b)
    rec = _Recorder(ops._fast)
    monkeypatch.setattr(ops, "_fast", rec)
    if what == "subclass":
        got = ops.quantized_matmul(x.as_subclass(_Sub), w, s, b)
    else:
        with Dispatch() if what == "dispatch mode" else Function():
            got = ops.quantized_matmul(x, w, s, b)
    assert rec.calls == [("quantized_matmul", False)] and torch.equal(got, want)


def test_fast_path_raises_the_librarys_refusal(gpu, monkeypatch):
    """A refused call is made once: the error comes from the C++ path, in the Python path's
    form, without a second attempt."""
    from fastmlx_amd import FmxqError, ops

    announce("fast path raises a refusal")
    w, s, b = _weights((64,), 256, 4, 64, gpu, 1)
    x = torch.zeros(256 + 8, dtype=torch.bfloat16, device=gpu)[1:257].view(1, 256)

    def second(*_):
        raise AssertionError("a second attempt")

    fast = ops._fast
    monkeypatch.setattr(ops, "_fast", None)
    with pytest.raises(FmxqError) as want:
        ops.quantized_matmul(x, w, s, b)
    monkeypatch.setattr(ops, "_fast", fast)
    monkeypatch.setattr(ops, "load", second)
    with pytest.raises(FmxqError) as got:
        ops.quantized_matmul(x, w, s, b)
    assert str(got.value) == str(want.value) and got.value.code == want.value.code
