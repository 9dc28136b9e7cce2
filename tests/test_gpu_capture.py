"""Calls captured into a graph on a stream that has run nothing before: no workspace of the
stream may grow then, so what needs none on some path is served by that path.  Each capture
is replayed with eager work between the replays and checked against the oracle."""
import ctypes

import numpy as np
import pytest
import torch

import parity
from gpu_util import announce, to_dev, to_np
from synth import make_quant, make_x

pytestmark = pytest.mark.gpu


def _new_stream():
    """A stream of its own (torch.cuda.Stream() hands out pooled ones, which an earlier test
    may have used); never destroyed, so its handle is not reused either."""
    hip = ctypes.CDLL("libamdhip64.so")
    s = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0  # non-blocking
    return torch.cuda.ExternalStream(s.value)


def _captured(f):
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=_new_stream()):
        f()
    return g


@pytest.mark.parametrize("bits,group,M,N,K", [
    (8, 32, 2, 256, 8192),      # long rows, a few x rows: the walk in K parts, dot2 GEMV without
    (8, 128, 4, 8192, 512),     # wide outputs likewise
    (8, 32, 16, 512, 512),
    (4, 32, 5, 512, 512),       # the walk in K parts, the prefill GEMM's 64-row tile without
    (4, 128, 33, 512, 512),
    (4, 32, 384, 512, 512),     # the wide GEMM's shared tiles, the prefill GEMM without
    (8, 128, 300, 14336, 4096),
])
def test_quantized_matmul_first_call_captured(gpu, oracle, bits, group, M, N, K):
    from fastmlx_amd import ops

    rng = np.random.default_rng(M + N)
    w, s, b = make_quant(rng, (N,), K, bits, group)
    x = make_x(rng, M, K)
    dw, ds, db, dx = (to_dev(t, gpu) for t in (w, s, b, x))
    y = torch.zeros(M, N, dtype=torch.bfloat16, device=gpu)
    announce(f"first call captured: bits={bits} group={group} M={M} N={N} K={K}")
    g = _captured(lambda: ops.quantized_matmul(dx, dw, ds, db, True, group, bits, None, y))
    ref = parity.DenseRef(x, w, s, b, group, bits)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        parity.check_dense(to_np(y), ref, what="captured")
        parity.check_dense(to_np(ops.quantized_matmul(dx, dw, ds, db, True, group, bits)), ref)


def _gather_case(rng, gpu, bits, group, E, S, xb, N, K):
    q = make_quant(rng, (E, N), K, bits, group)
    x = make_x(rng, xb, 1, K)
    rhs = rng.integers(0, E, size=S).astype(np.uint32)
    lhs = rng.integers(0, xb, size=S).astype(np.uint32)
    dev = [to_dev(t, gpu) for t in (x, *q, rhs, lhs)]
    from fastmlx_amd import ops

    call = lambda out=None: ops.gather_qmm(dev[0], *dev[1:4], dev[4], dev[5], 1, True, group, bits,
                                           False, out)
    sel = rng.choice(S, size=min(S, 200), replace=False)
    ref = parity.gather_refs(x.reshape(xb, K), *q, lhs[sel].astype(np.int32), rhs[sel].astype(np.int32),
                             group, bits)
    return call, lambda y: parity.check_dense(to_np(y).reshape(S, N)[sel], ref, what="gather_qmm")


@pytest.mark.parametrize("bits,group,E,S,N", [
    (4, 32, 8, 40, 1024), (8, 64, 4, 500, 128), (4, 128, 4, 4200, 64),
])
def test_gather_qmm_first_call_captured(gpu, oracle, bits, group, E, S, N):
    """Formats other than 4 bits in groups of 64: the sort's scratch cannot grow, the
    general kernels need none."""
    rng = np.random.default_rng(S)
    call, check = _gather_case(rng, gpu, bits, group, E, S, 64, N, 512)
    y = torch.zeros(S, 1, N, dtype=torch.bfloat16, device=gpu)
    announce(f"gather_qmm first call captured: bits={bits} group={group} S={S}")
    g = _captured(lambda: call(y))
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        check(y)
        check(call())


def _captured_after(stream, warm, f):
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        warm()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        f()
    return g


def test_gather_qmm_captured_within_walk_scratch(gpu, oracle):
    """A stream whose scratch holds the sorted walk of a batch but not the tiles' prepared x:
    captured on the walk."""
    rng = np.random.default_rng(3)
    warm, _ = _gather_case(rng, gpu, 4, 64, 4, 8192, 64, 300, 256)  # N % 32: no tiles
    call, check = _gather_case(rng, gpu, 4, 64, 4, 4200, 4200, 64, 512)
    y = torch.zeros(4200, 1, 64, dtype=torch.bfloat16, device=gpu)
    announce("gather_qmm captured within the walk's scratch")
    g = _captured_after(_new_stream(), warm, lambda: call(y))
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        check(y)
        check(call())


def test_switch_glu_captured_within_walk_scratch(gpu, oracle):
    """The same for SwitchGLU: 9.8 MB from 300 slots of I = 16384, 2.3 MB for the walk of 4200
    slots, 11.4 MB for its tiles."""
    from fastmlx_amd import ops
    from synth import topk_uniform

    rng = np.random.default_rng(4)

    def case(E, T, k, D, I):
        host = [make_quant(rng, (E, I), D, 4, 64), make_quant(rng, (E, I), D, 4, 64),
                make_quant(rng, (E, D), I, 4, 64)]
        x, inds = make_x(rng, T, D), topk_uniform(rng, T, E, k)
        dev = [tuple(to_dev(t, gpu) for t in q) for q in host]
        dx, di = to_dev(x, gpu), to_dev(inds.astype(np.uint32), gpu)
        return (x, inds, *host), lambda out=None: ops.switch_glu(dx, di, *dev, 64, 4, out)

    _, warm = case(8, 300, 1, 256, 16384)
    host, call = case(4, 2100, 2, 2048, 256)
    sel = np.array([0, 1000, 2099])
    sref = parity.SwitchRef(*host, 64, 4, token_sel=sel, fused=False)
    y = torch.zeros(2100, 2, 2048, dtype=torch.bfloat16, device=gpu)
    announce("switch_glu captured within the walk's scratch")
    g = _captured_after(_new_stream(), warm, lambda: call(y))
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        parity.check_switch(to_np(y)[sel], sref, what="captured")
        parity.check_switch(to_np(call())[sel], sref, what="eager")
