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
