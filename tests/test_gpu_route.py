"""GPU parity: the MoE routers (softmax top-k and DeepSeek's group-limited top-k)
against the oracle and the reference's own routing vectors.

The routers are fp32 on the device and fp64 in the oracle.  Picks must agree
exactly except where two candidates at the k-th place differ by less than fp32
can resolve (a near tie); weights agree to 1e-5 relative (fp32 output) or to
bf16 rounding (bf16 output).
"""
import json
import os

import numpy as np
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


def _picks_agree(got_i, want_i, key):
    """Same picks in the same order, or a swap at a near tie of `key`."""
    if np.array_equal(got_i, want_i):
        return True
    for g, w in zip(got_i, want_i):
        if g != w and abs(key[g] - key[w]) > 1e-5 * max(1.0, abs(key[w])):
            return False
    return set(got_i.tolist()) == set(want_i.tolist()) or abs(
        key[got_i[-1]] - key[want_i[-1]]) <= 1e-5


def _check_rows(gi, gw, oi, ow, key, wtol):
    bad = 0
    for t in range(gi.shape[0]):
        if not _picks_agree(gi[t], oi[t], key[t]):
            bad += 1
            continue
        if np.array_equal(gi[t], oi[t]):
            assert np.allclose(gw[t], ow[t], rtol=wtol, atol=wtol * 1e-3), (t, gw[t], ow[t])
    assert bad == 0, f"{bad} rows picked different experts"


def _w_np(w):
    return w.float().cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("T,E,k,in_dtype,out_dtype", [
    (512, 512, 10, torch.bfloat16, torch.bfloat16),   # C3 routing: 512 experts, top-10
    (128, 512, 10, torch.float32, torch.float32),
    (5, 64, 1, torch.float32, torch.float32),         # ragged T (not a multiple of 4 rows)
    (33, 1000, 16, torch.bfloat16, torch.float32),    # E not a multiple of 64
    (8, 1024, 64, torch.float32, torch.float32),      # the largest supported E and k
])
def test_softmax_router(gpu, oracle, T, E, k, in_dtype, out_dtype):
    from fastmlx_amd import ops

    announce(f"route_softmax_topk T={T} E={E} k={k} {in_dtype}->{out_dtype}")
    g = torch.Generator().manual_seed(T * 7 + E)
    logits = torch.randn(T, E, generator=g).to(in_dtype)
    for norm in (True, False):
        inds, w = ops.route_softmax_topk(logits.to(gpu), k, norm, out_dtype)
        torch.cuda.synchronize()
        x = logits.float().numpy()
        oi, ow = oracle.route_softmax_topk(x, k, norm=norm)
        gi = inds.cpu().numpy()
        wtol = 1e-5 if out_dtype == torch.float32 else 2 ** -8
        _check_rows(gi, _w_np(w), oi, ow, x.astype(np.float64), wtol)


@pytest.mark.parametrize("T,E,k,ng,tg,in_dtype,out_dtype", [
    (256, 256, 8, 8, 4, torch.float32, torch.float32),    # C4 routing: DeepSeek-V3 shape
    (256, 256, 8, 8, 4, torch.bfloat16, torch.bfloat16),
    (37, 64, 6, 8, 3, torch.float32, torch.float32),
    (16, 128, 4, 1, 1, torch.float32, torch.float32),     # no group restriction
    (16, 96, 5, 32, 7, torch.float32, torch.float32),     # groups of three experts
    (9, 64, 2, 64, 5, torch.float32, torch.float32),      # one expert per group
])
def test_group_router(gpu, oracle, T, E, k, ng, tg, in_dtype, out_dtype):
    from fastmlx_amd import ops

    announce(f"route_group_topk T={T} E={E} k={k} groups={ng}/{tg} {in_dtype}->{out_dtype}")
    g = torch.Generator().manual_seed(T * 11 + E + ng)
    gates = torch.randn(T, E, generator=g).to(in_dtype)
    bias = (torch.randn(E, generator=g) * 0.1).float()
    for norm, scale in ((True, 2.5), (False, 1.0)):
        inds, w = ops.route_group_topk(gates.to(gpu), bias.to(gpu), k, ng, tg, scale, norm,
                                       out_dtype)
        torch.cuda.synchronize()
        x = gates.float().numpy()
        oi, ow = oracle.route_group_topk(x, bias.numpy(), k, ng, tg, scale, norm)
        sig = 1.0 / (1.0 + np.exp(-x.astype(np.float64)))
        key = sig + bias.numpy().astype(np.float64)
        wtol = 1e-5 if out_dtype == torch.float32 else 2 ** -8
        _check_rows(inds.cpu().numpy(), _w_np(w), oi, ow, key, wtol)


@pytest.mark.parametrize("T,E,k,ng,tg", [
    (6, 1, 1, 0, 0),        # one expert
    (6, 63, 63, 0, 0),      # every expert picked, one lane idle
    (5, 65, 10, 0, 0),      # one expert past a whole wave
    (4, 1024, 64, 0, 0),    # the largest row
    (5, 96, 9, 3, 2),       # group counts that are no power of two
    (5, 130, 12, 5, 3),
    (3, 1024, 8, 2, 1),     # the longest groups: 32 lanes each
    (7, 64, 64, 64, 64),    # one lane per group, every expert picked
])
def test_router_ties(gpu, oracle, T, E, k, ng, tg):
    """Rows of few distinct values: equal scores go to the lower index, inside a lane's
    slots, across lanes and across groups.  Values 1/4 apart are far from any rounding,
    so the picks equal the oracle's exactly."""
    from fastmlx_amd import ops

    announce(f"router ties T={T} E={E} k={k} groups={ng}/{tg}")
    g = torch.Generator().manual_seed(E + k)
    x = torch.randint(-3, 4, (T, E), generator=g).float() * 0.25
    if ng:
        inds, w = ops.route_group_topk(x.to(gpu), None, k, ng, tg, 1.0, True)
        oi, ow = oracle.route_group_topk(x.numpy(), np.zeros(E, np.float32), k, ng, tg, 1.0, True)
    else:
        inds, w = ops.route_softmax_topk(x.to(gpu), k, True, torch.float32)
        oi, ow = oracle.route_softmax_topk(x.numpy(), k, norm=True)
    torch.cuda.synchronize()
    assert np.array_equal(inds.cpu().numpy(), oi)
    assert np.allclose(_w_np(w), ow, rtol=1e-5, atol=1e-7)


def test_router_masked_experts(gpu):
    """A correction bias of -inf takes an expert out; with fewer finite scores than
    picks the masked ones follow in index order, and a NaN score is never picked."""
    from fastmlx_amd import ops

    announce("router with -inf biases and a NaN")
    x = torch.zeros(1, 70)
    x[0, 3], x[0, 69], x[0, 40] = 2.0, 1.0, float("nan")
    bias = torch.full((70,), float("-inf"))
    bias[3] = bias[69] = bias[40] = 0.0
    inds, _ = ops.route_group_topk(x.to(gpu), bias.to(gpu), 4, 1, 1, 1.0, True)
    torch.cuda.synchronize()
    assert inds[0].cpu().tolist() == [3, 69, 0, 1]


def test_group_router_reference_vectors(gpu):
    """The reference fixture of TestDeepseekV3GroupExpertSelectParity
    (compute/models/deepseekv3_test.go:130-163) through the HIP router."""
    from fastmlx_amd import ops

    with open(os.path.join(HERE, "golden", "deepseek_routing.json")) as f:
        cases = json.load(f)["routing"]
    for c in cases:
        announce(f"route_group_topk fixture {c['label']}")
        gates = torch.tensor([c["gates"]], dtype=torch.float32, device=gpu)
        bias = torch.tensor(c["bias"], dtype=torch.float32, device=gpu)
        inds, w = ops.route_group_topk(gates, bias, c["top_k"], c["n_group"], c["topk_group"],
                                       c["routed_scaling_factor"], c["norm_topk_prob"])
        torch.cuda.synchronize()
        got = dict(zip(inds[0].cpu().tolist(), w[0].cpu().tolist()))
        want = dict(zip(c["inds"], c["scores"]))
        assert set(got) == set(want), (c["label"], got, want)
        for e, v in want.items():
            assert abs(got[e] - v) <= 1e-5 * abs(v), (c["label"], e, got[e], v)


def test_router_feeds_switch_glu_combine(gpu, oracle):
    """Router output drives the MoE pieces directly: softmax top-k weights in bf16
    into moe_combine give the oracle's weighted sum of the expert outputs."""
    from fastmlx_amd import ops

    announce("router -> moe_combine")
    T, E, k, D = 16, 64, 4, 256
    g = torch.Generator().manual_seed(5)
    logits = torch.randn(T, E, generator=g).to(torch.bfloat16).to(gpu)
    inds, w = ops.route_softmax_topk(logits, k, True, torch.bfloat16)
    y = torch.randn(T, k, D, generator=g).to(torch.bfloat16).to(gpu)
    out = ops.moe_combine(y, w)
    torch.cuda.synchronize()
    ref = (y.float() * w.float()[:, :, None]).sum(dim=1)
    assert torch.allclose(out.float(), ref, rtol=2e-2, atol=2e-2)
    assert (inds >= 0).all() and (inds < E).all()


def _butterfly(lanes):
    """fp32 sum of 64 lanes in the order of xor steps 32, 16, .. 1."""
    v = lanes.astype(np.float32)
    for off in (32, 16, 8, 4, 2, 1):
        v = v + v[..., np.arange(64) ^ off]
    return v[..., 0]


@pytest.mark.parametrize("E", [64, 512])
def test_softmax_denominator_order(gpu, E):
    """The softmax denominator adds the lanes as xor steps 32, 16, .. 1.  Three experts
    count in each row: 1 in lane 2^q and e = 0.75 * 2^-24 in lanes 0 and 2^p, the others
    exactly 0.  1 + e rounds to 1 and 1 + 2 e to 1 + 2^-23, so the sum shows which of the
    two steps came first."""
    from fastmlx_amd import ops

    announce(f"softmax denominator order E={E}")
    pq = [(p, q) for p in range(6) for q in range(6) if p != q]
    x = torch.full((len(pq), E), float("-inf"))
    for t, (p, q) in enumerate(pq):
        x[t, 2 ** q] = 0.0
        x[t, 0] = x[t, 2 ** p] = float(np.log(0.75 * 2.0 ** -24))
    inds, w = ops.route_softmax_topk(x.to(gpu), 1, False, torch.float32)
    torch.cuda.synchronize()
    w = w.cpu().numpy()[:, 0]
    for t, (p, q) in enumerate(pq):
        s = np.float32(1 + 2.0 ** -23) if p > q else np.float32(1)
        assert int(inds[t, 0]) == 2 ** q
        assert w[t] == np.float32(1) / s, (p, q, w[t])


@pytest.mark.parametrize("T,E,k", [(37, 512, 10), (37, 64, 8), (9, 1024, 64)])
def test_renormalization_order(gpu, T, E, k):
    """The picked weights are divided by their sum over lanes 0 .. k - 1, added as xor
    steps 32, 16, .. 1, in fp32: exact bits from the weights before the division."""
    from fastmlx_amd import ops

    announce(f"renormalization order T={T} E={E} k={k}")
    g = torch.Generator().manual_seed(T + E + k)
    x = torch.randn(T, E, generator=g).to(gpu)
    for route in (lambda norm: ops.route_softmax_topk(x, k, norm, torch.float32),
                  lambda norm: ops.route_group_topk(x, None, k, 8, 8, 1.0, norm, torch.float32)):
        i0, w0 = route(False)
        i1, w1 = route(True)
        torch.cuda.synchronize()
        assert torch.equal(i0, i1)
        w0, w1 = w0.cpu().numpy(), w1.cpu().numpy()
        lanes = np.zeros((T, 64), dtype=np.float32)
        lanes[:, :k] = w0
        assert np.array_equal(w1, w0 / _butterfly(lanes)[:, None])
