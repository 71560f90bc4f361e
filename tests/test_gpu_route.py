"""GPU parity of the routing kernels (moe_route.hip) against the CPU oracle
(oracle/route_ref.py), through the C ABI.

Bar: ids and token_expert_indices bit-exact (the ranking of topk_softmax and
topk_sigmoid compares the logits themselves); weights within rtol 2e-6. The
grouped modes rank by scores the GPU computes with its own exp, so a row may
differ from the oracle only where the oracle's keys tie to within 1e-6; every
such row must still be a valid top-k under the oracle's keys. The reference
tests compare ids after sorting and weights with checkAllclose
(op_tests/test_moeTopkSoftmax.py:102-125, 257-310).
"""
import numpy as np
import pytest
import torch

import aiter_amd as A
from oracle import route_ref as RR

pytestmark = pytest.mark.gpu


def _np(t):
    return t.detach().cpu().numpy()


def _logits(M, E, dtype, seed, dev):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, E, generator=g) * 2
    return x.to(dtype).to(dev)


def _strided(M, k, dtype, dev, pad):
    buf = torch.full((M, k + pad), -7, dtype=dtype, device=dev)
    return buf[:, :k], buf


@pytest.mark.parametrize("E,k", [(8, 2), (60, 6), (128, 8), (256, 8), (384, 8), (1024, 16)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("renorm", [True, False])
def test_topk_softmax_parity(cuda_device, E, k, dtype, renorm):
    M = 1000 if E <= 256 else 300
    x = _logits(M, E, dtype, E * 3 + k, cuda_device)
    w, wbuf = _strided(M, k, torch.float32, cuda_device, 10)   # row stride k+10, as the reference test
    ids, ibuf = _strided(M, k, torch.int32, cuda_device, 10)
    tei = torch.empty(M, k, dtype=torch.int32, device=cuda_device)
    A.topk_softmax(w, ids, tei, x, renorm)
    rw, rids, rtei = RR.topk_softmax_ref(_np(x.float()), k, renorm)
    assert np.array_equal(_np(ids), rids)
    assert np.array_equal(_np(tei), rtei)
    np.testing.assert_allclose(_np(w), rw, rtol=2e-6, atol=1e-9)
    # the padding columns of the strided outputs are untouched
    assert (_np(wbuf[:, k:]) == -7).all() and (_np(ibuf[:, k:]) == -7).all()


@pytest.mark.parametrize("E,S,k", [(256, 1, 8), (256, 2, 8), (128, 8, 6), (60, 4, 4),
                                   (512, 1, 8)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("renorm", [True, False])
def test_topk_softmax_shared_experts(cuda_device, E, S, k, dtype, renorm):
    """topk_softmax's shared-expert fusion against the oracle: routed ids and
    token_expert_indices bit-exact, weights (routed and shared sigmoid)
    within rtol 2e-6, through the Python op and the reference-shaped ctypes
    entry; the shared logits are raised so they would win if they were
    ranked; the padding columns of strided outputs stay untouched."""
    M = 700
    x = _logits(M, E + S, dtype, E * 5 + S, cuda_device)
    x[:, E:] += 8.0
    wbuf = torch.full((M, k + S + 3), -7.0, device=cuda_device)
    w = wbuf[:, :k + S]
    ids, ibuf = _strided(M, k, torch.int32, cuda_device, 5)
    tei = torch.empty(M, k, dtype=torch.int32, device=cuda_device)
    A.topk_softmax(w, ids, tei, x, renorm, S, "sigmoid")
    rw, rids, rtei = RR.topk_softmax_shared_ref(_np(x.float()), k, renorm, S)
    assert np.array_equal(_np(ids), rids)
    assert np.array_equal(_np(tei), rtei)
    np.testing.assert_allclose(_np(w), rw, rtol=2e-6, atol=1e-9)
    assert (_np(wbuf[:, k + S:]) == -7).all() and (_np(ibuf[:, k:]) == -7).all()
    from aiter_amd import ffi
    w2 = torch.empty(M, k + S, device=cuda_device)
    ids2 = torch.empty(M, k, dtype=torch.int32, device=cuda_device)
    ffi.topk_softmax(w2, ids2, None, x, renorm, S, "sigmoid")
    assert torch.equal(ids2, ids) and torch.equal(w2, w)


def test_topk_softmax_ties_and_fused_topk(cuda_device):
    M, E, k = 64, 256, 8
    x = torch.zeros(M, E, device=cuda_device)
    x[1::2, 100:] = 1.0                       # equal maxima: the lowest ids win
    w, ids = A.fused_topk(torch.empty(M, 16, device=cuda_device), x, k, True)
    assert (_np(ids[0::2]) == np.arange(k)).all()
    assert (_np(ids[1::2]) == np.arange(100, 100 + k)).all()
    np.testing.assert_allclose(_np(w), 1.0 / k, rtol=1e-6)
    with pytest.raises(ValueError, match="Number of tokens"):
        A.fused_topk(torch.empty(M + 1, 16, device=cuda_device), x, k, True)


@pytest.mark.parametrize("E,k", [(64, 1), (128, 4), (256, 8)])
def test_topk_sigmoid_parity(cuda_device, E, k):
    x = _logits(500, E, torch.bfloat16, E + k, cuda_device)
    w = torch.empty(500, k, dtype=torch.float32, device=cuda_device)
    ids = torch.empty(500, k, dtype=torch.int32, device=cuda_device)
    A.topk_sigmoid(w, ids, x)
    rw, rids = RR.topk_sigmoid_ref(_np(x.float()), k)
    assert np.array_equal(_np(ids), rids)
    np.testing.assert_allclose(_np(w), rw, rtol=2e-6)


def _check_grouped(x, w, ids, k, n_group, topk_group, renorm, softmax, scaling, bias):
    rw, rids = RR.grouped_topk_ref(x, k, n_group, topk_group, renorm, softmax, scaling, bias)
    gids, gw = _np(ids), _np(w)
    same = (gids == rids).all(axis=1)
    assert same.mean() >= 0.999, same.mean()
    np.testing.assert_allclose(gw[same], rw[same], rtol=2e-6)
    # rows that differ: the GPU's choice is a valid top-k of the oracle's keys
    s = RR.route_scores(x, softmax if bias is None else False)
    c = s if bias is None else s + bias[None, :]
    for r in np.nonzero(~same)[0]:
        chosen = set(gids[r].tolist())
        assert len(chosen) == k
        lo = min(c[r, list(chosen)])
        rest = [c[r, e] for e in rids[r] if e not in chosen]
        assert all(v <= lo + 1e-6 for v in rest), (r, gids[r], rids[r])


# 96 experts in 3 groups are the general kernel's: a wave per row under 1024 tokens,
# 16 lanes above
@pytest.mark.parametrize("M", [37, 2000])
@pytest.mark.parametrize("E,n_group,topk_group,k", [(256, 8, 4, 8), (64, 4, 2, 4), (96, 3, 1, 5)])
@pytest.mark.parametrize("softmax,renorm,scaling", [(True, True, 1.0), (False, False, 2.5),
                                                    (False, True, 1.5)])
def test_grouped_topk_parity(cuda_device, M, E, n_group, topk_group, k, softmax, renorm,
                             scaling):
    x = _logits(M, E, torch.float32, E + n_group, cuda_device)
    w = torch.empty(M, k, dtype=torch.float32, device=cuda_device)
    ids = torch.empty(M, k, dtype=torch.int32, device=cuda_device)
    A.grouped_topk(x, w, ids, n_group, topk_group, renorm, softmax, scaling)
    _check_grouped(_np(x), w, ids, k, n_group, topk_group, renorm, softmax, scaling, None)


@pytest.mark.parametrize("M", [37, 2000])
@pytest.mark.parametrize("E,n_group,topk_group,k", [(256, 8, 4, 8), (64, 4, 2, 6)])
@pytest.mark.parametrize("renorm,scaling", [(True, 2.5), (False, 1.0)])
def test_biased_grouped_topk_parity(cuda_device, M, E, n_group, topk_group, k, renorm, scaling):
    """The DeepSeek-V3 router shape (256 experts, 8 groups, 4 kept, top-8)."""
    x = _logits(M, E, torch.bfloat16, E * 7 + k, cuda_device)
    g = torch.Generator().manual_seed(E)
    bias = (torch.randn(E, generator=g) * 0.3).to(cuda_device)
    w = torch.empty(M, k, dtype=torch.float32, device=cuda_device)
    ids = torch.empty(M, k, dtype=torch.int32, device=cuda_device)
    A.biased_grouped_topk(x, bias, w, ids, n_group, topk_group, renorm, scaling)
    _check_grouped(_np(x.float()), w, ids, k, n_group, topk_group, renorm, False, scaling,
                   _np(bias))


def test_routing_feeds_the_layer(cuda_device):
    """Router logits -> fused_topk -> fused_moe at config A: the same output as
    routing computed by the oracle (bit-identical ids and weights)."""
    from aiter_amd import workloads as W
    cfg = W.CONFIG_A
    wts = W.make_weights(cfg, device=cuda_device, shuffle=True)
    x = W.make_hidden(cfg, device=cuda_device)
    logits = _logits(cfg.tokens, cfg.experts, torch.float32, 5, cuda_device)
    tw, ids = A.fused_topk(x, logits, cfg.topk, True)
    rw, rids, _ = RR.topk_softmax_ref(_np(logits), cfg.topk, True)
    assert np.array_equal(_np(ids), rids)
    out = A.fused_moe(x, wts["w1"], wts["w2"], tw, ids, quant_type=A.QuantType.per_128x128,
                      w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"])
    out2 = A.fused_moe(x, wts["w1"], wts["w2"], torch.from_numpy(rw).to(cuda_device),
                       torch.from_numpy(rids).to(cuda_device), quant_type=A.QuantType.per_128x128,
                       w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"])
    d = (out.float() - out2.float()).abs().max().item()
    assert d <= 2e-2 * out2.float().abs().max().item(), d


def _ranked(row, k):
    """Experts of a row by (value descending, index ascending), NaN and -inf
    never chosen (0x7fffffff past the last candidate); -0 ties with +0."""
    c = [e for e in range(len(row)) if row[e] > -np.inf]
    c.sort(key=lambda e: (-(row[e] + np.float32(0)), e))
    return (c + [0x7FFFFFFF] * k)[:k]


# both sides of every experts-per-lane step of the one-row-per-wave kernel, a
# narrow row on each side of the row count where it hands over
@pytest.mark.parametrize("M,E,k", [(5, 1, 1), (9, 64, 32), (9, 65, 8), (9, 128, 8), (9, 129, 8),
                                   (9, 192, 8), (9, 193, 7), (9, 256, 8), (9, 257, 9), (9, 320, 8),
                                   (9, 321, 8), (9, 384, 8), (9, 385, 8), (9, 512, 8), (9, 513, 8),
                                   (9, 768, 8), (9, 769, 8), (9, 1024, 32), (8191, 16, 3),
                                   (8192, 16, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_route_row_edges(cuda_device, M, E, k, dtype):
    """Ids exact (compared as whole rows, ties included) and weights within
    rtol 2e-6 (the bar above), with masked experts, rows with fewer candidates
    than ranks, NaN, infinities and both zeros."""
    g = torch.Generator().manual_seed(E)
    x = torch.randint(-6, 7, (M, E), generator=g).float() / 2       # many ties
    x[1::4, ::2] = float("-inf")
    x[2, 1:] = float("-inf")                                        # one candidate
    x[3, E // 2] = float("nan")
    x[4, :] = torch.where(torch.arange(E) % 2 == 0, -0.0, 0.0)
    x = x.to(dtype)
    w, ids = A.fused_topk(torch.empty(M, 1, device=cuda_device), x.to(cuda_device), k, True)
    xf, gid, gw = x.float().numpy(), _np(ids), _np(w)
    for r in list(range(min(M, 9))) + [M - 1]:
        want = _ranked(xf[r], k)
        assert gid[r].tolist() == want, r
        v = np.array([xf[r, e] if e < E else -np.inf for e in want], dtype=np.float64)
        with np.errstate(invalid="ignore"):                         # no candidate at all: NaN
            p = np.exp(v - v[0])
        np.testing.assert_allclose(gw[r], p / p.sum(), rtol=2e-6, atol=0)


# both sides of the row counts at which rows of few experts go to 16 lanes
@pytest.mark.parametrize("M,E,k,renorm", [
    (16383, 64, 8, False), (16384, 64, 8, False), (16385, 17, 3, False), (65535, 96, 4, False),
    (65537, 96, 4, False), (65535, 64, 2, True), (65536, 64, 2, True)])
def test_route_many_rows_of_few_experts(cuda_device, M, E, k, renorm):
    x = _logits(M, E, torch.bfloat16, M + E, cuda_device)
    w = torch.empty(M, k, dtype=torch.float32, device=cuda_device)
    ids = torch.empty(M, k, dtype=torch.int32, device=cuda_device)
    tei = torch.empty(M, k, dtype=torch.int32, device=cuda_device)
    A.topk_softmax(w, ids, tei, x, renorm)
    rw, rids, rtei = RR.topk_softmax_ref(_np(x.float()), k, renorm)
    assert np.array_equal(_np(ids), rids) and np.array_equal(_np(tei), rtei)
    np.testing.assert_allclose(_np(w), rw, rtol=2e-6, atol=1e-9)


# more ranks than a row has lanes, on 16 lanes (the last sizes of each form) and not
@pytest.mark.parametrize("M", [41, 1030, 16390])
@pytest.mark.parametrize("E,k", [(64, 17), (60, 32), (40, 31)])
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "grouped softmax", "grouped biased"])
def test_route_more_than_16_ranks(cuda_device, M, E, k, mode):
    x = _logits(M, E, torch.float32, M + E + k, cuda_device)
    w = torch.full((M, k), -7.0, dtype=torch.float32, device=cuda_device)
    ids = torch.full((M, k), -7, dtype=torch.int32, device=cuda_device)
    if mode == "softmax":
        tei = torch.full((M, k), -7, dtype=torch.int32, device=cuda_device)
        A.topk_softmax(w, ids, tei, x, False)
        rw, rids, rtei = RR.topk_softmax_ref(_np(x), k, False)
        assert np.array_equal(_np(tei), rtei)
    elif mode == "sigmoid":
        A.topk_sigmoid(w, ids, x)
        rw, rids = RR.topk_sigmoid_ref(_np(x), k)
    else:
        bias = None
        if mode == "grouped biased":
            bias = (torch.randn(E, generator=torch.Generator().manual_seed(E)) * 0.3).to(cuda_device)
            A.biased_grouped_topk(x, bias, w, ids, 2, 2, True, 1.5)
        else:
            A.grouped_topk(x, w, ids, 2, 2, True, True, 1.5)
        return _check_grouped(_np(x), w, ids, k, 2, 2, True, bias is None, 1.5,
                              None if bias is None else _np(bias))
    assert np.array_equal(_np(ids), rids)
    np.testing.assert_allclose(_np(w), rw, rtol=2e-6, atol=1e-9)


@pytest.mark.parametrize("M,n_group,topk_group", [(12287, 1, 1), (12288, 1, 1), (16383, 2, 1),
                                                  (16385, 2, 1), (16384, 4, 2)])
def test_grouped_many_rows_of_64_experts(cuda_device, M, n_group, topk_group):
    x = _logits(M, 64, torch.float32, M, cuda_device)
    w = torch.empty(M, 6, dtype=torch.float32, device=cuda_device)
    ids = torch.empty(M, 6, dtype=torch.int32, device=cuda_device)
    A.grouped_topk(x, w, ids, n_group, topk_group, True, True, 1.5)
    _check_grouped(_np(x), w, ids, 6, n_group, topk_group, True, True, 1.5, None)


@pytest.mark.parametrize("E,n_group,topk_group", [
    (64, 1, 1), (64, 32, 5), (128, 2, 1), (192, 4, 2), (256, 16, 16), (320, 8, 3), (384, 8, 4),
    (512, 32, 9), (768, 4, 3), (1024, 8, 4), (448, 8, 4), (96, 3, 2), (60, 4, 2)])
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "biased"])
def test_grouped_forms(cuda_device, E, n_group, topk_group, mode):
    """Every lanes-per-group form of the one-row-per-wave kernel, and groups
    that are not whole lanes (the general kernel), against the oracle: ids and
    weights of every rank."""
    _grouped_against_oracle(cuda_device, 41, E, n_group, topk_group, mode)


# one experts-per-lane form of the general kernel each: under 1024 rows a wave per
# row up to 64, 128, 256, 512 and 1024 experts, from there on 16 lanes up to 16, 64,
# 128 and 256 experts
@pytest.mark.parametrize("M", [41, 1030])
@pytest.mark.parametrize("E,n_group,topk_group", [(12, 2, 1), (60, 4, 2), (96, 3, 1), (160, 8, 4),
                                                  (448, 8, 4), (640, 8, 3)])
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "biased"])
def test_grouped_general_kernel(cuda_device, M, E, n_group, topk_group, mode):
    _grouped_against_oracle(cuda_device, M, E, n_group, topk_group, mode)


@pytest.mark.parametrize("E,n_group,topk_group", [
    (64, 1, 1), (64, 32, 5), (128, 2, 1), (192, 4, 2), (256, 16, 16), (320, 8, 3), (384, 8, 4),
    (512, 32, 9), (768, 4, 3), (1024, 8, 4), (448, 8, 4), (96, 3, 2), (60, 4, 2), (160, 8, 4)])
def test_biased_grouped_switched_off_experts(cuda_device, E, n_group, topk_group):
    """A bias of -inf takes an expert out: never chosen while the kept groups
    hold others, of which every rank's id and weight is checked."""
    per = E // n_group
    k = min(8, topk_group * (per - (per + 4) // 5))
    bias = (torch.randn(E, generator=torch.Generator().manual_seed(E)) * 0.3).to(cuda_device)
    bias[::5] = float("-inf")
    ids = _grouped_against_oracle(cuda_device, 41, E, n_group, topk_group, "biased", bias, k)
    assert (ids % 5 != 0).all()


def _grouped_against_oracle(dev, M, E, n_group, topk_group, mode, bias=None, k=None):
    k = k or min(8, topk_group * (E // n_group))
    x = _logits(M, E, torch.float32, E + n_group, dev)
    w = torch.empty(M, k, dtype=torch.float32, device=dev)
    ids = torch.empty(M, k, dtype=torch.int32, device=dev)
    if mode == "biased":
        if bias is None:
            bias = (torch.randn(E, generator=torch.Generator().manual_seed(E)) * 0.3).to(dev)
        A.biased_grouped_topk(x, bias, w, ids, n_group, topk_group, True, 1.5)
    else:
        A.grouped_topk(x, w, ids, n_group, topk_group, True, mode == "softmax", 1.5)
    _check_grouped(_np(x), w, ids, k, n_group, topk_group, True, mode == "softmax", 1.5,
                   None if bias is None else _np(bias))
    return ids
