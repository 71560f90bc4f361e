"""GPU parity of the HIP path against the CPU oracle (all through the C ABI).

Bar: sorting metadata and activation quantisation are bit-exact with the
oracle; the MoE outputs agree with the fp32-dequant oracle within the
normalised tolerance of the reference's MoE tests (max-rel <= 2e-2,
RMS-rel <= 4e-3, op_tests/triton_tests/moe/test_moe_gemm_a8w4.py:104-160).
"""
import importlib

import numpy as np
import pytest
import torch

import aiter_amd as A
from aiter_amd import workloads as W
from oracle import moe_ref as R

import _fullshape

pytestmark = pytest.mark.gpu

MAXTOL, RMSTOL = R.MAXTOL, R.RMSTOL


def _np(t):
    return t.detach().cpu().numpy()


def _routing_np(T, E, k, seed):
    rng = np.random.default_rng(seed)
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    w = rng.random((T, k), dtype=np.float32)
    return ids, w


# -------------------------------------------------------------- sorting ---
SORT_CASES = [
    # T, E, k, bm, masked, local_tokens
    (1, 256, 8, 16, False, None), (7, 32, 5, 32, False, None), (31, 32, 5, 32, True, None),
    (32, 256, 8, 16, False, None), (64, 8, 2, 16, False, None), (128, 256, 8, 32, False, None),
    (256, 256, 8, 64, True, None), (1000, 257, 9, 32, False, None),
    (2048, 256, 8, 64, False, None), (8192, 256, 8, 64, False, None),
    (8192, 256, 8, 32, True, None), (300, 256, 8, 32, False, 250), (33, 4096, 1, 16, False, None),
    (4096, 256, 8, 64, False, 4000), (163840, 32, 5, 32, False, None),
    (37, 32, 16, 16, False, None), (600, 64, 16, 32, True, None), (45, 1, 1, 64, False, None),
]


@pytest.mark.parametrize("T,E,k,bm,masked,local", SORT_CASES)
def test_sorting_bit_exact(cuda_device, T, E, k, bm, masked, local):
    ids, w = _routing_np(T, E, k, seed=T * 7 + E)
    mask = np.random.default_rng(T).integers(0, 2, E).astype(np.int32) if masked else None
    H = 256
    ids_t = torch.from_numpy(ids).to(cuda_device)
    w_t = torch.from_numpy(w).to(cuda_device)
    mask_t = torch.from_numpy(mask).to(cuda_device) if masked else None
    loc_t = torch.tensor([local], dtype=torch.int32, device=cuda_device) if local else None
    sid, sw, se, nv, buf = A.moe_sorting(ids_t, w_t, E, H, torch.bfloat16, bm, mask_t, loc_t)
    # moe_buf rows of local tokens are zeroed (it came from torch.empty)
    tokens = T if local is None else local
    assert torch.count_nonzero(buf[:tokens]).item() == 0
    ref = R.moe_sorting_argsort(ids, w, E, bm, mask, local)
    nv = _np(nv)
    assert np.array_equal(nv, ref[3])
    n = int(nv[0])
    assert np.array_equal(_np(sid)[:n], ref[0])
    assert np.array_equal(_np(sw)[:n].view(np.int32), ref[1].view(np.int32))
    assert np.array_equal(_np(se)[: n // bm], ref[2])


@pytest.mark.parametrize("ct", [1, 8, 32, 128])
def test_sorting_chunk_size_invariant(cuda_device, monkeypatch, ct):
    """The multi-chunk sort (AITER_AMD_SORT_CT forces tokens per chunk) gives
    the oracle's arrays bit for bit whatever the chunking: one token per
    chunk, a chunk per 8 tokens (one 64-bit word of slot masks), and larger
    ones; with a duplicated id inside a token's top-k, an out-of-range id and
    an expert mask."""
    monkeypatch.setenv("AITER_AMD_SORT_CT", str(ct))
    T, E, k, bm = 1000, 64, 6, 32
    ids, w = _routing_np(T, E, k, seed=ct + 5)
    ids[3, 1] = ids[3, 0]          # a duplicate expert inside one token's top-k
    ids[7, 2] = E + 3              # an id out of range
    mask = np.random.default_rng(ct).integers(0, 2, E).astype(np.int32)
    sid, sw, se, nv, buf = A.moe_sorting(torch.from_numpy(ids).to(cuda_device),
                                         torch.from_numpy(w).to(cuda_device), E, 256,
                                         torch.bfloat16, bm, torch.from_numpy(mask).to(cuda_device))
    ref = R.moe_sorting_argsort(ids, w, E, bm, mask, None)
    nv = _np(nv)
    assert np.array_equal(nv, ref[3])
    n = int(nv[0])
    assert np.array_equal(_np(sid)[:n], ref[0])
    assert np.array_equal(_np(sw)[:n].view(np.int32), ref[1].view(np.int32))
    assert np.array_equal(_np(se)[: n // bm], ref[2])
    assert torch.count_nonzero(buf).item() == 0


@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
@pytest.mark.parametrize("prequant", [False, True])   # bf16 and fp32 per-pair rows
@pytest.mark.parametrize("bm", [16, 64, 128])
def test_mask_with_more_experts_than_weights(cuda_device, weights, prequant, bm):
    """An expert_mask that sets more experts than the weights hold: the ones
    past the weights add nothing, on per-pair rows as on the accumulator. The
    workspace comes from memory that held NaN, so a row that is summed but
    never written shows."""
    cfg = W.MoEConfig("over", 400, 1024, 256, 4, 3, seed=bm, weights=weights)
    wts = W.make_weights(cfg, device=cuda_device)
    x = W.make_hidden(cfg, device=cuda_device)
    tw, _ = W.make_routing(cfg, device=cuda_device)
    g = torch.Generator().manual_seed(bm)
    ids = torch.rand(400, 8, generator=g).argsort(1)[:, :3].to(torch.int32).to(cuda_device)
    kw = dict(w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"], block_size_M=bm)
    if prequant:
        x, kw["a1_scale"] = A.per_group_quant_hip(x)

    def run(mask):
        junk = [torch.full((n,), float("nan"), device=cuda_device) for n in (1 << 22, 1 << 23)]
        del junk
        return W.run_layer(weights, x, wts["w1"], wts["w2"], tw, ids, **kw,
                           expert_mask=torch.tensor(mask, dtype=torch.int32, device=cuda_device))

    got, want = run([1] * 8), run([1] * 4 + [0] * 4)
    assert torch.count_nonzero(want).item() > 0
    # on the accumulator a token's three terms may add in another order
    tol = 0 if bm >= 64 else 4 * 2.0 ** -8
    assert ((got.float() - want.float()).abs() <= tol * want.float().abs().max()).all()


# both sides of every limit of the one-bit-per-pair sort: words of 32 pairs,
# 2048 pairs in one workgroup, 256 and 512 experts, its LDS table, one thread's
# second pair; block sizes that divide by 1 and by the largest; chunks of the
# scatter launch with a last partial one
@pytest.mark.parametrize("T,E,k,bm,masked,local", [
    (1, 1, 1, 1, False, None), (31, 7, 1, 16, True, None), (32, 64, 1, 1, False, None),
    (33, 65, 1, 256, True, None), (128, 64, 2, 32, True, 0), (129, 64, 2, 32, False, 77),
    (256, 256, 8, 16, True, 255), (257, 256, 8, 1, False, None), (227, 257, 9, 256, True, None),
    (228, 257, 9, 48, False, 200), (64, 512, 8, 16, True, None), (200, 512, 8, 16, False, None),
    (64, 513, 8, 16, True, None), (64, 40, 32, 16, False, None), (65, 40, 32, 16, True, 40),
    (700, 512, 8, 64, True, None), (701, 256, 8, 256, False, 650), (5000, 300, 8, 1, True, 4999),
    (700, 513, 8, 64, False, None)])
def test_sorting_bit_table_edges(cuda_device, T, E, k, bm, masked, local):
    ids, w = _routing_np(T, E, k, seed=T * 3 + E)
    if k > 1:
        ids[T // 2, 1] = ids[T // 2, 0]       # a duplicate inside one token's top-k
    ids[T - 1, k - 1] = E                     # out of range
    mask = np.random.default_rng(E).integers(0, 2, E).astype(np.int32) if masked else None
    dev = lambda a, dt=None: None if a is None else torch.as_tensor(a, dtype=dt, device=cuda_device)
    loc = dev([local], torch.int32) if local is not None else None
    sid, sw, se, nv, buf = A.moe_sorting(dev(ids), dev(w), E, 256, torch.bfloat16, bm, dev(mask), loc)
    ref = R.moe_sorting_argsort(ids, w, E, bm, mask, local)
    assert torch.count_nonzero(buf[:T if local is None else local]).item() == 0
    assert np.array_equal(_np(nv), ref[3])
    n = int(ref[3][0])
    assert np.array_equal(_np(sid)[:n], ref[0])
    assert np.array_equal(_np(sw)[:n].view(np.int32), ref[1].view(np.int32))
    assert np.array_equal(_np(se)[: n // bm], ref[2])


def test_sorting_worked_example(cuda_device):
    """The reference's worked example (csrc/include/moe_sorting_opus.h:277-339,
    fixture tests/golden/moe_sorting_worked_example.json), every output array."""
    from pathlib import Path
    import json

    g = json.loads((Path(__file__).resolve().parent / "golden" /
                    "moe_sorting_worked_example.json").read_text())
    ids = torch.tensor(g["topk_ids"], dtype=torch.int32, device=cuda_device)
    w = torch.tensor(g["topk_weights"], dtype=torch.float32, device=cuda_device)
    for variant in ("unmasked", "masked"):
        exp = g[variant]
        mask = exp.get("expert_mask")
        mask = None if mask is None else torch.tensor(mask, dtype=torch.int32, device=cuda_device)
        sid, sw, se, nv, _ = A.moe_sorting(ids, w, g["num_experts"], 128, torch.bfloat16,
                                            g["block_size"], mask)
        n = exp["num_valid_ids"][0]
        assert _np(nv).tolist() == exp["num_valid_ids"], variant
        assert _np(sid)[:n].tolist() == exp["sorted_token_ids"], variant
        assert _np(sw)[:n].tolist() == exp["sorted_weights"], variant
        assert _np(se)[:n // g["block_size"]].tolist() == exp["sorted_expert_ids"], variant


# ---------------------------------------------------------------- quant ---
@pytest.mark.parametrize("rows,cols,transpose,dtype", [
    (1, 4096, False, torch.bfloat16), (37, 1024, False, torch.bfloat16),
    (64, 4096, True, torch.bfloat16), (300, 2048, False, torch.float16),
])
def test_act_quant_bit_exact(cuda_device, rows, cols, transpose, dtype):
    g = torch.Generator().manual_seed(rows * 31 + cols)
    x = (torch.randn(rows, cols, generator=g) * 3).to(dtype)
    x[0, :128] = 0  # a zero group
    q, s = A.per_group_quant_hip(x.to(cuda_device), transpose_scale=transpose)
    qo, so = R.quant_1x128_kernel(x.float().numpy())
    if transpose:  # [cols/128, rows] data in the [rows, cols/128] buffer, as the reference
        so = np.ascontiguousarray(so.T)
    assert np.array_equal(_np(s).reshape(-1).view(np.int32), so.reshape(-1).view(np.int32))
    assert np.array_equal(_np(q.view(torch.uint8)), qo)


def test_act_quant_num_rows(cuda_device):
    x = torch.randn(16, 512).to(torch.bfloat16).to(cuda_device)
    nr = torch.tensor([5], dtype=torch.int32, device=cuda_device)
    y, s = A.per_group_quant_hip(x, num_rows=nr)
    qo, so = R.quant_1x128_kernel(x[:5].float().cpu().numpy())
    assert np.array_equal(_np(y.view(torch.uint8))[:5], qo)
    assert np.array_equal(_np(s)[:5], so)


# ------------------------------------------------------ fused MoE layer ---
def _make_layer(cfg, device, shuffle, doweight=False, activation="silu"):
    wts = W.make_weights(cfg, device="cpu", shuffle=False)
    x = W.make_hidden(cfg)
    tw, ids = W.make_routing(cfg)
    mask = W.make_expert_mask(cfg)
    w1u = wts["w1"].view(torch.uint8).numpy()
    w2u = wts["w2"].view(torch.uint8).numpy()
    ref = R.fused_moe_ref(x.float().numpy(), w1u, wts["w1_scale"].numpy(), w2u,
                          wts["w2_scale"].numpy(), ids.numpy(), tw.numpy(),
                          None if mask is None else mask.numpy(), doweight_stage1=doweight, activation=activation)
    w1, w2 = wts["w1"], wts["w2"]
    if shuffle:
        w1, w2 = A.shuffle_weight(w1), A.shuffle_weight(w2)
    dev = dict(x=x.to(device), w1=w1.to(device), w2=w2.to(device),
               s1=wts["w1_scale"].to(device), s2=wts["w2_scale"].to(device), tw=tw.to(device),
               ids=ids.to(device), mask=None if mask is None else mask.to(device))
    if shuffle:
        dev["w1"].is_shuffled = True
        dev["w2"].is_shuffled = True
    return dev, ref


def _run(dev, **kw):
    return A.fused_moe(dev["x"], dev["w1"], dev["w2"], dev["tw"], dev["ids"],
                       expert_mask=dev["mask"], quant_type=A.QuantType.per_128x128,
                       w1_scale=dev["s1"], w2_scale=dev["s2"], **kw)


def _check(ref_out, got, tag):
    mx, rms = R.normalized_errors(ref_out, got)
    print(f"[{tag}] max-rel {mx:.3e} rms-rel {rms:.3e}", flush=True)
    assert mx <= MAXTOL and rms <= RMSTOL, (mx, rms)


@pytest.mark.parametrize("shuffle", [True, False])
@pytest.mark.parametrize("bm", [16, 32, 64, 128])
def test_fused_moe_config_a(cuda_device, shuffle, bm):
    cfg = W.CONFIG_A
    dev, ref = _make_layer(cfg, cuda_device, shuffle)
    out = _run(dev, block_size_M=bm)
    assert out.dtype == torch.bfloat16 and out.shape == (cfg.tokens, cfg.model_dim)
    _check(ref["out"], _np(out.float()), f"A shuffle={shuffle} bm={bm}")


def test_stage1_fused_requant_matches_oracle(cuda_device):
    """a2 (fp8 + 1x128 scales) from stage 1 vs the oracle's h -> requant."""
    cfg = W.CONFIG_A
    dev, ref = _make_layer(cfg, cuda_device, True)
    T, k = cfg.tokens, cfg.topk
    a1, a1s = A.per_group_quant_hip(dev["x"])
    assert np.array_equal(_np(a1.view(torch.uint8)), ref["a1q"])
    sid, sw, se, nv, _ = A.moe_sorting(dev["ids"], dev["tw"], cfg.experts, cfg.model_dim,
                                        torch.float32, 32)
    a2, a2s = A.moe_stage1_fp8_blockscale(a1, a1s, dev["w1"], dev["s1"], sid, se, nv, k, 32, True)
    codes = _np(a2.view(torch.uint8)).reshape(T * k, -1)
    got = R.dequant_1x128(codes, _np(a2s).reshape(T * k, -1))
    want = R.dequant_1x128(ref["a2q"].reshape(T * k, -1), ref["a2s"].reshape(T * k, -1))
    # a2 is fp8: the GPU and the oracle sum stage 1 in different orders, so
    # an element sitting on an fp8 rounding tie may land one step apart
    # (one step = 2^-3 relative); everything else must be identical
    mx, rms = R.normalized_errors(want, got)
    print(f"[stage1 a2] max-rel {mx:.3e} rms-rel {rms:.3e}", flush=True)
    ref_codes = ref["a2q"].reshape(T * k, -1)
    flips = codes != ref_codes
    print(f"[stage1 a2] codes differing {flips.mean():.3%}", flush=True)
    assert flips.mean() <= 5e-3 and rms <= RMSTOL

    def signed_step(c):  # position on the e4m3fn number line (+0 and -0 both 0)
        c = c.astype(np.int32)
        return np.where(c & 0x80, -(c & 0x7F), c & 0x7F)

    assert np.abs(signed_step(codes) - signed_step(ref_codes)).max() <= 1
    # scales agree to fp32 rounding of the accumulation order
    np.testing.assert_allclose(_np(a2s), ref["a2s"], rtol=1e-2)


def test_fused_moe_fp8_input_path(cuda_device):
    """fp8 activations + caller a1_scale skip the quant step (fused_moe.py:256-265)."""
    cfg = W.CONFIG_A
    dev, ref = _make_layer(cfg, cuda_device, True)
    a1, a1s = A.per_group_quant_hip(dev["x"])
    out = A.fused_moe(a1, dev["w1"], dev["w2"], dev["tw"], dev["ids"],
                      quant_type=A.QuantType.per_128x128, w1_scale=dev["s1"], w2_scale=dev["s2"],
                      a1_scale=a1s, dtype=torch.bfloat16)
    _check(ref["out"], _np(out.float()), "fp8 input")


@pytest.mark.parametrize("bm", [16, 32, 64, 128])
def test_fused_moe_doweight_stage1(cuda_device, bm):
    """doweight_stage1: the routing weight scales gate and up before SiLU
    and stage 2 sums unweighted (aiter/fused_moe.py:1253, 1330, 1568-1571),
    on the stream (bm 16/32) and prefill (bm 64/128) stage-1 kernels; at bm 32
    also on the stage-wise fp8-input path. The layer with weights after the
    activation differs from it by far more than the tolerance."""
    cfg = W.CONFIG_A
    dev, ref = _make_layer(cfg, cuda_device, True, doweight=True)
    out = _np(_run(dev, block_size_M=bm, doweight_stage1=True).float())
    _check(ref["out"], out, f"doweight_stage1 bm={bm}")
    _, ref_late = _make_layer(cfg, cuda_device, True)
    assert R.normalized_errors(ref_late["out"], out)[0] > 10 * MAXTOL
    if bm == 32:
        a1, a1s = A.per_group_quant_hip(dev["x"])
        out8 = A.fused_moe(a1, dev["w1"], dev["w2"], dev["tw"], dev["ids"],
                           quant_type=A.QuantType.per_128x128, w1_scale=dev["s1"],
                           w2_scale=dev["s2"], a1_scale=a1s, dtype=torch.bfloat16,
                           block_size_M=bm, doweight_stage1=True)
        _check(ref["out"], _np(out8.float()), "doweight_stage1 fp8 input")


@pytest.mark.parametrize("bm", [16, 32, 64, 128])
def test_fused_moe_gelu(cuda_device, bm):
    """ActivationType.Gelu: exact-erf GELU(gate)·up (aiter/ops/quant.py:398-404)
    in every stage-1 kernel (stream at bm 16/32, prefill at bm 64/128); at bm
    64 also with doweight_stage1. The SiLU layer differs by far more than the
    tolerance."""
    cfg = W.CONFIG_A
    dev, ref = _make_layer(cfg, cuda_device, True, activation="gelu")
    out = _np(_run(dev, block_size_M=bm, activation=A.ActivationType.Gelu).float())
    _check(ref["out"], out, f"gelu bm={bm}")
    _fullshape.stagewise_vs_oracle(cfg, dev, ref, out, bm, A.ActivationType.Gelu)
    _, ref_silu = _make_layer(cfg, cuda_device, True)
    assert R.normalized_errors(ref_silu["out"], out)[0] > 10 * MAXTOL
    if bm == 64:
        dev, ref = _make_layer(cfg, cuda_device, True, doweight=True, activation="gelu")
        out = _run(dev, block_size_M=bm, activation=A.ActivationType.Gelu, doweight_stage1=True)
        _fullshape.stagewise_vs_oracle(cfg, dev, ref, _np(out.float()), bm,
                                       A.ActivationType.Gelu, doweight=True)


@pytest.mark.parametrize("bm", [32, 128])
def test_fused_moe_doweight_stage1_ep_share(cuda_device, bm):
    """doweight_stage1 with an expert mask (stream kernels at bm 32, the
    prefill kernels with per-pair stage-2 rows at bm 128). Weighting gate and
    up before SiLU shrinks a2 by about w^2 while the output keeps the
    unweighted sum, so one one-step fp8 requant flip of a2 moves a small
    output by more than the end-to-end max-rel bar; the check is therefore
    per stage, as for the full-size layers: stage 1's fp8 codes on the local
    pairs against the oracle's (at most 0.5% different, each within one
    top-binade e4m3 step of its group, 32/448 of the group amax), then
    the reference's own end-to-end bar (allclose rtol = atol = 0.05 on at
    least 95% of the outputs, op_tests/test_moe_blockscale.py:288) and
    RMS-rel <= 4e-3."""
    cfg = W.MoEConfig("ep_dw", 96, 512, 512, 16, 4, routing="sigmoid", local_experts=4, seed=4)
    dev, ref = _make_layer(cfg, cuda_device, True, doweight=True)
    a1, a1s = A.per_group_quant_hip(dev["x"])
    sid, sw, se, nv, _ = A.moe_sorting(dev["ids"], dev["tw"], cfg.experts, cfg.model_dim,
                                        torch.float32, bm, dev["mask"])
    a2, _ = A.moe_stage1_fp8_blockscale(a1, a1s, dev["w1"], dev["s1"], sid, se, nv, cfg.topk, bm,
                                        True, sorted_weights=sw)
    loc = ref["ids_local"] >= 0
    got = _np(a2.view(torch.uint8))[loc]
    exp = ref["a2q"][loc]
    print(f"[doweight_stage1 EP bm={bm}] stage 1 codes differing {(got != exp).mean():.3%}",
          flush=True)
    assert (got != exp).mean() <= 0.005
    # in the group's own units (codes span +-448): within one top-binade step
    assert np.abs(R.fp8_decode(got) - R.fp8_decode(exp)).max() <= 32
    out = _np(_run(dev, block_size_M=bm, doweight_stage1=True).float())
    far = (~np.isclose(out, ref["out"], rtol=0.05, atol=0.05)).mean()
    mx, rms = R.normalized_errors(ref["out"], out)
    print(f"[doweight_stage1 EP bm={bm}] outside allclose(0.05) {far:.4%} max-rel {mx:.2e} "
          f"rms-rel {rms:.2e}", flush=True)
    assert far <= 0.05 and rms <= RMSTOL


@pytest.mark.parametrize("bm", [None, 64, 128])
def test_fused_moe_ep_share_small(cuda_device, bm):
    """expert_mask: 4 local experts of 16 (sigmoid routing); tokens with no
    local expert give zero rows (op_tests/test_moe_ep.py:117-126). bm 64/128
    run stage 2 on the prefill kernel (per-pair rows summed over the local
    slots only)."""
    cfg = W.MoEConfig("ep_small", 96, 512, 512, 16, 4, routing="sigmoid", local_experts=4,
                      seed=3)
    dev, ref = _make_layer(cfg, cuda_device, True)
    out = _run(dev, block_size_M=bm)
    _check(ref["out"], _np(out.float()), "EP small")
    none_local = (ref["ids_local"] < 0).all(axis=1)
    assert none_local.any()
    assert torch.count_nonzero(out[torch.from_numpy(none_local).to(cuda_device)]).item() == 0


@pytest.mark.parametrize("bm", [16, 64])
def test_fused_moe_ep_share_fewer_experts_than_topk(cuda_device, bm):
    """An expert-parallel share holding fewer experts than topk (4 local
    experts of 32, top-8 routing, as 8 GPUs would hold them): the layer runs
    and matches the oracle; tokens with no local expert give zero rows."""
    cfg = W.MoEConfig("ep_few", 64, 512, 512, 32, 8, routing="sigmoid", local_experts=4,
                      seed=5)
    dev, ref = _make_layer(cfg, cuda_device, True)
    out = _run(dev, block_size_M=bm)
    _check(ref["out"], _np(out.float()), f"EP 4 of 32 experts, top-8, bm={bm}")
    none_local = (ref["ids_local"] < 0).all(axis=1)
    assert torch.count_nonzero(out[torch.from_numpy(none_local).to(cuda_device)]).item() == 0


@pytest.mark.parametrize("T,local,bm", [(80, 50, None), (80, 50, 64), (80, 50, 128),
                                         (600, 450, None), (600, 450, 16), (600, 290, 128)])
def test_fused_moe_num_local_tokens(cuda_device, T, local, bm):
    """num_local_tokens (a device scalar) limits the layer to the first rows;
    T=600 at E=8 is three sorting chunks, where the counting launch also
    quantises the activations and reads the row count from the device."""
    cfg = W.MoEConfig("local_tok", T, 512, 512, 8, 2, seed=4)
    dev, _ = _make_layer(cfg, cuda_device, True)
    loc = torch.tensor([local], dtype=torch.int32, device=cuda_device)
    out = _run(dev, num_local_tokens=loc, block_size_M=bm)
    wts = W.make_weights(cfg, device="cpu", shuffle=False)
    ref = R.fused_moe_ref(dev["x"].float().cpu().numpy(), wts["w1"].view(torch.uint8).numpy(),
                          wts["w1_scale"].numpy(), wts["w2"].view(torch.uint8).numpy(),
                          wts["w2_scale"].numpy(), _np(dev["ids"]), _np(dev["tw"]),
                          num_local_tokens=local)
    got = _np(out.float())
    if T <= 256:
        _check(ref["out"][:local], got[:local], f"num_local_tokens T={T} bm={bm}")
    else:
        # many more outputs: one of them sits next to an fp8 requant tie
        # (max-rel 5e-2 at RMS-rel 2.6e-3 measured), so the check is per stage
        got[local:] = 0
        ref["ids_local"][local:] = -1
        bm_used = bm or A.select_block_m(T, cfg.topk, cfg.experts, cfg.model_dim,
                                         cfg.inter_dim, False, cuda_device)
        _fullshape.stagewise_vs_oracle(cfg, dev, ref, got, bm_used, A.ActivationType.Silu)


@pytest.mark.parametrize("T,bm", [(40, None), (40, 128), (600, None), (600, 16)])
def test_fused_moe_fp16_io(cuda_device, T, bm):
    """fp16 in and out; T=600 at E=8 is three sorting chunks (the counting
    launch quantises the fp16 activations)."""
    cfg = W.MoEConfig("fp16", T, 512, 512, 8, 2, seed=6)
    dev, ref = _make_layer(cfg, cuda_device, True)
    dev["x"] = dev["x"].to(torch.float16)
    out = _run(dev, block_size_M=bm)
    assert out.dtype == torch.float16
    if T <= 256:
        _check(ref["out"], _np(out.float()), "fp16")
    else:   # per stage, as for num_local_tokens at this size
        bm_used = bm or A.select_block_m(T, cfg.topk, cfg.experts, cfg.model_dim,
                                         cfg.inter_dim, False, cuda_device)
        _fullshape.stagewise_vs_oracle(cfg, dev, ref, _np(out.float()), bm_used,
                                       A.ActivationType.Silu)


# ------------------------------------------- full MiMo shape (decode) ---
def _torch_ref_gpu(x, w1, s1, w2, s2, ids, tw, inter):
    """Plain torch fp32 reference on the GPU (tests/_fullshape.TorchChain)."""
    return _fullshape.torch_layer_ref(x, w1, s1, w2, s2, ids, tw)


@pytest.mark.parametrize("T", [1, 8, 32])
def test_fused_moe_mimo_decode(cuda_device, T):
    cfg = W.mimo_decode(T)
    wts = W.make_weights(cfg, device=cuda_device, shuffle=False)
    x = W.make_hidden(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    ref = _torch_ref_gpu(x, wts["w1"], wts["w1_scale"], wts["w2"], wts["w2_scale"], ids, tw,
                         cfg.inter_dim)
    w1s, w2s = A.shuffle_weight(wts["w1"]), A.shuffle_weight(wts["w2"])
    out = A.fused_moe(x, w1s, w2s, tw, ids, quant_type=A.QuantType.per_128x128,
                      w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"])
    _check(_np(ref), _np(out.float()), f"MiMo T={T}")
    # linearity in the routing weights: doubling them doubles the output
    # (to f32 atomic-order rounding and one bf16 rounding)
    out2 = A.fused_moe(x, w1s, w2s, tw * 2, ids, quant_type=A.QuantType.per_128x128,
                       w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"])
    mx, rms = R.normalized_errors(_np(out.float()) * 2, _np(out2.float()))
    assert mx <= 1e-2 and rms <= 1e-3


@pytest.mark.parametrize("bm", [16, 32, 64])
def test_fused_moe_odd_model_dim(cuda_device, bm):
    """model_dim 384 (3 K blocks; stage 2 cannot use 256-column tiles, so it
    takes the general kernels) with every small block size."""
    cfg = W.MoEConfig("odd_h", 48, 384, 256, 6, 2, seed=8)
    dev, ref = _make_layer(cfg, cuda_device, True)
    _check(ref["out"], _np(_run(dev, block_size_M=bm).float()), f"H=384 bm={bm}")


# ------------------------------------------- full MiMo shape (prefill) ---
@pytest.mark.parametrize("T,block_ms", [(2048, (128, 64, 32)), (8192, (128,))])
def test_fused_moe_mimo_prefill_stagewise(cuda_device, T, block_ms):
    """Full MiMo dims with Zipf routing (the register-B prefill kernels at
    K = 4096 / 2048; the default block_m is 128 at T=8192 and 64 at T=2048,
    below 16 rounds of 64-row workgroups), checked per stage."""
    cfg = W.mimo_prefill(T)
    assert A.default_block_m(cfg.tokens, cfg.topk, cfg.experts, cfg.model_dim,
                             cfg.inter_dim) == (128 if T == 8192 else 64)
    _fullshape.stagewise_check(cfg, cuda_device, block_ms)


@pytest.mark.parametrize("weights,bm", [("fp8", 64), ("fp8", 128), ("mxfp4", 128)])
@pytest.mark.parametrize("ntw", [2, 4])
def test_prefill_column_walk_bit_exact(cuda_device, monkeypatch, weights, bm, ntw):
    """A prefill workgroup that walks ntw column tiles in one pipelined K loop
    (AITER_AMD_PF_NTW1/2 force the count) computes every tile as a
    one-tile workgroup does: stage 1's a2 and the layer's output (per-pair
    rows summed in slot order) are bitwise equal. Stage 2 walks on its
    128-column tile (AITER_AMD_PF_WIDE2=0; the 256-column tile always takes
    one). Stage 1 has 8 column tiles and stage 2 16, so both the XCD order
    (8 column groups) and the plain order are walked."""
    cfg = W.MoEConfig("walk", 300, 2048, 1024, 16, 4, seed=21, weights=weights)
    wts = W.make_weights(cfg, device=cuda_device, shuffle=True)
    x = W.make_hidden(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    monkeypatch.setenv("AITER_AMD_PF_WIDE2", "0")

    def layer(c):
        monkeypatch.setenv("AITER_AMD_PF_NTW1", str(c))
        monkeypatch.setenv("AITER_AMD_PF_NTW2", str(c))
        out = W.run_layer(weights, x, wts["w1"], wts["w2"], tw, ids, w1_scale=wts["w1_scale"],
                          w2_scale=wts["w2_scale"], block_size_M=bm)
        a2 = None
        if weights == "fp8":
            a1, a1s = A.per_group_quant_hip(x)
            sid, sw, se, nv, _ = A.moe_sorting(ids, tw, cfg.experts, cfg.model_dim,
                                                torch.bfloat16, bm)
            a2, a2s = A.moe_stage1_fp8_blockscale(a1, a1s, wts["w1"], wts["w1_scale"], sid, se,
                                                  nv, cfg.topk, bm, True)
            a2 = (a2.view(torch.uint8).clone(), a2s.clone())
        torch.cuda.synchronize()
        return out, a2

    out1, a21 = layer(1)
    outc, a2c = layer(ntw)
    if a21 is not None:
        assert torch.equal(a21[0], a2c[0]) and torch.equal(a21[1], a2c[1])
    assert torch.equal(out1, outc), (out1.float() - outc.float()).abs().max().item()
    assert torch.count_nonzero(out1).item() > 0


@pytest.mark.parametrize("weights,bm,T", [("fp8", 64, 300), ("fp8", 128, 300),
                                         ("mxfp4", 64, 300), ("mxfp4", 128, 300),
                                         ("mxfp4", 64, 50), ("mxfp4", 128, 50)])
@pytest.mark.parametrize("order", [(2, 1, 2, 0, 1), (4, 0, 4, 1, 2), (8, 1, 1, 1, 1),
                                   (1, 1, 8, 0, 2)])
def test_prefill_xcd_order_bit_exact(cuda_device, monkeypatch, weights, bm, T, order):
    """The prefill and MXFP4 (v2) kernels' tile order (XCD groups along M,
    staggered walks; AITER_AMD_PF_MSPLIT1/2, AITER_AMD_PF_MROT1/2 and the
    AITER_AMD_V2_ ones force them) only moves tiles between XCDs and in
    time: stage 1's a2 and the layer output are bitwise equal to the plain
    order's (one group, no stagger). order = (groups 1, stagger 1, groups 2,
    stagger 2, stage-2 column walk); the walk of 2 leaves the prefill stage 2
    with 8 column groups instead of 16. MXFP4 at T=300 (75 routed rows per
    expert) runs on the prefill kernels, at T=50 (12.5) on v2, whose stage 2
    (at 64 rows) accumulates with fp32 atomics: their order differs between
    runs at top-4, so there the two outputs are compared at the layer bar
    instead (the plain order itself is checked against the oracle by the A8W4
    layer tests)."""
    cfg = W.MoEConfig("xcd", T, 2048, 1024, 16, 4, seed=23, weights=weights)
    wts = W.make_weights(cfg, device=cuda_device, shuffle=True)
    x = W.make_hidden(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)

    def layer(m1, r1, m2, r2, ntw2):
        for k, v in (("MSPLIT1", m1), ("MROT1", r1), ("MSPLIT2", m2), ("MROT2", r2)):
            monkeypatch.setenv("AITER_AMD_PF_" + k, str(v))
            monkeypatch.setenv("AITER_AMD_V2_" + k, str(v))
        monkeypatch.setenv("AITER_AMD_PF_NTW2", str(ntw2))
        out = W.run_layer(weights, x, wts["w1"], wts["w2"], tw, ids, w1_scale=wts["w1_scale"],
                          w2_scale=wts["w2_scale"], block_size_M=bm)
        a2 = None
        if weights == "fp8":
            a1, a1s = A.per_group_quant_hip(x)
            sid, sw, se, nv, _ = A.moe_sorting(ids, tw, cfg.experts, cfg.model_dim,
                                                torch.bfloat16, bm)
            a2, a2s = A.moe_stage1_fp8_blockscale(a1, a1s, wts["w1"], wts["w1_scale"], sid, se,
                                                  nv, cfg.topk, bm, True)
            a2 = (a2.view(torch.uint8).clone(), a2s.clone())
        torch.cuda.synchronize()
        return out, a2

    out1, a21 = layer(1, 0, 1, 0, order[4])
    outc, a2c = layer(*order)
    if a21 is not None:
        assert torch.equal(a21[0], a2c[0]) and torch.equal(a21[1], a2c[1])
    assert torch.count_nonzero(out1).item() > 0
    if weights == "mxfp4" and bm == 64 and T * cfg.topk < 48 * cfg.experts:
        _check(_np(out1.float()), _np(outc.float()), f"xcd order {order} vs plain")
    else:
        assert torch.equal(out1, outc), (out1.float() - outc.float()).abs().max().item()


@pytest.mark.parametrize("weights,bm", [("fp8", 64), ("fp8", 128), ("mxfp4", 128)])
@pytest.mark.parametrize("T,E", [(300, 64), (2000, 64), (700, 16)])
def test_prefill_pad_skip_bit_exact(cuda_device, monkeypatch, weights, bm, T, E):
    """Prefill stage-2 tiles with at most a quarter (or, in 128-row tiles,
    half) of their 16-row tiles routed run a copy of the kernel body that
    skips the padding tiles' MFMAs (AITER_AMD_PF_PADSKIP = 0 runs every tile
    on the full body). Routed rows get the same MFMAs and fold order either
    way, so the layer output is bitwise equal (and FP8 stage 1's a2, which
    has no such copy, too). Zipf routing over 64 experts leaves most experts
    a handful of rows, so tiles of 1-16, 17-32 and more rows all occur. MXFP4
    at bm 128 runs stage 2 (128-row tiles) and, from 16 routed rows per
    expert, stage 1 (with its own copy) on the prefill kernel."""
    cfg = W.MoEConfig("padskip", T, 2048, 1024, E, 4, routing="zipf", seed=27, weights=weights)
    wts = W.make_weights(cfg, device=cuda_device, shuffle=True)
    x = W.make_hidden(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    counts = torch.bincount(ids.flatten().long().cpu(), minlength=E)
    assert int(((counts > 0) & (counts <= 32)).sum()) > 0 and int((counts > 64).sum()) > 0

    def layer(skip):
        monkeypatch.setenv("AITER_AMD_PF_PADSKIP", str(skip))
        out = W.run_layer(weights, x, wts["w1"], wts["w2"], tw, ids, w1_scale=wts["w1_scale"],
                          w2_scale=wts["w2_scale"], block_size_M=bm)
        a2 = None
        if weights == "fp8":
            a1, a1s = A.per_group_quant_hip(x)
            sid, sw, se, nv, _ = A.moe_sorting(ids, tw, cfg.experts, cfg.model_dim,
                                                torch.bfloat16, bm)
            a2, a2s = A.moe_stage1_fp8_blockscale(a1, a1s, wts["w1"], wts["w1_scale"], sid, se,
                                                  nv, cfg.topk, bm, True)
            a2 = (a2.view(torch.uint8).clone(), a2s.clone())
        torch.cuda.synchronize()
        return out, a2

    out0, a20 = layer(0)
    out1, a21 = layer(1)
    if a20 is not None:
        assert torch.equal(a20[0], a21[0]) and torch.equal(a20[1], a21[1])
    assert torch.count_nonzero(out0).item() > 0
    assert torch.equal(out0, out1), (out0.float() - out1.float()).abs().max().item()


@pytest.mark.parametrize("weights,bm", [("fp8", 64), ("fp8", 128), ("mxfp4", 128)])
@pytest.mark.parametrize("T", [300, 2000])
def test_prefill_stage2_wide_tile_bit_exact(cuda_device, monkeypatch, weights, bm, T):
    """The prefill stage 2 as 64-row x 256-column workgroups (the FP8
    default; AITER_AMD_PF_WIDE2 forces either) and as block_m x 128-column
    ones compute every output element with the same MFMAs and the same
    scale-fold order, so the layer outputs (per-pair rows summed in slot
    order) are bitwise equal. T=2000 walks two column tiles in the narrow
    order (the wide one walks one)."""
    cfg = W.MoEConfig("wide", T, 2048, 1024, 16, 4, seed=25, weights=weights)
    wts = W.make_weights(cfg, device=cuda_device, shuffle=True)
    x = W.make_hidden(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)

    def layer(wide):
        monkeypatch.setenv("AITER_AMD_PF_WIDE2", str(wide))
        out = W.run_layer(weights, x, wts["w1"], wts["w2"], tw, ids, w1_scale=wts["w1_scale"],
                          w2_scale=wts["w2_scale"], block_size_M=bm)
        torch.cuda.synchronize()
        return out

    narrow, wide = layer(0), layer(1)
    assert torch.count_nonzero(narrow).item() > 0
    assert torch.equal(narrow, wide), (narrow.float() - wide.float()).abs().max().item()


@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
@pytest.mark.parametrize("bm", [16, 32])
@pytest.mark.parametrize("ntw", [2, 4])
def test_stream_stage2_column_walk(cuda_device, monkeypatch, weights, bm, ntw):
    """The decode kernel's stage 2 walking ntw 256-column groups per workgroup
    (AITER_AMD_ST_NTW2 forces the count). With one slot per token every
    output element gets exactly one atomic add, so the accumulator is
    bitwise equal to the one-group walk's; with top-4 the two differ only by
    the order of the fp32 atomic adds (the one-group path itself is checked
    against the oracle by the layer tests)."""
    st1 = A.moe_stage1_a8w4 if weights == "mxfp4" else A.moe_stage1_fp8_blockscale
    st2 = A.moe_stage2_a8w4 if weights == "mxfp4" else A.moe_stage2_fp8_blockscale
    for k, seed in ((1, 31), (4, 32)):
        cfg = W.MoEConfig("swalk", 40, 2048, 1024, 8, k, seed=seed, weights=weights)
        wts = W.make_weights(cfg, device=cuda_device, shuffle=True)
        x = W.make_hidden(cfg, device=cuda_device)
        tw, ids = W.make_routing(cfg, device=cuda_device)
        a1, a1s = A.per_group_quant_hip(x)
        sid, sw, se, nv, _ = A.moe_sorting(ids, tw, cfg.experts, cfg.model_dim, torch.float32,
                                            bm)
        a2, a2s = st1(a1, a1s, wts["w1"], wts["w1_scale"], sid, se, nv, k, bm, True)

        def stage2(c):
            monkeypatch.setenv("AITER_AMD_ST_NTW2", str(c))
            acc = torch.zeros(cfg.tokens, cfg.model_dim, dtype=torch.float32,
                              device=cuda_device)
            st2(a2, a2s, wts["w2"], wts["w2_scale"], sid, sw, se, nv, acc, bm, True)
            torch.cuda.synchronize()
            return acc

        acc1, accc = stage2(1), stage2(ntw)
        assert torch.count_nonzero(acc1).item() > 0
        if k == 1:
            assert torch.equal(acc1, accc)
        else:
            # four fp32 terms summed in another order: a few ulps of the largest
            tol = 4 * 2.0 ** -23 * acc1.abs().max().item()
            assert (acc1 - accc).abs().max().item() <= tol


@pytest.mark.parametrize("bm,splits", [(16, (2, 4)), (32, (2, 4, 8))])
def test_stream_stage1_split_k(cuda_device, monkeypatch, bm, splits):
    """Decode stage 1 with its K range split over 2, 4 or 8 workgroups per
    tile (AITER_AMD_ST_KSPLIT1 forces the count): the last workgroup of a
    tile to arrive adds the fp32 partial sums in split order and runs the
    SiLU*up + requant epilogue. Every split meets the oracle bar on two calls
    in a row (the arrival counters are left at zero), and so does the
    automatic choice (2 here: 32 tiles, fewer than 128). The two-launch
    layer is pinned, so stage 1's a2 goes through HBM."""
    monkeypatch.setenv("AITER_AMD_FUSED", "0")
    cfg = W.MoEConfig("ksplit", 5, 2048, 512, 8, 4, seed=41)
    dev, ref = _make_layer(cfg, cuda_device, True)
    for c in (1,) + splits:
        monkeypatch.setenv("AITER_AMD_ST_KSPLIT1", str(c))
        for call in range(2):
            out = _run(dev, block_size_M=bm)
            _check(ref["out"], _np(out.float()), f"split-K {c} bm={bm} call {call}")
    monkeypatch.delenv("AITER_AMD_ST_KSPLIT1")
    _check(ref["out"], _np(_run(dev, block_size_M=bm).float()), f"split-K auto bm={bm}")


@pytest.mark.parametrize("bm", [16, 32])
@pytest.mark.parametrize("shuffle", [True, False])
def test_fused_layer_one_launch(cuda_device, monkeypatch, bm, shuffle):
    """The one-launch layer (AITER_AMD_FUSED=1 forces it): each workgroup runs
    stage 1 for one 128-wide slice of the intermediate dim, keeps the slice's
    requantised rows (exactly one 1x128 quant group per row, as the
    reference's a2) in LDS and adds their down-GEMM share into the fp32
    accumulator. Config A against the oracle at the strict bar, with the
    plain, doweight_stage1 and Gelu variants, and with split-K (the last
    workgroup of a slice runs both the epilogue and the down GEMM)."""
    monkeypatch.setenv("AITER_AMD_FUSED", "1")
    cfg = W.CONFIG_A
    dev, ref = _make_layer(cfg, cuda_device, shuffle)
    _check(ref["out"], _np(_run(dev, block_size_M=bm).float()), f"one-launch bm={bm}")
    monkeypatch.setenv("AITER_AMD_ST_KSPLIT1", "2")
    _check(ref["out"], _np(_run(dev, block_size_M=bm).float()), f"one-launch split-K bm={bm}")
    monkeypatch.delenv("AITER_AMD_ST_KSPLIT1")
    if shuffle:
        dev, ref = _make_layer(cfg, cuda_device, True, doweight=True)
        out = _run(dev, block_size_M=bm, doweight_stage1=True)
        _check(ref["out"], _np(out.float()), f"one-launch doweight bm={bm}")
        dev, ref = _make_layer(cfg, cuda_device, True, activation="gelu")
        out = _run(dev, block_size_M=bm, activation=A.ActivationType.Gelu)
        _check(ref["out"], _np(out.float()), f"one-launch gelu bm={bm}")


@pytest.mark.parametrize("bm", [16, 32])
def test_fused_layer_one_launch_ep_share(cuda_device, monkeypatch, bm):
    """The one-launch layer with an expert mask: tokens with no local expert
    give zero rows, the rest match the oracle."""
    monkeypatch.setenv("AITER_AMD_FUSED", "1")
    cfg = W.MoEConfig("ep_small", 96, 512, 512, 16, 4, routing="sigmoid", local_experts=4,
                      seed=3)
    dev, ref = _make_layer(cfg, cuda_device, True)
    out = _run(dev, block_size_M=bm)
    _check(ref["out"], _np(out.float()), "one-launch EP small")
    none_local = (ref["ids_local"] < 0).all(axis=1)
    assert none_local.any()
    assert torch.count_nonzero(out[torch.from_numpy(none_local).to(cuda_device)]).item() == 0


@pytest.mark.parametrize("T", [1, 8, 32])
def test_fused_layer_one_launch_vs_two_stage_mimo(cuda_device, monkeypatch, T):
    """At MiMo decode dims the one-launch layer and the two-launch layer
    compute the same a2 (same kernel code, same requant) and differ only in
    the fp32 atomic order of the down GEMM: outputs agree to a few bf16 ulps
    of the largest element."""
    cfg = W.mimo_decode(T)
    wts = W.make_weights(cfg, device=cuda_device, shuffle=True)
    x = W.make_hidden(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)

    def layer(fused):
        monkeypatch.setenv("AITER_AMD_FUSED", str(fused))
        return A.fused_moe(x, wts["w1"], wts["w2"], tw, ids, quant_type=A.QuantType.per_128x128,
                           w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"]).float()

    one, two = layer(1), layer(0)
    torch.cuda.synchronize()
    mx, rms = R.normalized_errors(_np(two), _np(one))
    print(f"[one vs two launches T={T}] max-rel {mx:.3e} rms-rel {rms:.3e}", flush=True)
    assert mx <= 2e-2 and rms <= 2e-3 and torch.count_nonzero(one).item() > 0


def test_fused_moe_mimo_decode_t128_stagewise(cuda_device):
    """Decode T=128 at MiMo dims (the stream kernels, stage 2 walking two
    column groups per workgroup), checked per stage."""
    _fullshape.stagewise_check(W.mimo_decode(128), cuda_device, (16, 32))


def test_fused_moe_ep_share_full_stagewise(cuda_device):
    """The expert-parallel share at its benchmark shape: T=4096, 32 of 256
    experts local, sigmoid top-8 renormalised routing, checked per stage on
    the local pairs and end to end with the expert mask."""
    cfg = W.mimo_ep_share(4096)
    _fullshape.stagewise_check(cfg, cuda_device, (128, 64))


# --------------------------------------------------------- edge cases ---
def test_fused_moe_empty_batch(cuda_device):
    cfg = W.CONFIG_A
    dev, _ = _make_layer(cfg, cuda_device, True)
    out = A.fused_moe(dev["x"][:0], dev["w1"], dev["w2"], dev["tw"][:0], dev["ids"][:0],
                      quant_type=A.QuantType.per_128x128, w1_scale=dev["s1"], w2_scale=dev["s2"])
    assert out.shape == (0, cfg.model_dim) and out.dtype == torch.bfloat16


def test_fused_moe_beyond_4gib_operand(cuda_device):
    """A layer whose stage-2 activation operand (T*topk*inter fp8 bytes) is
    just over 4 GiB: the 64/128-row kernels address it with 32-bit offsets,
    so block_m falls back from 128 to 64 and stage 2 runs on the general
    kernel (64-bit addresses). Tokens are independent, so the oracle checks
    the first and last 16 tokens; the last ones' a2 rows lie past the 4 GiB
    offset."""
    T = (1 << 32) // (8 * 2048) + 64
    cfg = W.MoEConfig("big", T, 512, 2048, 16, 8, seed=21)
    wts = W.make_weights(cfg, device="cpu", shuffle=False)
    x = W.make_hidden(cfg)
    tw, ids = W.make_routing(cfg)
    dev = cuda_device
    w1, w2 = A.shuffle_weight(wts["w1"]).to(dev), A.shuffle_weight(wts["w2"]).to(dev)
    w1.is_shuffled = w2.is_shuffled = True
    fm = importlib.import_module("aiter_amd.fused_moe")
    assert fm.select_block_m(T, 8, 16, 512, 2048, False, torch.device(dev)) == 64
    out = A.fused_moe(x.to(dev), w1, w2, tw.to(dev), ids.to(dev),
                      quant_type=A.QuantType.per_128x128, w1_scale=wts["w1_scale"].to(dev),
                      w2_scale=wts["w2_scale"].to(dev))
    torch.cuda.synchronize()
    for rows in (slice(0, 16), slice(T - 16, T)):
        ref = R.fused_moe_ref(x[rows].float().numpy(), wts["w1"].view(torch.uint8).numpy(),
                              wts["w1_scale"].numpy(), wts["w2"].view(torch.uint8).numpy(),
                              wts["w2_scale"].numpy(), ids[rows].numpy(), tw[rows].numpy())
        _check(ref["out"], _np(out[rows].float()), f"T={T} rows {rows.start}..")
    del out, w1, w2
    torch.cuda.empty_cache()


@pytest.mark.parametrize("T,E,k,seed", [(37, 32, 16, 12), (45, 1, 1, 13), (1, 8, 8, 14)])
def test_fused_moe_topk_and_expert_extremes(cuda_device, T, E, k, seed):
    """topk 16 (32-bit slot masks in sorting), a single expert with top-1
    (a dense block-scale GEMM), and topk == E with one token, on every
    block size. Sixteen summed slots make the end-to-end error sensitive to
    one-ulp fp8 requant flips, so the layer is checked per stage."""
    cfg = W.MoEConfig("extreme", T, 512, 512, E, k, seed=seed)
    _fullshape.stagewise_check(cfg, cuda_device, (16, 32, 64, 128))


# ------------------------------------------------------- graph capture ---
@pytest.mark.parametrize("T,bm", [(32, 16), (512, 128)])
def test_fused_moe_hip_graph_replay(cuda_device, T, bm):
    """The one-call layer captured in a HIP graph (torch.cuda.CUDAGraph):
    the entry points allocate nothing and clear with kernels, not memsets.
    Each of three replays runs on new inputs copied into the captured
    buffers, with eager layers and synchronisation in between, and must
    match an eager call on the same inputs (the stream path's fp32 atomics
    may sum in another order; the per-pair path is deterministic). bm 16
    runs the stream kernels, bm 128 the prefill kernels with per-pair rows
    and the slot sum."""
    cfg = W.MoEConfig("graph", T, 1024, 512, 8, 2, seed=31)
    dev, ref = _make_layer(cfg, cuda_device, True)
    xs = [dev["x"]] + [torch.randn_like(dev["x"].float()).to(torch.bfloat16) for _ in range(2)]
    static_x = dev["x"].clone()
    run = lambda x: _run(dict(dev, x=x), block_size_M=bm)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            run(static_x)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static_out = run(static_x)
    for i, x in enumerate(xs):
        static_x.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        got = _np(static_out.float())
        eager = _np(run(x).float())
        torch.cuda.synchronize()
        if bm == 128:
            assert np.array_equal(got, eager), f"replay {i}"
        else:
            mx, rms = R.normalized_errors(eager, got)
            assert mx <= 1e-2 and rms <= 1e-3, (i, mx, rms)
        if i == 0:   # per stage: one fp8 requant tie moves a small output past max-rel here
            _fullshape.stagewise_vs_oracle(cfg, dev, ref, got, bm, A.ActivationType.Silu)


# ------------------------------------------- one token: direct M-blocks ---
def _bf16_close(a, b):
    """Within one bf16 rounding of each other: the two layers sum the same
    fp32 terms in different orders (the sorted layer with fp32 atomics, the
    direct layer per token in slot order)."""
    a, b = a.float(), b.float()
    return bool(((a - b).abs() <= 2.0 ** -7 * torch.maximum(a.abs(), b.abs()) + 1e-30).all())


def test_fused_moe_direct_t1_stagewise(cuda_device):
    """MiMo decode T=1 on direct M-blocks (no sorting launch: the GEMMs read
    the routing, stage 1 quantises the token, stage 2 sums the token's slots
    straight into the output row), checked per stage against the oracle."""
    _fullshape.stagewise_check(W.mimo_decode(1), cuda_device, (16,))


@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
def test_fused_moe_direct_matches_sorted(cuda_device, monkeypatch, weights):
    """At MiMo T=1 the direct layer's stage-1 output (fp8 a2 and its scales,
    read back from the layer's workspace) equals the sorted layer's bitwise:
    the in-kernel quant runs the quant kernel's arithmetic and each pair's
    M-block holds the same rows; the outputs agree to one bf16 rounding. The
    staggered K walk is off here (AITER_AMD_ST_ROT=0): its rotation follows
    the M-block index, which differs between the two layouts, and with it the
    order of stage 1's fp32 K sum."""
    monkeypatch.setenv("AITER_AMD_ST_ROT", "0")
    cfg = W.mimo_decode(1) if weights == "fp8" else W.mimo_a8w4(1)
    wts = W.make_weights(cfg, device=cuda_device, shuffle=False)
    x = W.make_hidden(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    w1s, w2s = A.shuffle_weight(wts["w1"]), A.shuffle_weight(wts["w2"])
    res = {}
    for direct in (1, 0):
        monkeypatch.setenv("AITER_AMD_DIRECT", str(direct))
        res[direct] = _fullshape.run_layer_keep_a2(cfg, x, w1s, w2s, wts["w1_scale"],
                                                   wts["w2_scale"], tw, ids, None, 16)
    torch.cuda.synchronize()
    (o1, a21, s21), (o0, a20, s20) = res[1], res[0]
    assert torch.equal(a21.view(torch.uint8), a20.view(torch.uint8))
    assert torch.equal(s21, s20)
    assert torch.count_nonzero(o1).item() > 0 and _bf16_close(o1, o0)


def _one_token_ref(cfg, x, ids, tw, doweight, activation):
    """The oracle layer for activations x and routing (ids, tw) on cfg's weights."""
    wts = W.make_weights(cfg, device="cpu", shuffle=False)
    return R.fused_moe_ref(x.float().cpu().numpy(), wts["w1"].view(torch.uint8).numpy(),
                           wts["w1_scale"].numpy(), wts["w2"].view(torch.uint8).numpy(),
                           wts["w2_scale"].numpy(), ids.cpu().numpy(), tw.cpu().numpy(),
                           None, doweight_stage1=doweight, activation=activation)


@pytest.mark.parametrize("case", ["plain", "fp16", "doweight", "gelu", "fp8_input", "dup_ids",
                                  "topk6", "topk8", "topk12"])
def test_fused_moe_direct_small(cuda_device, monkeypatch, case):
    """One token at a small shape (stage 1 kept to one K range, so the layer
    runs on direct M-blocks) against the oracle and against the sorted layer:
    fp16 activations, doweight_stage1, GeLU, a pre-quantised fp8 input, and
    both of the token's slots routed to one expert (two direct M-blocks of
    the same expert, where sorting puts both pairs in one). Stage 2's four
    waves take every fourth slot: top-2 leaves two waves without a slot,
    top-6 and top-12 give the waves unequal counts, top-8 two each. The
    oracle check is the stage-wise one of the other small layers: with one
    token a single one-step requant flip on a dominant a2 element moves the
    RMS of the whole output, so the output is held to the strict bar against
    the oracle's stage 2 on the kernel's own a2 (the staggered K walk off, so
    that the sorted stage 1 the check runs gives the layer's a2 bit for bit)."""
    monkeypatch.setenv("AITER_AMD_ST_KSPLIT1", "1")
    monkeypatch.setenv("AITER_AMD_ST_ROT", "0")
    k = int(case[4:]) if case.startswith("topk") else 2
    cfg = W.MoEConfig("one_token", 1, 1024, 512, 16, k, seed=31 + k)
    dw = case == "doweight"
    act = "gelu" if case == "gelu" else "silu"
    dev, _ = _make_layer(cfg, cuda_device, True, doweight=dw, activation=act)
    if case == "dup_ids":
        dev["ids"] = torch.full_like(dev["ids"], 3)
    if case == "fp16":
        dev["x"] = dev["x"].to(torch.float16)
    ref = _one_token_ref(cfg, dev["x"], dev["ids"], dev["tw"], dw, act)
    kw = dict(doweight_stage1=dw,
              activation=A.ActivationType.Gelu if act == "gelu" else A.ActivationType.Silu)
    outs = {}
    for direct in (1, 0):
        monkeypatch.setenv("AITER_AMD_DIRECT", str(direct))
        if case == "fp8_input":
            a1, a1s = A.per_group_quant_hip(dev["x"])
            outs[direct] = A.fused_moe(a1, dev["w1"], dev["w2"], dev["tw"], dev["ids"],
                                       quant_type=A.QuantType.per_128x128, w1_scale=dev["s1"],
                                       w2_scale=dev["s2"], a1_scale=a1s, dtype=torch.bfloat16,
                                       **kw)
        else:
            outs[direct] = _run(dev, block_size_M=16, **kw)
    torch.cuda.synchronize()
    _fullshape.stagewise_vs_oracle(cfg, dev, ref, _np(outs[1].float()), 16, kw["activation"],
                                   doweight=dw, e2e_rms=False)
    assert _bf16_close(outs[1], outs[0]), case


@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
@pytest.mark.parametrize("inter,variant", [(384, "plain"), (768, "plain"), (1536, "plain"),
                                           (768, "doweight_gelu")])
def test_fused_moe_direct_inter_sizes(cuda_device, monkeypatch, weights, inter, variant):
    """One token at K-step counts of 3, 6 and 12 per slot (inter 384, 768,
    1536): the one-token stage 2 then keeps 1, 2 or 4 steps in flight per
    wave (8 at MiMo), with fp8 or MXFP4 weights (e8m0 dwords loaded per
    group of steps), and once with doweight_stage1 and GeLU; stage-wise
    against the oracle and against the sorted layer."""
    monkeypatch.setenv("AITER_AMD_ST_KSPLIT1", "1")
    monkeypatch.setenv("AITER_AMD_ST_ROT", "0")
    mx4 = weights == "mxfp4"
    cfg = W.MoEConfig("one_token_k", 1, 1024, inter, 16, 6, seed=inter,
                      weights="mxfp4" if mx4 else "fp8")
    wts = W.make_weights(cfg, device="cpu", shuffle=False)
    x = W.make_hidden(cfg)
    tw, ids = W.make_routing(cfg)
    w1u = wts["w1"] if mx4 else wts["w1"].view(torch.uint8)
    w2u = wts["w2"] if mx4 else wts["w2"].view(torch.uint8)
    dw = variant == "doweight_gelu"
    act = A.ActivationType.Gelu if dw else A.ActivationType.Silu
    ref = R.fused_moe_ref(x.float().numpy(), w1u.numpy(), wts["w1_scale"].numpy(), w2u.numpy(),
                          wts["w2_scale"].numpy(), ids.numpy(), tw.numpy(), None,
                          weight_format="mxfp4" if mx4 else "fp8_128x128", doweight_stage1=dw,
                          activation="gelu" if dw else "silu")
    dev = dict(x=x.to(cuda_device), w1=A.shuffle_weight(wts["w1"]).to(cuda_device),
               w2=A.shuffle_weight(wts["w2"]).to(cuda_device), s1=wts["w1_scale"].to(cuda_device),
               s2=wts["w2_scale"].to(cuda_device), tw=tw.to(cuda_device), ids=ids.to(cuda_device),
               mask=None)
    dev["w1"].is_shuffled = dev["w2"].is_shuffled = True
    outs = {}
    for direct in (1, 0):
        monkeypatch.setenv("AITER_AMD_DIRECT", str(direct))
        if mx4:
            outs[direct] = A.fused_moe_a8w4(dev["x"], dev["w1"], dev["w2"], dev["tw"], dev["ids"],
                                            w1_scale=dev["s1"], w2_scale=dev["s2"],
                                            block_size_M=16, doweight_stage1=dw, activation=act)
        else:
            outs[direct] = _run(dev, block_size_M=16, doweight_stage1=dw, activation=act)
    torch.cuda.synchronize()
    _fullshape.stagewise_vs_oracle(cfg, dev, ref, _np(outs[1].float()), 16, act, doweight=dw,
                                   e2e_rms=False)
    assert _bf16_close(outs[1], outs[0]), (weights, inter, variant)


@pytest.mark.parametrize("shape", ["small", "mimo", "mimo_a8w4"])
def test_fused_moe_direct_hip_graph_replay(cuda_device, monkeypatch, shape):
    """One token on direct M-blocks captured in a HIP graph (two kernels,
    nothing else to record): each of three replays on new inputs, with eager
    layers and synchronisation in between, matches an eager call bit for bit
    (stage 2 sums each output in a fixed order, no atomics), FP8 and MXFP4."""
    if shape == "small":
        monkeypatch.setenv("AITER_AMD_ST_KSPLIT1", "1")   # one K range: direct M-blocks
        cfg = W.MoEConfig("graph_one_token", 1, 1024, 512, 8, 2, seed=37)
        dev, _ = _make_layer(cfg, cuda_device, True)
        run = lambda x: _run(dict(dev, x=x), block_size_M=16)
    else:
        w4 = shape == "mimo_a8w4"
        cfg = W.mimo_a8w4(1) if w4 else W.mimo_decode(1)
        wts = W.make_weights(cfg, device=cuda_device, shuffle=True)
        tw, ids = W.make_routing(cfg, device=cuda_device)
        dev = dict(x=W.make_hidden(cfg, device=cuda_device))
        if w4:
            run = lambda x: A.fused_moe_a8w4(x, wts["w1"], wts["w2"], tw, ids,
                                             w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"])
        else:
            run = lambda x: A.fused_moe(x, wts["w1"], wts["w2"], tw, ids,
                                        quant_type=A.QuantType.per_128x128,
                                        w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"])
    xs = [dev["x"]] + [torch.randn_like(dev["x"].float()).to(torch.bfloat16) for _ in range(2)]
    static_x = dev["x"].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            run(static_x)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static_out = run(static_x)
    for i, x in enumerate(xs):
        static_x.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        got = static_out.float().clone()
        eager = run(x).float()
        torch.cuda.synchronize()
        assert torch.count_nonzero(got).item() > 0 and torch.equal(got, eager), f"replay {i}"


@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
@pytest.mark.parametrize("tokens,bm,variant", [
    (1, 16, "plain"), (17, 16, "plain"), (65, 32, "plain"), (63, 64, "plain"), (300, 64, "plain"),
    (300, 128, "plain"), (300, 64, "mask"), (300, 64, "local_tokens"), (300, 128, "doweight"),
    (300, None, "fp16")])
def test_prequant_layer_matches_stage_calls(cuda_device, weights, tokens, bm, variant):
    """fp8 activations through the one-call entry against the stage calls with
    an fp32 accumulator. Both run the same stage-1 kernel and sum a token's
    rows in fp32, in another order, then round once: outputs differ by at most
    one 16-bit step (2^-8 relative for bf16), or by topk * 2^-23 of the largest
    sum where terms cancel."""
    cfg = W.MoEConfig("prequant", tokens, 1024, 512, 8, 3, seed=tokens, weights=weights,
                      local_experts=4 if variant == "mask" else None)
    wts = W.make_weights(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    a1, a1s = A.per_group_quant_hip(W.make_hidden(cfg, device=cuda_device))
    mask = W.make_expert_mask(cfg, device=cuda_device)
    E = cfg.experts
    n = torch.tensor([tokens - 9], dtype=torch.int32, device=cuda_device) \
        if variant == "local_tokens" else None
    dw = variant == "doweight"
    dt = torch.float16 if variant == "fp16" else torch.bfloat16
    out = W.run_layer(weights, a1, wts["w1"], wts["w2"], tw, ids, w1_scale=wts["w1_scale"],
                      w2_scale=wts["w2_scale"], a1_scale=a1s, expert_mask=mask, dtype=dt,
                      num_local_tokens=n, block_size_M=bm, doweight_stage1=dw)
    bm = bm or A.default_block_m(tokens, 3, E, 1024, 512)
    sid, sw, seid, nv, acc = A.moe_sorting(ids, tw, E, 1024, torch.float32, bm, mask, n)
    st1, st2 = ((A.moe_stage1_a8w4, A.moe_stage2_a8w4) if weights == "mxfp4" else
                (A.moe_stage1_fp8_blockscale, A.moe_stage2_fp8_blockscale))
    a2, a2s = st1(a1, a1s, wts["w1"], wts["w1_scale"], sid, seid, nv, 3, bm, True,
                  sorted_weights=sw if dw else None)
    st2(a2, a2s, wts["w2"], wts["w2_scale"], sid, None if dw else sw, seid, nv, acc, bm, True)
    rows = tokens - 9 if n is not None else tokens
    ref, got = acc[:rows], out[:rows].float()
    tol = ref.abs() * 2.0 ** (-10 if dt == torch.float16 else -8) + \
        3 * 2.0 ** -23 * ref.abs().max() * 8
    # stage 1 of the general and stream kernels may sum its K blocks from
    # another start, which moves a few fp8 codes of a2 by a step
    bad = ((got - ref).abs() > tol).float().mean().item()
    assert bad <= (0.0 if bm >= 64 else 0.02), bad
    _check(ref.cpu().numpy(), got.cpu().numpy(), "prequant")


def test_prequant_layer_beyond_the_row_limit(cuda_device):
    """The last token count on per-pair fp32 rows (1 GiB of them) and the first
    on the fp32 accumulator give the same output for the tokens they share. Both
    are rounded, so where their fp32 sums lie on two sides of a tie they differ
    by a whole bf16 spacing, 2^-7 of the value at the foot of a binade; the
    second term is the bound above."""
    T, k, E, H, I = 8193, 8, 8, 4096, 128
    cfg = W.MoEConfig("rows", T, H, I, E, k, seed=3)
    wts = W.make_weights(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    a1, a1s = A.per_group_quant_hip(W.make_hidden(cfg, device=cuda_device))
    run = lambda n: W.run_layer("fp8", a1[:n], wts["w1"], wts["w2"], tw[:n], ids[:n],
                                w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"],
                                a1_scale=a1s[:n], block_size_M=64).float()
    a, b = run(T)[:T - 1], run(T - 1)
    assert ((a - b).abs() <= b.abs() * 2.0 ** -7 + 8 * 2.0 ** -23 * b.abs().max() * 8).all()


@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
@pytest.mark.parametrize("prequant", [False, True])
@pytest.mark.parametrize("inter", [384, 1024])     # stage-2 depths 1 and 8
def test_fused_moe_direct_ids_out_of_range(cuda_device, monkeypatch, weights, prequant, inter):
    """One token some of whose slots name no expert (what routing gives past its
    last candidate, with any weight): they add nothing, as on the sorted layer,
    whatever the workspace held. Without the staggered K walk the two differ in
    the order of the fp32 sum alone: one bf16 rounding."""
    monkeypatch.setenv("AITER_AMD_ST_ROT", "0")
    monkeypatch.setenv("AITER_AMD_ST_KSPLIT1", "1")   # one K range: direct M-blocks
    k = 6
    cfg = W.MoEConfig("oor", 1, 1024, inter, 8, k, seed=inter, weights=weights)
    wts = W.make_weights(cfg, device=cuda_device)
    x = W.make_hidden(cfg, device=cuda_device)
    kw = dict(w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"], block_size_M=16)
    if prequant:
        x, kw["a1_scale"] = A.per_group_quant_hip(x)
    nan = float("nan")
    cases = [([3, -1, 5, 8, 0, 0x7fffffff], [0.5, nan, 0.25, nan, 0.125, nan]),
             ([-1, 2, -1, -1, 8, 7], [nan, 0.5, 1.0, nan, float("inf"), 0.25]),
             ([-1] * k, [nan] * k)]

    def run(ids, tw, direct):
        monkeypatch.setenv("AITER_AMD_DIRECT", direct)
        junk = torch.full((1 << 22,), nan, device=cuda_device)
        del junk
        return W.run_layer(weights, x, wts["w1"], wts["w2"],
                           torch.tensor([tw], device=cuda_device),
                           torch.tensor([ids], dtype=torch.int32, device=cuda_device), **kw)

    for ids, tw in cases:
        got, ref = run(ids, tw, "1"), run(ids, tw, "0")
        assert torch.isfinite(ref).all()
        assert (torch.count_nonzero(ref).item() > 0) == (max(i for i in ids if i < 8) >= 0)
        a, b = got.float(), ref.float()
        tol = 2.0 ** -7 * torch.maximum(a.abs(), b.abs()) + k * 2.0 ** -23 * b.abs().max() * 8
        assert ((a - b).abs() <= tol).all(), ids     # (the last term: where terms cancel)


@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
def test_prequant_layer_rows_per_expert(cuda_device, weights):
    """30 rows per expert sum on the fp32 accumulator, 35 on per-pair fp32 rows
    (39 and 46 MB of them): the tokens they share agree, within the bound above.
    The workspace held NaN."""
    T, k, E, H, I = 700, 8, 160, 2048, 128
    cfg = W.MoEConfig("rpe", T, H, I, E, k, seed=4, weights=weights)
    wts = W.make_weights(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    a1, a1s = A.per_group_quant_hip(W.make_hidden(cfg, device=cuda_device))

    def run(n):
        junk = torch.full((1 << 24,), float("nan"), device=cuda_device)
        del junk
        return W.run_layer(weights, a1[:n], wts["w1"], wts["w2"], tw[:n], ids[:n],
                           w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"],
                           a1_scale=a1s[:n], block_size_M=128).float()

    a, b = run(T)[:600], run(600)
    assert torch.count_nonzero(b).item() > 0
    assert ((a - b).abs() <= b.abs() * 2.0 ** -7 + 8 * 2.0 ** -23 * b.abs().max() * 8).all()


# column-tile counts that 8 divides and that it does not (stage 1 inter / 128,
# stage 2 model_dim / 256), M-blocks below, at and above the 32 of a whole round
# of groups, K-step counts of 1, 2, 3, 5, 6 and 8 in stage 2, experts with one
# M-block and with many (column walks: the two tests after this one)
@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
@pytest.mark.parametrize("bm", [16, 32])
@pytest.mark.parametrize("tokens,H,I,E", [
    (7, 512, 128, 3), (40, 1792, 256, 5), (150, 768, 384, 6), (400, 1792, 384, 9),
    (260, 512, 640, 40), (333, 2048, 768, 33), (512, 1024, 1024, 8), (90, 3584, 256, 64)])
def test_stream_shared_weights_and_tile_order(cuda_device, monkeypatch, weights, bm, tokens, H, I,
                                              E):
    """The stream kernel's workgroup order and weight-load policies against the prefill kernels (64-row blocks), which pass the oracle
    tests: with the staggered K walk off both sum K blocks in the same order,
    so stage 1 is bit for bit the same and a pair's stage-2 row too; a token's
    pairs then add in any order, (k - 1) * 2^-24 of the sum of their magnitudes."""
    monkeypatch.setenv("AITER_AMD_ST_ROT", "0")
    k = min(3, E)
    cfg = W.MoEConfig("order", tokens, H, I, E, k, seed=tokens, weights=weights, routing="zipf",
                      zipf_s=1.5)
    wts = W.make_weights(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    a1, a1s = A.per_group_quant_hip(W.make_hidden(cfg, device=cuda_device))
    st1, st2 = ((A.moe_stage1_a8w4, A.moe_stage2_a8w4) if weights == "mxfp4" else
                (A.moe_stage1_fp8_blockscale, A.moe_stage2_fp8_blockscale))
    monkeypatch.setenv("AITER_AMD_W4_PF_ROWS1", "0")     # MXFP4 on the prefill kernels too
    monkeypatch.setenv("AITER_AMD_W4_PF_ROWS2", "0")
    got = {}
    for b, dt in ((64, torch.float32), (bm, torch.float32), (bm, torch.bfloat16)):
        sid, sw, seid, nv, acc = A.moe_sorting(ids, tw, E, H, dt, b)
        a2, a2s = st1(a1, a1s, wts["w1"], wts["w1_scale"], sid, seid, nv, k, b, True)
        st2(a2, a2s, wts["w2"], wts["w2_scale"], sid, sw, seid, nv, acc, b, True)
        got[b, dt] = a2, a2s, acc
    (ra2, rs, racc), (a2, a2s, acc) = got[64, torch.float32], got[bm, torch.float32]
    assert torch.equal(a2s, rs)
    assert torch.equal(a2.view(torch.uint8), ra2.view(torch.uint8))
    # (terms that cancel may each be a few times the largest sum)
    tol = 4 * k * 2.0 ** -23 * racc.abs().max()
    assert ((acc - racc).abs() <= tol).all()
    # a bf16 moe_buf rounds after every add: half a spacing, 2^-8, per pair
    b16 = got[bm, torch.bfloat16][2].float()
    assert ((b16 - racc).abs() <= 2 * k * 2.0 ** -8 * racc.abs().max()).all()


def _walk_groups(w4, mv, groups, KB):
    """The stream kernel's own choice of stage 2's column groups per workgroup
    (walk_groups, moe_gemm_stream.hip), with the name of its line."""
    two, four = groups % 2 == 0 and 2 * KB <= 64, groups % 4 == 0 and 4 * KB <= 64
    w2 = mv * groups // 2
    w4_ = w2 // 2
    if KB <= 2:
        return (4, "short") if four and w4_ >= 256 else (2, "short") if two and w2 >= 448 else \
            (1, "short")
    if w4:
        return (4, "mxfp4") if four and w4_ >= 600 else (1, "mxfp4")
    if four and KB >= 8 and 384 <= w4_ <= 512:
        return 4, "fp8"
    if two and w2 >= 3 * 512:
        return 2, "fp8 many"
    return (2, "fp8 tail") if two and w2 >= 384 and w2 & 511 >= 256 else (1, "fp8")


# 600 pairs over 40 experts (more M-blocks than a round of 32 groups of four), K
# ranges of 3, 6, 2, 8 and 5 steps, 16, 12, 8 and 28 column groups: walks of two
# and four leave column counts that 8 divides and that it does not
@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
@pytest.mark.parametrize("bm", [16, 32])
@pytest.mark.parametrize("H,I", [(4096, 384), (3072, 768), (2048, 384), (7168, 256), (4096, 1024),
                                 (2048, 640)])
def test_stream_stage2_forced_walks(cuda_device, monkeypatch, weights, bm, H, I):
    """Stage 2 walking two and four column groups against one: with one slot per
    token every output element has one add, so they are equal bit for bit."""
    acc = _stage2_of(cuda_device, weights, 600, H, I, 40, bm)
    monkeypatch.setenv("AITER_AMD_ST_NTW2", "1")
    one, mv = acc()
    assert mv >= 40 and torch.count_nonzero(one).item() > 0
    for ntw in (2, 4):
        monkeypatch.setenv("AITER_AMD_ST_NTW2", str(ntw))
        assert torch.equal(acc()[0], one), ntw


# one case per line of the kernel's choice
@pytest.mark.parametrize("weights,tokens,H,I,E,want", [
    ("fp8", 700, 4096, 256, 8, (1, "short")), ("fp8", 850, 4096, 256, 8, (2, "short")),
    ("mxfp4", 850, 4096, 128, 8, (2, "short")), ("mxfp4", 1100, 4096, 256, 8, (4, "short")),
    ("mxfp4", 600, 4096, 384, 8, (1, "mxfp4")), ("mxfp4", 2500, 4096, 384, 8, (4, "mxfp4")),
    ("fp8", 1600, 4096, 1024, 8, (4, "fp8")), ("fp8", 3100, 4096, 384, 8, (2, "fp8 many")),
    ("fp8", 750, 4096, 384, 8, (2, "fp8 tail")), ("fp8", 750, 4096, 768, 8, (2, "fp8 tail")),
    ("fp8", 1050, 4096, 768, 8, (1, "fp8"))])
def test_stream_stage2_own_walk(cuda_device, monkeypatch, weights, tokens, H, I, E, want):
    monkeypatch.delenv("AITER_AMD_ST_NTW2", raising=False)
    acc = _stage2_of(cuda_device, weights, tokens, H, I, E, 16)
    own, mv = acc()
    assert _walk_groups(weights == "mxfp4", mv, H // 256, I // 128) == want, mv
    monkeypatch.setenv("AITER_AMD_ST_NTW2", "1")
    one = acc()[0]
    assert torch.count_nonzero(one).item() > 0 and torch.equal(own, one)


def _stage2_of(dev, weights, tokens, H, I, E, bm):
    """A call of stage 2 on one layer's a2, top-1: (accumulator, M-blocks)."""
    cfg = W.MoEConfig("walks", tokens, H, I, E, 1, seed=tokens + I, weights=weights)
    wts = W.make_weights(cfg, device=dev)
    tw, ids = W.make_routing(cfg, device=dev)
    a1, a1s = A.per_group_quant_hip(W.make_hidden(cfg, device=dev))
    st1, st2 = ((A.moe_stage1_a8w4, A.moe_stage2_a8w4) if weights == "mxfp4" else
                (A.moe_stage1_fp8_blockscale, A.moe_stage2_fp8_blockscale))
    sid, sw, seid, nv, acc = A.moe_sorting(ids, tw, E, H, torch.float32, bm)
    a2, a2s = st1(a1, a1s, wts["w1"], wts["w1_scale"], sid, seid, nv, 1, bm, True)

    def run():
        y = torch.zeros_like(acc)
        st2(a2, a2s, wts["w2"], wts["w2_scale"], sid, sw, seid, nv, y, bm, True)
        return y, nv[0].item() // bm

    return run


# stage 2 walks one, two and four column groups per workgroup (two K steps and 5,
# 60 and 70 M-blocks), stage 1 has 4, 2 and 3 column tiles and more than 32 M-blocks
@pytest.mark.parametrize("weights", ["fp8", "mxfp4"])
@pytest.mark.parametrize("bm", [16, 32])
@pytest.mark.parametrize("H,I,keep", [(1024, 512, 37), (512, 256, 5), (4096, 256, 60),
                                      (4096, 256, 70), (768, 384, 41)])
def test_stream_m_blocks_end_with_the_metadata(cuda_device, weights, bm, H, I, keep):
    """Stage calls given the first `keep` entries of sorted_expert_ids run the
    first `keep` M-blocks and no other, as if num_valid_ids ended there: the
    same a2 rows, and with one slot per token the same sums, bit for bit. Its
    entries past `keep` are left in memory, so a block run too many shows."""
    cfg = W.MoEConfig("short", 80 * bm, H, I, 8, 1, seed=keep, weights=weights)
    wts = W.make_weights(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    a1, a1s = A.per_group_quant_hip(W.make_hidden(cfg, device=cuda_device))
    st1, st2 = ((A.moe_stage1_a8w4, A.moe_stage2_a8w4) if weights == "mxfp4" else
                (A.moe_stage1_fp8_blockscale, A.moe_stage2_fp8_blockscale))
    sid, sw, seid, nv, acc = A.moe_sorting(ids, tw, 8, H, torch.float32, bm)
    assert nv[0].item() > keep * bm
    short = torch.tensor([keep * bm, cfg.tokens], dtype=torch.int32, device=cuda_device)
    done = sid[: keep * bm] & 0xFFFFFF
    done = done[done < cfg.tokens].long()
    rest = torch.ones(cfg.tokens, dtype=torch.bool, device=cuda_device)
    rest[done] = False
    out = {}
    for name, e, n in (("short", seid[:keep], nv), ("ref", seid, short)):
        a2, a2s = st1(a1, a1s, wts["w1"], wts["w1_scale"], sid, e, n, 1, bm, True)
        y = torch.zeros_like(acc)
        # rows that no block of this call wrote are anything: 0, for both
        a2.view(torch.uint8)[rest] = 0
        a2s[rest] = 0
        st2(a2, a2s, wts["w2"], wts["w2_scale"], sid, sw, e, n, y, bm, True)
        out[name] = a2.view(torch.uint8), a2s, y
    for got, want in zip(out["short"], out["ref"]):
        assert torch.equal(got, want)
    y = out["short"][2]
    assert torch.count_nonzero(y[rest]) == 0 and (y[done].abs().amax(1) > 0).all()


@pytest.mark.parametrize("H", [256, 1792, 2048, 2304, 4096, 7168])
@pytest.mark.parametrize("prequant", [False, True])   # bf16 and fp32 per-pair rows
def test_slot_sum_wave_spans(cuda_device, H, prequant):
    """The expert-parallel slot sum (a wave per span of a row) against the dense
    one: with every expert local both add the same rows in slot order, so the
    outputs are equal bit for bit; with some masked, a token without a local
    expert gets a zero row."""
    cfg = W.MoEConfig("spans", 131, H, 128, 8, 5, seed=H)
    wts = W.make_weights(cfg, device=cuda_device)
    tw, ids = W.make_routing(cfg, device=cuda_device)
    x = W.make_hidden(cfg, device=cuda_device)
    kw = dict(w1_scale=wts["w1_scale"], w2_scale=wts["w2_scale"], block_size_M=64)
    if prequant:
        x, kw["a1_scale"] = A.per_group_quant_hip(x)
    run = lambda **k: W.run_layer("fp8", x, wts["w1"], wts["w2"], tw, ids, **kw, **k)
    dense = run()
    assert torch.equal(run(expert_mask=torch.ones(8, dtype=torch.int32, device=cuda_device)), dense)
    n = torch.tensor([77], dtype=torch.int32, device=cuda_device)
    ones = torch.ones(8, dtype=torch.int32, device=cuda_device)
    assert torch.equal(run(expert_mask=ones, num_local_tokens=n)[:77], dense[:77])
    away = torch.full_like(ids, 11)                   # experts 8 .. 15 live on another GPU
    mixed = torch.where((torch.arange(131, device=cuda_device) % 3 == 0)[:, None], away, ids)
    mask = (torch.arange(16, device=cuda_device) < 8).to(torch.int32)
    got = W.run_layer("fp8", x, wts["w1"], wts["w2"], tw, mixed, expert_mask=mask, **kw)
    assert torch.count_nonzero(got[::3]) == 0
    assert torch.equal(got[1::3], dense[1::3]) and torch.equal(got[2::3], dense[2::3])
