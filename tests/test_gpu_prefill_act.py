"""The SwiGLU activations between the two GEMMs at prefill sizes: rounded to
bf16, each value with an exponent of its own, whatever else the batch holds."""
from __future__ import annotations

import pytest
import torch

from flashinfer_amd import kernel
from flashinfer_amd import workloads as W
from flashinfer_amd.shapes import DEFINITIONS
from _helpers import log, oracle_subset, run_gpu

pytestmark = pytest.mark.gpu

SMALL = DEFINITIONS[3]  # 16 of 128 experts, top-6, H = 4096, I = 1536
T_SMALL = 2816          # 11 row tiles of 256 rows for each chosen expert


def _concentrated(defn, T, seed):
    """Every token on the second shard's first top_k experts: T rows each."""
    wl = W.make_for(defn, f"rows_{T}", T, seed, local_expert_offset=defn.EL)
    wl.tensors["routing_logits"][:, defn.EL:defn.EL + defn.TOPK] += 12.0
    wl.tensors["routing_bias"].zero_()
    return wl


def _run_own_weights(wl):
    """run() on the workload's own weights (the cached device copies are the seeded ones)."""
    out = torch.full((wl.T, wl.tensors["gemm1_weights"].shape[2]), float("nan"),
                     dtype=torch.bfloat16, device="cuda")
    kernel.run(*wl.args("cuda"), out)
    torch.cuda.synchronize()
    return out


def test_small_values_beside_outlier_channels(monkeypatch):
    """One SwiGLU channel in 32 about 2^18 times the others, and no weight of
    GEMM2 reads it: the output is that of the other channels, each rounded
    relative to itself. Three bf16 roundings (activation, partial row, output)
    of at most 2^-9 of a value each, with independent errors: normwise
    sqrt(3) * 2^-9 at most."""
    from oracle import ref_moe as R
    log("test_small_values_beside_outlier_channels")
    monkeypatch.delenv("MI_MOE_VARIANT", raising=False)
    wl = _concentrated(SMALL, T_SMALL, 6100)
    t = wl.tensors
    w1, w2 = t["gemm1_weights"].clone(), t["gemm2_weights"].clone()
    outlier = torch.arange(SMALL.I) % 32 == 11
    gain = torch.where(outlier, 64.0, 0.125).repeat(2)[:, None]  # gate rows, up rows
    for e in range(SMALL.TOPK):
        w1[e] = (w1[e].float() * gain).clamp(-448.0, 448.0).to(W.FP8)
        w2[e] = w2[e].float().masked_fill(outlier, 0.0).to(W.FP8)
    t["gemm1_weights"], t["gemm2_weights"] = w1, w2
    out = _run_own_weights(wl)
    tokens = torch.cat([torch.arange(4), torch.arange(250, 262), torch.arange(T_SMALL - 8, T_SMALL)])
    rep = R.tolerance_report(out[tokens.cuda()].float().cpu(), oracle_subset(wl, tokens).acc)
    assert rep["n_bad"] == 0, rep
    assert rep["normwise_rel"] <= 3 ** 0.5 * 2 ** -9, rep


def test_single_infinity_meets_each_weight(monkeypatch):
    """One infinite SwiGLU value in one token's row: infinite where its weight
    is not zero, down to the smallest fp8 value, NaN where it is zero, as in the
    oracle; no other token's output changes by a bit."""
    log("test_single_infinity_meets_each_weight")
    monkeypatch.delenv("MI_MOE_VARIANT", raising=False)
    wl = _concentrated(SMALL, T_SMALL, 6200)
    t = wl.tensors
    tok, e, j, kb = 300, 2, 645, 3
    h = kb * 128 + 5
    # k-block kb is empty but for one product, whose scales carry it past fp32
    for name in ("hidden_states", "gemm1_weights", "gemm1_weights_scale", "gemm2_weights"):
        t[name] = t[name].clone()
    t["hidden_states"].view(torch.uint8)[:, kb * 128:(kb + 1) * 128] = 0
    t["gemm1_weights"].view(torch.uint8)[:, :, kb * 128:(kb + 1) * 128] = 0
    t["gemm1_weights"][e, j, h] = 448.0
    t["gemm1_weights_scale"][e, j // 128, kb] = 1e8
    t["hidden_states_scale"][kb, tok] = 1e30
    steps = torch.tensor([0.0, 2.0 ** -9, 2.0 ** -8, 1.0]).to(W.FP8)
    t["gemm2_weights"][e, :, j] = steps.repeat(SMALL.H // 4)
    plain = _run_own_weights(wl)
    assert torch.isfinite(plain).all()
    t["hidden_states"][tok, h] = 448.0
    out = _run_own_weights(wl)
    others = torch.arange(T_SMALL, device="cuda") != tok
    assert torch.equal(out[others].view(torch.int16), plain[others].view(torch.int16))
    want = oracle_subset(wl, torch.tensor([tok])).acc[0]
    zero = torch.arange(SMALL.H) % 4 == 0
    assert torch.equal(torch.isnan(want), zero) and torch.equal(torch.isinf(want), ~zero)
    got = out[tok].float().cpu()
    assert torch.equal(torch.isnan(got), zero)
    assert torch.equal(got[~zero], want[~zero])


@pytest.mark.parametrize("defn,T", [(SMALL, T_SMALL), (DEFINITIONS[1], 4100)],
                         ids=lambda x: x.name if hasattr(x, "name") else str(x))
def test_token_bits_do_not_depend_on_the_batch(defn, T, monkeypatch):
    """The same 65 tokens among T that all stay on the shard (full row tiles)
    and among T of which the others go elsewhere (65 rows an expert): the same
    bits."""
    log(f"test_token_bits_do_not_depend_on_the_batch[{defn.name}]")
    monkeypatch.delenv("MI_MOE_VARIANT", raising=False)
    wl = _concentrated(defn, T, 6300)
    full = run_gpu(wl, fill=float("nan")).clone()
    logits = wl.tensors["routing_logits"]
    logits[65:, defn.EL:defn.EL + defn.TOPK] -= 24.0
    logits[65:, :defn.TOPK] += 12.0  # the first shard's experts
    sparse = run_gpu(wl, fill=float("nan"))
    assert torch.isfinite(full.float()).all() and (full != 0).any(dim=1).all()
    assert (sparse[65:] == 0).all()
    assert torch.equal(full[:65].view(torch.int16), sparse[:65].view(torch.int16))


@pytest.mark.parametrize("scale", [float("nan"), float("inf"), 3e33, 1e-36, 0.0])
def test_nonfinite_and_extreme_rows(scale, monkeypatch):
    """A token whose activations are not finite, overflow, vanish or are zero
    has the bits of the plain LDS tiles (variants 3, 3), and so has every other."""
    log(f"test_nonfinite_and_extreme_rows[{scale}]")
    wl = _concentrated(SMALL, T_SMALL, 6000)
    wl.tensors["hidden_states_scale"][:, 300] = scale
    monkeypatch.delenv("MI_MOE_VARIANT", raising=False)
    out = run_gpu(wl, fill=1.0).clone()
    monkeypatch.setenv("MI_MOE_VARIANT", "3,3")
    plain = run_gpu(wl, fill=2.0)
    nan = torch.isnan(plain)
    assert torch.equal(torch.isnan(out), nan)
    assert torch.equal(out.view(torch.int16)[~nan], plain.view(torch.int16)[~nan])
